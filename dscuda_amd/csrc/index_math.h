// Integer arithmetic of the attention kernels that decides where data lives and
// which workgroup does what: LDS chunk permutations, tile-request offsets, the
// position of a dS block in the backward workspace, the work order of the
// persistent forward kernel and the split of the decode tile list.  Kept free
// of anything device-specific so that the same definitions compile for the
// host, where tests enumerate them exhaustively (coverage, uniqueness,
// fast path == general path).
#pragma once

#include <algorithm>
#include <vector>

#if defined(__HIPCC__)
#define DSCUDA_HOST_DEVICE __host__ __device__
#else
#define DSCUDA_HOST_DEVICE
#endif

namespace dscuda {
namespace index_math {

// ---- LDS chunk permutations -------------------------------------------------
// A row-major LDS tile keeps 16-byte chunk c of row r at position c ^ f(r).
// Row bytes = 0 (mod 256): the four bits of the row, pairs exchanged.
// Row bytes = 128 (mod 256): the three bits of row>>1, bits 0 and 2 exchanged.
template <int ROW_BYTES>
DSCUDA_HOST_DEVICE constexpr int tile_swizzle(int row) {
    if constexpr (ROW_BYTES % 256 == 0) {
        return ((row & 3) << 2) | ((row >> 2) & 3);
    } else {
        const int u = row >> 1;
        return ((u & 1) << 2) | (u & 2) | ((u >> 2) & 1);
    }
}

// ---- backward workspace -----------------------------------------------------
// Position of dS block (key block kb of 128 keys, query tile qt of 64 queries),
// qt >= 2*kb, key block major; and the number of such blocks of one head.
DSCUDA_HOST_DEVICE inline long long ds_block_index(int kb, int qt, int query_tiles) {
    return (long long)kb * query_tiles - (long long)kb * (kb - 1) + (qt - 2 * kb);
}

DSCUDA_HOST_DEVICE inline long long ds_block_count(int key_blocks, int query_tiles) {
    return (long long)key_blocks * query_tiles - (long long)key_blocks * (key_blocks - 1);
}

// ---- cut of the key blocks' walks (backward) -----------------------------------
// Key block kb of a (batch, key/value head) pair is walked in (query_tiles - 2 * kb) * sharing steps, one query tile of
// one query head each.  A walk may be cut into parts of at most part_steps steps, equal to within one, each a workgroup
// of its own.
DSCUDA_HOST_DEVICE inline int walk_parts(int steps, int part_steps) {
    return (int)(((unsigned)steps + (unsigned)part_steps - 1) / (unsigned)part_steps);
}

// First step of part `part` (part == parts: the end of the walk).
DSCUDA_HOST_DEVICE inline int part_begin(int steps, int parts, int part) {
    const unsigned each = (unsigned)steps / (unsigned)parts, more = (unsigned)steps % (unsigned)parts;
    return (int)(each * (unsigned)part + ((unsigned)part < more ? (unsigned)part : more));
}

struct WalkCut {
    int part_steps;   // 0: no walk is cut
    int items;        // workgroups per pair
    int cut_blocks;   // key blocks 0 .. cut_blocks - 1 have more than one part
};

inline long long walk_items(int key_blocks, int query_tiles, int sharing, int part_steps) {
    long long items = 0;
    for (int kb = 0; kb < key_blocks; ++kb) items += walk_parts((query_tiles - 2 * kb) * sharing, part_steps);
    return items;
}

// The cut for a launch of `pairs` pairs on `slots` workgroups at a time.  Costs are in steps of one workgroup.  A
// workgroup costs ITEM_STEPS besides its own (rows and first tile, the sums' way out, and for a part its share of the
// addition); one round of workgroups ends with the longest, several rounds some way into the last one: parts are alike
// and end together or not at all (half a part), whole walks start longest first and even out (a quarter of the
// longest).  Candidates: the shortest parts that still run as one round, and several rounds of parts of 1/2 .. 1/6 of
// the mean load.  Measured, whole walks -> cut (us for forward and backward): 128/128 columns, T=4096, 8 heads on 1:
// 908 -> 187 (32 walks of up to 512 steps); T=8192, 16 on 4: 1316 -> 1128 (256 walks, several rounds); 192/128 columns,
// T=4096, 4 heads: 224 -> 160, T=1000, 16 heads: 75 -> 64 (parts of 6).  Forced cuts of launches that the rule leaves
// whole: T=2000, 32 heads 235 -> 241 (parts of 24); T=8192, 8 heads 640 -> 686 (64); T=6000, 32 heads 1464 -> 1541.
// Walks below 12 steps stay whole: T=500, 8 heads 46 -> 45 with parts of 6.
inline WalkCut choose_walk_cut(long long pairs, int key_blocks, int query_tiles, int sharing, int slots) {
    constexpr int MIN_PART = 6;
    constexpr double ITEM_STEPS = 6;
    constexpr double GAIN = 0.9;   // of the cost of whole walks: what a cut has to stay below
    const WalkCut whole = {0, key_blocks, 0};
    const int longest = query_tiles * sharing;
    if (longest < 2 * MIN_PART || pairs * key_blocks >= 4LL * slots) return whole;
    const double mean = (double)pairs * key_blocks * (query_tiles - key_blocks + 1) * sharing / slots;
    auto cost = [&](long long items, int part, double tail) {
        return items * pairs <= slots ? part + ITEM_STEPS : mean + items * pairs * ITEM_STEPS / slots + tail * part;
    };
    const double uncut = cost(key_blocks, longest, 0.25);
    double best = GAIN * (uncut > longest ? uncut : longest);
    int part_steps = 0;
    auto consider = [&](int part) {
        if (part < MIN_PART || part >= longest) return;
        const double value = cost(walk_items(key_blocks, query_tiles, sharing, part), part, 0.5);
        if (value < best) {
            best = value;
            part_steps = part;
        }
    };
    for (int rounds = 2; rounds <= 6; ++rounds) consider((int)(mean / rounds));
    if (pairs * key_blocks <= slots) {
        int low = MIN_PART, high = longest;   // walk_items falls with the length of a part
        while (low < high) {
            const int middle = (low + high) / 2;
            if (pairs * walk_items(key_blocks, query_tiles, sharing, middle) <= slots) high = middle; else low = middle + 1;
        }
        consider(low);
    }
    if (part_steps == 0) return whole;
    WalkCut cut = {part_steps, (int)walk_items(key_blocks, query_tiles, sharing, part_steps), 0};
    while (cut.cut_blocks < key_blocks && (query_tiles - 2 * cut.cut_blocks) * sharing > part_steps) ++cut.cut_blocks;
    return cut;
}

// What a cut may ask of the workspace: at most `parts` parts, and `floats` floats for their sums and the dS blocks
// (`block_floats` each, one per step) together.  Both grow with every argument, as the dS blocks do, so that a workspace
// asked for the longest sequence and the most heads of a program also holds the sums of shorter calls that are cut where
// those are not.  No cut of choose_walk_cut comes near them (1827 parts and 1.33 blocks per slot and step of the longest
// walk at most, up to 40000 tokens and 32 heads sharing).
struct WalkCutRoom {
    long long parts;
    long long floats;
};

inline WalkCutRoom walk_cut_room(long long pairs, int key_blocks, int query_tiles, int sharing, int slots, long long block_floats) {
    constexpr int MIN_PART = 6;
    const long long longest = (long long)query_tiles * sharing;
    if (longest < 2 * MIN_PART) return WalkCutRoom{0, 0};
    const long long steps = pairs * sharing * ds_block_count(key_blocks, query_tiles);
    return WalkCutRoom{std::min(8LL * slots, steps / MIN_PART + pairs * key_blocks), 11 * slots * longest * block_floats / 8};
}

// ---- tile requests of the backward kernels ------------------------------------
// One wave's share of the global -> LDS requests of a [ROWS][ROW_BYTES] tile that
// WAVES waves fetch together.  LDS slot 64*load + lane (16 bytes each) holds chunk
// (slot % CHUNKS) ^ f(row) of row slot / CHUNKS.  PERIOD loads cover PERIOD_ROWS
// whole rows; from one period to the next only the low bits of f change, so load
// L = PERIOD*m + r reads at
//     tile + m * PERIOD_ROWS * row_stride  +  (offset of load r) ^ 16 * (m % XOR_STEPS)
// The periods of a wave's LOADS consecutive loads are m = wave * LOADS/PERIOD + j;
// LOADS/PERIOD and XOR_STEPS are powers of two, so the two parts of m touch
// different bits of the XOR term: the wave's part is folded into a per-lane base
// once and j's part is a compile-time constant.
template <int ROW_BYTES, int WAVES, int ROWS = 64>
struct TileRequestMath {
    static constexpr int CHUNKS = ROW_BYTES / 16;
    static constexpr int LOADS = ROWS * ROW_BYTES / 1024 / WAVES;
    static constexpr int PERIOD = CHUNKS == 24 ? 3 : 1;
    static constexpr int PERIOD_ROWS = 64 * PERIOD / CHUNKS;
    static constexpr int XOR_STEPS = CHUNKS == 16 ? 4 : 2;
    static constexpr int PERIODS = LOADS / PERIOD;   // per wave
    static_assert(CHUNKS == 8 || CHUNKS == 16 || CHUNKS == 24, "rows of 128, 256 or 384 bytes");
    static_assert(ROWS * ROW_BYTES % (1024 * WAVES) == 0 && LOADS % PERIOD == 0, "tile must divide evenly over the waves");
    static_assert(PERIODS == 1 || PERIODS == 2 || PERIODS == 4, "periods per wave must be a power of two");

    // general form: byte offset of lane `lane` of load `load` from the tile's first row; rows past
    // `row_limit` repeat that row
    DSCUDA_HOST_DEVICE static int row_of(int load, int lane) { return (64 * load + lane) / CHUNKS; }
    DSCUDA_HOST_DEVICE static int chunk_of(int load, int lane) {
        return ((64 * load + lane) % CHUNKS) ^ tile_swizzle<ROW_BYTES>(row_of(load, lane));
    }
    DSCUDA_HOST_DEVICE static unsigned offset_of(int load, int lane, unsigned row_stride, int row_limit) {
        const int row = row_of(load, lane);
        return (unsigned)(row_limit < row ? row_limit : row) * row_stride + 16u * chunk_of(load, lane);
    }
    // fast form, full tiles only: per-lane base of residue r (computed once per kernel) ...
    DSCUDA_HOST_DEVICE static unsigned base_of(int r, int lane, unsigned row_stride, int wave) {
        return offset_of(r, lane, row_stride, ROWS) ^ (16u * ((wave * PERIODS) % XOR_STEPS));
    }
    // ... the rows (from the tile's first) the uniform part of the address of the wave's load i skips ...
    DSCUDA_HOST_DEVICE static constexpr int rows_before(int i, int wave) {
        return wave * PERIODS * PERIOD_ROWS + i / PERIOD * PERIOD_ROWS;
    }
    // ... and the per-lane part of that load
    DSCUDA_HOST_DEVICE static constexpr unsigned lane_part(unsigned base, int i) {
        return base ^ (16u * ((i / PERIOD) % XOR_STEPS));
    }
};

// ---- fragment reads of the backward kernels ------------------------------------
// Per-lane byte offsets of the MFMA operand fragments inside a row-major swizzled
// LDS tile.  The swizzle only touches the low SPAN chunk positions of a row, so a
// handful of per-lane values plus compile-time constants reach every fragment.
//
//   natural(i, lane)        row lane%32, chunk (2i + g) ^ f(row), g = lane/32: the
//                           operand whose contraction index is the tile column;
//                           k-step ks = NAT*m + i lies NAT*32*m bytes further, 32
//                           rows down 32*ROW_BYTES (natural_constant)
//   transposed(h, i, lane)  for ds_read_b64_tr_b16: row 4g + s/4 + 8h (s = lane%16),
//                           chunk (4i + 2*((lane/16)%2) + (s%4)/2) ^ f(row), byte
//                           8*(s%2): the operand whose contraction index is the
//                           tile row; MFMA row/column lane%32 = tile column
//                           32*block + lane%32, k = rows {4g..4g+3, 8+4g..8+4g+3}
//                           of a 16-row step -- the order a C-layout register block
//                           carries; block = TR*m + i lies TR*64*m bytes further
//                           (transposed_constant)
//   quadrant(i, lane)       for the 16x16x32 products: row lane%16, chunk (4i + lane/16) ^ f(row):
//                           the operand whose contraction index is the tile column, 32 columns
//                           per step; step s = TR*m + i lies TR*64*m bytes further, 16 rows down
//                           16*ROW_BYTES (quadrant_constant; f repeats after 16 rows)
template <int ROW_BYTES>
struct TileReadMath {
    static constexpr int SPAN = (ROW_BYTES % 256 == 0) ? 16 : 8;
    static constexpr int NAT = SPAN / 2;
    static constexpr int TR = SPAN / 4;

    DSCUDA_HOST_DEVICE static unsigned natural(int i, int lane) {
        const int lq = lane % 32;
        const int g = lane / 32;
        return lq * ROW_BYTES + 16 * ((2 * i + g) ^ tile_swizzle<ROW_BYTES>(lq));
    }
    DSCUDA_HOST_DEVICE static unsigned transposed(int h, int i, int lane) {
        const int g = lane / 32;
        const int s = lane % 16;
        const int low = 2 * ((lane / 16) % 2) + (s % 4) / 2;
        const int row = 4 * g + s / 4 + 8 * h;
        return row * ROW_BYTES + 16 * ((4 * i + low) ^ tile_swizzle<ROW_BYTES>(row)) + 8 * (s % 2);
    }
    DSCUDA_HOST_DEVICE static unsigned quadrant(int i, int lane) {
        const int row = lane % 16;
        return row * ROW_BYTES + 16 * ((4 * i + lane / 16) ^ tile_swizzle<ROW_BYTES>(row));
    }
    DSCUDA_HOST_DEVICE static constexpr int quadrant_constant(int row0, int s) {
        return row0 * ROW_BYTES + (s / TR) * (TR * 64);
    }
    DSCUDA_HOST_DEVICE static constexpr int natural_constant(int row0, int ks) {
        return row0 * ROW_BYTES + (ks / NAT) * (NAT * 32);
    }
    DSCUDA_HOST_DEVICE static constexpr int transposed_constant(int row0, int block) {
        return row0 * ROW_BYTES + (block / TR) * (TR * 64);
    }
};

// ---- absorbed prefill forward with few rows ------------------------------------------
// 32 or 64 rows a workgroup (returned: 1, 2) where 64 rows are at most one round of the compute units.  64 rows take
// longer a unit of 32 keys, 32 rows may take two rounds, whose second pays a workgroup's start and end again; the
// sums (10 ns, from the times below) decide.  Forward in us, 32 / 64 rows: 100 tokens x 128 heads 14.5 / 12.1, 120 x 128
// 15.5 / 12.9, 250 x 64 18.8 / 16.9, 200 x 64 16.1 / 15.2, 3 x 300 x 16 22.2 / 18.3, 8 x 250 x 8 23.5 / 17.2, 500 x 32
// 25.5 / 24.4; 400 x 32 20.4 / 21.3, 300 x 32 15.6 / 17.8, 1000 x 16 38.6 / 39.4, 700 x 16 25.1 / 29.2, 2000 x 8 65 / 70.
DSCUDA_HOST_DEVICE inline int narrow_forward_row_blocks(int sequence_length, int heads, long long batch, int compute_units) {
    const long long blocks = ((long long)sequence_length * heads + 31) / 32 * batch;
    if (blocks <= compute_units) return 1;
    const long long keys = (sequence_length + 31LL) / 32;   // units of the longest walk
    const long long longest = 700 + 80 * keys;
    // the shortest walks of the first round and the longest of the second, one after the other
    const long long second = 1300 + 160 * keys * (blocks - compute_units) / blocks;
    return (longest > second ? longest : second) <= 900 + 94 * keys ? 1 : 2;
}

// How many 32-row blocks a workgroup of the absorbed prefill forward holds: 1 or 2 while 128 rows (0: four blocks, the
// kernels of mla_wide.hip) leave compute units idle.
//   * up to half a round of 128-row workgroups: 32 or 64 rows (forward in us, 64 / 128 rows: 130 tokens x 128 heads 15.2 / 17.2)
//   * up to one round, which 64 rows take in two: 128 rows for most of a round of walks of up to 160 keys (128 x 172 18.2 / 17.3,
//     2 x 123 x 98 18.3 / 17.4, 8 x 97 x 39 21.5 / 17.8), and up to 384 keys of many elements, whose heavy blocks 64 rows get late (3 x
//     172 x 46 21.1 / 20.0, 4 x 225 x 36 27.4 / 23.9, 16 x 379 x 4 33.8 / 28.3); 64 for longer ones, a unit of which takes them a third
//     less (512 x 64 32.0 / 33.8, 1000 x 32 47.9 / 56.2, 2000 x 16 82 / 100), and of one or two elements from 161 (192 x 126 19.8 / 20.5,
//     251 x 87 20.6 / 22.8, 344 x 64 21.3 / 26.8, 2 x 353 x 37 25.3 / 28.4; nearly a round of up to 224 keys 161 x 193 22.5 / 21.6,
//     256 x 114 24.7 / 24.2) or three from 225 (371 x 21 26.8 / 28.4, 236 x 34 23.7 / 23.0)
//   * up to a round and a fifth, one or two batch elements: the longest walk decides, which 64 rows take faster, where it is long
//     against the blocks of a second round (1 x 516 x 64, 258 workgroups, 40 / 37.5; 1 x 750 x 44, 258, 46.0 / 47.1; 1 x 2064 x 16,
//     258, 92 / 105; 1 x 8256 x 4, 258, 313 / 382; 2 x 1100 x 16, 276, 59.8 / 62.5; 1 x 1200 x 32, 300, 71.5 / 69; 1 x 2400 x 16, 300,
//     121 / 124; 1 x 5104 x 8, 319, 257 / 254); of more elements 64 rows get the heavy blocks late (3 x 2800 x 4, 264, 151 / 137,
//     4 x 8200 x 1 443 / 380)
//   * beyond: 128 rows, whose second item needs no second start (258 x 128 31.0 / 23.4, 300 x 128 33.9 / 26.1, 1200 x 32 71 / 67,
//     5 x 64 x 128 26.5 / 23.8, 1 x 5440 x 8, 340, 287 / 276), but for walks of one unit, of which they take two (300 x 1 x 40
//     13.4 / 17.1).
DSCUDA_HOST_DEVICE inline int forward_row_blocks(int sequence_length, int heads, long long batch, int compute_units) {
    const long long workgroups = ((long long)sequence_length * heads + 127) / 128 * batch;
    const int units = (sequence_length + 31) / 32;
    if (2 * workgroups <= compute_units) return narrow_forward_row_blocks(sequence_length, heads, batch, compute_units);
    if (workgroups <= compute_units) {
        if (units > 12 || 3 * workgroups <= 2LL * compute_units) return 2;
        if (units <= 5) return 0;
        if (batch <= 2) return units <= 7 && 8 * workgroups >= 7LL * compute_units ? 0 : 2;
        return batch == 3 && units >= 8 && 4 * workgroups < 3LL * compute_units ? 2 : 0;
    }
    if (units == 1) return 4 * workgroups <= 5LL * compute_units ? 2 : 0;
    return batch <= 2 && 5 * workgroups <= 6LL * compute_units && 2 * (units - 20) > workgroups - compute_units ? 2 : 0;
}

// ---- work order of the persistent forward kernel ------------------------------
struct ForwardItem {
    int batch_head;
    int query_block;
};

// Item `round` of workgroup `member` (of `members`) of a cluster that owns
// `cluster_heads` (batch, head) pairs (pairs cluster, cluster + clusters, ...);
// false past the end of the list.  Inside a cluster the items are laid out
// `abreast` heads at a time (0: two, or one if the count is odd), blocks from the heaviest (last) to
// the lightest, and cut into rounds of one item per workgroup; odd rounds are
// handed out in reverse.
DSCUDA_HOST_DEVICE inline bool forward_item(int round, int member, int members, int cluster, int clusters,
                                            int cluster_heads, int query_blocks, ForwardItem& item, int abreast = 0) {
    const int position = (round & 1) ? members - 1 - member : member;
    const int index = round * members + position;
    if (index >= cluster_heads * query_blocks) {
        return false;
    }
    const int interleave = abreast > 0 ? abreast : (cluster_heads % 2 == 0) ? 2 : 1;
    const int group = index / (interleave * query_blocks);
    const int rest = index % (interleave * query_blocks);
    item.batch_head = cluster + clusters * (interleave * group + rest % interleave);
    item.query_block = query_blocks - 1 - rest / interleave;
    return true;
}

// Tiles (64 keys x 256 queries) of the busiest workgroup of a cluster, an item's start and end counted as three more.
constexpr int FORWARD_ITEM_TILES = 3;

// One pass over the items in the order of forward_item: the rounds run through the workgroups there and back.
inline int forward_makespan(int members, int /* clusters: all alike */, int cluster_heads, int sequence_length, int abreast) {
    const int query_blocks = (sequence_length + 255) / 256;
    const int interleave = abreast > 0 ? abreast : (cluster_heads % 2 == 0) ? 2 : 1;
    std::vector<int> loads(members, 0);
    int position = 0, direction = 1;
    for (int group = 0; group < cluster_heads; group += interleave) {
        for (int block = query_blocks - 1; block >= 0; --block) {
            const int end = (block + 1) * 256;
            const int tiles = ((end < sequence_length ? end : sequence_length) + 63) / 64 + FORWARD_ITEM_TILES;
            for (int item = 0; item < interleave; ++item) {
                loads[position] += tiles;
                position += direction;
                if (position == members || position < 0) {
                    direction = -direction;
                    position += direction;
                }
            }
        }
    }
    return *std::max_element(loads.begin(), loads.end());
}

// How many heads a cluster takes abreast, and the cost of the launch in tiles.  Two at a time keep few keys live in the
// L2; where the rounds then do not come out even (2.5 rounds of items: the busiest workgroup has 1.4 times the mean),
// more heads sorted together do: 32 heads of 7168 tokens 570 -> 463 us, 128 heads of 1700 tokens 168 -> 147 us with all
// of a cluster's heads abreast.  Each doubling costs some 1.5 % through the L2 (128 heads of 4096 tokens, already even:
// 642 us with two, 652 with eight, 676 with sixteen), and more than that for short sequences, so a gain of less than 3 %
// is none (256 heads of 800 tokens, a gain of 0.1 %: 101.6 us with two, 106.5 with 32; 221 of 3700 1095 / 1137).
struct ForwardChoice {
    int abreast;
    double cost;
};

inline ForwardChoice forward_choice(int members, int clusters, int cluster_heads, int sequence_length) {
    const long long query_blocks = (sequence_length + 255) / 256;
    long long total = 0;   // of a head
    for (long long block = 0; block < query_blocks; ++block) {
        const long long end = (block + 1) * 256 < sequence_length ? (block + 1) * 256 : sequence_length;
        total += (end + 63) / 64 + FORWARD_ITEM_TILES;
    }
    const double mean = (double)total * cluster_heads / members;
    ForwardChoice best = {cluster_heads % 2 == 0 ? 2 : 1, 0.0};
    best.cost = forward_makespan(members, clusters, cluster_heads, sequence_length, best.abreast);
    const double worth = 0.97 * best.cost;
    double penalty = 1.0;
    for (int abreast = 4; best.cost > 1.03 * mean && abreast / 2 < cluster_heads; abreast *= 2) {
        penalty += 0.015;
        const int heads = abreast < cluster_heads ? abreast : cluster_heads;
        if (cluster_heads % heads != 0) continue;
        const double cost = penalty * forward_makespan(members, clusters, cluster_heads, sequence_length, heads);
        if (cost < best.cost && cost < worth) best = ForwardChoice{heads, cost};
    }
    return best;
}

// The cost of the split-key kernel with 128 queries a workgroup in the same tiles: steps (128 queries x 128 keys, start and
// end of a workgroup 2.5 more) of the mean or the longest workgroup, 1.15 tiles each.  Where the heads cannot be dealt to
// the XCDs every L2 reads every head's keys, and a workgroup of 128 queries fetches each key twice as often as one of 256:
// 1.17 times that (1.15 tiles throughout -> so, us, 192/128 columns: 171 heads of 1000 tokens 102 -> 92, 195 of 1300
// 194 -> 169, 156 of 1800 258 -> 226, 67 of 2500 183 -> 153, 300 of 3700 2057 -> 1588; 128/128: 171 of 768 67 -> 54).
inline double split_forward_steps(long long batch_heads, int sequence_length, int compute_units) {
    const long long blocks = (sequence_length + 127LL) / 128;
    return (double)batch_heads * (0.5 * blocks * (blocks + 1) + 2.5 * blocks) / compute_units;
}

inline double split_forward_cost(long long batch_heads, int sequence_length, int compute_units) {
    const double step_tiles = batch_heads % 8 == 0 ? 1.15 : 1.15 * 1.17;
    return step_tiles * std::max(split_forward_steps(batch_heads, sequence_length, compute_units),
                                 (sequence_length + 127LL) / 128 + 2.5);
}

// ---- work order of the split-key forward kernel ----------------------------------
// Division by a constant the host knows, as a multiply and a shift (n < 2^31).
struct FastDivision {
    unsigned multiplier;
    unsigned shift;
    unsigned divisor;
};

inline FastDivision fast_division(unsigned divisor) {
    FastDivision division;
    division.divisor = divisor;
    division.shift = 0;
    while ((1ULL << division.shift) < divisor) ++division.shift;
    division.multiplier = (unsigned)((((1ULL << division.shift) - divisor) << 32) / divisor + 1);
    return division;
}

DSCUDA_HOST_DEVICE inline unsigned divide(unsigned n, const FastDivision& by) {
    return (unsigned)(((((unsigned long long)n * by.multiplier) >> 32) + n) >> by.shift);
}

// Whether the 128-row forward numbers the row blocks of all batch elements together, from heavy to light, or one element
// after the other, which keeps few keys live in the L2s.  A workgroup takes a block of every round of `workgroups`, rounds there
// and back.  Numbered together the rounds even out; one element after the other they do only where elements fill rounds or rounds
// hold whole elements, and there is an even number of them.  Everywhere else a workgroup gets the heavy blocks of several elements.
// Forward in us, one after the other / together: 4 x 1957 x 16 372 / 241, 16 x 537 x 8 93 / 57, 8 x 1976 x 32 1323 / 994, 2 x 3000 x 32
// 631 / 523, 16 x 484 x 128 723 / 701, 9 x 800 x 64 452 / 457; even ones: 64 x 256 x 64 556 / 590, 12 x 1024 x 64 893 / 923, 2 x 2048 x
// 128 1031 / 1059, 40 x 1018 x 16 756 / 774.
DSCUDA_HOST_DEVICE inline bool forward_interleaves(int sequence_length, long long batch, long long row_blocks, long long workgroups) {
    if (batch * sequence_length * 2 * (512 + 64) <= (3 << 20)) return true;   // the keys of all fit an L2
    const bool whole = row_blocks % workgroups == 0 || workgroups % row_blocks == 0;
    return !whole || batch * row_blocks % (2 * workgroups) != 0;
}

// Item `index` of that order: the batch element and its row block, the heaviest first.  by_order: divides by the number of batch
// elements (interleaved) or of row blocks.
DSCUDA_HOST_DEVICE inline void forward_item(unsigned index, bool interleaved, const FastDivision& by_order, unsigned row_blocks,
                                            unsigned& batch, unsigned& row_block) {
    const unsigned quotient = divide(index, by_order);
    const unsigned rest = index - quotient * by_order.divisor;
    batch = interleaved ? rest : quotient;
    row_block = row_blocks - 1 - (interleaved ? quotient : rest);
}

// Index of the item that `workgroup` takes in a round.
DSCUDA_HOST_DEVICE inline unsigned forward_index(unsigned round, unsigned workgroup, unsigned workgroups) {
    return round * workgroups + (round & 1 ? workgroups - 1 - workgroup : workgroup);
}

// The workgroup's index if every XCD took a run of consecutive ones; they go to the eight XCDs round-robin by linear id.
DSCUDA_HOST_DEVICE inline unsigned run_index(unsigned workgroup, unsigned workgroups) {
    const unsigned xcd = workgroup % 8, more = workgroups % 8;   // the first `more` XCDs have one more
    return xcd * (workgroups / 8) + (xcd < more ? xcd : more) + workgroup / 8;
}

// Items (batch, query head, query block), numbered so that what runs at one time shares keys and ends together.
// Workgroups go to the XCDs round-robin by linear id and every XCD has an L2 of its own, so the query heads that read
// one key/value head stay on one XCD; with too few key/value heads for that, query heads are dealt to the XCDs one by
// one; with too few of those there is no dealing.  An XCD takes a number of its groups together, the longest query
// blocks of all of them first: all its groups while they make at most four rounds of its compute units (what decides
// then is that no long block starts late), beyond that two rounds' worth at a time (what decides then is that few
// heads' keys are live in the L2).
struct SplitOrder {
    FastDivision turn;       // items an XCD takes together
    FastDivision abreast;    // (group, query head) pairs among them
    FastDivision members;    // query heads of a group
    FastDivision groups;     // groups per batch element
    FastDivision sharing;    // query heads per key/value head
    int clusters;
    int together;            // groups an XCD takes together
    int query_blocks;
    int batch;
    long long workgroups;    // of the launch; items with a batch index past the last one are nobody's
};

// Whether heads that are no multiple of eight are dealt to the XCDs all the same, the last turn to some of them only.
// Undealt, every L2 reads every head's keys, which is slow as soon as they do not fit (64 columns, four waves with the heads
// in turn / undealt / so, us: 221 heads of 448 tokens 25 / 25 / 20, 67 of 1728 66 / 65 / 46, 115 of 2368 145 / 193 / 124, 189 of
// 3392 425 / 628 / 391, 250 of 5952 1620 / 2490 / 1467); with few heads the idle slots of the last turn, at most seven
// heads, would weigh more.
inline bool split_spreads(long long batch_heads, int sequence_length) {
    return batch_heads % 8 != 0 && batch_heads >= 64 && batch_heads * sequence_length >= 50000;
}

inline SplitOrder split_order(int batch, int query_heads, int key_value_heads, int query_blocks, bool spread = false) {
    constexpr int XCDS = 8, UNITS = 32;
    SplitOrder order;
    order.batch = batch;
    const int sharing = query_heads / key_value_heads;
    const bool by_group = (long long)batch * key_value_heads % XCDS == 0;
    order.clusters = by_group || spread || (long long)batch * query_heads % XCDS == 0 ? XCDS : 1;
    const int members = by_group ? sharing : 1;
    const long long groups = ((long long)batch * query_heads / members + order.clusters - 1) / order.clusters;   // of an XCD
    const long long inner = (long long)members * query_blocks;
    long long together = groups;
    if (order.clusters > 1 && groups * inner > 4 * UNITS) {
        together = (2 * UNITS + inner - 1) / inner;
        while (groups % together != 0) ++together;
    }
    order.together = (int)together;
    order.workgroups = order.clusters * groups * inner;
    order.turn = fast_division((unsigned)(together * inner));
    order.abreast = fast_division((unsigned)(together * members));
    order.members = fast_division((unsigned)members);
    order.groups = fast_division((unsigned)(query_heads / members));
    order.sharing = fast_division((unsigned)sharing);
    order.query_blocks = query_blocks;
    return order;
}

struct SplitItem {
    int batch, head, key_value_head, query_block;
};

DSCUDA_HOST_DEVICE inline SplitItem split_item(unsigned linear, const SplitOrder& order) {
    SplitItem item;
    const unsigned slot = order.clusters > 1 ? linear / 8 : linear;
    const unsigned turn = divide(slot, order.turn);
    const unsigned rest = slot - turn * order.turn.divisor;
    const unsigned rank = divide(rest, order.abreast);
    const unsigned pair = rest - rank * order.abreast.divisor;
    const unsigned group_of_turn = divide(pair, order.members);
    const unsigned local = turn * (unsigned)order.together + group_of_turn;
    const unsigned group = order.clusters > 1 ? linear % 8 + 8 * local : local;
    const unsigned batch = divide(group, order.groups);
    item.batch = (int)batch;
    item.head = (int)((group - batch * order.groups.divisor) * order.members.divisor + pair - group_of_turn * order.members.divisor);
    item.key_value_head = (int)divide((unsigned)item.head, order.sharing);
    item.query_block = order.query_blocks - 1 - (int)rank;
    return item;
}

// ---- decode: tile loads -------------------------------------------------------
// A [4 * ROWS_PER_WAVE][ROW_BYTES] tile of consecutive rows is fetched by four waves,
// wave w filling rows ROWS_PER_WAVE*w .. +ROWS_PER_WAVE-1 with 1 KB instructions: LDS
// slot 64*i + lane of the wave's share (16 bytes each) holds chunk (slot % CHUNKS) ^
// f(row) of local row slot / CHUNKS.  With i a compile-time constant a wave
// instruction spans at most two rows, so the row part of the offset is wave-uniform
// and the lane part costs an add, an xor and a shift-add per candidate row.  Rows
// past `row_limit` (of the tile) repeat that row.  ROWS_PER_WAVE = 16 is the 64-key
// tile, 8 the 32-key unit.
template <int ROW_BYTES, int ROWS_PER_WAVE = 16>
DSCUDA_HOST_DEVICE inline unsigned contiguous_load_offset(int wave, int i, int lane, int row_limit) {
    constexpr int CHUNKS = ROW_BYTES / 16;
    const int first_row = (64 * i) / CHUNKS;                 // row of lane 0 (within the wave's rows)
    const int boundary = CHUNKS * (first_row + 1) - 64 * i;  // first lane of the next row (may be >= 64)
    const int tile_row_a = ROWS_PER_WAVE * wave + first_row;
    const unsigned row_a = (unsigned)(tile_row_a < row_limit ? tile_row_a : row_limit) * ROW_BYTES;
    unsigned offset = row_a + 16u * (unsigned)((lane + 64 * i - CHUNKS * first_row) ^ tile_swizzle<ROW_BYTES>(tile_row_a));
    if (boundary < 64) {
        const int tile_row_b = tile_row_a + 1;
        const unsigned row_b = (unsigned)(tile_row_b < row_limit ? tile_row_b : row_limit) * ROW_BYTES;
        const unsigned other =
            row_b + 16u * (unsigned)((lane + 64 * i - CHUNKS * (first_row + 1)) ^ tile_swizzle<ROW_BYTES>(tile_row_b));
        offset = lane >= boundary ? other : offset;
    }
    return offset;
}

// ---- decode: cutting the work list ---------------------------------------------
// Every sequence with tokens contributes `overhead` + tiles positions to one list
// (sequence after sequence): its 64-token tiles, preceded by positions that stand for
// what a workgroup spends on a segment besides its tiles (query rows, the first
// requests, filling and draining the pipeline, storing the result), so that ranges of
// equal length take about equal time.  The list is cut into W = min(workgroups, total)
// ranges, none empty, whose lengths differ by at most one: range w is
// [w * total / W, (w + 1) * total / W).  A
// range computes the tiles whose positions it holds; a range that holds only part of
// the tiles of a sequence leaves a partial result in slot workgroup + sequence: ranges
// and sequences both advance monotonically, so no two (range, sequence) pairs that
// intersect share a slot, and every slot is below workgroups + sequences.
constexpr int SEGMENT_OVERHEAD = 6;   // in tiles: what a segment costs before, between and after its tiles

DSCUDA_HOST_DEVICE inline int positions_of(int tiles, int overhead) { return tiles > 0 ? tiles + overhead : 0; }

DSCUDA_HOST_DEVICE inline int ranges_of(int total, int workgroups) { return total < workgroups ? total : workgroups; }

// Whether what the two functions below divide fits 32 bits (a 64-bit division is some 500 cycles of a kernel's start).
DSCUDA_HOST_DEVICE inline bool products_fit(int total, int ranges) {
    return (unsigned long long)(unsigned)total * (unsigned)ranges <= 0xffffffffull;
}

// First position of range `range` (0 .. ranges: the last one is the end of the list).
DSCUDA_HOST_DEVICE inline int range_begin_of(int total, int ranges, int range) {
    if (products_fit(total, ranges)) return (int)((unsigned)range * (unsigned)total / (unsigned)ranges);
    return (int)((long long)range * total / ranges);
}

// The range that holds position `position` (0 <= position < total).
DSCUDA_HOST_DEVICE inline int range_of_position(int total, int ranges, int position) {
    if (products_fit(total, ranges)) return (int)((((unsigned)position + 1) * (unsigned)ranges - 1) / (unsigned)total);
    return (int)((((long long)position + 1) * ranges - 1) / total);
}

// Tiles [first, last) that the positions [begin, end) hold of a sequence whose positions
// start at `before`; last <= first when they hold none.
DSCUDA_HOST_DEVICE inline void tiles_in_positions(int begin, int end, int before, int overhead, int& first, int& last) {
    const int low = begin - before - overhead;
    const int high = end - before - overhead;
    first = low > 0 ? low : 0;
    last = high > 0 ? high : 0;
}

// First and last range that hold tiles of a sequence of `positions` > 0 positions that starts at `before`.
DSCUDA_HOST_DEVICE inline void ranges_of_sequence(int total, int ranges, int before, int positions, int overhead,
                                                  int& first, int& last) {
    first = range_of_position(total, ranges, before + overhead);
    last = range_of_position(total, ranges, before + positions - 1);
}

// ---- absorbed backward: the list of (key block, row tile) visits -----------------
// Rows are the (token, head) pairs of one batch element in memory order, 32 to a row
// tile (`row_tiles` of them); key block kb (32 keys) is seen by the row tiles from
// kb * heads (the tile of row 32 * kb * heads, the first row of token 32 * kb) to the
// last.  The visits of all key blocks of all batch elements, in that order, form one
// list that the key-gradient kernel cuts into ranges of equal length (+-1); a range
// that holds only part of a key block's visits leaves an fp32 partial result in slot
// range + (batch * key_blocks + key block): ranges and key blocks both advance
// monotonically along the list, so the sums are distinct and below ranges + blocks.
struct KeyVisits {
    int key_blocks;
    int row_tiles;
    int heads;

    DSCUDA_HOST_DEVICE long long before(int key_block) const {   // visits of key blocks 0 .. key_block-1
        return (long long)key_block * row_tiles - (long long)heads * key_block * (key_block - 1) / 2;
    }
    DSCUDA_HOST_DEVICE long long per_batch() const { return before(key_blocks); }
    DSCUDA_HOST_DEVICE int first_tile(int key_block) const { return key_block * heads; }
    // the key block that holds visit `visit` (0 <= visit < per_batch())
    DSCUDA_HOST_DEVICE int block_of(long long visit) const {
        int low = 0, high = key_blocks - 1;
        while (low < high) {
            const int middle = (low + high + 1) / 2;
            if (before(middle) <= visit) low = middle; else high = middle - 1;
        }
        return low;
    }
};

// `key_tiles`: key blocks of 32 * key_tiles keys.  Such a block is seen from the tile of row 32 * key_tiles * kb * heads
// on, which is what blocks of 32 keys and key_tiles * heads heads give: `heads` holds that product.
DSCUDA_HOST_DEVICE inline KeyVisits key_visits(int sequence_length, int heads, int key_tiles = 1) {
    KeyVisits visits;
    visits.key_blocks = (sequence_length + 32 * key_tiles - 1) / (32 * key_tiles);
    visits.row_tiles = (int)(((long long)sequence_length * heads + 31) / 32);
    visits.heads = heads * key_tiles;
    return visits;
}

// Where the key-gradient kernels keep dS for the query-gradient product, when they have a workspace: a block of 2 KB
// per (32-key tile, row tile) that a key block of 32 * key_tiles keys visits, in the order of the visits, so that the
// blocks of neighbouring row tiles lie one behind the other.  Inside a block key k has bytes 64k .. 64k + 63: bf16 of
// row 16r + 4q + e at 16q + 8r + 2e, which both sides move as whole 16-byte pieces of consecutive lanes.
struct KeptGradients {
    static constexpr int BLOCK_BYTES = 2048;
    KeyVisits visits;
    int key_tiles;

    DSCUDA_HOST_DEVICE long long bytes() const { return visits.per_batch() * key_tiles * BLOCK_BYTES; }
    DSCUDA_HOST_DEVICE long long at(int tile, int row_tile) const {
        const int block = tile / key_tiles;
        const long long visit = visits.before(block) + row_tile - visits.first_tile(block);
        return (visit * key_tiles + tile % key_tiles) * BLOCK_BYTES;
    }
};

DSCUDA_HOST_DEVICE inline KeptGradients kept_gradients(int sequence_length, int heads, int key_tiles) {
    return KeptGradients{key_visits(sequence_length, heads, key_tiles), key_tiles};
}

// Bytes that hold dS of one batch element for key blocks of either size.
DSCUDA_HOST_DEVICE inline long long kept_gradient_bytes(int sequence_length, int heads) {
    const long long narrow = kept_gradients(sequence_length, heads, 1).bytes();
    const long long wide = kept_gradients(sequence_length, heads, 2).bytes();
    return narrow > wide ? narrow : wide;
}

DSCUDA_HOST_DEVICE inline long long wide_range_begin(long long total, long long ranges, long long range) {
    return range * total / ranges;
}

DSCUDA_HOST_DEVICE inline long long wide_range_of(long long total, long long ranges, long long position) {
    return ((position + 1) * ranges - 1) / total;
}

// Large inputs (the query and dO rows of a batch element no longer stay in the caches): equal ranges would have
// every workgroup stream its own stretch of rows from memory, one pass over all rows per key block.  Instead the
// row tiles are cut into intervals of `length` tiles and the work into items (interval, key block), numbered
// interval by interval, so that the workgroups running at any time walk the same few intervals and all but
// the first of them find the rows in the caches.  Item (i, kb) exists when the block sees the interval
// (kb * heads < end of interval i), covers the block's tiles inside it, and leaves its partial result in the
// slot of its own number (none when it is the block's only item, i.e. the block starts in the last interval).
struct KeyIntervals {
    int length;      // row tiles per interval
    int intervals;
    int heads;
    int key_blocks;
    int row_tiles;

    DSCUDA_HOST_DEVICE int end_of(int interval) const {
        const long long end = (long long)(interval + 1) * length;
        return end < row_tiles ? (int)end : row_tiles;
    }
    DSCUDA_HOST_DEVICE int blocks_in(int interval) const {   // key blocks 0 .. blocks_in-1 see the interval
        const int seen = (end_of(interval) + heads - 1) / heads;
        return seen < key_blocks ? seen : key_blocks;
    }
    DSCUDA_HOST_DEVICE long long items_before(int interval) const {
        long long items = 0;
        for (int i = 0; i < interval; ++i) items += blocks_in(i);
        return items;
    }
    DSCUDA_HOST_DEVICE long long items() const { return items_before(intervals); }
    DSCUDA_HOST_DEVICE int first_interval(int key_block) const { return (int)((long long)key_block * heads / length); }
    // item number (within its batch element) -> interval, key block
    DSCUDA_HOST_DEVICE void locate(long long item, int& interval, int& key_block) const {
        interval = 0;
        while (item >= blocks_in(interval)) {
            item -= blocks_in(interval);
            ++interval;
        }
        key_block = (int)item;
    }
};

DSCUDA_HOST_DEVICE inline KeyIntervals key_intervals(int sequence_length, int heads, int length, int key_tiles = 1) {
    KeyIntervals cut;
    cut.length = length;
    cut.heads = heads * key_tiles;   // as in key_visits
    cut.key_blocks = (sequence_length + 32 * key_tiles - 1) / (32 * key_tiles);
    cut.row_tiles = (int)(((long long)sequence_length * heads + 31) / 32);
    cut.intervals = (cut.row_tiles + length - 1) / length;
    return cut;
}

constexpr long long KEY_PARTIAL_BYTES = 32LL * 576 * 4;   // one slot: [32 keys][576] fp32

// Interval length (row tiles) of the cut into items: the shortest of the ladder 24, 32, 48, 64, 96, ... whose items,
// over `batch` batch elements, number at most twelve rounds of the compute units and have a slot each (shorter
// intervals give more, shorter items: a fuller last round, as long as the slots last).  0: even that many items
// are fewer than two rounds, or no length of the ladder fits; equal ranges balance the units better then.
DSCUDA_HOST_DEVICE inline int key_interval_choice(int sequence_length, int heads, long long batch, long long slots,
                                                  int compute_units, int key_tiles) {
    const long long rounds = 12LL * compute_units;
    const long long most = rounds < slots ? rounds : slots;
    const long long row_tiles = ((long long)sequence_length * heads + 31) / 32;
    for (long long base = 8; ; base *= 2) {
        for (int multiple = 3; multiple <= 4; ++multiple) {
            const long long tiles = base * multiple;
            if (tiles >= (1 << 24)) return 0;
            const long long items = key_intervals(sequence_length, heads, (int)tiles, key_tiles).items() * batch;
            if (items <= most) return items >= 2LL * compute_units ? (int)tiles : 0;
            if (tiles >= row_tiles) return 0;
        }
    }
}

// The same where dS is kept in a workspace, which has room for slots as well: the length whose items take the least
// time, r rounds of the compute units of `length` + ITEM_OVERHEAD steps each (the keys, the first tile, the partial
// result and its share of the reduction), over the shortest length whose items number at most r rounds, r = 1 .. 12.
// Backward in us by rounds 1, 2, 3, 5, 7, 12: 2048 tokens x 128 heads 1786 1721 1744 1791 1862 2116, 4096 x 128 7260 6892
// 6598 6397 6318 6519, 8000 x 16 3283 2942 2933 2927 2936 3009, 1024 x 128 535 554 594 683 804 1201, which is what the
// sum predicts to 3 %; the ladder above: 1898, 6471, 605 (1024 x 128).
// 0: so few visits a unit that ranges of 32-key blocks, which need no whole rounds, are the better cut (ranges / items:
// 480 x 16 54 / 69, 200 x 32 43 / 65, 226 x 128 77 / 91; 1000 x 4 68 / 69, 4 x 512 x 8 78 / 73, 2 x 592 x 16 95 / 83,
// 2048 x 4 137 / 117, 2845 x 4 x 3 583 / 385).
constexpr int ITEM_OVERHEAD = 12;
constexpr int MOST_ROUNDS = 12;

DSCUDA_HOST_DEVICE inline int key_interval_fit(int sequence_length, int heads, long long batch, long long slots,
                                               int compute_units, int key_tiles) {
    const long long visits = key_visits(sequence_length, heads, key_tiles).per_batch() * batch;
    if (slots <= 0 || visits < (heads < 16 ? 5LL : 10LL) * compute_units) return 0;
    const long long row_tiles = ((long long)sequence_length * heads + 31) / 32;
    long long best = 0, best_cost = 0;
    for (int rounds = 1; rounds <= MOST_ROUNDS; ++rounds) {
        const long long most = (long long)rounds * compute_units < slots ? (long long)rounds * compute_units : slots;
        long long length = (visits + most - 1) / most;
        while (length < row_tiles && key_intervals(sequence_length, heads, (int)length, key_tiles).items() * batch > most) {
            length += 1 + length / 64;
        }
        if (length > row_tiles) length = row_tiles;
        if (length >= (1 << 24)) continue;
        const long long items = key_intervals(sequence_length, heads, (int)length, key_tiles).items() * batch;
        const long long cost = (items + compute_units - 1) / compute_units * (length + ITEM_OVERHEAD);
        if (items <= slots && (best == 0 || cost < best_cost)) {
            best = length;
            best_cost = cost;
        }
    }
    return (int)best;
}

// How many ranges the list is cut into when `scratch_bytes` are there for the slots: one per compute unit if the
// slots allow.  0: every key block is one range and writes its result itself (too few slots for a cut whose
// longest range is shorter than the longest key block, `row_tiles` visits).
DSCUDA_HOST_DEVICE inline long long key_gradient_ranges(long long total, long long blocks, int row_tiles,
                                                        long long scratch_bytes, int compute_units) {
    const long long slots = scratch_bytes / KEY_PARTIAL_BYTES;
    long long ranges = slots - blocks;
    if (ranges > compute_units) ranges = compute_units;
    if (ranges > total / 2) ranges = total / 2;    // at least two visits per range
    if (ranges < 2) return 0;
    const long long longest = (total + ranges - 1) / ranges;
    return (longest < row_tiles || blocks > compute_units) ? ranges : 0;
}

// ---- absorbed backward where dS is kept: short walks ----------------------------------
// A range that runs from one key block into the next ends one walk and begins another, and partial results take one launch
// more (a range over the border costs some 6 us: 6 x 58 x 8 30, 6 x 64 x 8 26).  Ranges of two visits, which every call of at
// most two a compute unit has, do not cross where the blocks' walks are even.
DSCUDA_HOST_DEVICE inline bool ranges_stay_in_blocks(const KeyVisits& visits, long long batch, int compute_units) {
    if (visits.per_batch() * batch > 2LL * compute_units) return false;
    return visits.key_blocks * batch == 1 || (visits.row_tiles % 2 == 0 && (visits.key_blocks == 1 || visits.heads % 2 == 0));
}

// Whether a workgroup walks a key block from its first row tile to its last, writes its gradients itself and there is no
// reduction, or the walks are cut into ranges.  In steps of a walk, fitted to 6100 shapes of up to 60000 rows (the choice
// costs 0.3 % against the better of the two): beginning and end of a walk 7, the reduction 3.  Backward in us, cut /
// whole: 512 x 1 token x 1 head 38 / 25, 2000 x 1 x 1 125 / 82, 128 x 5 x 16 37 / 30, 300 x 158 x 1 180 / 151, 64 x 49 x 5 40 / 36;
// 1 x 142 x 40 36 / 227, 8 x 121 x 16 46 / 98, 16 x 21 x 16 31.0 / 29.6, 3 x 11 x 36 23.3 / 27.7.
constexpr int WALK_ENDS = 7;
constexpr int REDUCTION_STEPS = 3;
constexpr int SHORT_WALK = 12;   // row tiles up to which items of 64-key blocks are never the better cut (300 x 158 x 1 180)

DSCUDA_HOST_DEVICE inline bool whole_key_walks(int sequence_length, int heads, long long batch, int compute_units) {
    const KeyVisits visits = key_visits(sequence_length, heads);
    const long long total = visits.per_batch() * batch, blocks = (long long)visits.key_blocks * batch;
    const long long ranges = key_gradient_ranges(total, blocks, visits.row_tiles, (blocks + compute_units) * KEY_PARTIAL_BYTES, compute_units);
    if (visits.row_tiles <= 2 || ranges == 0) return true;
    const long long whole = blocks <= compute_units ? visits.row_tiles + WALK_ENDS
                                                    : (total + WALK_ENDS * blocks) / compute_units + visits.row_tiles / 2;
    const long long crossings = ranges_stay_in_blocks(visits, batch, compute_units) ? 0 : blocks > ranges ? blocks / ranges : 1;
    // (an odd list of visits in ranges of two has one of three, which crosses no border)
    const long long longest = total == 2 * ranges + 1 ? 2 : (total + ranges - 1) / ranges;
    return whole <= longest + WALK_ENDS * (1 + crossings) + REDUCTION_STEPS;
}

// How the key gradients of a call are cut: items of 64-key blocks in intervals of `length` row tiles, or (length 0) ranges of
// 32-key blocks, or (ranges 0) whole 32-key blocks, and the bytes of slots that takes.
struct KeyCut {
    int length;
    long long items;
    long long ranges;
    long long slot_bytes;
};
constexpr int KEY_PAIR = 2;   // 32-key tiles of an item

DSCUDA_HOST_DEVICE inline KeyCut key_cut_of_length(int sequence_length, int heads, long long batch, int length) {
    const KeyIntervals intervals = key_intervals(sequence_length, heads, length, KEY_PAIR);
    const long long items = intervals.items() * batch;
    return KeyCut{length, items, 0, intervals.intervals > 1 ? items * KEY_PAIR * KEY_PARTIAL_BYTES : 0};   // one interval: no partial results
}

DSCUDA_HOST_DEVICE inline KeyCut key_cut_of_ranges(int sequence_length, int heads, long long batch, long long slot_bytes, int compute_units) {
    const KeyVisits visits = key_visits(sequence_length, heads);
    const long long blocks = (long long)visits.key_blocks * batch;
    const long long ranges = key_gradient_ranges(visits.per_batch() * batch, blocks, visits.row_tiles, slot_bytes, compute_units);
    return KeyCut{0, 0, ranges, ranges > 0 ? (ranges + blocks) * KEY_PARTIAL_BYTES : 0};
}

// Where dS is kept and there is room for `slot_bytes` of slots.
DSCUDA_HOST_DEVICE inline KeyCut kept_cut(int sequence_length, int heads, long long batch, long long slot_bytes, int compute_units) {
    const KeyVisits visits = key_visits(sequence_length, heads, KEY_PAIR);
    if (visits.row_tiles > SHORT_WALK) {
        // whole blocks, which take no slots, are as many items as there are blocks, and every cut of them is more
        const long long blocks = (long long)visits.key_blocks * batch, slots = slot_bytes / (KEY_PAIR * KEY_PARTIAL_BYTES);
        const int length = key_interval_fit(sequence_length, heads, batch, slots > blocks ? slots : blocks, compute_units, KEY_PAIR);
        if (length > 0) return key_cut_of_length(sequence_length, heads, batch, length);
    }
    if (whole_key_walks(sequence_length, heads, batch, compute_units)) return KeyCut{0, 0, 0, 0};
    return key_cut_of_ranges(sequence_length, heads, batch, slot_bytes, compute_units);
}

// The slots that a cut may ask of a workspace where the latent query gradients hold fewer: three rounds of items, more
// than the blocks and ranges of any call that is cut into ranges.
constexpr long long WORKSPACE_SLOT_BYTES = 3LL * 256 * KEY_PAIR * KEY_PARTIAL_BYTES;   // 113 MB

DSCUDA_HOST_DEVICE inline long long query_gradient_bytes(int sequence_length, int heads, long long batch) {
    return (long long)sequence_length * heads * batch * 1024;
}

// A batch in passes of at most `most` elements, as equal as they can be: pass p has elements first(p) .. first(p + 1) - 1.
// (64 x 4096 tokens x 4 heads, whose dS allows 63 elements a pass: 17.0 ms with a last pass of one element, 15.5 in halves.)
struct BatchPasses {
    long long batch;
    long long passes;

    DSCUDA_HOST_DEVICE long long first(long long pass) const { return batch * pass / passes; }
    DSCUDA_HOST_DEVICE long long largest() const { return (batch + passes - 1) / passes; }   // the others have one less, or as many
};

DSCUDA_HOST_DEVICE inline BatchPasses batch_passes(long long batch, long long most) {
    return BatchPasses{batch, (batch + most - 1) / most};
}

// Whether a call's slots lie in its workspace: where the latent query gradients might not hold them.  (They can for
// 300 tokens x 64 heads, 20 MB: 72 us there, 69 in the workspace; equal from 35 MB on.)
DSCUDA_HOST_DEVICE inline bool slots_in_workspace(int sequence_length, int heads, long long batch) {
    return query_gradient_bytes(sequence_length, heads, batch) < WORKSPACE_SLOT_BYTES;
}

// Slots to choose the cut of a call by that has a workspace of the size it asks for.
DSCUDA_HOST_DEVICE inline long long slot_bytes_of_workspace(int sequence_length, int heads, long long batch) {
    const long long scratch = query_gradient_bytes(sequence_length, heads, batch);
    return scratch > WORKSPACE_SLOT_BYTES ? scratch : WORKSPACE_SLOT_BYTES;
}

// ---- absorbed backward of short sequences: where P is kept ------------------------
// Row `row` = token * heads + head of a batch element with `blocks` blocks of 32 tokens (the last one possibly short)
// keeps dS of key block b (32 keys, 64 bytes) in chunk b of its own 16 chunks of the latent query gradient, b = 0 ..
// its token block.  P of key block b: for a row of token block i < blocks - 1 in chunk kept_chunk of row kept_row, a
// row of block blocks - 2 - i, behind that row's dS; for a row of the last block in the rope query gradient (one
// chunk a row) of row kept_row, a row of block b.
constexpr int SHORT_TOKENS = 512;

// Which calls keep P and dS instead of partial key gradients.  More tokens do not fit.  The key-gradient launch walks
// all rows of a batch element per 32 keys x 32 columns, so many rows, or many heads on few keys, are better off with
// the other kernels; so are calls whose key blocks alone occupy half the chip there, and those with one row tile a batch
// element or with batch elements enough to fill the chip, where one launch more is what counts.  Forward and backward,
// partial results -> kept (us): 512 tokens x 8 heads 106 -> 71, 300 x 4 106 -> 46, 350 x 16 82 -> 70, 128 x 32 56 -> 49,
// 3 x 500 x 4 142 -> 81, 8 x 500 x 4 169 -> 152.  Backward alone, kept / partial results, of calls left to the others:
// 200 x 32 and 480 x 16 equal, 4 x 512 x 8 1.04, 2 x 174 x 32 1.06, 2 x 278 x 20 1.13, 3 x 302 x 16 1.10, 14 x 337 x 3 1.15,
// 13 x 359 x 2 1.11, 13 x 4 x 1 1.31, 64 x 2 x 20 1.41, 24 x 2 x 17 1.14, 16 x 4 x 9 1.05, 64 x 8 x 8 1.25, 64 x 48 x 4 1.17,
// 24 x 100 x 1 1.11; of calls that keep them: 2 x 219 x 20 0.92, 4 x 113 x 20 0.81, 8 x 338 x 3 0.84, 9 x 301 x 3 0.87,
// 1 x 3 x 16 0.93, 8 x 4 x 9 0.97, 32 x 16 x 8 0.91, 32 x 64 x 4 0.91, 16 x 100 x 1 1.00.
DSCUDA_HOST_DEVICE inline bool short_backward(long long batch, int tokens, int heads) {
    const long long rows = (long long)tokens * heads;
    if (tokens > SHORT_TOKENS || heads > 32 || rows > 6000 || rows * batch > 16000 || rows <= 32) return false;
    if (batch > (rows < 64 ? 12 : heads == 1 ? 16 : 32)) return false;
    if (heads <= 3) return batch * ((tokens + 31) / 32) <= 110;
    return heads < 16 || rows * batch * tokens <= (heads <= 20 ? 2000000 : 1600000);
}

// Which of them still do where a workspace could hold dS: those of a few hundred visits whose key blocks are neither short
// walks (whole_key_walks) nor cut into ranges that stay inside them.  Backward in us, P and dS kept / dS in a workspace:
// 6 x 58 x 8 24 / 30, 3 x 121 x 8 27 / 34, 9 x 26 x 11 22 / 28, 1 x 49 x 17 23 / 27; 1 x 157 x 32 46 / 41;
// taken by the workspace form: 2 x 219 x 20 53 / 43, 8 x 338 x 3 63 / 49, 512 x 8 50 / 46, 64 x 32 28 / 24, 32 x 64 x 4 34 / 29,
// 12 x 2 x 17 20 / 15, 6 x 60 x 32 38 / 41, 9 x 168 x 4 39 / 43.
DSCUDA_HOST_DEVICE inline bool short_without_workspace(long long batch, int tokens, int heads) {
    const KeyVisits visits = key_visits(tokens, heads);
    const long long blocks = (long long)visits.key_blocks * batch;
    if (visits.row_tiles <= 2 || visits.per_batch() * batch > 512) return false;
    if (ranges_stay_in_blocks(visits, batch, 256) && (heads > 4 || visits.row_tiles <= 5 || blocks > 16)) return false;
    if (visits.row_tiles <= 5) return blocks <= 12 && heads <= 10;
    if (visits.row_tiles <= 8) return blocks <= 20;
    return visits.row_tiles > 12 || blocks <= 32;
}

DSCUDA_HOST_DEVICE inline bool kept_in_rope(int token_block, int blocks) { return token_block == blocks - 1; }

DSCUDA_HOST_DEVICE inline int kept_row(int row, int token_block, int key_block, int blocks, int heads) {
    const int block = kept_in_rope(token_block, blocks) ? key_block : blocks - 2 - token_block;
    return row + (block - token_block) * 32 * heads;
}

DSCUDA_HOST_DEVICE inline int kept_chunk(int token_block, int key_block, int blocks) {
    return blocks - 1 - token_block + key_block;
}

// ---- projections: do results lie over inputs ---------------------------------------
// Rows of `width` elements, `tokens` x `heads` of them.
struct ProjectionRows {
    long long token_stride, head_stride;   // in elements
    int width;

    DSCUDA_HOST_DEVICE long long extent(long long tokens, int heads) const {
        return (tokens - 1) * token_stride + (heads - 1) * head_stride + width;
    }
};

// Whether no element of `y`, whose first row starts `offset` elements behind the first row of `x`, is one of `x`: apart in
// memory, or different columns of the same rows.  False where that is not plain to see.
DSCUDA_HOST_DEVICE inline bool rows_apart(const ProjectionRows& x, const ProjectionRows& y, long long offset,
                                          long long tokens, int heads) {
    if (offset >= x.extent(tokens, heads) || -offset >= y.extent(tokens, heads)) return true;
    if (x.token_stride != y.token_stride || x.head_stride != y.head_stride || x.token_stride % x.head_stride != 0) return false;
    const long long column = (offset % x.head_stride + x.head_stride) % x.head_stride;
    return column >= x.width && column + y.width <= x.head_stride;
}

// ---- decode: the plan and how a call uses the caller's workspace ---------------
// The plan is what a decode call needs to know about the lengths of its batch
// before any workgroup starts: an int table
//     [0] total positions   [1] workgroups   [2] overhead positions per sequence   [3] mode (below)
//     [4] ranges the list is cut into (<= workgroups)
//     [5 .. 5+B]        inclusive prefix of positions per sequence (B + 1 entries)
//     [.. + W]          first sequence whose positions reach past the start of each range
// It is read-only once built.
constexpr int PLAN_TOTAL = 0;
constexpr int PLAN_WORKGROUPS = 1;
constexpr int PLAN_OVERHEAD = 2;
constexpr int PLAN_MODE = 3;
constexpr int PLAN_RANGES = 4;
constexpr int PLAN_HEADER = 5;

// Modes: ranges cut sequences, whose parts are kept in bf16 or (wide) in fp32, or there is a workgroup per sequence.
constexpr int PLAN_PARTS = 0;
constexpr int PLAN_WHOLE = 1;
constexpr int PLAN_WIDE_PARTS = 2;

DSCUDA_HOST_DEVICE inline long long plan_prefix_at() { return PLAN_HEADER; }
DSCUDA_HOST_DEVICE inline long long plan_first_sequence_at(int batch) { return PLAN_HEADER + (long long)batch + 1; }
DSCUDA_HOST_DEVICE inline long long plan_elements(int batch, int workgroups) {
    return plan_first_sequence_at(batch) + workgroups;
}
// Thread `thread` of `threads` copies its share of a plan's prefix, which has an entry more than there are sequences.
DSCUDA_HOST_DEVICE inline void leave_prefix(int* plan, const int* prefix, int batch, int thread, int threads) {
    for (int s = thread; s <= batch; s += threads) plan[plan_prefix_at() + s] = prefix[s];
}
// Size of a plan buffer that fits whatever device builds the plan: a call cuts its list into at
// most one range per compute unit (the host clamps the count it asks the device for to
// PLAN_MAX_WORKGROUPS), or runs one workgroup per sequence.
constexpr int PLAN_MAX_WORKGROUPS = 1024;
DSCUDA_HOST_DEVICE inline long long plan_elements_bound(int batch) {
    return plan_elements(batch, batch > PLAN_MAX_WORKGROUPS ? batch : PLAN_MAX_WORKGROUPS);
}

// The caller's workspace holds batch * heads * splits * (rank + 2) floats.  A
// range that holds only part of a sequence leaves its unnormalised result there:
// slot workgroup + sequence (slots = workgroups + batch), each slot one bf16 row of
// `rank` values plus two floats (reference exponent, sum) per head, heads rounded up
// to whole waves of 32.  A call without a caller-provided plan keeps its plan behind
// the slots.  The number of workgroups is the largest (up to one per compute unit)
// for which all of that fits; when fewer than two fit, no sequence is cut: one
// workgroup per sequence, no slots.
struct DecodeLayout {
    int workgroups;
    int whole_sequences;
    int head_groups;
    long long slot_floats;
    long long slots;
    long long plan_offset;   // in floats from the start of the workspace
    long long plan_ints;
    // Fallback of narrow_decode_layout, for batches with sequences that `reference_ranges` ranges leave uncut (0: none):
    // `wide_ranges` ranges with fp32 parts or, if that is 0, `reference_ranges` with bf16 parts.
    int reference_ranges;
    int wide_ranges;
    long long wide_slot_floats;
};

DSCUDA_HOST_DEVICE inline DecodeLayout decode_layout(int batch, int heads, int splits, int compute_units,
                                                     int rows_per_group, int rank) {
    DecodeLayout layout;
    layout.head_groups = (heads + rows_per_group - 1) / rows_per_group;
    const long long padded_rows = (long long)((heads + 31) / 32) * 32;
    layout.slot_floats = padded_rows * (rank / 2 + 2);
    const long long workspace = (long long)batch * heads * splits * (rank + 2);
    // (W + batch) * slot_floats + plan_elements(batch, W) <= workspace, W <= compute_units
    const long long fixed = (long long)batch * layout.slot_floats + plan_elements(batch, 0);
    long long cutting = workspace >= fixed ? (workspace - fixed) / (layout.slot_floats + 1) : 0;
    if (cutting > compute_units) cutting = compute_units;
    layout.whole_sequences = (splits <= 1 || cutting < 2) ? 1 : 0;
    if (layout.whole_sequences) {
        layout.workgroups = batch;
        layout.slots = 0;
    } else {
        layout.workgroups = (int)cutting;
        layout.slots = (long long)layout.workgroups + batch;
    }
    layout.plan_offset = layout.slots * layout.slot_floats;
    layout.plan_ints = plan_elements(batch, layout.workgroups);
    layout.reference_ranges = layout.wide_ranges = 0;
    layout.wide_slot_floats = 0;
    return layout;
}

// The same for the kernels that take 32 * row_blocks rows (heads) per workgroup: slots hold the real heads only, one
// bf16 row of `rank` values plus two floats per head, rounded up to 16 bytes, and the compute units are shared by the
// head groups.
//
// Fewer padded heads a slot means more ranges than decode_layout finds slots for, and so cuts through sequences that its
// ranges hold whole.  A whole sequence stays in fp32 until its result is rounded; as bf16 parts it is rounded once more
// (relative error against fp64 of one sequence of 400 tokens, 8 heads: 2.4e-3 whole, 2.8e-3 in parts).  So bf16 parts are
// for batches all of whose sequences the ranges of decode_layout (`reference_ranges`) cut as well; any other batch is
// cut into `wide_ranges` ranges with fp32 parts, for which slots of twice the size leave room, or as decode_layout would
// (wide_ranges 0) if that makes more ranges; a workgroup per sequence where decode_layout has that and the ranges would be
// fewer than the sequences (ranges / workgroups: two sequences of 13 tokens, 16 heads, 2 splits 16.6 / 7.3 us).  bf16 parts
// throughout -> so, us: eight heads, 8 splits, eight sequences of 1024..8192 tokens 24.7 -> 35.1, 1 of 400 11.0 -> 13.4;
// 16 heads, 2 splits, eight of 1024..8192 62.8 -> 171.
DSCUDA_HOST_DEVICE inline DecodeLayout narrow_decode_layout(int batch, int heads, int splits, int compute_units,
                                                            int row_blocks, int rank) {
    DecodeLayout layout;
    const int rows_per_group = 32 * row_blocks;
    layout.head_groups = (heads + rows_per_group - 1) / rows_per_group;
    layout.slot_floats = ((long long)heads * (rank / 2 + 2) + 3) / 4 * 4;
    const long long workspace = (long long)batch * heads * splits * (rank + 2);
    const long long fixed = (long long)batch * layout.slot_floats + plan_elements(batch, 0);
    long long cutting = workspace >= fixed ? (workspace - fixed) / (layout.slot_floats + 1) : 0;
    const int most = compute_units > layout.head_groups ? compute_units / layout.head_groups : 1;
    if (cutting > most) cutting = most;
    layout.whole_sequences = (splits <= 1 || cutting < 2) ? 1 : 0;
    layout.workgroups = layout.whole_sequences ? batch : (int)cutting;
    layout.slots = layout.whole_sequences ? 0 : (long long)layout.workgroups + batch;
    layout.plan_offset = layout.slots * layout.slot_floats;
    layout.plan_ints = plan_elements(batch, layout.workgroups);
    layout.reference_ranges = layout.wide_ranges = 0;
    layout.wide_slot_floats = ((long long)heads * (rank + 2) + 3) / 4 * 4;
    if (layout.whole_sequences) return layout;
    const DecodeLayout reference = decode_layout(batch, heads, splits, compute_units, 128, rank);
    const int reference_ranges = reference.whole_sequences ? 1 : reference.workgroups;
    if (reference_ranges < layout.workgroups) {
        layout.reference_ranges = reference_ranges;
        long long wide = (workspace - layout.plan_ints) / layout.wide_slot_floats - batch;
        if (wide > layout.workgroups) wide = layout.workgroups;
        if (wide < 1) wide = 1;   // a single range cuts nothing and needs no slot
        if (reference.whole_sequences && wide < batch) {   // decode_layout runs every sequence on its own: not fewer at a time
            layout.whole_sequences = 1;
            layout.workgroups = batch;
            layout.slots = layout.plan_offset = 0;
            layout.plan_ints = plan_elements(batch, batch);
            layout.reference_ranges = 0;
            return layout;
        }
        if (wide >= reference_ranges) {
            layout.wide_ranges = (int)wide;
            const long long wide_end = wide > 1 ? (wide + batch) * layout.wide_slot_floats : 0;
            if (wide_end > layout.plan_offset) layout.plan_offset = wide_end;   // the plan goes behind either slots
        }
    }
    return layout;
}

// Which kernel takes a decode call, and how its list is cut.
struct DecodeForm {
    int row_blocks;   // 32 * row_blocks rows per workgroup; 0: 128 rows
    DecodeLayout layout;
};

constexpr int DECODE_ROWS = 128;
constexpr int NARROW_SEQUENCE_GROUPS = 48;

// Depends on the batch, the head count and the splits only, so that a plan built for them fits the call.  The line
// between the kernels (times of the whole call, 1024..8192 tokens a sequence unless stated, 8 splits):
//   * 32 rows when one head group holds all heads (64 sequences, 16 heads: 69 us against 75 with 64 rows and 104 with
//     128; 32 heads: 75 / 76 / 104), or when every range the partial-result slots allow finds a compute unit for each
//     of its head groups anyway (4 sequences, 128 heads: 31 / 32 / 53; 1 sequence of 200 tokens: 13 / 14 / 21);
//   * 64 rows up to 64 heads (64 sequences, 64 heads: 109 / 83 / 109) and beyond while sequences x head groups stay
//     few: the 128-row kernel is then held back by its slots and its start (16 sequences, 128 heads: 63 / 50 / 64);
//   * 128 rows otherwise (32 sequences, 128 heads: 101 / 78 / 79; 64 sequences: 183 / 136 / 117).
inline DecodeForm decode_form(int batch, int heads, int splits, int compute_units, int rank) {
    const long long groups32 = (heads + 31) / 32, groups64 = (heads + 63) / 64;
    const long long ranges = (long long)batch * (2LL * splits - 1);
    DecodeForm form;
    if (groups32 == 1 || groups32 * ranges <= compute_units) {
        form.row_blocks = 1;
    } else if (groups64 == 1 || batch * groups64 <= NARROW_SEQUENCE_GROUPS) {
        form.row_blocks = 2;
    } else {
        form.row_blocks = 0;
    }
    form.layout = form.row_blocks == 0 ? decode_layout(batch, heads, splits, compute_units, DECODE_ROWS, rank)
                                       : narrow_decode_layout(batch, heads, splits, compute_units, form.row_blocks, rank);
    return form;
}

// The form a call with `page_size` tokens a page takes.  Pages that do not hold whole units of 32 keys are looked up key
// by key, nine round trips a unit that bound the call, and head groups of 64 each do so for the whole cache.  Where
// 128 rows make more ranges than those groups have, they take over (64 / 128 rows, pages of one token: 20 sequences of
// 14913 tokens, 128 heads, 32 splits 446 / 284 us, 19 of 18668, 96 heads 519 / 332; of 48 tokens: 16 of 16051, 96 heads
// 360 / 237).  A plan built for the other form serves: its positions are the same, the ranges are counted anew.
inline DecodeForm decode_form_of_call(int batch, int heads, int splits, int page_size, int compute_units, int rank) {
    const DecodeForm form = decode_form(batch, heads, splits, compute_units, rank);
    if (form.row_blocks != 2 || page_size % 32 == 0 || form.layout.whole_sequences) return form;
    const DecodeForm wide = {0, decode_layout(batch, heads, splits, compute_units, DECODE_ROWS, rank)};
    return wide.layout.head_groups < form.layout.head_groups && !wide.layout.whole_sequences &&
            wide.layout.workgroups > form.layout.workgroups ? wide : form;
}

// Whether `ranges` ranges cut the sequence with `positions` positions from `before` on.
DSCUDA_HOST_DEVICE inline bool sequence_is_cut(int total, int ranges, int before, int positions, int overhead) {
    int first, last;
    ranges_of_sequence(total, ranges, before, positions, overhead, first, last);
    return first != last;
}

}  // namespace index_math
}  // namespace dscuda
