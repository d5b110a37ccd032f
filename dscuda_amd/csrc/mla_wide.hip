// Absorbed MLA attention, 128 query rows a workgroup: the causal prefill forward, and the decode over pages that hold whole
// units.  Takes the place of the reference's mla_forward_kernel and mla_decode_split_kernel
// (kernels/attention/mla/sm89.cu:156-291, 413-477); the decomposition below is built around 64-lane MFMA waves and the 160 KB LDS and
// shares nothing with their per-head scalar loops.
//
// Rows and units
//   A workgroup owns 128 rows, consecutive (token, head) pairs (decode: heads of a sequence), and walks
//   a stream of keys in units of 32.  Every row reads the same keys, so a unit is fetched once for 128 rows x (576 + 512)
//   x 2 flop per key.
//
// Eight waves, two a SIMD
//   scores     S^T (32 keys x 16 rows) = K Q^T: a wave has 16 rows, their 576 columns as operands in 72 registers
//              (16x16x32 MFMA, two key halves, 18 steps), the exponentials of its scores, and leaves P as bf16 in LDS
//   products   O^T (64 columns x 128 rows) += V^T P^T: a wave has 64 of the 512 columns of all rows, 128 registers
//              (32x32x16 MFMA, 16 a unit); a V fragment is read once in the workgroup, P by all waves
//   In a step the products of unit n and the scores of unit n + 1 go side by side: waves 0..3 take the products first,
//   waves 4..7 (on the same SIMDs) the scores, so that one's exponentials run beside the other's MFMAs; one barrier ends
//   the step.  With four waves of 32 rows each, 512 registers a wave and one wave a SIMD, a wave's scores, exponentials,
//   LDS reads and products queue up behind each other: a step takes 3800 to 4100 cycles there and 3200 here, of which
//   2176 are MFMAs (forward in us, four waves -> here, 128 heads: 1024 tokens 176 -> 153, 2048 590 -> 519, 4096 2129 -> 1916;
//   3 x 700 x 33 86 -> 66, 40 x 130 x 16 57 -> 39, 7 x 257 x 128 169 -> 139).
//
// The stream runs on over the ends of items
//   A workgroup takes several items (blocks of 128 rows; decode: the segments of its range of the work list), one a compute unit being all that the
//   registers and the LDS hold.  Units are requested three steps ahead, the next item's among them; the query rows of the
//   next item are asked for as the last scores of this one release their registers.  An item used to cost 12 to 20 us
//   besides its units (a workgroup's start, query rows and first units, its rows on their way out), now some 7, of which
//   the query rows take most: 147 KB at the 21 bytes a cycle that a compute unit draws.
//
// LDS
//   Four slots of 32 latent rows, three of 32 rope rows (a unit's rope rows are only read for its scores, a step before
//   its values), P of two units: 156 of 160 KB.  A latent row is one 1 KB request
//   (global_load_lds, 16 bytes a lane): its address is a scalar, the swizzle of index_math::tile_swizzle a lane's constant.
//   Bank conflicts: ds_read_b128 serves lanes 0-3, 12-15, 20-27 together, then 4-11, 16-19, 28-31, and the same of the
//   upper half.  The 16x16x32 operand (row lane % 16, chunk lane / 16) meets itself there under the tiles' swizzle; with
//   the four chunks of a step dealt to the lane groups in the order 0, 3, 1, 2 -- in the query rows as well, the sum over
//   them is the same -- it does not: 1430 of 3100 LDS cycles a unit were conflicts, 80 of 1710 are (2048 tokens x 128 heads 575 -> 525 us).
//
// What bounds the decode
//   64 sequences of 1024..8192 tokens, 128 heads: 13 us until the loop (plan, block table, query rows and the first units of
//   all workgroups at once), 44 units in 80 us, 6 us of parts stored.  1.83 us a unit are 4.9 TB/s and 1.25 PFLOP/s,
//   what the power limit leaves: 1.55 with a zero cache and query, 1.43 with its rows in the L2s as well.  So four waves
//   (mla_decode_split_kernel when it took such pages) come to nearly the same there, and cutting the list by units or counting
//   fewer positions for a segment gains nothing.  us, four waves / here, 128 heads: 64 x 1024..8192 tokens 116.9 / 116.3,
//   32 x 1024..8192 76.3 / 74.4, 64 x 512..4096 66.7 / 65.6; short sequences, whose start and end count, 64 x 200..1000 37.6 / 35.0,
//   64 x 100..200 30.1 / 27.1, 300 x 300..900 91.8 / 87.3; but 180 to 257 x 300..900, a sequence or two a workgroup, 75 / 76.6, and long
//   sequences in one piece (one split) 64 x 1024..8192 243 / 249.
//
// Softmax reference
//   Exponentials are taken against a fixed reference, the maximum of the row's first unit plus 40 in the log2 domain.  A row
//   whose scores outrun that by more than 80 (120 above its first 32 keys: next to never) has its item walked a second time,
//   against the maxima found.  That is what it costs: with such a row in every block of the later half 2048 tokens x 128 heads take
//   916 us instead of 549; four waves, which scaled their sums in place, took 609 either way.
#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "latent_stream.h"

#include <algorithm>
#include <cstdint>

namespace dscuda {
namespace {

constexpr int WIDE_WAVES = 8;
constexpr int WIDE_THREADS = 64 * WIDE_WAVES;
constexpr int WIDE_ROWS = index_math::DECODE_ROWS;
constexpr int ROW_TILES = WIDE_ROWS / 32;                    // 4
constexpr int WAVE_COLUMNS = RANK / WIDE_WAVES;              // 64 output columns of a wave
constexpr int WAVE_BLOCKS = WAVE_COLUMNS / 32;               // 2
constexpr int LATENT_BYTES = 2 * RANK;                       // of a latent row
constexpr int ROPE_BYTES = 2 * ROPE;
constexpr int LATENT_SLOT = UNIT * LATENT_BYTES;             // 32 KB
constexpr int ROPE_SLOT = UNIT * ROPE_BYTES;                 // 4 KB
constexpr int ROPE_SLOTS = UNIT_SLOTS - 1;
constexpr int ROPE_AT = UNIT_SLOTS * LATENT_SLOT;
constexpr int LATENT_STEPS = RANK / 32;                      // 16
constexpr int SCORE_STEPS = WIDTH / 32;                      // 18
constexpr int P_BYTES = UNIT * WIDE_ROWS * 2;                // 8 KB: [16 keys][32 rows][lane g][row][8 keys]
constexpr int P_HALF = P_BYTES / 2;
constexpr int P_AT = ROPE_AT + ROPE_SLOTS * ROPE_SLOT;
constexpr int SUMS_AT = P_AT + 2 * P_BYTES;                  // [128] reciprocal sums of the rows
constexpr int WIDE_LDS_BYTES = SUMS_AT + WIDE_ROWS * 4;
static_assert(WIDE_LDS_BYTES <= 160 * 1024, "all there is");
static_assert(LATENT_SLOT + ROPE_SLOT == UNIT_BYTES, "a unit");

// Fragments read ahead of the MFMA that takes them (1024 / 2048 tokens x 128 heads: three 159 / 537 us, two 161 / 551,
// four 160 / 542, six, which spill, 163 / 550).
constexpr int KEY_RING = 3;
// The 18 loads of the next query rows: 9 beside the last scores, 8 beside the last products, the last one behind them.
// All beside the last scores, the waves stood at a full request queue for 6500 cycles (1024 x 128 147 -> 139 us).
constexpr int QUERY_SCORES = 9;
constexpr int QUERY_PRODUCTS = 17;

constexpr float HEADROOM = 40.0f;
constexpr float OUTRUN = 80.0f;

typedef short wide_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) wide_s16x4* wide_tr_pointer;

using LatentReads = index_math::TileReadMath<LATENT_BYTES>;
using RopeReads = index_math::TileReadMath<ROPE_BYTES>;

// The order of the k-steps: of a row's 256-byte groups, the two lines of 128 bytes one after the other (steps of one line
// are neighbours for the query loads; at most two chunk positions are live in the key reads).
__device__ constexpr int step_of(int place) {
    return place < LATENT_STEPS ? 4 * (place % 8 / 2) + 2 * (place / 8) + place % 2 : place;
}

// Chunk of a k-step that lane group q = lane / 16 of a 16x16x32 operand holds (see above).
__device__ __forceinline__ int chunk_of_group(int q) {
    return (q >> 1) ^ (3 * (q & 1));   // 0, 3, 1, 2
}

// The value of lane l ^ 16, by a swizzle whose pattern is a constant (0x401f: exclusive or with 16 within 32 lanes): __shfl_xor
// computes with the lane's number, which the decode then kept in scratch.
__device__ __forceinline__ float of_lane_xor_16(float value) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, value), 0x401f));
}

// over the lanes l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ float wide_quarter_max(float value) {
    return half_wave_max(fmaxf(value, of_lane_xor_16(value)));
}

__device__ __forceinline__ float wide_quarter_sum(float value) {
    return half_wave_sum(value + of_lane_xor_16(value));
}

// ---- what a workgroup walks ---------------------------------------------------------------------------------------
//
// A Work is a kernel's argument.  It names the items of a workgroup, one after the other (Iterator), the rows of an item, and where the keys of its
// units lie (Keys: first row of the unit at hand and the last row that holds a visible token, which those behind it
// repeat).  An item has at least two units; one past its keys is masked as a whole.

// A kernel's argument, read anew from the constant memory at every use: held in scalar registers from the kernel's start to
// its end, its fields pushed what the loops use out into lanes of vector registers, and those into scratch.
template <typename Work>
struct Argument {
    const __attribute__((address_space(4))) Work* place;

    __device__ __forceinline__ Argument() {
        place = (const __attribute__((address_space(4))) Work*)__builtin_amdgcn_kernarg_segment_ptr();   // the first argument
    }
    __device__ __forceinline__ const Work& operator*() const {
        const __attribute__((address_space(4))) Work* fresh = place;
        asm volatile("" : "+s"(fresh));
        return *(const Work*)fresh;
    }
    __device__ __forceinline__ const Work* operator->() const { return &**this; }
};

// Prefill: 128 consecutive (token, head) pairs of a batch element.
struct ForwardWork {
    static constexpr int LATENT_STRIDE = 2 * RANK;   // bytes, of keys and query rows
    static constexpr int ROPE_STRIDE = 2 * ROPE;
    static constexpr bool STREAMING = false;         // keys are read by many workgroups

    bf16_t* output;
    float* logsumexp;
    const bf16_t* query_latent;
    const bf16_t* query_rope;
    const bf16_t* kv_latent;
    const bf16_t* key_rope;
    int sequence_length;
    int heads;
    unsigned rows;                       // (token, head) pairs of a batch element
    unsigned items;
    unsigned row_blocks;
    bool interleaved;                    // the batch elements' blocks are numbered together
    index_math::FastDivision by_heads;
    index_math::FastDivision by_order;   // batch elements (interleaved), row blocks of one
    float c;

    struct Place {};                     // what a workgroup knows of itself

    struct Item {
        int batch;
        unsigned row0;
        int tokens;                      // keys that any of its rows sees
        int unit_begin;
        int units;
    };

    // The heaviest blocks first, rounds there and back (index_math::forward_interleaves).
    struct Iterator {
        int round;

        __device__ __forceinline__ bool next(const ForwardWork& work, const Place&, Item& item) {
            const unsigned index = index_math::forward_index((unsigned)round, blockIdx.x, gridDim.x);
            ++round;
            if (index >= work.items) return false;
            unsigned batch, row_block;
            index_math::forward_item(index, work.interleaved, work.by_order, work.row_blocks, batch, row_block);
            item.batch = (int)batch;
            item.row0 = row_block * WIDE_ROWS;
            const unsigned last_row = min(work.rows, item.row0 + WIDE_ROWS) - 1;
            item.tokens = (int)index_math::divide(last_row, work.by_heads) + 1;
            item.unit_begin = 0;
            item.units = max((item.tokens + UNIT - 1) / UNIT, 2);
            return true;
        }
    };

    struct Keys {
        const unsigned char* latent;
        const unsigned char* rope_rows;
        int limit;

        __device__ __forceinline__ const unsigned char* rope() const { return rope_rows; }
        __device__ __forceinline__ void open(const ForwardWork& work, const Item& item) {
            const size_t first = (size_t)item.batch * work.sequence_length;
            latent = reinterpret_cast<const unsigned char*>(work.kv_latent + first * RANK);
            rope_rows = reinterpret_cast<const unsigned char*>(work.key_rope + first * ROPE);
            limit = item.tokens - 1;
        }
        __device__ __forceinline__ int look_up() const { return 0; }
        __device__ __forceinline__ void next(const ForwardWork&, int) {
            const int rows = min(limit, UNIT);   // fewer: no visible token behind them, the last row stands for the unit
            latent += rows * LATENT_STRIDE;
            rope_rows += rows * ROPE_STRIDE;
            limit -= rows;
        }
    };

    __device__ __forceinline__ unsigned valid_rows(const Place&, const Item& item) const {
        return min(rows - item.row0, (unsigned)WIDE_ROWS);
    }
    __device__ __forceinline__ size_t query_row(const Place&, const Item& item, unsigned row) const {
        return (size_t)item.batch * rows + item.row0 + row;
    }
    __device__ __forceinline__ const bf16_t* latent_row(const Place& place, const Item& item, unsigned row) const {
        return query_latent + query_row(place, item, row) * RANK;
    }
    __device__ __forceinline__ const bf16_t* rope_row(const Place& place, const Item& item, unsigned row) const {
        return query_rope + query_row(place, item, row) * ROPE;
    }
    __device__ __forceinline__ void store_logsumexp(const Place&, const Item& item, unsigned row, float value) const {
        const unsigned token = index_math::divide(item.row0 + row, by_heads);
        const unsigned head = item.row0 + row - token * heads;
        logsumexp[((size_t)item.batch * heads + head) * sequence_length + token] = value;
    }
    // keys that a row of the item sees
    __device__ __forceinline__ int visible(const Item& item, unsigned row) const {
        return (int)index_math::divide(item.row0 + row, by_heads) + 1;
    }
    __device__ __forceinline__ static constexpr bool is_part(const Item&) { return false; }
    __device__ __forceinline__ float* part_statistics(const Place&, const Item&) const { return nullptr; }
    __device__ __forceinline__ unsigned char* part_rows(const Place&, const Item&) const { return nullptr; }
};

// What is the same for all lanes, by the scalar unit: its wait is that of the LDS reads, not of the requests on their way.
__device__ __forceinline__ int scalar_load(const int* place) {
    return *(const __attribute__((address_space(4))) int*)place;
}

// The lengths' plan that a workgroup works out for itself (latent_stream.h) lies behind the LDS of the walk.
constexpr int OWN_PREFIX_AT = WIDE_LDS_BYTES;
constexpr int OWN_LENGTHS_AT = OWN_PREFIX_AT + 4 * (SELF_PLAN_BATCH + 4);
constexpr int OWN_TOTALS_AT = OWN_LENGTHS_AT + 4 * SELF_PLAN_BATCH;
constexpr int OWN_RANGE_AT = OWN_TOTALS_AT + 4 * (2 * SELF_PLAN_BATCH / 64);   // end of the range, overhead of a sequence
constexpr int DECODE_LDS_BYTES = OWN_RANGE_AT + 8;
static_assert(DECODE_LDS_BYTES <= 160 * 1024, "all there is");

__device__ __forceinline__ int own_value(int at, int index) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    return __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(lds + at + 4 * index));
}

// Decode: 128 heads of a sequence, the tiles of it that a range of the work list holds.  Pages hold whole units.
struct DecodeWork {
    static constexpr int LATENT_STRIDE = 2 * WIDTH;
    static constexpr int ROPE_STRIDE = 2 * WIDTH;
    static constexpr bool STREAMING = true;          // each head group reads the cache once

    bf16_t* output;
    float* logsumexp;
    const bf16_t* query;
    const bf16_t* cache;
    const int* block_table;
    const int* cache_lengths;
    float* workspace;
    int* plan;
    int batch_size;
    int heads;
    int page_size;
    int pages_per_sequence;
    long long slot_floats;
    int padded_rows;
    bool own_plan;
    DecodeCut cut;
    float c;

    struct Place {};                     // its range lies in the LDS: scalar registers are scarce

    struct Item {
        int sequence;
        int tokens;
        int unit_begin;
        int units;
        bool part;                       // of its sequence
    };

    struct Iterator {
        int position;
        int sequence;

        __device__ __forceinline__ bool next(const DecodeWork& work, const Place&, Item& item) {
            const int end = own_value(OWN_RANGE_AT, 0);
            while (position < end) {
                const int overhead = own_value(OWN_RANGE_AT, 1);
                const int at = sequence++;
                int before, after, tokens;
                if (work.batch_size <= 64 || work.own_plan) {
                    before = own_value(OWN_PREFIX_AT, at);
                    after = own_value(OWN_PREFIX_AT, at + 1);
                    tokens = own_value(OWN_LENGTHS_AT, at);
                } else {
                    const int* prefix = work.plan + index_math::plan_prefix_at() + at;
                    before = scalar_load(prefix);
                    after = scalar_load(prefix + 1);
                    tokens = scalar_load(work.cache_lengths + at);
                }
                const int segment_end = min(end, after);
                if (segment_end <= position) continue;   // a sequence without tiles
                int tile_begin, tile_end;
                index_math::tiles_in_positions(position, segment_end, before, overhead, tile_begin, tile_end);
                position = segment_end;
                item.sequence = at;
                item.tokens = tokens;
                item.unit_begin = (BN / UNIT) * tile_begin;
                item.units = min((BN / UNIT) * tile_end, (tokens + UNIT - 1) / UNIT) - item.unit_begin;
                item.part = tile_begin != 0 || tile_end != after - before - overhead;
                if (item.units <= 0) continue;           // nothing but positions that stand for the sequence's overhead
                item.units = max(item.units, 2);
                return true;
            }
            return false;
        }
    };

    struct Keys {
        const unsigned char* latent;
        const int* entry;                // of the block table, of the page behind the unit's
        int limit;
        int left;                        // units of the page from this one on

        __device__ __forceinline__ const unsigned char* rope() const { return latent + 2 * RANK; }
        __device__ __forceinline__ void open(const DecodeWork& work, const Item& item) {
            const int key0 = item.unit_begin * UNIT;
            const int page = __builtin_amdgcn_readfirstlane((unsigned)key0 / (unsigned)work.page_size);
            const int inside = key0 - page * work.page_size;
            entry = work.block_table + (size_t)item.sequence * work.pages_per_sequence + page;
            const long long id = scalar_load(entry);
            latent = reinterpret_cast<const unsigned char*>(work.cache + (id * work.page_size + inside) * WIDTH);
            ++entry;
            left = (work.page_size - inside) / UNIT;
            limit = item.tokens - 1 - key0;
        }
        // The next unit's page, if that is another one: asked for ahead of the products, used behind them.  No entry past
        // the last page with a visible token is read.
        __device__ __forceinline__ int look_up() const { return left == 1 && limit >= UNIT ? scalar_load(entry) : 0; }
        __device__ __forceinline__ void next(const DecodeWork& work, int ahead) {
            if (limit < UNIT) {          // no visible token behind them, the last row stands for the unit
                latent += limit * LATENT_STRIDE;
                limit = 0;
                return;
            }
            limit -= UNIT;
            latent += UNIT * LATENT_STRIDE;
            if (--left == 0) {
                latent = reinterpret_cast<const unsigned char*>(work.cache + (long long)ahead * work.page_size * WIDTH);
                left = work.page_size / UNIT;
                ++entry;
            }
        }
    };

    // Workgroups go to the eight XCDs round-robin by linear id.  Neighbouring ranges are mostly parts of the same
    // sequence and fetch the same query rows, so each XCD takes a run of consecutive ranges.
    __device__ __forceinline__ static int workgroup() {
        return gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    }
    __device__ __forceinline__ static unsigned head0() { return blockIdx.y * WIDE_ROWS; }
    __device__ __forceinline__ unsigned valid_rows(const Place&, const Item&) const {
        return min((unsigned)heads - head0(), (unsigned)WIDE_ROWS);
    }
    __device__ __forceinline__ size_t query_row(const Place&, const Item& item, unsigned row) const {
        return (size_t)item.sequence * heads + head0() + row;
    }
    __device__ __forceinline__ const bf16_t* latent_row(const Place& place, const Item& item, unsigned row) const {
        return query + query_row(place, item, row) * WIDTH;
    }
    __device__ __forceinline__ const bf16_t* rope_row(const Place& place, const Item& item, unsigned row) const {
        return query + query_row(place, item, row) * WIDTH + RANK;
    }
    __device__ __forceinline__ void store_logsumexp(const Place& place, const Item& item, unsigned row, float value) const {
        logsumexp[query_row(place, item, row)] = value;
    }
    __device__ __forceinline__ int visible(const Item& item, unsigned) const { return item.tokens; }
    __device__ __forceinline__ static bool is_part(const Item& item) { return item.part; }
    // A part's slot: 32 KB for every 32 rows, in the order of the accumulators' registers, then (reference, sum) of a head.
    __device__ __forceinline__ float* slot(const Place& place, const Item& item) const {
        return workspace + ((long long)workgroup() + item.sequence) * slot_floats;
    }
    __device__ __forceinline__ float* part_statistics(const Place& place, const Item& item) const {
        return slot(place, item) + (size_t)padded_rows * (RANK / 2) + 2 * head0();
    }
    __device__ __forceinline__ unsigned char* part_rows(const Place& place, const Item& item) const {
        return reinterpret_cast<unsigned char*>(slot(place, item)) + (size_t)head0() * (2 * RANK);
    }
};

// The unit requested next; runs ahead of the products, over the ends of items.
template <typename Work>
struct WideCursor {
    typename Work::Iterator items;
    typename Work::Keys keys;
    int left;   // units of the item from this one on; 0: no more items

    __device__ __forceinline__ bool enabled() const { return left > 0; }
    __device__ __forceinline__ void open(const Argument<Work>& work, const typename Work::Item& item) {
        left = __builtin_amdgcn_readfirstlane(item.units);
        keys.open(*work, item);
    }
    // (ahead: what keys.look_up returned)
    __device__ __forceinline__ void advance(const Argument<Work>& work, const typename Work::Place& place, int ahead) {
        if (left == 0) return;
        if (--left > 0) {
            keys.next(*work, ahead);
            return;
        }
        typename Work::Item item;
        if (items.next(*work, place, item)) open(work, item);
    }
};

// A workgroup's stream: the item at hand and those that `items` names after it.  LATE: waves 4..7, scores before products.
template <typename Work, bool LATE>
__device__ __forceinline__ void wide_stream(const typename Work::Place place, typename Work::Item item,
                                            typename Work::Iterator items, unsigned char* lds, const int wave) {
    using Item = typename Work::Item;
    constexpr int REQUESTS = LATE ? 4 : 5;    // of a wave and unit
    const unsigned lds0 = lds_offset_of(lds);
    const Argument<Work> work;
    const float c = work->c;

    WideCursor<Work> cursor;
    // request I (0..3 a latent row, 4 eight rope rows, of the early waves) of the cursor's unit, the stream's unit n
    auto issue = [&](int n, auto tag) {
        constexpr int I = decltype(tag)::value;
        if (!cursor.enabled()) return;
        auto load = [&](const unsigned char* base, unsigned offset, unsigned target) {
            if constexpr (Work::STREAMING) direct_load_16_offset_streaming(base, offset, target);
            else direct_load_16_offset(base, offset, target);
        };
        const int lane = fresh_lane_id();
        if constexpr (I < 4) {
            const int line = 4 * wave + I;
            const unsigned target = lds0 + ((unsigned)n % UNIT_SLOTS) * LATENT_SLOT + line * LATENT_BYTES;
            const unsigned chunk = 16 * (lane ^ (wave & 3)) ^ (64u * I);   // 16 * (lane ^ tile_swizzle(line))
            load(cursor.keys.latent + min(line, cursor.keys.limit) * Work::LATENT_STRIDE, chunk, target);
        } else if constexpr (!LATE) {
            const int line = 8 * wave + lane / 8;
            const unsigned chunk = 16 * ((lane % 8) ^ index_math::tile_swizzle<ROPE_BYTES>(line));
            const unsigned target = lds0 + ROPE_AT + ((unsigned)n % ROPE_SLOTS) * ROPE_SLOT + wave * 1024;
            load(cursor.keys.rope(), min(line, cursor.keys.limit) * Work::ROPE_STRIDE + chunk, target);
        }
    };
    auto issue_all = [&](int n) {
        const int ahead = cursor.keys.look_up();
        unrolled<0, 5>([&](auto tag) { issue(n, tag); });
        cursor.advance(work, place, ahead);
    };

    f32x16 out[ROW_TILES][WAVE_BLOCKS];   // 32 rows x 32 columns each
    bf16x8 qf[SCORE_STEPS];
    // of the lane's row 16 * wave + lane % 16
    float reference, row_sum, highest;
    const bf16_t* next_latent = nullptr;   // the lane's part of the query row that is loaded next
    const bf16_t* next_rope = nullptr;
    // (needed: there is a next item; otherwise the loads, which stay in the code, fetch a line each for all lanes)
    auto find_query = [&](const Item& of, bool needed) {
        const int lane = fresh_lane_id();
        const int first = needed ? 8 * chunk_of_group(lane / 16) : 0;
        // rows past the end repeat the last one, nothing of theirs is stored
        const unsigned row = needed ? min((unsigned)(16 * wave + lane % 16), work->valid_rows(place, of) - 1) : 0;
        next_latent = work->latent_row(place, of, row) + first;
        next_rope = work->rope_row(place, of, row) + first;
    };
    auto load_query = [&](auto place) {
        constexpr int S = step_of(decltype(place)::value);
        qf[S] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                               S < LATENT_STEPS ? next_latent + 32 * S : next_rope + 32 * (S - LATENT_STEPS)));
    };

    // Offsets of the fragment reads in the slot at hand; the other chunks of a 256-byte group are one XOR away.
    unsigned key_at, rope_at, value_at[2];
    {
        const int lane = fresh_lane_id();
        const int operand = 16 * chunk_of_group(lane / 16) + lane % 16;
        key_at = LatentReads::quadrant(0, operand);
        rope_at = ROPE_AT + RopeReads::quadrant(0, operand);
        // lanes 32..63 take the two key groups of their four rows in the other order, as P has them
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            value_at[h] = LatentReads::transposed(h ^ (lane / 32), 2 * (wave & 1), lane) + (wave >> 1) * 256;
        }
    }
    auto latent_step = [&](int n) {   // from a unit's slot to the next one's
        return (unsigned)n % UNIT_SLOTS == UNIT_SLOTS - 1 ? 0u - (UNIT_SLOTS - 1) * LATENT_SLOT : (unsigned)LATENT_SLOT;
    };
    auto rope_step = [&](int n) {
        return (unsigned)n % ROPE_SLOTS == ROPE_SLOTS - 1 ? 0u - (ROPE_SLOTS - 1) * ROPE_SLOT : (unsigned)ROPE_SLOT;
    };

    int all_visible = 0;   // keys that all rows of the item see
    f32x4 scores[2];
    // Scores of the stream's unit n, unit `unit` of its item.  LAST: of its item; the query rows of the next one are asked
    // for as those of this one have been used.
    auto form_scores = [&](const Item& of, int n, int unit, auto last) {
        // fragment F: key half F % 2 of the k-step in place F / 2
        auto fragment = [&](auto tag) -> bf16x8 {
            constexpr int F = decltype(tag)::value;
            constexpr int S = step_of(F / 2);
            if constexpr (S < LATENT_STEPS) {
                return *reinterpret_cast<const bf16x8*>(lds + (key_at ^ (64 * (S % 4))) + (S / 4) * 256 + (F % 2) * 16 * LATENT_BYTES);
            } else {
                return *reinterpret_cast<const bf16x8*>(lds + (rope_at ^ (64 * (S % 2))) + (F % 2) * 16 * ROPE_BYTES);
            }
        };
        constexpr int COUNT = 2 * SCORE_STEPS;
        bf16x8 ring[KEY_RING];
        unrolled<0, KEY_RING>([&](auto tag) { ring[decltype(tag)::value] = fragment(tag); });
        scores[0] = scores[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        // The chain of scores is what a step waits for: its MFMAs go first (531 against 550 us, 2048 tokens x 128 heads).
        __builtin_amdgcn_s_setprio(1);
        unrolled<0, COUNT>([&](auto tag) {
            constexpr int F = decltype(tag)::value;
            scores[F % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[F % KEY_RING], qf[step_of(F / 2)], scores[F % 2], 0, 0, 0);
            if constexpr (F + KEY_RING < COUNT) ring[F % KEY_RING] = fragment(std::integral_constant<int, F + KEY_RING>{});
            if constexpr (decltype(last)::value && F % 2 == 1 && F / 2 < QUERY_SCORES) load_query(std::integral_constant<int, F / 2>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        __builtin_amdgcn_s_setprio(0);
        key_at += latent_step(n);
        rope_at += rope_step(n);
        const int first = (of.unit_begin + unit) * UNIT;
        if (first + UNIT > all_visible) {
            const int lane = fresh_lane_id();
            const unsigned row = min((unsigned)(16 * wave + lane % 16), work->valid_rows(place, of) - 1);
            const int hidden = work->visible(of, row) - first - 4 * (lane / 16);   // the lane's keys 16 * k + i from there on
#pragma unroll
            for (int k = 0; k < 2; ++k) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (16 * k + i >= hidden) scores[k][i] = -INFINITY;
                }
            }
        }
    };
    auto lane_max = [&]() {
        float value = fmaxf(scores[0][0], scores[1][0]);
#pragma unroll
        for (int i = 1; i < 4; ++i) value = fmaxf(value, fmaxf(scores[0][i], scores[1][i]));
        return value;
    };
    auto write_probabilities = [&](int n) {
        // Keys 4q .. 4q + 3 of a half: the 8 bytes q / 2 of lane group g = q % 2 of the product's operand, the other way
        // round for g = 1, so that the two groups write to different banks.
        const int lane = fresh_lane_id();
        const unsigned to = P_AT + (n & 1) * P_BYTES + (wave / 2) * 1024 + (wave & 1) * 256 + (lane & 15) * 16 +
                            ((lane >> 4) & 1) * 512 + (((lane >> 5) ^ (lane >> 4)) & 1) * 8;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[i] = __builtin_amdgcn_exp2f(fmaf(scores[k][i], c, -reference));
                row_sum += p[i];
            }
            const u32x2 packed = {pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
            *reinterpret_cast<u32x2*>(lds + to + k * P_HALF) = packed;
        }
    };
    auto score_phase = [&](const Item& of, int n, int unit, auto last) {
        form_scores(of, n, unit, last);
        highest = fmaxf(highest, lane_max());
        write_probabilities(n);
    };
    // Products of the stream's unit n, and the requests of unit n + 3 into the slot that unit n - 1 has left.
    auto output_phase = [&](int n, auto last) {
        const int ahead = cursor.keys.look_up();
        const unsigned p_at = P_AT + 16 * fresh_lane_id() + (n & 1) * P_BYTES;
        auto value_fragment = [&](auto half, auto d) -> bf16x8 {
            constexpr int AT = decltype(half)::value * 16 * LATENT_BYTES;
            constexpr int D = decltype(d)::value;
            const wide_s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((wide_tr_pointer)(lds + (value_at[0] ^ (64 * D)) + AT));
            const wide_s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((wide_tr_pointer)(lds + (value_at[1] ^ (64 * D)) + AT));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        auto p_fragment = [&](int half, int b) -> bf16x8 {
            return *reinterpret_cast<const bf16x8*>(lds + p_at + half * P_HALF + b * 1024);
        };
        using Zero = std::integral_constant<int, 0>;
        using One = std::integral_constant<int, 1>;
        bf16x8 vf[WAVE_BLOCKS], pf[ROW_TILES];
        vf[0] = value_fragment(Zero{}, Zero{});
#pragma unroll
        for (int b = 0; b < ROW_TILES; ++b) pf[b] = p_fragment(0, b);
        vf[1] = value_fragment(Zero{}, One{});
        unrolled<0, 16>([&](auto tag) {
            constexpr int M = decltype(tag)::value;
            constexpr int HALF = M / 8, D = (M / 4) % 2, B = M % 4;
            out[B][D] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[D], pf[B], out[B][D], 0, 0, 0);
            if constexpr (HALF == 0 && D == 1) pf[B] = p_fragment(1, B);
            if constexpr (M == 3) vf[0] = value_fragment(One{}, Zero{});
            if constexpr (M == 7) vf[1] = value_fragment(One{}, One{});
            if constexpr (M % 3 == 1 && M / 3 < 5) issue(n + 3, std::integral_constant<int, M / 3>{});
            if constexpr (decltype(last)::value && M % 2 == 1 && QUERY_SCORES + M / 2 < QUERY_PRODUCTS) {
                load_query(std::integral_constant<int, QUERY_SCORES + M / 2>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        value_at[0] += latent_step(n);
        value_at[1] += latent_step(n);
        cursor.advance(work, place, ahead);
    };

    int n = 0;              // unit of the stream
    bool restart = true;    // the stream starts (again) with the item at hand
    bool again = false;     // the item is walked a second time, against the maxima of its rows
    // Scores of an item's first unit, and the reference every exponential of its walk is taken against.
    auto first_scores = [&](const Item& of, int at) {
        all_visible = work->visible(of, 0);
        form_scores(of, at, 0, std::false_type{});
        reference = again ? wide_quarter_max(highest) * c : wide_quarter_max(lane_max()) * c + HEADROOM;
        highest = lane_max();
        row_sum = 0.f;
        write_probabilities(at);
    };
    while (true) {
        if (restart) {
            // At the start of the kernel every workgroup asks at once and the answers come at the rate of the memory: what
            // the first scores need is asked for first.
            cursor.items = items;
            cursor.open(work, item);
            find_query(item, true);
            unrolled<0, SCORE_STEPS>(load_query);
            issue_all(n);
            wait_vector_memory<0>();
            workgroup_barrier();
            issue_all(n + 1);
            const bool third = cursor.enabled();
            issue_all(n + 2);
            first_scores(item, n);
            if (third) wait_vector_memory<REQUESTS>(); else wait_vector_memory<0>();   // unit n + 1 has landed
            restart = false;
        }
        workgroup_barrier();   // the first probabilities are there
#pragma unroll
        for (int b = 0; b < ROW_TILES; ++b) {
#pragma unroll
            for (int d = 0; d < WAVE_BLOCKS; ++d) {
#pragma unroll
                for (int i = 0; i < 16; ++i) out[b][d][i] = 0.f;
            }
        }
        const int units = __builtin_amdgcn_readfirstlane(item.units);
        int unit = 0;
        for (; unit + 2 < units; ++unit, ++n) {
            const bool requested = cursor.enabled();
            if (LATE) score_phase(item, n + 1, unit + 1, std::false_type{});
            output_phase(n, std::false_type{});
            if (!LATE) score_phase(item, n + 1, unit + 1, std::false_type{});
            // unit n + 2 has landed; only this wave's share of unit n + 3 may still be on its way
            if (requested) wait_vector_memory<REQUESTS>(); else wait_vector_memory<0>();
            workgroup_barrier();
        }
        bool more;
        {
            typename Work::Iterator ahead = items;   // which stays: a second walk starts the stream from there
            Item next = item;
            more = ahead.next(*work, place, next);
            find_query(next, more);
        }
        {
            const bool requested = cursor.enabled();
            if (LATE) score_phase(item, n + 1, unit + 1, std::true_type{});
            output_phase(n, std::false_type{});
            if (!LATE) score_phase(item, n + 1, unit + 1, std::true_type{});
            if (requested) wait_vector_memory<REQUESTS + QUERY_SCORES>(); else wait_vector_memory<0>();
            workgroup_barrier();
            ++n;
        }
        float* inverses = reinterpret_cast<float*>(lds + SUMS_AT);
        const float total = wide_quarter_sum(row_sum);
        {
            // (not twice: of scores beyond 2^24 the maximum itself is that far from its rounded product with c)
            const bool outrun = !again && fmaf(wide_quarter_max(highest), c, -reference) > OUTRUN;
            const int lane = fresh_lane_id();
            if (lane < 16) inverses[16 * wave + lane] = outrun ? -1.0f : 1.0f / total;
            const bool requested = cursor.enabled();
            output_phase(n, std::true_type{});
            // behind unit n + 2's requests: query rows (early waves: of both phases), the requests of unit n + 3
            if (!requested) wait_vector_memory<0>();
            else if (LATE) wait_vector_memory<REQUESTS + QUERY_PRODUCTS - QUERY_SCORES>();
            else wait_vector_memory<REQUESTS + QUERY_PRODUCTS>();
            workgroup_barrier();
        }
        unrolled<QUERY_PRODUCTS, SCORE_STEPS>(load_query);
        const int lane = fresh_lane_id();
        const int lq = lane % 32;
        float inverse[ROW_TILES];
#pragma unroll
        for (int b = 0; b < ROW_TILES; ++b) inverse[b] = inverses[32 * b + lq];
        const float least = fminf(fminf(inverse[0], inverse[1]), fminf(inverse[2], inverse[3]));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(least < 0.f) != 0, 0)) {
            wait_vector_memory<0>();
            workgroup_barrier();   // what was on its way has arrived, everybody has read the verdict
            again = restart = true;
            ++n;
            continue;
        }
        again = false;
        const unsigned valid = work->valid_rows(place, item);
        const unsigned own_row = 16 * wave + lane;   // of lanes 0..15
        if (work->is_part(item)) {
            if (lane < 16 && own_row < valid) {
                float* statistics = work->part_statistics(place, item) + 2 * own_row;
                statistics[0] = reference;
                statistics[1] = total;
            }
            // 16-byte piece j of a lane: registers 8 * (j % 2) .. + 7 of column block j / 2
            unsigned char* pieces = work->part_rows(place, item) + wave * (2 * WAVE_BLOCKS * 1024) + 16 * lane;
#pragma unroll
            for (int b = 0; b < ROW_TILES; ++b) {
                if (32u * b >= valid) break;
#pragma unroll
                for (int j = 0; j < 2 * WAVE_BLOCKS; ++j) {
                    u32x4 packed;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        packed[k] = pack_bf16(out[b][j / 2][8 * (j % 2) + 2 * k], out[b][j / 2][8 * (j % 2) + 2 * k + 1]);
                    }
                    *reinterpret_cast<u32x4*>(pieces + b * (32 * 2 * RANK) + j * 1024) = packed;
                }
            }
        } else {
        if (lane < 16 && own_row < valid) work->store_logsumexp(place, item, own_row, (reference + __builtin_amdgcn_logf(total)) * LN2);
        // The rows leave through the slot of the last unit, a tile of 32 rows x the wave's 128 bytes at a time, eight whole
        // lines an instruction.  (With the hint for streams the kernel by itself is 10 us shorter at 1024 tokens x 128 heads,
        // but the un-absorb that reads the rows 20 longer: the layer 245 against 234 us.)
        unsigned char* staged = lds + ((unsigned)n % UNIT_SLOTS) * LATENT_SLOT + wave * (32 * 2 * WAVE_COLUMNS);
        bf16_t* rows = work->output + work->query_row(place, item, 0) * RANK + wave * WAVE_COLUMNS;
        const int to = lq * 128 + 8 * (lane / 32), flip = (lq >> 1) & 7;
        const int line8 = lane / 8, piece = lane % 8;
#pragma unroll
        for (int b = 0; b < ROW_TILES; ++b) {
#pragma unroll
            for (int d = 0; d < WAVE_BLOCKS; ++d) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    u32x2 packed;
                    packed.x = pack_bf16(out[b][d][4 * i4 + 0] * inverse[b], out[b][d][4 * i4 + 1] * inverse[b]);
                    packed.y = pack_bf16(out[b][d][4 * i4 + 2] * inverse[b], out[b][d][4 * i4 + 3] * inverse[b]);
                    *reinterpret_cast<u32x2*>(staged + to + 16 * ((4 * d + i4) ^ flip)) = packed;
                }
            }
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's LDS writes have landed
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int line = 8 * j + line8;
                if ((unsigned)(32 * b + line) < valid) {
                    const u32x4 bits = *reinterpret_cast<const u32x4*>(staged + line * 128 + 16 * (piece ^ ((line >> 1) & 7)));
                    *reinterpret_cast<u32x4*>(rows + (size_t)(32 * b + line) * RANK + 8 * piece) = bits;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        }
        if (!more) break;
        ++n;
        items.next(*work, place, item);
        first_scores(item, n);
    }
}

__global__ __launch_bounds__(WIDE_THREADS) void mla_wide_forward_kernel(ForwardWork) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const Argument<ForwardWork> work;
    ForwardWork::Item item;
    ForwardWork::Iterator items = {0};
    if (!items.next(*work, {}, item)) return;
    if (wave >= 4) {
        wide_stream<ForwardWork, true>({}, item, items, lds, wave);
    } else {
        wide_stream<ForwardWork, false>({}, item, items, lds, wave);
    }
}

// A workgroup's range of the work list (index_math.h).  Its parts of sequences go to slot workgroup + sequence of the workspace.
__global__ __launch_bounds__(WIDE_THREADS) void mla_wide_decode_kernel(DecodeWork) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const Argument<DecodeWork> work;
    DecodeCut cut = work->cut;
    cut.reference_ranges = 0;   // decode_layout has none; the vote over them would take LDS in front of the slots
    const DecodeRange range = decode_range(
        work->plan, work->cache_lengths, work->batch_size, work->own_plan, false, cut,
        reinterpret_cast<int*>(lds + OWN_PREFIX_AT), reinterpret_cast<int*>(lds + OWN_LENGTHS_AT),
        reinterpret_cast<int*>(lds + OWN_TOTALS_AT), threadIdx.x, WIDE_THREADS, DecodeWork::workgroup(), blockIdx.x == 0 && blockIdx.y == 0);
    if (range.begin >= range.end) return;
    int* own_range = reinterpret_cast<int*>(lds + OWN_RANGE_AT);
    own_range[0] = range.end;     // the same from every wave, which reads what it wrote
    own_range[1] = range.overhead;
    DecodeWork::Iterator items = {__builtin_amdgcn_readfirstlane(range.begin), __builtin_amdgcn_readfirstlane(range.sequence)};
    DecodeWork::Item item;
    if (!items.next(*work, {}, item)) return;
    if (wave >= 4) {
        wide_stream<DecodeWork, true>({}, item, items, lds, wave);
    } else {
        wide_stream<DecodeWork, false>({}, item, items, lds, wave);
    }
}

template <typename Kernel>
void allow_wide_lds(Kernel kernel, int bytes) {
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
}

}  // namespace

void mla_wide_forward_launch(bf16_t* output, float* logsumexp, const bf16_t* query_latent, const bf16_t* query_rope,
                             const bf16_t* kv_latent, const bf16_t* key_rope, int batch_size, int sequence_length,
                             int heads, float scale, hipStream_t stream) {
    static hip_common::OncePerDevice prepared;
    prepared.run([] { allow_wide_lds(mla_wide_forward_kernel, WIDE_LDS_BYTES); });
    ForwardWork work;
    work.output = output;
    work.logsumexp = logsumexp;
    work.query_latent = query_latent;
    work.query_rope = query_rope;
    work.kv_latent = kv_latent;
    work.key_rope = key_rope;
    work.sequence_length = sequence_length;
    work.heads = heads;
    work.rows = (unsigned)((long long)sequence_length * heads);
    work.row_blocks = (work.rows + WIDE_ROWS - 1) / WIDE_ROWS;
    work.items = work.row_blocks * batch_size;
    const unsigned workgroups = std::min(work.items, (unsigned)std::max(hip_common::compute_units_of_current_device(), 1));
    work.interleaved = index_math::forward_interleaves(sequence_length, batch_size, work.row_blocks, workgroups);
    work.by_heads = index_math::fast_division((unsigned)heads);
    work.by_order = index_math::fast_division(work.interleaved ? (unsigned)batch_size : work.row_blocks);
    work.c = scale * LOG2E;
    hipLaunchKernelGGL(mla_wide_forward_kernel, dim3(workgroups), dim3(WIDE_THREADS), WIDE_LDS_BYTES, stream, work);
    HIP_CHECK(hipGetLastError());
}

void mla_wide_decode_launch(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* paged_kv_cache,
                            const int* block_table, const int* cache_lengths, float* workspace, int* plan, int batch_size,
                            int heads, int page_size, int pages_per_sequence, const index_math::DecodeLayout& layout,
                            bool own_plan, float scale, hipStream_t stream) {
    static hip_common::OncePerDevice prepared;
    prepared.run([] { allow_wide_lds(mla_wide_decode_kernel, DECODE_LDS_BYTES); });
    DecodeWork work;
    work.output = output;
    work.logsumexp = logsumexp;
    work.query = query;
    work.cache = paged_kv_cache;
    work.block_table = block_table;
    work.cache_lengths = cache_lengths;
    work.workspace = workspace;
    work.plan = plan;
    work.batch_size = batch_size;
    work.heads = heads;
    work.page_size = page_size;
    work.pages_per_sequence = pages_per_sequence;
    work.slot_floats = layout.slot_floats;
    work.padded_rows = (heads + 31) / 32 * 32;
    work.own_plan = own_plan;
    work.cut = DecodeCut{layout.workgroups, layout.whole_sequences, layout.reference_ranges, layout.wide_ranges};
    work.c = scale * LOG2E;
    hipLaunchKernelGGL(mla_wide_decode_kernel, dim3(layout.workgroups, layout.head_groups), dim3(WIDE_THREADS),
                       DECODE_LDS_BYTES, stream, work);
    HIP_CHECK(hipGetLastError());
}

}  // namespace dscuda
