// Absorbed MLA backward of short sequences (at most 512 tokens) with few rows: the gradients of
// mla_absorbed.hip, from probabilities and dS that are formed once and kept.
//
// There the key gradients are cut into parts whose fp32 sums lie in the query-gradient buffers
// until the last launch, 72 KB each: 512 tokens of 8 heads have room for 40 parts, 300 tokens of
// 4 heads for none, on 256 compute units.  The same buffers hold something smaller that needs no
// sums at all: P and dS as bf16, which is how they enter the products anyway.  Three launches
// after the row statistics:
//
//   probabilities     64 rows x 128 keys a workgroup, a 32 x 32 block a wave: S and dP over 64
//                     columns at a time, P and dS to the buffers below
//   key gradients     dK = dS^T Q + P^T dO: 32 keys x 32 columns a workgroup; its four waves take
//                     row tiles in turn, each through LDS of its own (no barriers), and add up
//                     their sums at the end, in wave order
//   query gradients   dQ = dS K: 64 rows a workgroup, over the key tiles they see
//
// "Rows" are the (token, head) pairs of a batch element, token major, as in mla_absorbed.hip.  A
// row's dS lies in its own 1024 bytes of the latent query gradient, 64 bytes per block of 32 keys
// up to the row's own block of tokens: the last launch reads the dS of exactly the rows it
// overwrites.  With n blocks of tokens the rows of block i leave 64 * (16 - i - 1) bytes free.
// P, 64 * (i + 1) bytes of a row of block i, lies behind the dS of the row that many heads
// further in block n - 2 - i (i < n - 1); P of the last block, n chunks a row, chunk c in bytes
// 64..127 of the rope query gradient of the row of block c (bytes 0..3 hold the row's delta).
// Only the last block of tokens may be short, and its rows receive chunks of their own P alone.
//
// Bound by the bytes a compute unit draws, some 30 cycles per KB of whole lines.  T = 512, H = 8:
// key gradients, reduction and query gradients of mla_absorbed.hip 51 + 5 + 28 us -> 10 + 20 + 17
// here.  The key gradients read 64 bytes of each row: 33 us with the column blocks dealt to the
// XCDs in turn (every L2 then fetches every row whole), 20 with two neighbouring ones per XCD.
// The query gradients' dS straight from memory, 16 bytes of 32 rows per load, cost 16 us; through
// LDS with the key tiles 2.
#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "lds_tiles.h"

#include <cstdint>
#include <type_traits>

namespace dscuda {
namespace {

constexpr int RANK = 512;
constexpr int ROPE = 64;
constexpr int TILE = 32;
constexpr int CHUNK_BYTES = 2 * TILE;          // P or dS of a row and 32 keys
constexpr int DELTA_STRIDE = ROPE / 2;         // floats between the deltas of two rows

// Where P and dS lie, in the query gradients of one batch element.
struct KeptScores {
    unsigned char* latent;
    unsigned char* rope;
    int heads;
    int blocks;   // of 32 tokens

    __device__ __forceinline__ unsigned char* ds(int row, int key_block) const {
        return latent + (size_t)row * (2 * RANK) + CHUNK_BYTES * key_block;
    }
    __device__ __forceinline__ unsigned char* p(int row, int token_block, int key_block) const {
        return index_math::kept_in_rope(token_block, blocks)
            ? rope + (size_t)index_math::kept_row(row, token_block, key_block, blocks, heads) * (2 * ROPE) + CHUNK_BYTES
            : latent + (size_t)index_math::kept_row(row, token_block, key_block, blocks, heads) * (2 * RANK) +
                CHUNK_BYTES * index_math::kept_chunk(token_block, key_block, blocks);
    }
};

__device__ __forceinline__ f32x16 zeros() {
    return f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
}

// ---- P and dS --------------------------------------------------------------------

constexpr int SCORE_THREADS = 512;
constexpr int SCORE_ROWS = 64;
constexpr int SCORE_KEYS = 128;

struct ScoreLayout {
    static constexpr int COLUMNS = 64;                      // of a step
    static constexpr int ROW = 2 * COLUMNS;
    static constexpr int Q_AT = 0;
    static constexpr int DO_AT = Q_AT + SCORE_ROWS * ROW;
    static constexpr int K_AT = DO_AT + SCORE_ROWS * ROW;
    static constexpr int STAGE_BYTES = K_AT + SCORE_KEYS * ROW;   // 32 KB
    static constexpr int STAGES = 4;
    static constexpr int LDS_BYTES = STAGES * STAGE_BYTES;
    static constexpr int OUT_PITCH = CHUNK_BYTES + 16;      // of a staged chunk, in the place of the stages
    static_assert(8 * 2 * TILE * OUT_PITCH <= LDS_BYTES, "the staged chunks must fit");
};

__global__ __launch_bounds__(SCORE_THREADS) void mla_short_probabilities_kernel(
    unsigned char* latent_gradient, unsigned char* rope_gradient, const bf16_t* __restrict__ output_gradient,
    const float* __restrict__ logsumexp, const bf16_t* __restrict__ query_latent, const bf16_t* __restrict__ query_rope,
    const bf16_t* __restrict__ kv_latent, const bf16_t* __restrict__ key_rope, int sequence_length, int heads, float scale) {
    using L = ScoreLayout;
    constexpr int STEPS = (RANK + ROPE) / L::COLUMNS;   // 9, the last one the rope columns
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int T = sequence_length;
    const int rows = T * heads;
    const int batch = blockIdx.z;
    const int row0 = blockIdx.x * SCORE_ROWS;
    const int key0 = blockIdx.y * SCORE_KEYS;
    if (key0 > (min(row0 + SCORE_ROWS, rows) - 1) / heads) {
        return;   // no row of the workgroup sees these keys
    }
    const size_t batch_row = (size_t)batch * rows + row0;
    const unsigned char* q = reinterpret_cast<const unsigned char*>(query_latent + batch_row * RANK);
    const unsigned char* qr = reinterpret_cast<const unsigned char*>(query_rope + batch_row * ROPE);
    const unsigned char* dout = reinterpret_cast<const unsigned char*>(output_gradient + batch_row * RANK);
    const unsigned char* k = reinterpret_cast<const unsigned char*>(kv_latent + ((size_t)batch * T + key0) * RANK);
    const unsigned char* kr = reinterpret_cast<const unsigned char*>(key_rope + ((size_t)batch * T + key0) * ROPE);

    // rows and keys past the end repeat the last one: their P and dS are not kept, or zero
    TileRequests<L::ROW, 8, SCORE_ROWS> wide_rows, rope_rows;
    TileRequests<L::ROW, 8, SCORE_KEYS> wide_keys, rope_keys;
    wide_rows.init(2 * RANK, wave, lane);
    rope_rows.init(2 * ROPE, wave, lane);
    wide_keys.init(2 * RANK, wave, lane);
    rope_keys.init(2 * ROPE, wave, lane);
    constexpr int LOADS = 2 * TileRequests<L::ROW, 8, SCORE_ROWS>::LOADS + TileRequests<L::ROW, 8, SCORE_KEYS>::LOADS;
    const int row_limit = rows - 1 - row0;
    const int key_limit = T - 1 - key0;
    const unsigned lds_base = lds_offset_of(lds);
    auto request_step = [&](int step) {
        const unsigned target = lds_base + step % L::STAGES * L::STAGE_BYTES;
        if (step < STEPS - 1) {
            wide_rows.request(q + step * L::ROW, 2 * RANK, row_limit, target + L::Q_AT, wave);
            wide_rows.request(dout + step * L::ROW, 2 * RANK, row_limit, target + L::DO_AT, wave);
            wide_keys.request(k + step * L::ROW, 2 * RANK, key_limit, target + L::K_AT, wave);
        } else {
            rope_rows.request(qr, 2 * ROPE, row_limit, target + L::Q_AT, wave);
            rope_rows.request(qr, 2 * ROPE, row_limit, target + L::DO_AT, wave);   // not read: as many loads as any step
            rope_keys.request(kr, 2 * ROPE, key_limit, target + L::K_AT, wave);
        }
    };
    request_step(0);
    request_step(1);
    request_step(2);

    // the lane's row
    const int row_half = wave % 2;
    const int key_block = wave / 2;   // of the workgroup's four
    const int row = row0 + TILE * row_half + lq;
    const bool valid = row < rows;
    int token = -1;
    float lse2 = 0.f, delta = 0.f;
    if (valid) {
        token = row / heads;
        lse2 = logsumexp[((size_t)batch * heads + row % heads) * T + token] * LOG2E;
        delta = reinterpret_cast<const float*>(rope_gradient)[((size_t)batch * rows + row) * DELTA_STRIDE];
    }

    TileReads<L::ROW> reads;
    reads.init(lane);
    f32x16 s_acc = zeros(), dp_acc = zeros();
    // S^T and dP^T (keys x rows) over the step's columns
    auto multiply = [&](int step, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        const unsigned stage = step % L::STAGES * L::STAGE_BYTES;
        unsigned q_at[TileReads<L::ROW>::NAT], do_at[TileReads<L::ROW>::NAT], k_at[TileReads<L::ROW>::NAT];
        rebase(q_at, reads.natural, stage + L::Q_AT + row_half * TILE * L::ROW);
        rebase(do_at, reads.natural, stage + L::DO_AT + row_half * TILE * L::ROW);
        rebase(k_at, reads.natural, stage + L::K_AT + key_block * TILE * L::ROW);
        unrolled<0, L::COLUMNS / 16>([&](auto tag) {
            constexpr int KS = decltype(tag)::value;
            const bf16x8 key_fragment = natural_fragment<L::ROW, 0, KS>(lds, k_at);
            s_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(key_fragment, natural_fragment<L::ROW, 0, KS>(lds, q_at), s_acc, 0, 0, 0);
            if constexpr (!LAST) {
                dp_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(key_fragment, natural_fragment<L::ROW, 0, KS>(lds, do_at), dp_acc,
                                                                 0, 0, 0);
            }
        });
    };
    for (int step = 0; step < STEPS - 1; ++step) {
        if (step + 2 < STEPS) {
            wait_vector_memory<2 * LOADS>();   // steps step + 1 and step + 2 may stay in flight
        } else {
            wait_vector_memory<LOADS>();
        }
        workgroup_barrier();
        if (step + 3 < STEPS) request_step(step + 3);
        multiply(step, std::false_type{});
    }
    wait_vector_memory<0>();
    workgroup_barrier();
    multiply(STEPS - 1, std::true_type{});
    workgroup_barrier();   // the stages have been read

    // lane holds row lq and keys 8*i4 + 4*g .. +3 of the wave's block: chunks of 64 bytes through LDS
    unsigned char* staged = lds + wave * 2 * TILE * L::OUT_PITCH;
    const float c = scale * LOG2E;
    const int first_key = key0 + TILE * key_block;
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
        float p[4], ds[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[e] = __builtin_amdgcn_exp2f(fmaf(s_acc[4 * i4 + e], c, -lse2));
            if (first_key + 8 * i4 + 4 * g + e > token) p[e] = 0.f;
            ds[e] = p[e] * (dp_acc[4 * i4 + e] - delta) * scale;
        }
        unsigned char* at = staged + lq * L::OUT_PITCH + 16 * i4 + 8 * g;
        *reinterpret_cast<u32x2*>(at) = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
        *reinterpret_cast<u32x2*>(at + TILE * L::OUT_PITCH) = u32x2{pack_bf16(ds[0], ds[1]), pack_bf16(ds[2], ds[3])};
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's LDS writes have landed
    __builtin_amdgcn_wave_barrier();
    const KeptScores kept = {latent_gradient + (size_t)batch * rows * (2 * RANK), rope_gradient + (size_t)batch * rows * (2 * ROPE),
                             heads, (T + TILE - 1) / TILE};
    const int block = first_key / TILE;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int out_row = 16 * j + lane / 4;   // four lanes a row, 16 bytes each
        const int piece = lane % 4;
        const int global_row = row0 + TILE * row_half + out_row;
        const int token_block = global_row / heads / TILE;
        if (global_row < rows && block <= token_block) {
            const unsigned char* at = staged + out_row * L::OUT_PITCH + 16 * piece;
            *reinterpret_cast<u32x4*>(kept.p(global_row, token_block, block) + 16 * piece) = *reinterpret_cast<const u32x4*>(at);
            *reinterpret_cast<u32x4*>(kept.ds(global_row, block) + 16 * piece) =
                *reinterpret_cast<const u32x4*>(at + TILE * L::OUT_PITCH);
        }
    }
}

// ---- key gradients ----------------------------------------------------------------

constexpr int KEY_THREADS = 256;
constexpr int XCDS = 8;
static_assert(RANK / TILE == 2 * XCDS && ROPE / TILE == 2, "two column blocks per XCD, and two of the rope columns");

struct KeyLayout {
    static constexpr int PART = TILE * CHUNK_BYTES;      // [32 rows][64 bytes]: dS, P, query or dO columns
    static constexpr int SLOT_BYTES = 4 * PART;
    static constexpr int SLOTS = 4;                      // of a wave
    static constexpr int WAVE_BYTES = SLOTS * SLOT_BYTES;
    static constexpr int LDS_BYTES = 4 * WAVE_BYTES;     // 128 KB: no two of the heaviest workgroups on one compute unit
    static constexpr int SUM_PITCH = TILE + 1;           // floats
    static_assert(4 * TILE * SUM_PITCH * 4 <= LDS_BYTES, "the sums take the place of the slots");
};

// Operand with the row of a [32][64 bytes] tile as the contraction index: column lane % 32, rows {16*STEP + 4g .. +3,
// 16*STEP + 8 + 4g .. +3}.  The 64 lanes of a read cover 512 bytes in a row: no bank conflicts without a swizzle.
template <int STEP>
__device__ __forceinline__ bf16x8 chunk_fragment(const unsigned char* tile, int lane_at) {
    const unsigned char* at = tile + lane_at + 16 * STEP * CHUNK_BYTES;
    const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)at);
    const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(at + 8 * CHUNK_BYTES));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
}

__global__ __launch_bounds__(KEY_THREADS) void mla_short_key_gradient_kernel(
    bf16_t* __restrict__ kv_latent_gradient, bf16_t* __restrict__ key_rope_gradient, unsigned char* latent_gradient,
    unsigned char* rope_gradient, const bf16_t* __restrict__ output_gradient, const bf16_t* __restrict__ query_latent,
    const bf16_t* __restrict__ query_rope, int sequence_length, int heads) {
    using L = KeyLayout;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int T = sequence_length;
    const int rows = T * heads;
    const int batch = blockIdx.y;
    // Which key block and columns.  An XCD takes two neighbouring latent column blocks of every key block, so that its
    // L2 fetches 128 of a row's 1024 bytes, and an eighth of the (cheaper) rope blocks; key block 0, which sees every
    // row, first.
    const int blocks = (T + TILE - 1) / TILE;
    const int slot_of_xcd = blockIdx.x / XCDS;
    int key_block, column_block;
    if (slot_of_xcd < 2 * blocks) {
        key_block = slot_of_xcd / 2;
        column_block = 2 * (blockIdx.x % XCDS) + slot_of_xcd % 2;
    } else {
        const int item = (slot_of_xcd - 2 * blocks) * XCDS + blockIdx.x % XCDS;
        key_block = item / 2;
        column_block = RANK / TILE + item % 2;
        if (key_block >= blocks) return;
    }
    const bool latent_columns = column_block < RANK / TILE;
    const size_t batch_row = (size_t)batch * rows;
    const KeptScores kept = {latent_gradient + batch_row * (2 * RANK), rope_gradient + batch_row * (2 * ROPE), heads,
                             blocks};
    const unsigned char* query = latent_columns
        ? reinterpret_cast<const unsigned char*>(query_latent + batch_row * RANK) + CHUNK_BYTES * column_block
        : reinterpret_cast<const unsigned char*>(query_rope + batch_row * ROPE) + CHUNK_BYTES * (column_block - RANK / TILE);
    const int query_stride = latent_columns ? 2 * RANK : 2 * ROPE;
    const unsigned char* dout = reinterpret_cast<const unsigned char*>(output_gradient + batch_row * RANK) +
        CHUNK_BYTES * (latent_columns ? column_block : 0);

    const int first_tile = key_block * heads;   // of 32 rows: tokens 32 * key_block on
    const int end_tile = (rows + TILE - 1) / TILE;
    const unsigned lds_base = lds_offset_of(lds) + wave * L::WAVE_BYTES;
    const int s = lane % 16;
    const int lane_at = (4 * g + s / 4) * CHUNK_BYTES + 32 * ((lane / 16) % 2) + 8 * (s % 4);
    f32x16 sum = zeros();
    auto walk = [&](auto latent_tag) {
        constexpr bool LATENT = decltype(latent_tag)::value;
        constexpr int LOADS = LATENT ? 8 : 4;   // of a row tile, 1 KB each: 16 rows, four lanes a row
        auto request_tile = [&](int tile, int slot) {
            const unsigned target = lds_base + slot * L::SLOT_BYTES;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                // rows past the end repeat the last one; the products leave them out
                const int row = min(TILE * tile + 16 * j + lane / 4, rows - 1);
                const int token_block = row / heads / TILE;
                const int byte = 16 * (lane % 4);
                direct_load_16(kept.ds(row, key_block) + byte, target + 0 * L::PART + 1024 * j);
                direct_load_16(query + (size_t)row * query_stride + byte, target + 1 * L::PART + 1024 * j);
                if constexpr (LATENT) {
                    direct_load_16(kept.p(row, token_block, key_block) + byte, target + 2 * L::PART + 1024 * j);
                    direct_load_16(dout + (size_t)row * (2 * RANK) + byte, target + 3 * L::PART + 1024 * j);
                }
            }
        };

        // the wave's tiles, three of them asked for ahead of the one in use
        const int count = (end_tile - first_tile - wave + 3) / 4;
        for (int ahead = 0; ahead < min(count, 3); ++ahead) request_tile(first_tile + wave + 4 * ahead, ahead);
        for (int index = 0; index < count; ++index) {
            const int tile = first_tile + wave + 4 * index;
            const int slot = index % L::SLOTS;
            if (index + 3 < count) {
                request_tile(tile + 12, (index + 3) % L::SLOTS);
                wait_vector_memory<3 * LOADS>();
            } else if (index + 2 < count) {
                wait_vector_memory<2 * LOADS>();
            } else if (index + 1 < count) {
                wait_vector_memory<LOADS>();
            } else {
                wait_vector_memory<0>();
            }
            asm volatile("" ::: "memory");   // the slot is read below, not above
            const unsigned char* at = lds + wave * L::WAVE_BYTES + slot * L::SLOT_BYTES;
            const int valid_rows = rows - TILE * tile;
            unrolled<0, 2>([&](auto tag) {
                constexpr int N = decltype(tag)::value;
                bf16x8 ds = chunk_fragment<N>(at, lane_at);
                const bf16x8 query_columns = chunk_fragment<N>(at + 1 * L::PART, lane_at);
                bf16x8 p, do_columns;
                if constexpr (LATENT) {
                    p = chunk_fragment<N>(at + 2 * L::PART, lane_at);
                    do_columns = chunk_fragment<N>(at + 3 * L::PART, lane_at);
                }
                if (valid_rows < TILE) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (16 * N + 4 * g + (e < 4 ? e : 4 + e) >= valid_rows) ds[e] = p[e] = (__bf16)0.f;
                    }
                }
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ds, query_columns, sum, 0, 0, 0);
                if constexpr (LATENT) sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p, do_columns, sum, 0, 0, 0);
            });
            __builtin_amdgcn_s_waitcnt(0xc07f);   // the slot has been read before it is asked for again
            asm volatile("" ::: "memory");
        }
    };
    if (latent_columns) walk(std::true_type{}); else walk(std::false_type{});

    // lane holds column lq and keys 8*(i/4) + 4*g + i%4
    __syncthreads();
    float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[(wave * TILE + 8 * (i / 4) + 4 * g + i % 4) * L::SUM_PITCH + lq] = sum[i];
    __syncthreads();
    const int key = tid / 8;
    const int column = 4 * (tid % 8);
    float total[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        total[e] = sums[key * L::SUM_PITCH + column + e];
#pragma unroll
        for (int w = 1; w < 4; ++w) total[e] += sums[(w * TILE + key) * L::SUM_PITCH + column + e];
    }
    const int token = TILE * key_block + key;
    if (token < T) {
        bf16_t* target = latent_columns
            ? kv_latent_gradient + ((size_t)batch * T + token) * RANK + TILE * column_block + column
            : key_rope_gradient + ((size_t)batch * T + token) * ROPE + TILE * (column_block - RANK / TILE) + column;
        *reinterpret_cast<u32x2*>(target) = u32x2{pack_bf16(total[0], total[1]), pack_bf16(total[2], total[3])};
    }
}

// ---- query gradients ---------------------------------------------------------------

constexpr int QUERY_THREADS = 512;
constexpr int QUERY_ROWS = 64;

struct QueryLayout {
    static constexpr int WIDE_ROW = 2 * RANK;
    static constexpr int NARROW_ROW = 2 * ROPE;
    static constexpr int ROPE_AT = TILE * WIDE_ROW;
    static constexpr int DS_AT = ROPE_AT + TILE * NARROW_ROW;
    static constexpr int STAGE_BYTES = DS_AT + QUERY_ROWS * CHUNK_BYTES;   // 40 KB: [32 keys][512], [32 keys][64], dS [64 rows][32 keys]
    static constexpr int STAGES = 4;
    static constexpr int LDS_BYTES = STAGES * STAGE_BYTES;
    static constexpr int OUT_PITCH = 2 * (RANK + ROPE) + 16;               // of a staged gradient row
    static_assert(LDS_BYTES <= 160 * 1024 && QUERY_ROWS * OUT_PITCH <= LDS_BYTES, "LDS of a compute unit");
    // 16-byte piece of a row's dS chunk -> its place: rows four apart share their banks
    static __device__ __forceinline__ int ds_piece(int row, int piece) { return piece ^ (row / 4 % 4); }
};

__global__ __launch_bounds__(QUERY_THREADS) void mla_short_query_gradient_kernel(
    bf16_t* latent_gradient, bf16_t* rope_gradient, const bf16_t* __restrict__ kv_latent, const bf16_t* __restrict__ key_rope,
    int sequence_length, int heads) {
    using L = QueryLayout;
    using Wide = index_math::TileReadMath<L::WIDE_ROW>;
    using Narrow = index_math::TileReadMath<L::NARROW_ROW>;
    constexpr int LATENT_BLOCKS = RANK / TILE / 4;   // 32-column blocks of a wave
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int T = sequence_length;
    const int rows = T * heads;
    const int batch = blockIdx.y;
    const int row0 = (gridDim.x - 1 - blockIdx.x) * QUERY_ROWS;   // latest rows (most keys) first
    const size_t batch_row = (size_t)batch * rows;
    const unsigned char* latent = reinterpret_cast<const unsigned char*>(kv_latent + (size_t)batch * T * RANK);
    const unsigned char* rope = reinterpret_cast<const unsigned char*>(key_rope + (size_t)batch * T * ROPE);
    const int tiles = (min(row0 + QUERY_ROWS, rows) - 1) / heads / TILE + 1;   // key tiles the rows see

    // wave w: rows of tile w / 4, latent column blocks 4v .. 4v + 3 (v = w % 4) and, v < 2, rope block v
    const int v = wave % 4;
    const int row = row0 + TILE * (wave / 4) + lq;
    const int own_tiles = row < rows ? row / heads / TILE + 1 : 0;   // whose dS the lane's row has
    const unsigned char* ds_rows = reinterpret_cast<const unsigned char*>(latent_gradient) + batch_row * (2 * RANK);

    // a wave requests key rows 4*wave .. +3 of the wide tile, waves 0 .. 3 also eight rows of the narrow one, waves 4 .. 7
    // dS of 16 rows
    const unsigned lds_base = lds_offset_of(lds);
    auto request_tile = [&](int tile) {
        const unsigned target = lds_base + tile % L::STAGES * L::STAGE_BYTES;
        const int last = min(T - tile * TILE, TILE) - 1;   // keys past the end repeat the last one: their dS is zero
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int key = 4 * wave + j;
            direct_load_16_offset(latent + (size_t)tile * TILE * L::WIDE_ROW,
                                  (unsigned)(min(key, last) * L::WIDE_ROW + 16 * (lane ^ index_math::tile_swizzle<L::WIDE_ROW>(key))),
                                  target + key * L::WIDE_ROW);
        }
        if (wave < 4) {
            const int key = 8 * wave + lane / 8;
            direct_load_16_offset(rope + (size_t)tile * TILE * L::NARROW_ROW,
                                  (unsigned)(min(key, last) * L::NARROW_ROW +
                                             16 * ((lane % 8) ^ index_math::tile_swizzle<L::NARROW_ROW>(key))),
                                  target + L::ROPE_AT + 8 * wave * L::NARROW_ROW);
        } else {
            const int ds_row = 16 * (wave - 4) + lane / 4;
            direct_load_16(ds_rows + (size_t)min(row0 + ds_row, rows - 1) * (2 * RANK) + CHUNK_BYTES * tile +
                               16 * L::ds_piece(ds_row, lane % 4),
                           target + L::DS_AT + 16 * (wave - 4) * CHUNK_BYTES);
        }
    };
    constexpr int LOADS = 5;   // of a wave and tile
    request_tile(0);
    if (tiles > 1) request_tile(1);
    if (tiles > 2) request_tile(2);

    unsigned wide_at[2][LATENT_BLOCKS], narrow_at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < LATENT_BLOCKS; ++j) wide_at[h][j] = Wide::transposed(h, j, lane) + 256 * v;
        narrow_at[h] = L::ROPE_AT + Narrow::transposed(h, v % 2, lane);
    }
    f32x16 sum[LATENT_BLOCKS + 1];
#pragma unroll
    for (int j = 0; j <= LATENT_BLOCKS; ++j) sum[j] = zeros();
    for (int tile = 0; tile < tiles; ++tile) {
        if (tile + 2 < tiles) {
            wait_vector_memory<2 * LOADS>();   // tiles tile + 1 and tile + 2 may stay in flight
        } else if (tile + 1 < tiles) {
            wait_vector_memory<LOADS>();
        } else {
            wait_vector_memory<0>();
        }
        workgroup_barrier();
        if (tile + 3 < tiles) request_tile(tile + 3);
        const unsigned char* stage = lds + tile % L::STAGES * L::STAGE_BYTES;
        // dS of the lane's row: keys {16n + 4g .. +3, 16n + 8 + 4g .. +3}; a chunk past the row's own block holds something else
        const unsigned char* own_ds = stage + L::DS_AT + (TILE * (wave / 4) + lq) * CHUNK_BYTES + 8 * g;
        unrolled<0, 2>([&](auto tag) {
            constexpr int N = decltype(tag)::value;
            const u32x2 low_ds = *reinterpret_cast<const u32x2*>(own_ds + 16 * L::ds_piece(lq, 2 * N));
            const u32x2 high_ds = *reinterpret_cast<const u32x2*>(own_ds + 16 * L::ds_piece(lq, 2 * N + 1));
            u32x4 bits = {0, 0, 0, 0};
            if (tile < own_tiles) bits = u32x4{low_ds[0], low_ds[1], high_ds[0], high_ds[1]};
            const bf16x8 dsf = __builtin_bit_cast(bf16x8, bits);
            auto fragment = [&](unsigned low_at, unsigned high_at, int row_bytes) {
                const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(stage + low_at + 16 * N * row_bytes));
                const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(stage + high_at + 16 * N * row_bytes));
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
            };
#pragma unroll
            for (int j = 0; j < LATENT_BLOCKS; ++j) {
                sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fragment(wide_at[0][j], wide_at[1][j], L::WIDE_ROW), dsf, sum[j], 0, 0, 0);
            }
            if (v < 2) {
                sum[LATENT_BLOCKS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fragment(narrow_at[0], narrow_at[1], L::NARROW_ROW), dsf,
                                                                             sum[LATENT_BLOCKS], 0, 0, 0);
            }
        });
    }

    // Every dS of the workgroup's rows has arrived.  A lane holds row lq and columns 32*block + 8*(i/4) + 4*g + i%4: rows
    // through LDS, so that a store instruction writes whole lines
    workgroup_barrier();
    unsigned char* staged = lds + (TILE * (wave / 4) + lq) * L::OUT_PITCH;
    auto stage_block = [&](const f32x16& values, int block) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            *reinterpret_cast<u32x2*>(staged + CHUNK_BYTES * block + 16 * i4 + 8 * g) =
                u32x2{pack_bf16(values[4 * i4 + 0], values[4 * i4 + 1]), pack_bf16(values[4 * i4 + 2], values[4 * i4 + 3])};
        }
    };
#pragma unroll
    for (int j = 0; j < LATENT_BLOCKS; ++j) stage_block(sum[j], LATENT_BLOCKS * v + j);
    if (v < 2) stage_block(sum[LATENT_BLOCKS], RANK / TILE + v);
    workgroup_barrier();
    for (int out_row = wave; out_row < min(QUERY_ROWS, rows - row0); out_row += QUERY_THREADS / 64) {
        const size_t target = batch_row + row0 + out_row;
        *reinterpret_cast<u32x4*>(latent_gradient + target * RANK + 8 * lane) =
            *reinterpret_cast<const u32x4*>(lds + out_row * L::OUT_PITCH + 16 * lane);
        if (lane < ROPE / 8) {
            *reinterpret_cast<u32x4*>(rope_gradient + target * ROPE + 8 * lane) =
                *reinterpret_cast<const u32x4*>(lds + out_row * L::OUT_PITCH + 2 * RANK + 16 * lane);
        }
    }
}

template <typename Kernel>
void raise_lds_limit(Kernel kernel, int bytes) {
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
}

}  // namespace

void mla_absorbed_short_backward_launch(bf16_t* query_latent_gradient, bf16_t* query_rope_gradient, bf16_t* kv_latent_gradient,
                                        bf16_t* key_rope_gradient, const bf16_t* output_gradient, const float* logsumexp,
                                        const bf16_t* query_latent, const bf16_t* query_rope, const bf16_t* kv_latent,
                                        const bf16_t* key_rope, int batch_size, int sequence_length, int heads, float scale,
                                        hipStream_t stream) {
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        raise_lds_limit(mla_short_probabilities_kernel, ScoreLayout::LDS_BYTES);
        raise_lds_limit(mla_short_key_gradient_kernel, KeyLayout::LDS_BYTES);
        raise_lds_limit(mla_short_query_gradient_kernel, QueryLayout::LDS_BYTES);
    });
    const int rows = sequence_length * heads;
    const int blocks = (sequence_length + TILE - 1) / TILE;
    unsigned char* latent = reinterpret_cast<unsigned char*>(query_latent_gradient);
    unsigned char* rope = reinterpret_cast<unsigned char*>(query_rope_gradient);
    hipLaunchKernelGGL(mla_short_probabilities_kernel,
                       dim3((unsigned)((rows + SCORE_ROWS - 1) / SCORE_ROWS), (unsigned)((sequence_length + SCORE_KEYS - 1) / SCORE_KEYS),
                            (unsigned)batch_size),
                       dim3(SCORE_THREADS), ScoreLayout::LDS_BYTES, stream, latent, rope, output_gradient, logsumexp, query_latent,
                       query_rope, kv_latent, key_rope, sequence_length, heads, scale);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(mla_short_key_gradient_kernel,
                       dim3((unsigned)(XCDS * (2 * blocks + (2 * blocks + XCDS - 1) / XCDS)), (unsigned)batch_size),
                       dim3(KEY_THREADS), KeyLayout::LDS_BYTES, stream, kv_latent_gradient, key_rope_gradient, latent, rope,
                       output_gradient, query_latent, query_rope, sequence_length, heads);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(mla_short_query_gradient_kernel, dim3((unsigned)((rows + QUERY_ROWS - 1) / QUERY_ROWS), (unsigned)batch_size),
                       dim3(QUERY_THREADS), QueryLayout::LDS_BYTES, stream, query_latent_gradient, query_rope_gradient, kv_latent,
                       key_rope, sequence_length, heads);
    HIP_CHECK(hipGetLastError());
}

}  // namespace dscuda
