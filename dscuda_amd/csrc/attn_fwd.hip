// Causal attention forward for gfx950: S^T = K Q^T and O^T = V^T P^T on bf16
// MFMA 32x32x16 tiles, online softmax in fp32, natural-log LSE.
//
// Three kernels serve the flash-attention forward (D = 64 / 128, GQA) and the
// per-head MLA prefill forward (d_qk = 128 nope + 64 rope = 192, d_v = 128):
// split keys for short and medium problems, a persistent one for large ones,
// and small independent workgroups (four waves) for many heads of 64 columns or
// of one tile of keys.
// They take the place of the reference's
// flash_attention_forward_tensor_core_kernel
// (kernels/attention/flash_attention/sm89_forward.cu:99-205); the tiling is
// chosen for 64-lane waves and the 160 KB LDS, not taken from there.
//
// Transposed formulation
//   Scores are produced as S^T (keys x queries): A = K tile (LDS), B = Q
//   (registers, loaded once).  In the MFMA C layout a lane then holds one
//   query column (lane % 32) and 32 of the tile's 64 keys, so the softmax
//   statistics are per-lane scalars and the only cross-lane step is one
//   exchange with the lane 32 away.  The same registers, rounded to bf16, are
//   directly the B operand of O^T += V^T P^T (k index = key), so P never
//   moves between lanes or through LDS.
//
// Tiles: global -> LDS without registers
//   K and V tiles arrive by global_load_lds (16 bytes per lane, 1 KB of
//   consecutive LDS per wave instruction), both row-major.  No
//   thread holds tile data in registers and nothing is written to LDS with
//   store instructions.  With no padding possible inside the 1 KB a wave
//   instruction fills, bank spread comes from a swizzle applied on the global
//   side: which 16-byte chunk a lane fetches.  The split-key kernel takes that of
//   lds_tiles.h, the others
//     K  : chunk c of row r sits at position c ^ fK(r).  A fragment read is 16
//          lanes x 16 B down a column of rows; fK(r) = (r>>1)&7 for rows that
//          are 128 (mod 256) bytes long, r&15 for rows that are 0 (mod 256).
//     V  : MFMA wants the contraction index (key) contiguous per lane, V has
//          d_v contiguous.  ds_read_b64_tr_b16 transposes a 4 keys x 16 columns
//          block across 16 lanes while reading, so the row-major tile is used
//          as it is.  Such a read touches 4 rows x 64 bytes; rows are 64*NG
//          bytes long (NG = d_v/32 column groups), so the 64-byte group index
//          of row r is XORed with r&3 (NG = 4) or (r>>1)&1 (NG = 2), and the
//          lane that addresses row r undoes it in its own address.
//   A tile is requested while the previous one is consumed; arrival is ordered
//   by s_waitcnt vmcnt + one workgroup barrier per tile.
#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "lds_tiles.h"

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <string>
#include <type_traits>

namespace dscuda {
namespace {

template <int DQK, int DV, int NWAVES>
struct FwdConfig {
    static constexpr int BN = 64;
    static constexpr int BM = 32 * NWAVES;
    static constexpr int THREADS = 64 * NWAVES;
    static constexpr int K_ROW = DQK * 2;                  // bytes
    static constexpr int K_CHUNKS = DQK / 8;               // 16-byte chunks per row
    static constexpr int K_BYTES = BN * K_ROW;
    static constexpr int V_ROW = DV * 2;
    static constexpr int V_CHUNKS = DV / 8;
    static constexpr int V_GROUPS = DV / 32;               // 64-byte column groups per row
    static constexpr int V_BYTES = BN * V_ROW;
    static constexpr int STAGE_BYTES = K_BYTES + V_BYTES;
    static constexpr int K_LOADS_PER_WAVE = K_BYTES / 1024 / NWAVES;   // wave instructions
    static constexpr int V_LOADS_PER_WAVE = V_BYTES / 1024 / NWAVES;
    // four-wave kernel: two stages, then the output rows in their place
    static constexpr int O_PITCH = DV * 2 + 16;            // bytes
    static constexpr int O_BYTES = BM * O_PITCH;
    static constexpr int LDS_BYTES = (2 * STAGE_BYTES > O_BYTES) ? 2 * STAGE_BYTES : O_BYTES;
    static_assert(K_BYTES % (1024 * NWAVES) == 0 && V_BYTES % (1024 * NWAVES) == 0,
                  "tile loads must divide evenly over the waves");
    static_assert(K_ROW % 128 == 0, "K rows must be a multiple of 128 bytes");
    static_assert(V_GROUPS == 2 || V_GROUPS == 4, "d_v must be 64 or 128");

    __device__ static constexpr int k_swizzle(int row) {
        return (K_ROW % 256 == 0) ? (row & 15) : ((row >> 1) & 7);
    }
    __device__ static constexpr int v_flip(int row) {
        return V_GROUPS == 4 ? (row & 3) : ((row >> 1) & 1);
    }
};

// ---------------------------------------------------------------------------
// Four waves, 128 queries.
//
// Each wave owns 32 query rows for the whole key loop; keys are walked in tiles of 64 from key 0 up to the diagonal, two
// stages.  A walk is one dependent chain of scores, softmax and output products per tile, twice to four times as long as
// in the split-key kernel, but a workgroup of 64 columns takes 32 KB of LDS and a quarter of the waves of a compute unit:
// with enough of them the others cover each chain, no output part crosses LDS, and start and end of a workgroup, 8000
// cycles there, are cheap.  Bound by issue (matrix, softmax and LDS reads of two to four workgroups a unit).
// Split keys -> four waves (us): 64 columns, 2048 heads of 128 tokens 35.9 -> 26.3, of 1024 tokens 592 -> 486; 512 heads
// of 2048 tokens 463 -> 418; one tile of keys: 2048 heads of 64 tokens, 64 columns 18.1 -> 15.9, 192/128 columns
// 51.7 -> 48.8, of one token 45.3 -> 34.2.
template <int DQK, int DV, int NWAVES>
__global__ __launch_bounds__(64 * NWAVES) void attention_forward_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp,
    const bf16_t* __restrict__ query, const bf16_t* __restrict__ key, const bf16_t* __restrict__ value,
    int sequence_length, int query_heads, int key_value_heads, int query_blocks, float scale) {
    using C = FwdConfig<DQK, DV, NWAVES>;
    constexpr int BN = C::BN;
    constexpr int KSTEPS = DQK / 16;
    constexpr int DBLOCKS = DV / 32;

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;

    // (batch, head) groups are dealt across XCDs; inside a group the heaviest
    // (last) query blocks are issued first.
    int bh, qb_rank;
    xcd_order(blockIdx.x, gridDim.x / query_blocks, query_blocks, bh, qb_rank);
    const int qb = query_blocks - 1 - qb_rank;
    const int b = bh / query_heads;
    const int h = bh % query_heads;
    const int hk = h / (query_heads / key_value_heads);
    const int S = sequence_length;

    const int q0 = qb * C::BM;
    const int wave_q0 = q0 + 32 * wave;
    const int q_row = wave_q0 + lq;

    const size_t q_stride = (size_t)query_heads * DQK;
    const unsigned k_stride_bytes = (unsigned)key_value_heads * DQK * 2;
    const unsigned v_stride_bytes = (unsigned)key_value_heads * DV * 2;
    const bf16_t* q_base = query + ((size_t)b * S * query_heads + h) * DQK;
    const unsigned char* k_base =
        reinterpret_cast<const unsigned char*>(key + ((size_t)b * S * key_value_heads + hk) * DQK);
    const unsigned char* v_base =
        reinterpret_cast<const unsigned char*>(value + ((size_t)b * S * key_value_heads + hk) * DV);

    // ---- Q fragments (B operand: column = query lq, k = 16*ks + 8*g + j)
    bf16x8 qf[KSTEPS];
    {
        const bool valid = q_row < S;
        const bf16_t* row = q_base + (size_t)(valid ? q_row : 0) * q_stride + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            u32x4 bits = {0, 0, 0, 0};
            if (valid) {
                bits = *reinterpret_cast<const u32x4*>(row + 16 * ks);
            }
            qf[ks] = __builtin_bit_cast(bf16x8, bits);
        }
    }

    const int last_key = min(S, q0 + C::BM) - 1;
    const int tiles = last_key / BN + 1;
    const unsigned lds_base = lds_offset_of(lds);

    // Requests this wave's share of tile `tile` into `stage`.  Rows past the end
    // of the sequence are clamped to the last one: such keys are invisible to
    // every stored query, the data only has to be finite.
    auto request_tile = [&](int tile, int stage) {
        const int key0 = tile * BN;
        const int row_limit = S - 1 - key0;
        const unsigned char* k_tile = k_base + (size_t)key0 * k_stride_bytes;
        const unsigned char* v_tile = v_base + (size_t)key0 * v_stride_bytes;
        const unsigned stage_base = lds_base + stage * C::STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < C::K_LOADS_PER_WAVE; ++i) {
            const int load = wave * C::K_LOADS_PER_WAVE + i;
            const int slot = 64 * load + lane;
            const int row = slot / C::K_CHUNKS;
            const int chunk = (slot % C::K_CHUNKS) ^ C::k_swizzle(row);
            const unsigned offset = (unsigned)min(row, row_limit) * k_stride_bytes + 16u * chunk;
            direct_load_16_offset(k_tile, offset, stage_base + load * 1024);
        }
#pragma unroll
        for (int i = 0; i < C::V_LOADS_PER_WAVE; ++i) {
            const int load = wave * C::V_LOADS_PER_WAVE + i;
            const int slot = 64 * load + lane;
            const int row = slot / C::V_CHUNKS;
            const int chunk = (slot % C::V_CHUNKS) ^ (C::v_flip(row) << 2);
            const unsigned offset = (unsigned)min(row, row_limit) * v_stride_bytes + 16u * chunk;
            direct_load_16_offset(v_tile, offset, stage_base + C::K_BYTES + load * 1024);
        }
    };

    f32x16 o_acc[DBLOCKS];
#pragma unroll
    for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o_acc[d][i] = 0.f;
    }
    float row_max = -INFINITY;  // reference point of the exponent, raw score units
    float row_sum = 0.f;        // this lane's share (its 32 keys per tile) of the normaliser
    const float c = scale * LOG2E;

    // Per-lane pieces of the LDS read addresses.
    const int k_swz = C::k_swizzle(lq);                        // rows lq and lq+32 share it
    const int s16 = lane % 16;
    const int v_row = 4 * g + s16 / 4;                          // + 16*n, + 8 for the second read
    const int v_in_group = 32 * ((lane / 16) % 2) + 8 * (s16 % 4);
    const int v_flip = C::v_flip(v_row);                        // rows v_row + 8*m share it

    wait_vector_memory<0>();   // the query loads: no wait for them may remain inside the loop
    request_tile(0, 0);

    for (int tile = 0; tile < tiles; ++tile) {
        const int stage = tile & 1;
        wait_vector_memory<0>();   // this wave's share of the tile has landed
        workgroup_barrier();       // ... and everybody's; every wave has left the previous tile
        if (tile + 1 < tiles) {
            request_tile(tile + 1, stage ^ 1);
        }
        const int key0 = tile * BN;
        if (key0 <= wave_q0 + 31) {  // otherwise every key of the tile is in this wave's future
            const unsigned char* k_lds = lds + stage * C::STAGE_BYTES;
            const unsigned char* v_lds = k_lds + C::K_BYTES;

            f32x16 s_acc[2];
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s_acc[mb][i] = 0.f;
            }
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
                const int position = (2 * ks + g) ^ k_swz;
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const bf16x8 a =
                        *reinterpret_cast<const bf16x8*>(k_lds + (32 * mb + lq) * C::K_ROW + 16 * position);
                    s_acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[ks], s_acc[mb], 0, 0, 0);
                }
            }

            if (key0 + BN - 1 > wave_q0) {  // tile crosses this wave's diagonal
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int k = key0 + 32 * mb + 8 * (i / 4) + 4 * g + (i % 4);
                        if (k > q_row) s_acc[mb][i] = -INFINITY;
                    }
                }
            }

            float tile_max = s_acc[0][0];
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                for (int i = 0; i < 16; ++i) tile_max = fmaxf(tile_max, s_acc[mb][i]);
            }
            tile_max = half_wave_max(tile_max);

            // The reference point only moves when some row's maximum grew by
            // more than 2^8 in the exponent; until then probabilities may
            // exceed one, which fp32 sums and bf16 operands hold without loss.
            const float new_max = fmaxf(row_max, tile_max);
            const bool grew = (new_max - row_max) * c > 8.0f;
            if (__any(grew)) {
                const float alpha = __builtin_amdgcn_exp2f((row_max - new_max) * c);
                row_max = new_max;
                row_sum *= alpha;
#pragma unroll
                for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) o_acc[d][i] *= alpha;
                }
            }

            const float offset = row_max * c;
            bf16x8 pf[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                u32x4 packed;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int i = 8 * (n % 2) + 2 * j;
                    const float p0 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i], c, -offset));
                    const float p1 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i + 1], c, -offset));
                    row_sum += p0 + p1;
                    packed[j] = pack_bf16(p0, p1);
                }
                pf[n] = __builtin_bit_cast(bf16x8, packed);
            }

            // V^T operand through transposing reads.  In a block of 16 lanes, lane s
            // points at key row 16n + 4g + s/4 (+8 for the second read) and columns
            // 4*(s%4)..+3 of the 16-column half (block%2) of column group d; the
            // instruction hands lane i column i of the four rows.  Together: MFMA row
            // lane%32, keys {4g..4g+3, 8+4g..8+4g+3} of the 16-key step, the k-order
            // P^T carries from the C layout.
#pragma unroll
            for (int n = 0; n < 4; ++n) {
#pragma unroll
                for (int d = 0; d < DBLOCKS; ++d) {
                    const unsigned char* first =
                        v_lds + (16 * n + v_row) * C::V_ROW + 64 * (d ^ v_flip) + v_in_group;
                    const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)first);
                    const s16x4 high =
                        __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(first + 8 * C::V_ROW));
                    const s16x8 both = __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7);
                    o_acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, both), pf[n],
                                                                       o_acc[d], 0, 0, 0);
                }
            }
        }
    }

    // ---- epilogue: normalise, stage O through LDS for 16-byte row stores
    workgroup_barrier();   // every wave is done reading the tile stages
    const float total = half_wave_sum(row_sum);
    const float inverse = 1.0f / total;
    if (g == 0 && q_row < S) {
        logsumexp[((size_t)b * query_heads + h) * S + q_row] = row_max * scale + __logf(total);
    }
    unsigned char* o_lds = lds + (32 * wave) * C::O_PITCH;
#pragma unroll
    for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            u32x2 packed;
            packed.x = pack_bf16(o_acc[d][4 * i4 + 0] * inverse, o_acc[d][4 * i4 + 1] * inverse);
            packed.y = pack_bf16(o_acc[d][4 * i4 + 2] * inverse, o_acc[d][4 * i4 + 3] * inverse);
            const int dv = 32 * d + 8 * i4 + 4 * g;
            *reinterpret_cast<u32x2*>(o_lds + lq * C::O_PITCH + 2 * dv) = packed;
        }
    }
    __syncthreads();
    constexpr int ROW_CHUNKS = DV / 8;          // 16-byte chunks per output row
    constexpr int ROWS_PER_PASS = 64 / ROW_CHUNKS;
    const size_t o_stride = (size_t)query_heads * DV;
    bf16_t* o_base = output + ((size_t)b * S * query_heads + h) * DV;
#pragma unroll
    for (int pass = 0; pass < 32 / ROWS_PER_PASS; ++pass) {
        const int row = pass * ROWS_PER_PASS + lane / ROW_CHUNKS;
        const int chunk = lane % ROW_CHUNKS;
        const int q = wave_q0 + row;
        if (q < S) {
            const u32x4 bits = *reinterpret_cast<const u32x4*>(o_lds + row * C::O_PITCH + 16 * chunk);
            *reinterpret_cast<u32x4*>(o_base + (size_t)q * o_stride + 8 * chunk) = bits;
        }
    }
}

// ---------------------------------------------------------------------------
// Split-key variant for short and medium problems.
//
// A workgroup of eight waves (two per SIMD) takes 32 * QG queries and walks the keys in tiles of 128; the eight waves
// are QG query groups x KG key groups, a wave holds 32 queries and TILE / KG keys of every tile, with softmax statistics
// and output sums of its own.  After the last tile the KG parts of a query meet in LDS: every wave hands the column
// blocks it does not own to their owners, which scale the parts to the common maximum and add them up.
// The walk of a workgroup is half (KG = 2) or a quarter (KG = 4) as many dependent rounds of scores, softmax and
// output products as with one wave for all keys, and the two waves of a SIMD cover each other's latencies.
// Queries arrive as a tile of their own (whole rows, then operand reads from LDS): loaded by the lanes that need them,
// 16 bytes of 32 different rows per instruction and once per key group, they took longer than a tile of keys.
//
// What bounds it: a step of 128 queries and 128 keys (head size 128, stamps) takes 4000 cycles -- requests 600 to 850 (64
// pieces of 1 KB at the 13 cycles the address unit takes for one), scores 1150 and output products 1170 for the two
// waves of a SIMD (1024 of matrix time each), softmax 250 to 550, barrier -- and start and end of a workgroup some 8000.
// Moving the requests into the product streams, setting the waves of a SIMD half a step apart, leaving the requests to
// four of the waves, touching the keys ahead of time for the L2: each within 5 % of this order, or slower.
// With one wave for all keys (128 queries, four waves) before: 8 heads of 512 tokens, 64 columns 12.0 -> 7.3 us; 32 x 8
// heads of 2048 tokens, 128 columns 58 -> 41 us (830 TFLOP/s); 16 heads of 1000 tokens, 192 / 128 columns 31 -> 16 us.
template <int DQK, int DV, int QG, int KG>
struct SplitConfig {
    static constexpr int TILE = 128;
    static constexpr int WAVES = QG * KG;
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int BN = TILE / KG;                   // keys per wave and tile
    static constexpr int BM = 32 * QG;
    static constexpr int K_ROW = DQK * 2;                  // bytes
    static constexpr int K_BYTES = TILE * K_ROW;
    static constexpr int V_ROW = DV * 2;
    static constexpr int V_BYTES = TILE * V_ROW;
    static constexpr int STAGE_BYTES = K_BYTES + V_BYTES;
    static constexpr int DBLOCKS = DV / 32;
    // after the walk: parts on their way to their owners (4 KB per 32 x 32 block), statistics, output rows
    static constexpr int PART_BYTES = QG * DBLOCKS * (KG - 1) * 4096;
    static constexpr int MAX_AT = PART_BYTES;              // [KG][BM]
    static constexpr int SUM_AT = MAX_AT + KG * BM * 4;    // [KG][BM]
    static constexpr int O_AT = SUM_AT + KG * BM * 4;
    static constexpr int O_PITCH = DV * 2 + 16;
    static constexpr int MERGE_BYTES = O_AT + BM * O_PITCH;
    static constexpr int LDS_BYTES = 2 * STAGE_BYTES > MERGE_BYTES ? 2 * STAGE_BYTES : MERGE_BYTES;
    static_assert(WAVES == 8 && BN % 32 == 0 && BM <= TILE && LDS_BYTES <= 160 * 1024, "");

    __device__ static constexpr int owner(int block) { return block * KG / DBLOCKS; }
};

template <int DQK, int DV, int QG, int KG>
__global__ __launch_bounds__(64 * QG * KG) void attention_forward_split_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp,
    const bf16_t* __restrict__ query, const bf16_t* __restrict__ key, const bf16_t* __restrict__ value,
    int sequence_length, int query_heads, int key_value_heads, index_math::SplitOrder order, float scale) {
    using C = SplitConfig<DQK, DV, QG, KG>;
    using KReads = TileReads<C::K_ROW>;
    using VReads = TileReads<C::V_ROW>;
    constexpr int BN = C::BN;
    constexpr int MB = BN / 32;
    constexpr int KSTEPS = DQK / 16;
    constexpr int NSTEPS = BN / 16;
    constexpr int DBLOCKS = C::DBLOCKS;
    constexpr int QK_MFMAS = MB * KSTEPS;
    constexpr int PV_MFMAS = NSTEPS * DBLOCKS;
    constexpr int RING = QK_MFMAS >= 8 ? 8 : 4;            // fragments read ahead of the product that takes them

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int query_group = wave % QG;
    const int key_group = wave / QG;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;

    const index_math::SplitItem item = index_math::split_item(blockIdx.x, order);
    if (item.batch >= order.batch) return;   // a slot of the last turn without a head
    const int h = item.head;
    const int qb = item.query_block;
    const int b = item.batch;
    const int hk = item.key_value_head;
    const int S = sequence_length;

    const int q0 = qb * C::BM;
    const int wave_q0 = q0 + 32 * query_group;
    const int q_row = wave_q0 + lq;
    const unsigned k_stride_bytes = (unsigned)key_value_heads * DQK * 2;
    const unsigned v_stride_bytes = (unsigned)key_value_heads * DV * 2;
    const unsigned char* k_base =
        reinterpret_cast<const unsigned char*>(key + ((size_t)b * S * key_value_heads + hk) * DQK);
    const unsigned char* v_base =
        reinterpret_cast<const unsigned char*>(value + ((size_t)b * S * key_value_heads + hk) * DV);
    const unsigned lds_base = lds_offset_of(lds);

    // Rows past the end of the sequence repeat the last one: such keys are invisible to every stored query.
    TileRequests<C::K_ROW, C::WAVES, C::TILE> k_requests;
    TileRequests<C::V_ROW, C::WAVES, C::TILE> v_requests;
    k_requests.init(k_stride_bytes, wave, lane);
    v_requests.init(v_stride_bytes, wave, lane);
    auto request_tile = [&](int tile) {
        const int key0 = tile * C::TILE;
        const unsigned target = lds_base + (tile & 1) * C::STAGE_BYTES;
        k_requests.request(k_base + (size_t)key0 * k_stride_bytes, k_stride_bytes, S - 1 - key0, target, wave);
        v_requests.request(v_base + (size_t)key0 * v_stride_bytes, v_stride_bytes, S - 1 - key0, target + C::K_BYTES, wave);
    };

    KReads k_reads;
    VReads v_reads;
    k_reads.init(lane);
    v_reads.init(lane);

    // The queries go where tile 1 will go, tile 0 to its own stage.
    bf16x8 qf[KSTEPS];   // B operand: column = query lq, k = 16*ks + 8*g + j
    {
        using Requests = TileRequests<C::K_ROW, C::WAVES, C::BM>;
        const unsigned char* q_base = reinterpret_cast<const unsigned char*>(query + (((size_t)b * S + q0) * query_heads + h) * DQK);
        if ((unsigned)query_heads <= 0xffffffffu / (C::BM * C::K_ROW)) {
            const unsigned q_stride_bytes = (unsigned)query_heads * DQK * 2;
            Requests q_requests;
            q_requests.init(q_stride_bytes, wave, lane);
            q_requests.request(q_base, q_stride_bytes, S - 1 - q0, lds_base + C::STAGE_BYTES, wave);
        } else {   // rows of one tile more than 4 GiB apart
            Requests::request_far(q_base, (size_t)query_heads * DQK * 2, S - 1 - q0, lds_base + C::STAGE_BYTES, wave);
        }
        request_tile(0);
        wait_vector_memory<TileRequests<C::K_ROW, C::WAVES, C::TILE>::LOADS + TileRequests<C::V_ROW, C::WAVES, C::TILE>::LOADS>();
        workgroup_barrier();   // the query tile has landed
        unsigned q_at[KReads::NAT];
        rebase(q_at, k_reads.natural, C::STAGE_BYTES + query_group * 32 * C::K_ROW);
        unrolled<0, KSTEPS>([&](auto tag) { qf[decltype(tag)::value] = natural_fragment<C::K_ROW, 0, decltype(tag)::value>(lds, q_at); });
    }

    f32x16 o_acc[DBLOCKS];
#pragma unroll
    for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o_acc[d][i] = 0.f;
    }
    // Reference point of the exponent, raw score units.  Parts and query groups start at multiples of 32, so a part that
    // is walked shows every row a key and leaves a number here; -inf stays only with a key group that walked none.
    float row_max = -INFINITY;
    float row_sum = 0.f;       // this lane's share of the normaliser
    const float c = scale * LOG2E;

    const int tiles = (min(S, q0 + C::BM) - 1) / C::TILE + 1;
    for (int tile = 0; tile < tiles; ++tile) {
        wait_vector_memory<0>();   // this wave's share of the tile has landed
        workgroup_barrier();       // ... and everybody's; every wave has left the previous tile (or its queries)
        if (tile + 1 < tiles) request_tile(tile + 1);
        const int key0 = tile * C::TILE + key_group * BN;
        if (key0 > wave_q0 + 31) continue;   // every key of this wave's part is in its queries' future

        const unsigned stage = (tile & 1) * C::STAGE_BYTES;
        unsigned k_at[KReads::NAT], v_at[2][VReads::TR];
        rebase(k_at, k_reads.natural, stage + key_group * BN * C::K_ROW);
        rebase(v_at, v_reads.transposed, stage + C::K_BYTES + key_group * BN * C::V_ROW);
        // fragment I of the stream: k-step I / MB of key block I % MB, then 16-key step and column block of V
        auto fragment = [&](auto tag) -> bf16x8 {
            constexpr int I = decltype(tag)::value;
            if constexpr (I < QK_MFMAS) {
                return natural_fragment<C::K_ROW, 32 * (I % MB), I / MB>(lds, k_at);
            } else {
                constexpr int J = I - QK_MFMAS;
                return transposed_fragment<C::V_ROW, 16 * (J / DBLOCKS), J % DBLOCKS>(lds, v_at);
            }
        };

        f32x16 s_acc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s_acc[mb][i] = 0.f;
        }
        bf16x8 ring[RING];
        static_assert(QK_MFMAS >= RING && PV_MFMAS >= RING, "the first V fragments are read behind the last K fragments");
        unrolled<0, RING>([&](auto tag) { ring[decltype(tag)::value] = fragment(tag); });
        unrolled<0, QK_MFMAS>([&](auto tag) {
            constexpr int I = decltype(tag)::value;
            s_acc[I % MB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[I % RING], qf[I / MB], s_acc[I % MB], 0, 0, 0);
            ring[I % RING] = fragment(std::integral_constant<int, I + RING>{});
            __builtin_amdgcn_sched_barrier(0);
        });

        if (key0 + BN - 1 > wave_q0) {  // the part reaches past this wave's first query
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int k = key0 + 32 * mb + 8 * (i / 4) + 4 * g + (i % 4);
                    if (k > q_row) s_acc[mb][i] = -INFINITY;
                }
            }
        }
        float tile_max = s_acc[0][0];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) tile_max = fmaxf(tile_max, s_acc[mb][i]);
        }
        tile_max = half_wave_max(tile_max);
        // The reference point only moves when some row's maximum grew by more than 2^8 in the exponent.
        const float new_max = fmaxf(row_max, tile_max);
        const bool grew = (new_max - row_max) * c > 8.0f;
        if (__any(grew)) {
            const float alpha = __builtin_amdgcn_exp2f((row_max - new_max) * c);
            row_max = new_max;
            row_sum *= alpha;
#pragma unroll
            for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
                for (int i = 0; i < 16; ++i) o_acc[d][i] *= alpha;
            }
        }
        const float offset = row_max * c;
        bf16x8 pf[NSTEPS];
#pragma unroll
        for (int n = 0; n < NSTEPS; ++n) {
            u32x4 packed;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = 8 * (n % 2) + 2 * j;
                const float p0 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i], c, -offset));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i + 1], c, -offset));
                row_sum += p0 + p1;
                packed[j] = pack_bf16(p0, p1);
            }
            pf[n] = __builtin_bit_cast(bf16x8, packed);
        }
        unrolled<QK_MFMAS, QK_MFMAS + PV_MFMAS>([&](auto tag) {
            constexpr int I = decltype(tag)::value;
            constexpr int J = I - QK_MFMAS;
            o_acc[J % DBLOCKS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[I % RING], pf[J / DBLOCKS], o_acc[J % DBLOCKS], 0, 0, 0);
            if constexpr (I + RING < QK_MFMAS + PV_MFMAS) ring[I % RING] = fragment(std::integral_constant<int, I + RING>{});
            __builtin_amdgcn_sched_barrier(0);
        });
    }

    // ---- the KG parts of a query: statistics and foreign blocks into LDS, then every owner puts its blocks together
    float* maxima = reinterpret_cast<float*>(lds + C::MAX_AT);
    float* sums = reinterpret_cast<float*>(lds + C::SUM_AT);
    const int q_local = 32 * query_group + lq;
    // part of a block: 16-byte pieces [i4][lane] as the registers hold them
    auto part_of = [&](int block, int from) {
        const int index = from < C::owner(block) ? from : from - 1;
        return lds + ((query_group * DBLOCKS + block) * (KG - 1) + index) * 4096 + 16 * lane;
    };
    row_sum = half_wave_sum(row_sum);
    workgroup_barrier();   // every wave is done with the tile stages
    if (g == 0) {
        maxima[key_group * C::BM + q_local] = row_max;
        sums[key_group * C::BM + q_local] = row_sum;
    }
#pragma unroll
    for (int d = 0; d < DBLOCKS; ++d) {
        if (C::owner(d) != key_group) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                *reinterpret_cast<f32x4*>(part_of(d, key_group) + 1024 * i4) =
                    f32x4{o_acc[d][4 * i4], o_acc[d][4 * i4 + 1], o_acc[d][4 * i4 + 2], o_acc[d][4 * i4 + 3]};
            }
        }
    }
    workgroup_barrier();
    float highest = maxima[q_local];
#pragma unroll
    for (int k = 1; k < KG; ++k) highest = fmaxf(highest, maxima[k * C::BM + q_local]);
    float weight[KG];
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < KG; ++k) {
        weight[k] = __builtin_amdgcn_exp2f((maxima[k * C::BM + q_local] - highest) * c);
        total = fmaf(sums[k * C::BM + q_local], weight[k], total);
    }
    if (key_group == 0 && g == 0 && q_row < S) {
        logsumexp[((size_t)b * query_heads + h) * S + q_row] = highest * scale + __logf(total);
    }
    const float inverse = 1.0f / total;
#pragma unroll
    for (int k = 0; k < KG; ++k) weight[k] *= inverse;
#pragma unroll
    for (int d = 0; d < DBLOCKS; ++d) {
        if (C::owner(d) == key_group) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                f32x4 sum;
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[j] = o_acc[d][4 * i4 + j] * weight[C::owner(d)];
#pragma unroll
                for (int k = 0; k < KG; ++k) {
                    if (k == C::owner(d)) continue;
                    const f32x4 part = *reinterpret_cast<const f32x4*>(part_of(d, k) + 1024 * i4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum[j] = fmaf(part[j], weight[k], sum[j]);
                }
                const u32x2 packed = {pack_bf16(sum[0], sum[1]), pack_bf16(sum[2], sum[3])};
                *reinterpret_cast<u32x2*>(lds + C::O_AT + q_local * C::O_PITCH + 2 * (32 * d + 8 * i4 + 4 * g)) = packed;
            }
        }
    }
    workgroup_barrier();
    constexpr int ROW_CHUNKS = DV / 8;          // 16-byte chunks per output row
    const size_t o_stride = (size_t)query_heads * DV;
    bf16_t* o_base = output + ((size_t)b * S * query_heads + h) * DV;
#pragma unroll
    for (int pass = 0; pass < C::BM * ROW_CHUNKS / C::THREADS; ++pass) {
        const int piece = pass * C::THREADS + tid;
        const int row = piece / ROW_CHUNKS;
        const int chunk = piece % ROW_CHUNKS;
        if (q0 + row < S) {
            *reinterpret_cast<u32x4*>(o_base + (size_t)(q0 + row) * o_stride + 8 * chunk) =
                *reinterpret_cast<const u32x4*>(lds + C::O_AT + row * C::O_PITCH + 16 * chunk);
        }
    }
}

// ---------------------------------------------------------------------------
// Persistent two-phase ("ping-pong") variant for long sequences.
//
// One workgroup of 8 waves (2 per SIMD) per compute unit walks a list of work
// items, an item being one block of 256 queries of one (batch, head).
//
// Phases.  A SIMD's matrix pipeline idles while its waves run the softmax, and
// with one barrier per tile both waves of a SIMD run it at the same time.  Here
// every wave alternates between two phases that end in a workgroup barrier:
//     X(j): request later tiles, softmax of S(j) -> P(j)          (VALU, exp)
//     Y(j): O += V(j)^T P(j), then S(j+1) = K(j+1) Q^T            (MFMA, LDS reads)
// Waves 4..7 run one extra barrier before their first phase, so they are in X
// while waves 0..3 (the other wave of each SIMD) are in Y and the reverse: the
// matrix pipeline always has a wave feeding it.  Y raises its wave priority.
//
// Y is one stream of MFMAs (PV then QK), each with one A fragment from LDS.
// Fragments go through a ring of RING register sets that runs RING MFMAs ahead
// of their use; the first RING fragments (of V(j)) are read at the end of X(j),
// before the barrier, so that Y starts with its operands in registers.
//
// Tiles.  K tiles sit in a ring of three slots, V tiles in a ring of four, and
// the tiles of all items of a workgroup form one stream: a wave requests stream
// tile t+2 during X of stream tile t, whether it belongs to this item or to the
// next one, and waits for its own requests at the end of that tile's Y; the
// barrier that ends Y of the later group publishes them.  K(t+2) is first read
// in Y(t+1), V(t+2) at the end of X(t+2); the slots they overwrite (K(t-1),
// V(t-2)) were last read in Y(t-2).  So a new item finds its first two tiles in
// LDS; what stays exposed at an item switch is the load of the new queries.
//
// Work order.  Workgroup w belongs to cluster w % 8 (workgroups are dealt
// round-robin to the 8 XCDs, each with its own L2) and the (batch, head) pairs
// are dealt to the clusters the same way.  Inside a cluster the items are laid
// out `abreast` heads at a time (index_math::forward_choice: two where that comes
// out even), blocks from the heaviest (last) to the lightest, and cut into rounds
// of one item per workgroup; odd rounds are handed out in reverse, so a
// workgroup's heavy and light blocks add up to the same total while the cluster
// works on few heads at any time.
struct PingPong {
    static constexpr int K_SLOTS = 3;
    static constexpr int V_SLOTS = 4;
    static constexpr int RING = 8;
    static constexpr int CLUSTERS = 8;
    // Output rows leave through LDS, half a row (64 columns, one 128-byte line) at a time: 32 rows of
    // 128 + 16 bytes per wave, for the four waves of one group (the two groups store in different phases).
    static constexpr int O_HALF_COLUMNS = 64;
    static constexpr int O_PITCH = O_HALF_COLUMNS * 2 + 16;
    static constexpr int O_WAVE_BYTES = 32 * O_PITCH;
    static constexpr int O_BYTES = 4 * O_WAVE_BYTES;
};

using index_math::forward_item;
using index_math::ForwardItem;

template <int DQK, int DV>
__global__ __launch_bounds__(512) void attention_forward_pingpong_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp,
    const bf16_t* __restrict__ query, const bf16_t* __restrict__ key, const bf16_t* __restrict__ value,
    int sequence_length, int query_heads, int key_value_heads, int query_blocks, int batch_heads, int clusters,
    int abreast, float scale) {
    using C = FwdConfig<DQK, DV, 8>;
    constexpr int BN = C::BN;
    constexpr int KSTEPS = DQK / 16;
    constexpr int DBLOCKS = DV / 32;
    constexpr int SPAN = (C::K_ROW % 256 == 0) ? 16 : 8;   // chunk positions the K swizzle permutes
    constexpr int KLOW = SPAN / 2;                          // k-steps with distinct swizzled addresses
    constexpr int V_RING = PingPong::K_SLOTS * C::K_BYTES;  // byte offset of the V slots
    constexpr int O_STAGE = V_RING + PingPong::V_SLOTS * C::V_BYTES;   // byte offset of the output staging rows
    static_assert(DV % PingPong::O_HALF_COLUMNS == 0, "output rows leave in halves of 64 columns");
    constexpr int RING = PingPong::RING;
    constexpr int PV_MFMAS = 4 * DBLOCKS;
    constexpr int QK_MFMAS = 2 * KSTEPS;
    constexpr int REQUESTS = C::K_LOADS_PER_WAVE + C::V_LOADS_PER_WAVE;
    static_assert(REQUESTS <= 5, "X issues five tile requests");
    static_assert(PV_MFMAS >= RING, "the fragments read ahead in X must all belong to V");

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int group = wave / 4;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int S = sequence_length;

    __builtin_assume(abreast > 0);
    const int cluster = blockIdx.x % clusters;
    const int member = blockIdx.x / clusters;
    const int members = gridDim.x / clusters;
    const int cluster_heads = batch_heads / clusters;

    const size_t q_stride = (size_t)query_heads * DQK;
    const size_t o_stride = (size_t)query_heads * DV;
    const unsigned k_stride_bytes = (unsigned)key_value_heads * DQK * 2;
    const unsigned v_stride_bytes = (unsigned)key_value_heads * DV * 2;
    const unsigned lds_base = lds_offset_of(lds);

    // operands of an item
    auto key_base = [&](const ForwardItem& item) {
        const int b = item.batch_head / query_heads;
        const int hk = (item.batch_head % query_heads) / (query_heads / key_value_heads);
        return reinterpret_cast<const unsigned char*>(key + ((size_t)b * S * key_value_heads + hk) * DQK);
    };
    auto value_base = [&](const ForwardItem& item) {
        const int b = item.batch_head / query_heads;
        const int hk = (item.batch_head % query_heads) / (query_heads / key_value_heads);
        return reinterpret_cast<const unsigned char*>(value + ((size_t)b * S * key_value_heads + hk) * DV);
    };
    auto tile_count = [&](const ForwardItem& item) { return (min(S, (item.query_block + 1) * C::BM) - 1) / BN + 1; };

    // One 1 KB piece (index `part` of this wave's share) of the K and V tiles that
    // start at key `key0` of the head at (k_head, v_head): parts below
    // K_LOADS_PER_WAVE belong to K, the rest to V.  Rows past the end of the
    // sequence are clamped to the last one: such keys are invisible to every
    // stored query, the data only has to be finite.
    auto request_part = [&](const unsigned char* k_head, const unsigned char* v_head, int key0, int k_slot,
                            int v_slot, int part) {
        const int row_limit = S - 1 - key0;
        if (part < C::K_LOADS_PER_WAVE) {
            const unsigned char* k_tile = k_head + (size_t)key0 * k_stride_bytes;
            const int load = wave * C::K_LOADS_PER_WAVE + part;
            const int position = 64 * load + lane;
            const int row = position / C::K_CHUNKS;
            const int chunk = (position % C::K_CHUNKS) ^ C::k_swizzle(row);
            const unsigned offset = (unsigned)min(row, row_limit) * k_stride_bytes + 16u * chunk;
            direct_load_16_offset(k_tile, offset, lds_base + k_slot * C::K_BYTES + load * 1024);
        } else {
            const unsigned char* v_tile = v_head + (size_t)key0 * v_stride_bytes;
            const int load = wave * C::V_LOADS_PER_WAVE + (part - C::K_LOADS_PER_WAVE);
            const int position = 64 * load + lane;
            const int row = position / C::V_CHUNKS;
            const int chunk = (position % C::V_CHUNKS) ^ (C::v_flip(row) << 2);
            const unsigned offset = (unsigned)min(row, row_limit) * v_stride_bytes + 16u * chunk;
            direct_load_16_offset(v_tile, offset, lds_base + V_RING + v_slot * C::V_BYTES + load * 1024);
        }
    };

    // Per-lane byte offsets of the fragment reads inside a slot.  K: chunk
    // 2*ks + g of row lq sits at position (2*ks + g) ^ swizzle; the XOR only
    // touches the low bits, so KLOW addresses plus immediates cover all k-steps.
    unsigned k_read[KLOW];
    {
        const int t = g ^ C::k_swizzle(lq);
#pragma unroll
        for (int i = 0; i < KLOW; ++i) k_read[i] = lq * C::K_ROW + 16 * ((2 * i) ^ t);
    }
    unsigned v_read[DBLOCKS];
    {
        const int s16 = lane % 16;
        const int v_row = 4 * g + s16 / 4;
        const int in_group = 32 * ((lane / 16) % 2) + 8 * (s16 % 4);
#pragma unroll
        for (int d = 0; d < DBLOCKS; ++d) v_read[d] = v_row * C::V_ROW + 64 * (d ^ C::v_flip(v_row)) + in_group;
    }
    auto k_fragment = [&](const unsigned char* k_tile, int ks, int mb) -> bf16x8 {
        return *reinterpret_cast<const bf16x8*>(k_tile + k_read[ks % KLOW] + (ks / KLOW) * (SPAN * 16) +
                                                mb * 32 * C::K_ROW);
    };
    auto v_fragment = [&](const unsigned char* v_tile, int n, int d) -> bf16x8 {
        const unsigned char* first = v_tile + v_read[d] + n * 16 * C::V_ROW;
        const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)first);
        const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(first + 8 * C::V_ROW));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // fragment i of the Y stream: PV_MFMAS fragments of V (16-key step i / DBLOCKS,
    // column block i % DBLOCKS), then QK_MFMAS fragments of K (k-step, key half)
    auto stream_fragment = [&](const unsigned char* v_tile, const unsigned char* k_tile, int i) -> bf16x8 {
        if (i < PV_MFMAS) {
            return v_fragment(v_tile, i / DBLOCKS, i % DBLOCKS);
        }
        return k_fragment(k_tile, (i - PV_MFMAS) / 2, (i - PV_MFMAS) % 2);
    };

    bf16x8 qf[KSTEPS];
    f32x16 o_acc[DBLOCKS];
    f32x16 s_acc[2];
    bf16x8 pf[4];
    bf16x8 ring[RING];
    float row_max, row_sum;
    const float c = scale * LOG2E;
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // Q fragments of an item (B operand: column = query lq, k = 16*ks + 8*g + j)
    auto load_queries = [&](const ForwardItem& item) {
        const int row_index = item.query_block * C::BM + 32 * wave + lq;
        const bool valid = row_index < S;
        const int b = item.batch_head / query_heads;
        const int h = item.batch_head % query_heads;
        const bf16_t* row = query + ((size_t)b * S * query_heads + h) * DQK + (size_t)(valid ? row_index : 0) * q_stride + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            u32x4 bits = {0, 0, 0, 0};
            if (valid) {
                bits = *reinterpret_cast<const u32x4*>(row + 16 * ks);
            }
            qf[ks] = __builtin_bit_cast(bf16x8, bits);
        }
    };

    ForwardItem item, next_item;
    if (!forward_item(0, member, members, cluster, clusters, cluster_heads, query_blocks, item, abreast)) {
        return;   // uniform over the workgroup
    }
    bool has_next = forward_item(1, member, members, cluster, clusters, cluster_heads, query_blocks, next_item, abreast);

    // ---- prologue of the first item: its queries and its tiles 0 and 1
    load_queries(item);
    wait_vector_memory<0>();
    {
        const unsigned char* k_head = key_base(item);
        const unsigned char* v_head = value_base(item);
#pragma unroll
        for (int part = 0; part < REQUESTS; ++part) request_part(k_head, v_head, 0, 0, 0, part);
#pragma unroll
        for (int part = 0; part < REQUESTS; ++part) request_part(k_head, v_head, BN, 1, 1, part);
    }
    wait_vector_memory<0>();
    workgroup_barrier();

    int k_slot = 0;     // slot of K of the current stream tile (stream index % 3)
    int v_slot = 0;     // slot of V of the current stream tile (stream index % 4)
    int round = 0;
    bool shifted = false;
    while (true) {
        const int tiles = tile_count(item);
        const int wave_q0 = item.query_block * C::BM + 32 * wave;
        const int q_row = wave_q0 + lq;
        const unsigned char* k_head = key_base(item);
        const unsigned char* v_head = value_base(item);
        const unsigned char* next_k_head = has_next ? key_base(next_item) : k_head;
        const unsigned char* next_v_head = has_next ? value_base(next_item) : v_head;

        // S(0) of the item; its K tile was requested two tiles ago
        {
            const unsigned char* k_tile = lds + k_slot * C::K_BYTES;
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    s_acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_fragment(k_tile, ks, mb), qf[ks],
                                                                        ks == 0 ? zero : s_acc[mb], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o_acc[d][i] = 0.f;
        }
        row_max = -INFINITY;
        row_sum = 0.f;
        if (!shifted) {
            shifted = true;
            if (group == 1) {
                workgroup_barrier();
            }
        }

        // X(tile): the requests for stream tile + 2, then the softmax.
        // A wave whose rows all lie before this tile runs it like any other: the
        // mask turns its scores into zeros, and the phases are barrier-locked, so
        // skipping would not end the tile sooner.  (Branching around the
        // arithmetic of such tiles was tried: the extra control flow made the
        // register allocator spill some 200 registers.)
        auto phase_x = [&](int tile) {
            const int key0 = tile * BN;
            const int k_slot2 = k_slot == 0 ? 2 : k_slot - 1;      // (slot + 2) % 3
            const int v_slot2 = (v_slot + 2) & 3;
            const bool from_next = tile + 2 >= tiles;
            const unsigned char* request_k = from_next ? next_k_head : k_head;
            const unsigned char* request_v = from_next ? next_v_head : v_head;
            const int request_key0 = (from_next ? tile + 2 - tiles : tile + 2) * BN;
            auto request_next = [&](int part) {
                if (part < REQUESTS) {
                    request_part(request_k, request_v, request_key0, k_slot2, v_slot2, part);
                }
            };
            // all of this wave's requests first: they have the whole phase and the next to arrive
            request_next(0);
            request_next(1);
            request_next(2);
            request_next(3);
            request_next(4);
            if (key0 + BN - 1 > wave_q0) {  // tile reaches past this wave's first row
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int k = key0 + 32 * mb + 8 * (i / 4) + 4 * g + (i % 4);
                        if (k > q_row) s_acc[mb][i] = -INFINITY;
                    }
                }
            }
            float tile_max = s_acc[0][0];
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                for (int i = 0; i < 16; ++i) tile_max = fmaxf(tile_max, s_acc[mb][i]);
            }
            tile_max = half_wave_max(tile_max);
            // The reference point only moves when some row's maximum grew by
            // more than 2^8 in the exponent; until then probabilities may
            // exceed one, which fp32 sums and bf16 operands hold without loss.
            const float new_max = fmaxf(row_max, tile_max);
            const bool grew = (new_max - row_max) * c > 8.0f;
            if (__any(grew)) {
                const float alpha = __builtin_amdgcn_exp2f((row_max - new_max) * c);
                row_max = new_max;
                row_sum *= alpha;
#pragma unroll
                for (int d = 0; d < DBLOCKS; ++d) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) o_acc[d][i] *= alpha;
                }
            }
            const float offset = row_max * c;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                u32x4 packed;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int i = 8 * (n % 2) + 2 * j;
                    const float p0 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i], c, -offset));
                    const float p1 = __builtin_amdgcn_exp2f(fmaf(s_acc[n / 2][i + 1], c, -offset));
                    row_sum += p0 + p1;   // unrounded: the logsumexp tolerance leaves no room for bf16 sums
                    packed[j] = pack_bf16(p0, p1);
                }
                pf[n] = __builtin_bit_cast(bf16x8, packed);
            }
        };
        // Y(tile): O += V^T P, and with FULL the next S.  The first RING fragments
        // are read before the barrier that separates X from Y.
        auto phase_y = [&](auto full_tag) {
            constexpr bool FULL = decltype(full_tag)::value;
            constexpr int COUNT = FULL ? PV_MFMAS + QK_MFMAS : PV_MFMAS;
            const int k_slot1 = k_slot == 2 ? 0 : k_slot + 1;
            const unsigned char* k_tile = lds + k_slot1 * C::K_BYTES;           // K(tile + 1)
            const unsigned char* v_tile = lds + V_RING + v_slot * C::V_BYTES;   // V(tile)
#pragma unroll
            for (int i = 0; i < RING; ++i) ring[i] = stream_fragment(v_tile, k_tile, i);
            workgroup_barrier();
            __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int i = 0; i < COUNT; ++i) {
                if (i < PV_MFMAS) {
                    o_acc[i % DBLOCKS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i % RING], pf[i / DBLOCKS],
                                                                                 o_acc[i % DBLOCKS], 0, 0, 0);
                } else {
                    const int ks = (i - PV_MFMAS) / 2;
                    const int mb = (i - PV_MFMAS) % 2;
                    s_acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i % RING], qf[ks],
                                                                        ks == 0 ? zero : s_acc[mb], 0, 0, 0);
                }
                if (i + RING < COUNT) {
                    ring[i % RING] = stream_fragment(v_tile, k_tile, i + RING);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            wait_vector_memory<0>();   // this wave's requests of X(tile)
            workgroup_barrier();
            k_slot = k_slot1;
            v_slot = (v_slot + 1) & 3;
        };

        for (int tile = 0; tile + 1 < tiles; ++tile) {
            phase_x(tile);
            phase_y(std::true_type{});
        }
        // Last tile: its scores exist already, so the query registers are free: the next item's queries load
        // while this tile finishes.
        if (has_next) {
            load_queries(next_item);
        }
        phase_x(tiles - 1);
        phase_y(std::false_type{});

        // ---- epilogue: normalise, round, and store rows and logsumexp.  A lane holds, per column block, four
        // runs of four columns of one query; the rows go through this wave's staging rows in LDS, 64 columns
        // at a time, so that every store instruction writes eight whole 128-byte lines.  Only this wave touches
        // its staging rows; the two groups come through here in different phases and share them.
        {
            const int fresh = fresh_lane_id();   // nothing of the address arithmetic below is carried through the tile loop
            const int row = fresh % 32;
            const int half_wave = fresh / 32;
            const float total = half_wave_sum(row_sum);
            const float inverse = 1.0f / total;
            const int b = item.batch_head / query_heads;
            const int h = item.batch_head % query_heads;
            if (half_wave == 0 && wave_q0 + row < S) {
                logsumexp[((size_t)b * query_heads + h) * S + wave_q0 + row] = row_max * scale + __logf(total);
            }
            bf16_t* o_head = output + ((size_t)b * S * query_heads + h) * DV;
            unsigned char* o_lds = lds + O_STAGE + (wave % 4) * PingPong::O_WAVE_BYTES;
            constexpr int HALVES = DV / PingPong::O_HALF_COLUMNS;
            constexpr int HALF_BLOCKS = PingPong::O_HALF_COLUMNS / 32;
#pragma unroll
            for (int half = 0; half < HALVES; ++half) {
#pragma unroll
                for (int db = 0; db < HALF_BLOCKS; ++db) {
                    const int d = half * HALF_BLOCKS + db;
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        u32x2 packed;
                        packed.x = pack_bf16(o_acc[d][4 * i4 + 0] * inverse, o_acc[d][4 * i4 + 1] * inverse);
                        packed.y = pack_bf16(o_acc[d][4 * i4 + 2] * inverse, o_acc[d][4 * i4 + 3] * inverse);
                        *reinterpret_cast<u32x2*>(o_lds + row * PingPong::O_PITCH + 2 * (32 * db + 8 * i4 + 4 * half_wave)) = packed;
                    }
                }
                __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes have landed
                __builtin_amdgcn_wave_barrier();
                // 32 rows x 128 bytes: eight lanes per row, eight rows per pass
#pragma unroll
                for (int pass = 0; pass < 4; ++pass) {
                    const int r = 8 * pass + fresh / 8;
                    const u32x4 bits = *reinterpret_cast<const u32x4*>(o_lds + r * PingPong::O_PITCH + 16 * (fresh % 8));
                    if (wave_q0 + r < S) {
                        *reinterpret_cast<u32x4*>(o_head + (size_t)(wave_q0 + r) * o_stride +
                                                  half * PingPong::O_HALF_COLUMNS + 8 * (fresh % 8)) = bits;
                    }
                }
                __builtin_amdgcn_wave_barrier();   // the reads above precede the next half's writes
            }
        }
        if (!has_next) {
            break;
        }
        item = next_item;
        ++round;
        has_next = forward_item(round + 1, member, members, cluster, clusters, cluster_heads, query_blocks, next_item, abreast);
    }
    if (group == 0) {
        workgroup_barrier();
    }
}

template <int DQK, int DV>
void launch_forward_four_waves(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* key, const bf16_t* value,
                               int batch_size, int sequence_length, int query_heads, int key_value_heads, float scale,
                               hipStream_t stream) {
    using C = FwdConfig<DQK, DV, 4>;
    const int query_blocks = (sequence_length + C::BM - 1) / C::BM;
    auto kernel = attention_forward_kernel<DQK, DV, 4>;
    if (C::LDS_BYTES > 64 * 1024) {
        static hip_common::OncePerDevice raised;
        raised.run([&] {
            HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES));
        });
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)((long long)batch_size * query_heads * query_blocks)), dim3(C::THREADS),
                       C::LDS_BYTES, stream, output, logsumexp, query, key, value, sequence_length, query_heads,
                       key_value_heads, query_blocks, scale);
    HIP_CHECK(hipGetLastError());
}

template <int DQK, int DV, int QG, int KG>
void launch_forward_split(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* key, const bf16_t* value,
                          int batch_size, int sequence_length, int query_heads, int key_value_heads, float scale,
                          hipStream_t stream) {
    using C = SplitConfig<DQK, DV, QG, KG>;
    const int query_blocks = (sequence_length + C::BM - 1) / C::BM;
    const long long batch_heads = (long long)batch_size * query_heads;
    // 64 columns: for 128 the dispatch below has the persistent kernel there
    const bool spread = DV == 64 && index_math::split_spreads(batch_heads, sequence_length) &&
        (batch_heads + 7) * query_blocks <= 0x7fffffffLL;
    const index_math::SplitOrder order = index_math::split_order(batch_size, query_heads, key_value_heads, query_blocks, spread);
    auto kernel = attention_forward_split_kernel<DQK, DV, QG, KG>;
    static hip_common::OncePerDevice raised;
    raised.run([&] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES));
    });
    hipLaunchKernelGGL(kernel, dim3((unsigned)order.workgroups), dim3(C::THREADS), C::LDS_BYTES, stream, output, logsumexp,
                       query, key, value, sequence_length, query_heads, key_value_heads, order, scale);
    HIP_CHECK(hipGetLastError());
}

// How the persistent kernel would take a problem: its clusters and workgroups, and what index_math::forward_choice
// makes of them.  The choice walks the work list, 1 to 2 ns an item: 0.1 us for 64 heads of 2048 tokens, 14 us for 127 heads
// of 16384, whose call takes 9 ms (36 us with a division per item).  Each thread remembers the eight shapes it asked about
// last: a program that alternates between layers or prompt lengths does not pay on each call.
struct PingPongPlan {
    int clusters;
    int grid;
    index_math::ForwardChoice choice;
};

PingPongPlan pingpong_plan(long long batch_heads, int sequence_length) {
    struct Memory {
        long long batch_heads = 0;
        int sequence_length = 0, compute_units = 0;
        PingPongPlan plan = {};
    };
    constexpr int SHAPES = 8;
    thread_local Memory shapes[SHAPES];
    thread_local int oldest = 0;
    const int compute_units = hip_common::compute_units_of_current_device();
    for (const Memory& known : shapes) {
        if (known.batch_heads == batch_heads && known.sequence_length == sequence_length && known.compute_units == compute_units) {
            return known.plan;
        }
    }
    // one workgroup per compute unit (the LDS footprint admits no second one)
    PingPongPlan plan;
    plan.clusters = (batch_heads % PingPong::CLUSTERS == 0 && compute_units >= PingPong::CLUSTERS) ? PingPong::CLUSTERS : 1;
    const long long query_blocks = (sequence_length + 255) / 256;
    const long long members = std::min<long long>(compute_units / plan.clusters, batch_heads / plan.clusters * query_blocks);
    plan.grid = (int)(members * plan.clusters);
    plan.choice = index_math::forward_choice((int)members, plan.clusters, (int)(batch_heads / plan.clusters), sequence_length);
    shapes[oldest] = Memory{batch_heads, sequence_length, compute_units, plan};
    oldest = (oldest + 1) % SHAPES;
    return plan;
}

template <int DQK, int DV>
void launch_forward_pingpong(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* key,
                             const bf16_t* value, int batch_size, int sequence_length, int query_heads,
                             int key_value_heads, const PingPongPlan& plan, float scale, hipStream_t stream) {
    using C = FwdConfig<DQK, DV, 8>;
    constexpr int LDS_BYTES = PingPong::K_SLOTS * C::K_BYTES + PingPong::V_SLOTS * C::V_BYTES + PingPong::O_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "the tile slots and the output staging rows must fit the LDS");
    const int query_blocks = (sequence_length + C::BM - 1) / C::BM;
    auto kernel = attention_forward_pingpong_kernel<DQK, DV>;
    static hip_common::OncePerDevice raised;
    raised.run([&] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES));
    });
    hipLaunchKernelGGL(kernel, dim3((unsigned)plan.grid), dim3(C::THREADS), LDS_BYTES, stream, output, logsumexp, query,
                       key, value, sequence_length, query_heads, key_value_heads, query_blocks, batch_size * query_heads,
                       plan.clusters, plan.choice.abreast, scale);
    HIP_CHECK(hipGetLastError());
}

}  // namespace

void attention_forward_dispatch(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* key,
                                const bf16_t* value, int batch_size, int sequence_length, int query_heads,
                                int key_value_heads, int qk_head_size, int v_head_size, float scale,
                                hipStream_t stream) {
    // Offsets of the lanes inside a tile of 128 keys are 32-bit; items and workgroups are counted in ints.
    if (2LL * std::max(qk_head_size, v_head_size) * key_value_heads * 64 > 0x7fffffffLL) {
        throw std::invalid_argument("attention forward: key_value_heads * head size is too large");
    }
    const long long batch_heads = (long long)batch_size * query_heads;
    const long long blocks64 = (sequence_length + 63LL) / 64, blocks128 = (sequence_length + 127LL) / 128;
    if (batch_heads * blocks64 > 0x7fffffffLL) {
        throw std::invalid_argument("attention forward: batch*heads*query_blocks exceeds the grid limit");
    }
    const int compute_units = hip_common::compute_units_of_current_device();
#define DSCUDA_FWD_SPLIT(DQK, DV, QG, KG)                                                                          \
    launch_forward_split<DQK, DV, QG, KG>(output, logsumexp, query, key, value, batch_size, sequence_length,       \
                                          query_heads, key_value_heads, scale, stream)
#define DSCUDA_FWD_FOUR_WAVES(DQK, DV)                                                                             \
    launch_forward_four_waves<DQK, DV>(output, logsumexp, query, key, value, batch_size, sequence_length,          \
                                       query_heads, key_value_heads, scale, stream)
#define DSCUDA_FWD_CASE(DQK, DV)                                                                                   \
    if (qk_head_size == DQK && v_head_size == DV) {                                                                \
        if (one_tile) {                                                                                            \
            DSCUDA_FWD_FOUR_WAVES(DQK, DV);                                                                        \
        } else if (persistent) {                                                                                          \
            launch_forward_pingpong<DQK, DV>(output, logsumexp, query, key, value, batch_size, sequence_length,    \
                                             query_heads, key_value_heads, plan, scale, stream);                   \
        } else if (quarters) {                                                                                     \
            DSCUDA_FWD_SPLIT(DQK, DV, 2, 4);                                                                       \
        } else {                                                                                                   \
            DSCUDA_FWD_SPLIT(DQK, DV, 4, 2);                                                                       \
        }                                                                                                          \
        return;                                                                                                    \
    }
    // One tile of keys: the split-key kernel's tiles of 128 keys are half repeated rows, which half a compute unit's worth
    // of heads and more have to wait for (split / four waves: 64 heads 6.3 / 6.4 us, 256 heads 7.1 / 6.3, 512 heads of 192
    // columns 12.6 / 14.6).
    const bool one_tile = sequence_length <= 64 && 2 * batch_heads >= compute_units;
    if (qk_head_size == 64 && v_head_size == 64) {
        // With 64 columns the softmax outweighs the products, and the persistent kernel's phases do not come out even.  Four
        // waves from one and a half heads per compute unit on (split / four waves, of 1024 tokens, in us: 128 heads equal,
        // 256 heads 66.3 / 67.3, 384 heads 4 % less, 512 heads 132 / 121; of 512 tokens: 64 heads 8.0 / 11.9, 256 heads
        // 24.6 / 26.9, 512 heads 46.2 / 43.6), from one head per unit on for long sequences (256 heads of 2048 tokens
        // 213 / 206, of 4608 972 / 931), and at seven eighths to one head per unit where full rounds of workgroups of 64
        // queries (two a unit) are followed by a short one (256 heads of 192 tokens 9.2 / 8.6, of 384 tokens 18.1 / 16.1; of
        // 128 and 448 tokens 3 and 17 % more).
        const bool heads_enough = 2 * batch_heads >= 3LL * compute_units || (batch_heads >= compute_units && sequence_length >= 2048);
        const bool uneven = 8 * batch_heads >= 7LL * compute_units && batch_heads <= compute_units && sequence_length > 128 &&
            sequence_length <= 384;
        if (one_tile || heads_enough || uneven) {
            DSCUDA_FWD_FOUR_WAVES(64, 64);
        } else {
            // 64 queries per workgroup (128: 22.7 against 16.3 us for 8 heads of 2048 tokens, 203 against 205 us for 64
            // heads of 4352)
            DSCUDA_FWD_SPLIT(64, 64, 2, 4);
        }
        return;
    }
    // Persistent kernel or split keys: the tiles of the busiest workgroup against index_math::split_forward_cost.  Measured with either kernel
    // forced, split / persistent in us, 192/128 columns: 16 heads of 1000 tokens 15.5 / 31.6, 128 of 1152 75.6 / 78.3,
    // 32 of 3313 120 / 109, 64 of 2048 97 / 90, 128 of 1700 157 / 144.  Where the two costs are within 5 %: 16 of 6573
    // 232 / 217, 40 of 5137 352 / 334, 32 of 5137 284 / 271, 48 of 3545 205 / 198, 128 of 2154 235 / 227, but 64 of 1301
    // 53 / 55 and 96 of 2154 165 / 167; 128/128 columns: 40 of 5120 274 / 256, 32 of 5120 220 / 211, but 96 of 1664
    // 86 / 89.
    PingPongPlan plan = {};
    bool persistent = false;
    // the persistent kernel streams two tiles ahead across items: every item needs two tiles
    if (sequence_length >= 128 && index_math::split_forward_steps(batch_heads, sequence_length, compute_units) > blocks128) {
        plan = pingpong_plan(batch_heads, sequence_length);
        persistent = plan.choice.cost <= index_math::split_forward_cost(batch_heads, sequence_length, compute_units);
    }
    // 64 queries instead of 128 while that finds idle compute units, for long sequences up to one workgroup of 128 per
    // unit (64 / 128: 16 heads of 1000 tokens 16.3 / 20.6 us, 8 of 4096 47.5 / 57.6, 64 of 512 16.3 / 15.4, 32 of 1500
    // 41.5 / 32.0).
    const long long workgroups = batch_heads * blocks128;
    const bool quarters = 2 * workgroups <= compute_units || (workgroups <= compute_units && sequence_length >= 1024);
    DSCUDA_FWD_CASE(192, 128)
    DSCUDA_FWD_CASE(128, 128)
#undef DSCUDA_FWD_CASE
#undef DSCUDA_FWD_FOUR_WAVES
#undef DSCUDA_FWD_SPLIT
    throw std::invalid_argument("attention forward: unsupported head sizes (d_qk,d_v) = (" +
                                std::to_string(qk_head_size) + "," + std::to_string(v_head_size) + ")");
}

}  // namespace dscuda
