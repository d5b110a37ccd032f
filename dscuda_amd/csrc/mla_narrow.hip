// Absorbed MLA attention with few query rows per workgroup (32 or 64), for work that the
// 128-row kernels of mla_decode.hip leave most of the chip idle on: decode with few heads
// (one rank of a head-sharded server), decode of a small batch, short absorbed prefills.
// Same mathematics and same key stream (latent_stream.h) as there; what differs is how a
// workgroup splits a unit of 32 keys over its waves.
//
// Two roles, eight waves, two waves per SIMD.  A 128-row workgroup gives every wave 32 rows
// and the whole unit: 68 MFMAs, one dependent stream of some 4000 cycles, whatever the number
// of rows that are real.  With few rows the unit is split instead:
//   score waves 0..3   S(u+1)^T = K(u+1) Q^T as 16 x 16 blocks (16x16x32 MFMA, 18 k-steps),
//                      each wave RB blocks; exp2 against a fixed reference; P(u+1) as bf16
//                      into LDS, in the order the output products take it
//   output waves 4..7  the requests of unit u+3, then O^T += V(u)^T P(u), each wave 128 of
//                      the 512 output columns (32x32x16 MFMA, 8 * RB products)
// one barrier per unit.  Stamps of a step (prefill, T = 512, H = 8): 32 rows 1640 cycles, of
// which the requests of a unit take 1100 (the rate at which a compute unit draws 1 KB pieces
// into LDS) and score and output streams 600 and 370 beside and behind them; 64 rows 2000.
// A 128-row workgroup takes 4000 a unit, so 32 rows win while the chip has idle compute
// units, 64 rows where the key stream (one 36 KB unit per workgroup) is the bound and 128
// where everything is busy.  Measured, 128-row kernels -> these: decode of 16 sequences
// x 16 heads x 1024..4096 tokens 44 -> 22 us, 64 x 16 x 1024..8192 104 -> 69 us (384 MB at
// 5.7 TB/s under the profiler), 16 x 128 x 1024..8192 64 -> 47 us; prefill T = 512, H = 8
// 39 -> 19 us.
//
// Softmax reference.  As in mla_decode.hip the exponentials are taken against the first
// unit's maximum plus a head room, and the reference is raised when a row outruns it (next to
// never).  Here the rows of a unit are spread over waves, so a score wave that sees a row
// outrun its reference raises a flag beside the P tile; every wave reads the flag with the
// operands of its next step and all of them take the rare path together.
#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "latent_stream.h"

#include <cstdint>
#include <stdexcept>

namespace dscuda {
namespace {

constexpr int NARROW_THREADS = 512;
constexpr int SCORE_STEPS = WIDTH / 32;       // 18
constexpr int OUT_BLOCKS = RANK / 32 / 4;     // 32-column blocks of an output wave: 4
constexpr int STAGE_PITCH = 2 * RANK + 16;    // bytes per staged output row ...
constexpr int WIDE_PITCH = 4 * RANK + 16;     // ... and per fp32 row of a part
constexpr int SCORE_RING = 6;                 // key fragments read ahead of the product that takes them
constexpr int VALUE_RING = 4;

// Head room (log2 units) between the first unit's maximum and the reference of a walk, and the
// excess over the reference at which it is raised.
constexpr float HEADROOM = 40.0f;
constexpr float OUTRUN = 80.0f;

template <int RB>
struct NarrowLayout {
    static constexpr int ROWS = 32 * RB;
    static constexpr int P_BYTES = UNIT * ROWS * 2;                     // P of one unit, bf16
    static constexpr int P_AT = UNIT_SLOTS * UNIT_BYTES;                // two buffers
    static constexpr int MAX_AT = P_AT + 2 * P_BYTES;                   // [2 key halves][ROWS]
    static constexpr int FACTOR_AT = MAX_AT + 2 * ROWS * 4;             // [ROWS]
    static constexpr int SUM_AT = FACTOR_AT + ROWS * 4;                 // [2][ROWS]
    static constexpr int FLAG_AT = SUM_AT + 2 * ROWS * 4;               // [2]
    static constexpr int LDS_BYTES = FLAG_AT + 16;
    static_assert(ROWS * WIDE_PITCH <= UNIT_SLOTS * UNIT_BYTES, "the staged rows take the place of the units");
};

__device__ __forceinline__ float quarter_max(float value) {   // over the lanes l, l ^ 16, l ^ 32, l ^ 48
    value = fmaxf(value, __shfl_xor(value, 16));
    return half_wave_max(value);
}

__device__ __forceinline__ float quarter_sum(float value) {
    value += __shfl_xor(value, 16);
    return half_wave_sum(value);
}

// The rows of a workgroup as the walk needs them: what a score wave's lane reads and sees.
struct NarrowRow {
    const bf16_t* latent;   // of the lane's row (16 rows per wave, row lane % 16)
    const bf16_t* rope;
    int visible;            // keys the row sees (>= 1)
    bool valid;
};

// One walk over tiles [tile_begin, tile_end) of one key stream for ROWS rows.  On return the
// staged rows lie in LDS at row * STAGE_PITCH (bf16, normalised if `normalise`) or, if `wide`,
// at row * WIDE_PITCH (fp32, not normalised), `reference` and `total` are set in the lanes of the
// score waves (of row 16 * group + lane % 16), all waves have passed a barrier, and the caller
// owes one more before the next walk.
template <int RB, bool PREFILL>
__device__ __forceinline__ void narrow_walk(const NarrowRow& row, unsigned char* lds, const KeyStream& keys, int tile_begin,
                                            int tile_end, int tokens, float c, bool normalise, bool wide, int wave,
                                            float& reference, float& total) {
    using L = NarrowLayout<RB>;
    constexpr int ROWS = L::ROWS;
    const int last_token = tokens - 1;
    const int unit_begin = (BN / UNIT) * tile_begin;
    const int unit_end = min((BN / UNIT) * tile_end, (tokens + UNIT - 1) / UNIT);   // > unit_begin
    const int lane = fresh_lane_id();
    auto slot_of = [&](int unit) { return lds + ((unsigned)unit % UNIT_SLOTS) * UNIT_BYTES; };
    float* maxima = reinterpret_cast<float*>(lds + L::MAX_AT);
    float* factors = reinterpret_cast<float*>(lds + L::FACTOR_AT);
    float* sums = reinterpret_cast<float*>(lds + L::SUM_AT);
    volatile int* flags = reinterpret_cast<volatile int*>(lds + L::FLAG_AT);

    if (wave < 4) {
        // ================= score wave =================
        const int group = RB == 1 ? wave % 2 : wave;       // 16 rows
        const int half0 = RB == 1 ? wave / 2 : 0;          // first of the RB key halves this wave takes
        const int r = lane % 16;
        const int q = lane / 16;
        bf16x8 qf[SCORE_STEPS];   // B operand: column = row r, k = 32*s + 8*q + j
#pragma unroll
        for (int s = 0; s < SCORE_STEPS; ++s) {
            u32x4 bits = {0, 0, 0, 0};
            if (row.valid) {
                bits = *reinterpret_cast<const u32x4*>(s < RANK / 32 ? row.latent + 32 * s + 8 * q
                                                                     : row.rope + 32 * (s - RANK / 32) + 8 * q);
            }
            qf[s] = __builtin_bit_cast(bf16x8, bits);
        }
        using Read = index_math::TileReadMath<ROW_BYTES>;
        unsigned key_at[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) key_at[i] = Read::quadrant(i, lane) + half0 * 16 * ROW_BYTES;
        // where this lane's four keys of block `half` go in a P tile: [half][row][8-byte pieces q = 0, 2, 1, 3]
        const unsigned p_at = L::P_AT + (16 * group + r) * 32 + (q & 1) * 16 + (q >> 1) * 8 + half0 * (ROWS * 32);

        f32x4 scores[RB];
        // fragment F of the stream: key half F % RB, k-step F / RB
        auto form_scores = [&](int unit) {
            const unsigned char* base = slot_of(unit);
            auto fragment = [&](auto tag) -> bf16x8 {
                constexpr int F = decltype(tag)::value;
                constexpr int S = F / RB;
                return *reinterpret_cast<const bf16x8*>(base + key_at[S % 2] + (S / 2) * 128 + (F % RB) * 16 * ROW_BYTES);
            };
            constexpr int COUNT = SCORE_STEPS * RB;
            bf16x8 ring[SCORE_RING];
            unrolled<0, SCORE_RING>([&](auto tag) { ring[decltype(tag)::value] = fragment(tag); });
            f32x4 odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < RB; ++k) scores[k] = f32x4{0.f, 0.f, 0.f, 0.f};
            unrolled<0, COUNT>([&](auto tag) {
                constexpr int F = decltype(tag)::value;
                f32x4& chain = RB == 1 && F % 2 == 1 ? odd : scores[F % RB];   // two chains either way
                chain = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[F % SCORE_RING], qf[F / RB], chain, 0, 0, 0);
                if constexpr (F + SCORE_RING < COUNT) ring[F % SCORE_RING] = fragment(std::integral_constant<int, F + SCORE_RING>{});
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (RB == 1) {
#pragma unroll
                for (int i = 0; i < 4; ++i) scores[0][i] += odd[i];
            }
            if ((unit + 1) * UNIT > (PREFILL ? 0 : tokens)) {   // uniform; in prefill every row has its own limit
#pragma unroll
                for (int k = 0; k < RB; ++k) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (unit * UNIT + 16 * (half0 + k) + 4 * q + i >= row.visible) scores[k][i] = -INFINITY;
                    }
                }
            }
        };
        auto lane_max = [&]() {
            float value = scores[0][0];
#pragma unroll
            for (int k = 0; k < RB; ++k) {
#pragma unroll
                for (int i = 0; i < 4; ++i) value = fmaxf(value, scores[k][i]);
            }
            return value;
        };
        float pending = 0.f;   // this lane's share of the sum of the unit whose P was written last
        auto write_probabilities = [&](int unit) {
            pending = 0.f;
#pragma unroll
            for (int k = 0; k < RB; ++k) {
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = __builtin_amdgcn_exp2f(fmaf(scores[k][i], c, -reference));
                    pending += p[i];
                }
                const u32x2 packed = {pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
                *reinterpret_cast<u32x2*>(lds + p_at + (unit & 1) * L::P_BYTES + k * (ROWS * 32)) = packed;
            }
        };
        auto publish_max = [&]() {
            const float value = quarter_max(lane_max());
            if (q == 0) maxima[half0 * ROWS + 16 * group + r] = value;
        };
        auto row_max = [&]() {
            return RB == 1 ? fmaxf(maxima[16 * group + r], maxima[ROWS + 16 * group + r]) : maxima[16 * group + r];
        };

        wait_vector_memory<0>();   // the query rows: no wait for them may remain inside the loop
        workgroup_barrier();       // the first unit has landed
        form_scores(unit_begin);
        publish_max();
        workgroup_barrier();
        reference = row_max() * c + HEADROOM;
        float row_sum = 0.f;
        write_probabilities(unit_begin);
        workgroup_barrier();
        for (int unit = unit_begin; unit < unit_end; ++unit) {
            if (__builtin_expect(__builtin_amdgcn_readfirstlane(flags[unit & 1]) != 0, 0)) {
                publish_max();
                workgroup_barrier();
                const float highest = row_max() * c;
                const float raised = highest - reference > OUTRUN ? highest + HEADROOM : reference;
                const float factor = __builtin_amdgcn_exp2f(reference - raised);   // 1 for the rows that stay
                reference = raised;
                row_sum *= factor;
                if (half0 == 0 && q == 0) factors[16 * group + r] = factor;
                if (wave == 0 && lane == 0) flags[unit & 1] = 0;
                write_probabilities(unit);
                workgroup_barrier();
            }
            row_sum += pending;
            if (unit + 1 < unit_end) {
                form_scores(unit + 1);
                write_probabilities(unit + 1);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(fmaf(lane_max(), c, -reference) > OUTRUN) != 0, 0)) {
                    if (lane == 0) flags[(unit + 1) & 1] = 1;
                }
            }
            workgroup_barrier();
        }
        row_sum = quarter_sum(row_sum);
        if (q == 0) sums[half0 * ROWS + 16 * group + r] = row_sum;
        workgroup_barrier();
        total = RB == 1 ? sums[16 * group + r] + sums[ROWS + 16 * group + r] : sums[16 * group + r];
    } else {
        // ================= output wave =================
        const int v = wave - 4;
        const int lq = lane % 32;
        const int g = lane / 32;
        UnitCursor cursor;
        cursor.init(keys, unit_begin, last_token);
        if constexpr (PREFILL) {
            cursor.contiguous = false;   // latent and rope parts come from tensors of their own
            cursor.split = keys.latent_stride < ((size_t)1 << 24) && keys.rope_stride < ((size_t)1 << 24);
        }
        FullUnitOffsets offsets;
        offsets.init(v, lane);
        auto request = [&]() { issue_unit(cursor.next(lds, keys, last_token, v, unit_end), offsets, keys, v); };
        // all of this wave's requests but those of the youngest `outstanding` units have landed
        auto wait_for = [&](int outstanding) {
            if (outstanding >= 2) wait_vector_memory<2 * UNIT_LOADS>();
            else if (outstanding == 1) wait_vector_memory<UNIT_LOADS>();
            else wait_vector_memory<0>();
        };
        request();
        request();
        request();
        f32x16 out[OUT_BLOCKS][RB];
#pragma unroll
        for (int d = 0; d < OUT_BLOCKS; ++d) {
#pragma unroll
            for (int b = 0; b < RB; ++b) {
#pragma unroll
                for (int i = 0; i < 16; ++i) out[d][b][i] = 0.f;
            }
        }
        UnitReads reads;
        reads.init(lane);
        wait_for(min(unit_end - unit_begin, 3) - 1);
        workgroup_barrier();
        workgroup_barrier();   // the score waves agree on the reference
        wait_for(min(unit_end - unit_begin, 3) - 2);
        workgroup_barrier();
        for (int unit = unit_begin; unit < unit_end; ++unit) {
            if (__builtin_expect(__builtin_amdgcn_readfirstlane(flags[unit & 1]) != 0, 0)) {
                workgroup_barrier();   // the score waves settle on the raised references ...
                workgroup_barrier();   // ... and have formed the probabilities again
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const float factor = factors[32 * b + lq];
#pragma unroll
                    for (int d = 0; d < OUT_BLOCKS; ++d) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) out[d][b][i] *= factor;
                    }
                }
            }
            // Unit + 3, into the slot that unit - 1 left.  All nine requests go out before the products: what a compute
            // unit draws from the L2s into LDS (36 KB in some 1500 cycles) is what bounds a step, and requests placed
            // between the products instead made it 8 % longer.
            request();
            const unsigned char* base = slot_of(unit) + v * (OUT_BLOCKS * 64);
            bf16x8 pf[2][RB];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    pf[n][b] = *reinterpret_cast<const bf16x8*>(lds + L::P_AT + (unit & 1) * L::P_BYTES +
                                                                n * (ROWS * 32) + (32 * b + lq) * 32 + 16 * g);
                }
            }
            constexpr int COUNT = 2 * OUT_BLOCKS;
            bf16x8 ring[VALUE_RING];
            unrolled<0, VALUE_RING>([&](auto tag) {
                constexpr int F = decltype(tag)::value;
                ring[F] = unit_value_fragment<F / OUT_BLOCKS, F % OUT_BLOCKS>(base, reads);
            });
            unrolled<0, COUNT>([&](auto tag) {
                constexpr int F = decltype(tag)::value;
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    out[F % OUT_BLOCKS][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[F % VALUE_RING], pf[F / OUT_BLOCKS][b],
                                                                                     out[F % OUT_BLOCKS][b], 0, 0, 0);
                }
                if constexpr (F + VALUE_RING < COUNT) {
                    constexpr int N = F + VALUE_RING;
                    ring[F % VALUE_RING] = unit_value_fragment<N / OUT_BLOCKS, N % OUT_BLOCKS>(base, reads);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            wait_for(unit + 3 < unit_end ? 1 : 0);   // unit + 2 has landed
            workgroup_barrier();
        }
        workgroup_barrier();   // the sums are there, the unit slots are free
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            float inverse = 1.f;
            if (normalise) {
                inverse = 1.0f / (RB == 1 ? sums[32 * b + lq] + sums[ROWS + 32 * b + lq] : sums[32 * b + lq]);
            }
            if (wide) {
                unsigned char* row_parts = lds + (32 * b + lq) * WIDE_PITCH + 4 * (128 * v + 4 * g);
#pragma unroll
                for (int d = 0; d < OUT_BLOCKS; ++d) {
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        *reinterpret_cast<f32x4*>(row_parts + 4 * (32 * d + 8 * i4)) =
                            f32x4{out[d][b][4 * i4], out[d][b][4 * i4 + 1], out[d][b][4 * i4 + 2], out[d][b][4 * i4 + 3]};
                    }
                }
                continue;
            }
            unsigned char* staged = lds + (32 * b + lq) * STAGE_PITCH + 2 * (128 * v + 4 * g);
#pragma unroll
            for (int d = 0; d < OUT_BLOCKS; ++d) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    u32x2 packed;
                    packed.x = pack_bf16(out[d][b][4 * i4 + 0] * inverse, out[d][b][4 * i4 + 1] * inverse);
                    packed.y = pack_bf16(out[d][b][4 * i4 + 2] * inverse, out[d][b][4 * i4 + 3] * inverse);
                    *reinterpret_cast<u32x2*>(staged + 2 * (32 * d + 8 * i4)) = packed;
                }
            }
        }
    }
    workgroup_barrier();   // the staged rows are complete
}

// Staged rows -> destination(row) (nullptr: none), one 1 KB row per wave instruction.
template <int ROWS, typename RowPointer>
__device__ __forceinline__ void store_staged_rows(const unsigned char* lds, int wave, RowPointer destination) {
    const int lane = fresh_lane_id();
#pragma unroll
    for (int i = 0; i < ROWS / 8; ++i) {
        const int row = 8 * i + wave;
        bf16_t* to = destination(row);
        if (to != nullptr) {
            *reinterpret_cast<u32x4*>(to + 8 * lane) = *reinterpret_cast<const u32x4*>(lds + row * STAGE_PITCH + 16 * lane);
        }
    }
}

// The same for fp32 rows, two instructions a row.
template <int ROWS, typename RowPointer>
__device__ __forceinline__ void store_wide_rows(const unsigned char* lds, int wave, RowPointer destination) {
    const int lane = fresh_lane_id();
#pragma unroll
    for (int i = 0; i < ROWS / 8; ++i) {
        const int row = 8 * i + wave;
        float* to = destination(row);
        if (to != nullptr) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                *reinterpret_cast<f32x4*>(to + 256 * half + 4 * lane) =
                    *reinterpret_cast<const f32x4*>(lds + row * WIDE_PITCH + 1024 * half + 16 * lane);
            }
        }
    }
}

// ----------------------------------------------------------------------------
// decode
// ----------------------------------------------------------------------------

// A partial result lies in slot range + sequence of the workspace (index_math.h): one row of 512 per head, bf16 or, in
// a wide plan, fp32, then (reference, sum) per head.
template <int RB>
__global__ __launch_bounds__(NARROW_THREADS) void mla_narrow_decode_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp, const bf16_t* __restrict__ query,
    const bf16_t* __restrict__ paged_kv_cache, const int* __restrict__ block_table,
    const int* __restrict__ cache_lengths, float* __restrict__ workspace, int* __restrict__ plan, int batch_size,
    int heads, int page_size, int pages_per_sequence, long long slot_floats, long long wide_slot_floats, float scale,
    bool own_plan, DecodeCut cut) {
    using L = NarrowLayout<RB>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ int own_prefix[SELF_PLAN_BATCH + 1];
    __shared__ int own_lengths[SELF_PLAN_BATCH];
    __shared__ int own_wave_totals[2 * SELF_PLAN_BATCH / 64];

    const int tid = threadIdx.x;
    const int lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int workgroup = gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int head0 = blockIdx.y * L::ROWS;
    const float c = scale * LOG2E;

    if (tid < 2) *reinterpret_cast<volatile int*>(lds + L::FLAG_AT + 4 * tid) = 0;
    const DecodeRange range = decode_range(plan, cache_lengths, batch_size, own_plan, false, cut, own_prefix, own_lengths,
                                           own_wave_totals, tid, NARROW_THREADS, workgroup, blockIdx.x == 0 && blockIdx.y == 0);
    if (range.begin >= range.end) return;

    int sequence = range.sequence;
    int position = range.begin;
    while (position < range.end) {
        int sequence_begin, sequence_end, tokens;
        if (range.local) {
            sequence_begin = own_prefix[sequence];
            sequence_end = own_prefix[sequence + 1];
            tokens = own_lengths[sequence];
        } else {
            sequence_begin = range.prefix[sequence];
            sequence_end = range.prefix[sequence + 1];
            tokens = cache_lengths[sequence];
        }
        sequence_begin = __builtin_amdgcn_readfirstlane(sequence_begin);
        sequence_end = __builtin_amdgcn_readfirstlane(sequence_end);
        tokens = __builtin_amdgcn_readfirstlane(tokens);
        const int segment_end = min(range.end, sequence_end);
        if (segment_end <= position) {  // a sequence without tiles (length < 1) owns nothing
            ++sequence;
            continue;
        }
        int tile_begin, tile_end;
        index_math::tiles_in_positions(position, segment_end, sequence_begin, range.overhead, tile_begin, tile_end);
        if (tile_end <= tile_begin) {   // the range ends among the positions that stand for the sequence's overhead
            position = segment_end;
            ++sequence;
            continue;
        }
        const bool whole = tile_begin == 0 && tile_end == sequence_end - sequence_begin - range.overhead;

        KeyStream keys;
        keys.latent = paged_kv_cache;
        keys.rope = paged_kv_cache + RANK;
        keys.latent_stride = WIDTH;
        keys.rope_stride = WIDTH;
        keys.block_table = block_table + (size_t)sequence * pages_per_sequence;
        keys.page_size = page_size;
        const int head = head0 + 16 * (RB == 1 ? wave % 2 : wave % 4) + lane % 16;   // of a score wave's lane
        NarrowRow row;
        row.valid = head < heads;
        row.latent = query + ((size_t)sequence * heads + (row.valid ? head : 0)) * WIDTH;
        row.rope = row.latent + RANK;
        row.visible = tokens;
        float reference = 0.f, total = 1.f;
        narrow_walk<RB, false>(row, lds, keys, tile_begin, tile_end, tokens, c, whole, !whole && range.wide, wave, reference,
                               total);

        const bool writer = wave < (RB == 1 ? 2 : 4) && lane < 16 && row.valid;
        if (whole) {
            if (writer) logsumexp[(size_t)sequence * heads + head] = (reference + __builtin_amdgcn_logf(total)) * LN2;
            store_staged_rows<L::ROWS>(lds, wave, [&](int r) -> bf16_t* {
                return head0 + r < heads ? output + ((size_t)sequence * heads + head0 + r) * RANK : nullptr;
            });
        } else {
            float* slot = workspace + ((size_t)workgroup + sequence) * (range.wide ? wide_slot_floats : slot_floats);
            if (writer) {
                float* statistics = slot + (size_t)heads * (range.wide ? RANK : RANK / 2) + 2 * head;
                statistics[0] = reference;
                statistics[1] = total;
            }
            if (range.wide) {
                store_wide_rows<L::ROWS>(lds, wave, [&](int r) -> float* {
                    return head0 + r < heads ? slot + (size_t)(head0 + r) * RANK : nullptr;
                });
            } else {
                store_staged_rows<L::ROWS>(lds, wave, [&](int r) -> bf16_t* {
                    return head0 + r < heads ? reinterpret_cast<bf16_t*>(slot) + (size_t)(head0 + r) * RANK : nullptr;
                });
            }
        }
        workgroup_barrier();   // the staged rows have been read: the next segment's units may come
        position = segment_end;
        ++sequence;
    }
}

// Merge of the parts of every sequence that a range boundary cut: a wave per (sequence, head),
// eight columns per lane.  The statistics of 64 parts (a lane each) and the rows of the first
// AHEAD come in one round trip, further rows AHEAD at a time (sixteen bf16 rows or eight fp32
// rows: 64 registers).  Against statistics first and rows four at a time, whole calls: 64 sequences
// x 16 heads x 1024..8192 tokens 71.3 -> 68.7 us, 16 x 128 50.4 -> 48.8, 8 x 8 x 3336 19.7 -> 18.9,
// one of 200 tokens x 128 heads 12.7 -> 12.0.
constexpr int MERGE_WAVES = 4;

struct MergedRow {
    float sums[8];       // not normalised
    float highest;       // reference of the sums
    float normaliser;
};

template <bool WIDE>
__device__ __forceinline__ MergedRow merge_parts(const float* slots, long long slot_floats, int parts, int heads, int head,
                                                 int lane) {
    constexpr int AHEAD = WIDE ? 8 : 16;
    constexpr int PIECES = WIDE ? 2 : 1;   // of 16 bytes per lane and row
    static_assert(64 % AHEAD == 0, "the statistics change between two requests of rows");
    const size_t stats_offset = (size_t)heads * (WIDE ? RANK : RANK / 2) + 2 * head;
    // the lane's eight columns of part 0
    const float* rows = slots + (WIDE ? (size_t)head * RANK + 8 * lane : (size_t)head * (RANK / 2) + 4 * lane);
    u32x4 bits[AHEAD][PIECES];
    auto request = [&](int part) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            if (part + i < parts) {
#pragma unroll
                for (int j = 0; j < PIECES; ++j) {
                    bits[i][j] = *reinterpret_cast<const u32x4*>(rows + (part + i) * slot_floats + 4 * j);
                }
            }
        }
    };
    // lane: statistics of part base + lane; those of the first 64 parts stay in registers
    float lane_highest = -INFINITY, lane_sum = 0.f;
    auto load_statistics = [&](int base) {
        lane_highest = -INFINITY;
        lane_sum = 0.f;
        if (base + lane < parts) {
            const float* stats = slots + (base + lane) * slot_floats + stats_offset;
            lane_highest = stats[0];
            lane_sum = stats[1];
        }
    };
    MergedRow row;
    float highest = -INFINITY;
    for (int base = 64; base < parts; base += 64) {
        load_statistics(base);
        highest = fmaxf(highest, lane_highest);
    }
    load_statistics(0);
    request(0);
    highest = fmaxf(highest, lane_highest);
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) highest = fmaxf(highest, __shfl_xor(highest, offset));
    float normaliser = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) row.sums[k] = 0.f;
    float weight = 0.f;
    for (int part = 0; part < parts; part += AHEAD) {
        if (part > 0) request(part);
        if (part % 64 == 0) {
            if (part > 0) load_statistics(part);
            weight = __builtin_amdgcn_exp2f(lane_highest - highest);   // 0 in lanes without a part
            normaliser = fmaf(weight, lane_sum, normaliser);
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            if (part + i < parts) {
                const float w = __shfl(weight, (part + i) % 64);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if constexpr (WIDE) {
                        row.sums[k] = fmaf(w, __uint_as_float(bits[i][0][k]), row.sums[k]);
                        row.sums[4 + k] = fmaf(w, __uint_as_float(bits[i][1][k]), row.sums[4 + k]);
                    } else {
                        row.sums[2 * k] = fmaf(w, __uint_as_float(bits[i][0][k] << 16), row.sums[2 * k]);
                        row.sums[2 * k + 1] = fmaf(w, __uint_as_float(bits[i][0][k] & 0xffff0000u), row.sums[2 * k + 1]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) normaliser += __shfl_xor(normaliser, offset);
    row.highest = highest;
    row.normaliser = normaliser;
    return row;
}

__global__ __launch_bounds__(64 * MERGE_WAVES) void mla_narrow_merge_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp, const float* __restrict__ workspace,
    const int* __restrict__ plan, int batch_size, int heads, long long slot_floats, long long wide_slot_floats) {
    const int lane = threadIdx.x % 64;
    const int head = blockIdx.x * MERGE_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int sequence = blockIdx.y;
    if (head >= heads) return;
    const int total = plan[PLAN_TOTAL];
    const int overhead = plan[PLAN_OVERHEAD];
    const int ranges = plan[PLAN_RANGES];
    const int mode = plan[PLAN_MODE];
    const int* prefix = plan + index_math::plan_prefix_at();
    const int sequence_begin = prefix[sequence];
    const int sequence_end = prefix[sequence + 1];
    asm volatile("" ::"s"(total), "s"(overhead), "s"(ranges), "s"(mode), "s"(sequence_end));   // one round trip, not two
    if (sequence_end <= sequence_begin) return;   // no tiles: nothing was computed for it
    int first, last;
    index_math::ranges_of_sequence(total, ranges, sequence_begin, sequence_end - sequence_begin, overhead, first, last);
    if (first == last) return;                    // finished in place

    const size_t slot = (size_t)first + sequence;
    const int parts = last - first + 1;
    const MergedRow row = mode == PLAN_WIDE_PARTS
        ? merge_parts<true>(workspace + slot * wide_slot_floats, wide_slot_floats, parts, heads, head, lane)
        : merge_parts<false>(workspace + slot * slot_floats, slot_floats, parts, heads, head, lane);
    const float inverse = 1.0f / row.normaliser;
    u32x4 packed;
#pragma unroll
    for (int k = 0; k < 4; ++k) packed[k] = pack_bf16(row.sums[2 * k] * inverse, row.sums[2 * k + 1] * inverse);
    *reinterpret_cast<u32x4*>(output + ((size_t)sequence * heads + head) * RANK + 8 * lane) = packed;
    if (lane == 0) logsumexp[(size_t)sequence * heads + head] = (row.highest + __builtin_amdgcn_logf(row.normaliser)) * LN2;
}

// ----------------------------------------------------------------------------
// absorbed causal prefill forward
// ----------------------------------------------------------------------------

template <int RB>
__global__ __launch_bounds__(NARROW_THREADS) void mla_narrow_forward_kernel(
    bf16_t* __restrict__ output, float* __restrict__ logsumexp, const bf16_t* __restrict__ query_latent,
    const bf16_t* __restrict__ query_rope, const bf16_t* __restrict__ kv_latent, const bf16_t* __restrict__ key_rope,
    int sequence_length, int heads, int row_blocks, float scale) {
    using L = NarrowLayout<RB>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const float c = scale * LOG2E;
    if (tid < 2) *reinterpret_cast<volatile int*>(lds + L::FLAG_AT + 4 * tid) = 0;

    // heaviest (latest) row blocks first
    const int batch = blockIdx.x / row_blocks;
    const int row_block = row_blocks - 1 - blockIdx.x % row_blocks;
    const long long rows = (long long)sequence_length * heads;   // (token, head) pairs of one batch element
    const long long row0 = (long long)row_block * L::ROWS;
    const long long last_row = min(rows, row0 + L::ROWS) - 1;
    const int visible = (int)(last_row / heads) + 1;             // keys any row of this block may see

    KeyStream keys;
    keys.latent = kv_latent + (size_t)batch * sequence_length * RANK;
    keys.rope = key_rope + (size_t)batch * sequence_length * ROPE;
    keys.latent_stride = RANK;
    keys.rope_stride = ROPE;
    keys.block_table = nullptr;
    keys.page_size = 0;
    const long long at = row0 + 16 * (RB == 1 ? wave % 2 : wave % 4) + lane % 16;   // of a score wave's lane
    NarrowRow row;
    row.valid = at < rows;
    const int token = row.valid ? (int)(at / heads) : 0;
    const long long global_row = (long long)batch * rows + (row.valid ? at : 0);
    row.latent = query_latent + global_row * RANK;
    row.rope = query_rope + global_row * ROPE;
    row.visible = row.valid ? token + 1 : visible;
    float reference = 0.f, total = 1.f;
    narrow_walk<RB, true>(row, lds, keys, 0, tiles_of(visible), visible, c, true, false, wave, reference, total);

    if (wave < (RB == 1 ? 2 : 4) && lane < 16 && row.valid) {
        logsumexp[((size_t)batch * heads + (int)(at % heads)) * sequence_length + token] =
            (reference + __builtin_amdgcn_logf(total)) * LN2;
    }
    store_staged_rows<L::ROWS>(lds, wave, [&](int r) -> bf16_t* {
        return row0 + r < rows ? output + ((long long)batch * rows + row0 + r) * RANK : nullptr;
    });
}

template <int RB>
void allow_narrow_lds() {
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_narrow_decode_kernel<RB>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, NarrowLayout<RB>::LDS_BYTES));
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_narrow_forward_kernel<RB>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, NarrowLayout<RB>::LDS_BYTES));
}

void prepare_narrow() {
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        allow_narrow_lds<1>();
        allow_narrow_lds<2>();
    });
}

}  // namespace

void mla_narrow_decode_launch(bf16_t* output, float* logsumexp, const bf16_t* query, const bf16_t* paged_kv_cache,
                              const int* block_table, const int* cache_lengths, float* workspace, int* plan,
                              int batch_size, int heads, int page_size, int pages_per_sequence, int row_blocks,
                              const index_math::DecodeLayout& layout, bool own_plan, float scale, hipStream_t stream) {
    prepare_narrow();
    const int rows = 32 * row_blocks;
    const dim3 grid(layout.workgroups, (heads + rows - 1) / rows);
    const DecodeCut cut = {layout.workgroups, layout.whole_sequences, layout.reference_ranges, layout.wide_ranges};
    auto launch = [&](auto kernel, int lds_bytes) {
        hipLaunchKernelGGL(kernel, grid, dim3(NARROW_THREADS), lds_bytes, stream, output, logsumexp, query, paged_kv_cache,
                           block_table, cache_lengths, workspace, plan, batch_size, heads, page_size, pages_per_sequence,
                           layout.slot_floats, layout.wide_slot_floats, scale, own_plan, cut);
        HIP_CHECK(hipGetLastError());
    };
    if (row_blocks == 1) {
        launch(mla_narrow_decode_kernel<1>, NarrowLayout<1>::LDS_BYTES);
    } else {
        launch(mla_narrow_decode_kernel<2>, NarrowLayout<2>::LDS_BYTES);
    }
    if (!layout.whole_sequences) {
        hipLaunchKernelGGL(mla_narrow_merge_kernel, dim3((heads + MERGE_WAVES - 1) / MERGE_WAVES, batch_size),
                           dim3(64 * MERGE_WAVES), 0, stream, output, logsumexp, workspace, plan, batch_size, heads,
                           layout.slot_floats, layout.wide_slot_floats);
        HIP_CHECK(hipGetLastError());
    }
}

void mla_narrow_forward_launch(bf16_t* output, float* logsumexp, const bf16_t* query_latent, const bf16_t* query_rope,
                               const bf16_t* kv_latent, const bf16_t* key_rope, int batch_size, int sequence_length,
                               int heads, int row_blocks, float scale, hipStream_t stream) {
    prepare_narrow();
    const int rows = 32 * row_blocks;
    const long long blocks = ((long long)sequence_length * heads + rows - 1) / rows;
    auto launch = [&](auto kernel, int lds_bytes) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(blocks * batch_size)), dim3(NARROW_THREADS), lds_bytes, stream, output,
                           logsumexp, query_latent, query_rope, kv_latent, key_rope, sequence_length, heads, (int)blocks,
                           scale);
        HIP_CHECK(hipGetLastError());
    };
    if (row_blocks == 1) {
        launch(mla_narrow_forward_kernel<1>, NarrowLayout<1>::LDS_BYTES);
    } else {
        launch(mla_narrow_forward_kernel<2>, NarrowLayout<2>::LDS_BYTES);
    }
}

}  // namespace dscuda
