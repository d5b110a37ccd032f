// Rotary position embedding applied in place to a slice of the last dimension of a
// [B, S, H, W] bf16 tensor: the step that precedes the attention kernels in an MLA
// layer (the rope parts of Q and K) and that the reference leaves to its caller
// (reference/python/sources.json:2 lists "model projections" and position encoding
// among the things it does not contain).
//
// Convention: interleaved pairs.  Within the slice of `rope` columns, columns
// (2i, 2i + 1) form pair i, rotated by the angle position * theta^(-2i / rope):
//     x'[2i]     = x[2i] * cos - x[2i + 1] * sin
//     x'[2i + 1] = x[2i] * sin + x[2i + 1] * cos
// with position = s (+ positions[b] when a per-sequence start is given, as for the one
// new token of a decode step).  Frequencies and angles are formed in double precision
// and the sine and cosine rounded to fp32 once, the products and the sum each rounded to
// fp32 without fusing, the result rounded to bf16: the same sequence of roundings as
// forming the rotation with fp32 tensors on the host.
//
// Layout on the chip: one wave per (batch, position) and slice of the heads.  A lane owns
// pair lane % (rope/2) and computes its sine and cosine once; the 64 / (rope/2) groups of
// lanes then walk the heads, so every access of a group is one contiguous run of
// 2 * rope bytes.  The kernel moves 4 * rope bytes per (b, s, h) and is bound by memory:
// BATCH heads of a group are fetched before the first is stored (in place, so the loads
// would otherwise wait for the stores, a round trip per head), and where the rows alone
// leave the chip idle the heads are sliced so that one batch covers a wave.  The last batch
// asks for its own heads only (repeating the last head instead: 60 x 804 rows of 17 heads
// 40.1 us, so 34.1).  64 rows of 128 heads 11.9 -> 3.5 us, 1024 rows 14.4 -> 8.0, 4096 rows
// 28.9 -> 22.6 (134 MB at 6 TB/s).

#include "attn_kernels.h"
#include "hip_common.h"

#include <cmath>
#include <cstdint>
#include <stdexcept>
#include <string>

namespace dscuda {
namespace {

constexpr int ROPE_THREADS = 256;
constexpr int ROPE_ROWS = ROPE_THREADS / 64;   // (batch, position) rows per workgroup

// BATCH: heads a group of lanes has in flight
template <int BATCH>
__global__ __launch_bounds__(ROPE_THREADS) void rope_apply_kernel(bf16_t* __restrict__ tensor,
                                                                  const int* __restrict__ positions, long long rows,
                                                                  int sequence_length, int heads, int slice, int width,
                                                                  int rope_offset, int rope, double log2_theta) {
    const long long row = (long long)blockIdx.x * ROPE_ROWS + threadIdx.x / 64;
    if (row >= rows) return;
    const int lane = threadIdx.x % 64;
    const int pairs = rope / 2;            // a power of two, at most 64
    const int pair = lane % pairs;
    const int group = lane / pairs;
    const int groups = 64 / pairs;
    const long long b = row / sequence_length;
    const int s = (int)(row % sequence_length);
    const int position = s + (positions ? positions[b] : 0);
    const double frequency = exp2(-log2_theta * (2.0 * pair / rope));
    const double angle = (double)position * frequency;
    const float cosine = (float)cos(angle);
    const float sine = (float)sin(angle);
    unsigned* base = reinterpret_cast<unsigned*>(tensor + (size_t)row * heads * width + rope_offset) + pair;
    const int end = min(heads, (int)(blockIdx.y + 1) * slice);
    auto rotate = [&](int h, unsigned bits) {
        const float even = __uint_as_float(bits << 16);
        const float odd = __uint_as_float(bits & 0xffff0000u);
        const float rotated_even = __fsub_rn(__fmul_rn(even, cosine), __fmul_rn(odd, sine));
        const float rotated_odd = __fadd_rn(__fmul_rn(even, sine), __fmul_rn(odd, cosine));
        base[(size_t)h * (width / 2)] = pack_bf16(rotated_even, rotated_odd);
    };
    for (int first = blockIdx.y * slice + group; first < end; first += groups * BATCH) {
        unsigned bits[BATCH];
        if (first + (BATCH - 1) * groups < end) {
#pragma unroll
            for (int j = 0; j < BATCH; ++j) bits[j] = base[(size_t)(first + j * groups) * (width / 2)];
#pragma unroll
            for (int j = 0; j < BATCH; ++j) rotate(first + j * groups, bits[j]);
        } else {
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                if (first + j * groups < end) bits[j] = base[(size_t)(first + j * groups) * (width / 2)];
            }
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                if (first + j * groups < end) rotate(first + j * groups, bits[j]);
            }
        }
    }
}

}  // namespace

void rope_apply_dispatch(bf16_t* tensor, const int* positions, int batch_size, int sequence_length, int heads, int width,
                         int rope_offset, int rope_size, float theta, hipStream_t stream) {
    if (batch_size <= 0 || sequence_length <= 0 || heads <= 0) {
        throw std::invalid_argument("rope: batch, sequence length and heads must be positive");
    }
    const bool power_of_two = rope_size >= 2 && (rope_size & (rope_size - 1)) == 0;
    if (!power_of_two || rope_size > 128) {
        throw std::invalid_argument("rope: the rotated slice must be 2, 4, ..., 128 columns wide, got " +
                                    std::to_string(rope_size));
    }
    // pairs are moved as 32-bit words: the slice must start at an even column of rows of even width
    if (width <= 0 || width % 2 != 0 || rope_offset < 0 || rope_offset % 2 != 0 || rope_offset + rope_size > width) {
        throw std::invalid_argument("rope: columns " + std::to_string(rope_offset) + ".." +
                                    std::to_string(rope_offset + rope_size) + " do not fit rows of " +
                                    std::to_string(width) + " columns (even offset and width required)");
    }
    if (!(theta > 0.f)) {
        throw std::invalid_argument("rope: theta must be positive");
    }
    if (tensor == nullptr || reinterpret_cast<uintptr_t>(tensor) % 4 != 0) {
        throw std::invalid_argument("rope: the tensor must be a non-null pointer aligned to 4 bytes");
    }
    const long long rows = (long long)batch_size * sequence_length;
    const long long blocks = (rows + ROPE_ROWS - 1) / ROPE_ROWS;
    if (blocks > 0x7fffffffLL) {
        throw std::invalid_argument("rope: batch * sequence length exceeds the grid limit");
    }
    // below four workgroups per compute unit the heads are sliced, one batch of every group of lanes a slice
    constexpr int BATCH = 8;
    const int groups = 64 / (rope_size / 2);
    const int batch_heads = groups * BATCH;
    const bool sliced = blocks < 4LL * hip_common::compute_units_of_current_device() && (heads - 1) / batch_heads < 65535;
    const int slice = sliced ? batch_heads : heads;
    const unsigned slices = (unsigned)((heads + (long long)slice - 1) / slice);
    // One head at a time where rows abound and a group of lanes has few heads: the rows cover the round trips, and the
    // comparisons of a batch are time (eight in flight / one, us: 204845 rows of one head 87.7 / 81.7, 16384 rows of one
    // 9.1 / 8.5, of two 9.6 / 8.9, 35742 rows of four 21.3 / 20.4; 16000 rows of eight 11.4 / 11.9).
    const auto kernel = !sliced && heads < 4 * groups ? rope_apply_kernel<1> : rope_apply_kernel<BATCH>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, slices), dim3(ROPE_THREADS), 0, stream, tensor, positions, rows,
                       sequence_length, heads, slice, width, rope_offset, rope_size, std::log2((double)theta));
    HIP_CHECK(hipGetLastError());
}

}  // namespace dscuda
