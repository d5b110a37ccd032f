// The two per-head projections either side of absorbed MLA attention, which the reference
// leaves to its caller (reference/python/sources.json:2: "No ... model projections"):
//
//     absorb     q_latent[t, h, c] = sum_d q_nope[t, h, d]  * W_UK[h, d, c]      (d < 128, c < 512)
//     un-absorb  out[t, h, d]      = sum_c o_latent[t, h, c] * W_UV[h, d, c]
//
// with both weights in the layout of the two halves of DeepSeek-V3's wkv_b viewed as
// [heads, 128 + 128, 512] (inference/model.py of deepseek-ai/DeepSeek-V3: the absorbed
// attention path multiplies q_nope by wkv_b[:, :128] before and the latent output by
// wkv_b[:, -128:] after the attention).  BF16 in and out, FP32 accumulation on the
// 32x32x16 MFMA.
//
// Whole weights: a head's weight (128 KB) is staged once per workgroup in LDS, row-major as 32-row tiles;
// a wave then takes 32 tokens at a time, holds their input rows in registers straight from
// memory (lane = token, as the operand whose column is the token) and forms the transposed
// product y^T = W x^T; a lane ends up with one token and groups of four neighbouring output
// columns, which leave through a small LDS stage as whole 128-byte lines.
//   absorb:    W_UK[h] is [d][c]; the contraction index d is the tile row, so the weight
//              operand comes through transposing reads (ds_read_b64_tr_b16), which deliver
//              rows {4g..4g+3, 8+4g..8+4g+3} of a 16-row step: the token operand is brought
//              into the same order by one lane exchange per step.
//   un-absorb: W_UV[h] is [d][c]; the contraction index c is the tile column: plain 16-byte
//              row reads on both sides.
// Which calls take it, and the kernels for few tokens, for quarters of the columns and for streams of token tiles: below.
// Either way a token tile costs 128 MFMAs per wave against 8 + 32 KB (absorb) or 32 + 8 KB
// of memory traffic: the kernels are bound by memory.

#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "lds_tiles.h"

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <type_traits>

namespace dscuda {
namespace {

constexpr int RANK = 512;       // c
constexpr int HEAD = 128;       // d
constexpr int THREADS = 256;
constexpr int TILE = 32;
constexpr int PITCH = 2 * RANK + 16;            // bytes per weight row in LDS: 16 bytes apart modulo 256
constexpr int TILE_BYTES = TILE * PITCH;
constexpr int WEIGHT_BYTES = (HEAD / TILE) * TILE_BYTES;   // 133 120
constexpr int AHEAD = 6;

// W[h] ([128][512], `weight`) -> LDS, 16-byte pieces
// (sixteen loads in flight per thread and round trip: one at a time, the 32 round trips of a thread's share were a
// third of the kernel's time)
__device__ __forceinline__ void stage_weight(unsigned char* lds, const bf16_t* weight, int tid) {
    constexpr int PIECES = HEAD * RANK / 8;
    constexpr int PER_THREAD = PIECES / THREADS;   // 32
    constexpr int BATCH = 16;
    static_assert(PER_THREAD * THREADS == PIECES && PER_THREAD % BATCH == 0, "the weight must divide evenly");
#pragma unroll
    for (int first = 0; first < PER_THREAD; first += BATCH) {
        u32x4 bits[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
            bits[j] = *reinterpret_cast<const u32x4*>(weight + 8 * (tid + (first + j) * THREADS));
        }
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
            const int piece = tid + (first + j) * THREADS;
            const int row = piece / (RANK / 8);
            const int chunk = piece % (RANK / 8);
            *reinterpret_cast<u32x4*>(lds + (row / TILE) * TILE_BYTES + (row % TILE) * PITCH + 16 * chunk) = bits[j];
        }
    }
}

// A wave's results leave through LDS, two 32-column blocks (one 128-byte line per token) at a time: a lane holds
// one token and scattered groups of four columns, and stores straight from the accumulators would touch 32
// different rows with 16 bytes each.
constexpr int STAGE_PITCH = 128 + 16;
constexpr int STAGE_BYTES = TILE * STAGE_PITCH;              // per wave
constexpr int LDS_BYTES = WEIGHT_BYTES + 4 * STAGE_BYTES;

// blocks `first`, `first + 1` of the accumulators -> columns 32 * first .. + 63 of the tile's tokens
template <int BLOCKS>
__device__ __forceinline__ void store_block_pair(const f32x16 (&acc)[BLOCKS], int first, unsigned char* stage, bf16_t* y_head,
                                                 long long y_token_stride, long long tile0, long long tokens, int lane) {
    const int lq = lane % 32;
    const int g = lane / 32;
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            u32x2 packed;
            packed.x = pack_bf16(acc[first + pair][4 * i4 + 0], acc[first + pair][4 * i4 + 1]);
            packed.y = pack_bf16(acc[first + pair][4 * i4 + 2], acc[first + pair][4 * i4 + 3]);
            *reinterpret_cast<u32x2*>(stage + lq * STAGE_PITCH + 64 * pair + 16 * i4 + 8 * g) = packed;
        }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's LDS writes have landed
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 8 * r + lane / 8;
        const int chunk = lane % 8;
        const u32x4 bits = *reinterpret_cast<const u32x4*>(stage + row * STAGE_PITCH + 16 * chunk);
        if (tile0 + row < tokens) {
            *reinterpret_cast<u32x4*>(y_head + (tile0 + row) * y_token_stride + 32 * first + 8 * chunk) = bits;
        }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);   // the reads are done before the next pair overwrites the stage
    __builtin_amdgcn_wave_barrier();
}

// The 16 bytes at 16ks + 8g of a token's row for every k-step (zeros for a token past the end).
template <int KSTEPS>
__device__ __forceinline__ void fetch_token_row(u32x4 (&bits)[KSTEPS], const bf16_t* row, bool valid, int g) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        bits[ks] = u32x4{0, 0, 0, 0};
        if (valid) bits[ks] = *reinterpret_cast<const u32x4*>(row + 16 * ks + 8 * g);
    }
}

struct Strides {
    long long x_token, x_head, y_token, y_head, w_head;   // in elements
};

// q_latent = q_nope W_UK
__global__ __launch_bounds__(THREADS) void mla_absorb_query_kernel(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
                                                                   const bf16_t* __restrict__ weight, long long tokens,
                                                                   long long tokens_per_workgroup, Strides strides) {
    constexpr int KSTEPS = HEAD / 16;      // 8
    constexpr int BLOCKS = RANK / 32;      // 16 output column blocks
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = tid / 64;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int head = blockIdx.y;
    stage_weight(lds, weight + head * strides.w_head, tid);
    unsigned char* stage = lds + WEIGHT_BYTES + wave * STAGE_BYTES;
    __syncthreads();

    // transposing reads: in a block of 16 lanes, lane s points at row 4*g + s/4 (+8), columns 4*(s%4)..+3 of
    // the block's 16 columns
    const int s = lane % 16;
    const int half = (lane / 16) % 2;
    const int lane_offset = (4 * g + s / 4) * PITCH + 32 * half + 8 * (s % 4);
    auto weight_fragment = [&](auto tag) {
        constexpr int I = decltype(tag)::value;   // k-step I / BLOCKS, column block I % BLOCKS
        constexpr int KS = I / BLOCKS;
        constexpr int BLOCK = I % BLOCKS;
        const unsigned char* at = lds + (KS / 2) * TILE_BYTES + (KS % 2) * 16 * PITCH + lane_offset + 64 * BLOCK;
        const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)at);
        const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(at + 8 * PITCH));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    // a wave's tiles: tile0, tile0 + 128, ... below `end`; the rows of the next tile are fetched while this one is multiplied
    const long long first = (long long)blockIdx.x * tokens_per_workgroup;
    const long long end = min(first + tokens_per_workgroup, tokens);
    const bf16_t* x_head = x + head * strides.x_head;
    auto row_of = [&](long long tile0) { return x_head + min(tile0 + lq, tokens - 1) * strides.x_token; };
    u32x4 next_bits[KSTEPS];
    fetch_token_row(next_bits, row_of(first + TILE * wave), first + TILE * wave + lq < tokens, g);
    for (long long tile0 = first + TILE * wave; tile0 < end; tile0 += TILE * 4) {
        // The token operand has to hold columns {16ks + 4g .. +3, 16ks + 8 + 4g .. +3}, the order of the transposing
        // reads.  Each lane loads the 16 bytes at 16ks + 8g; exchanging the second half of the g = 0 lane's with the
        // first half of the g = 1 lane's (v_permlane32_swap on the two dwords of each half) gives that order.
        bf16x8 xf[KSTEPS];
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            const auto first_pair = __builtin_amdgcn_permlane32_swap(next_bits[ks][0], next_bits[ks][2], false, false);
            const auto second_pair = __builtin_amdgcn_permlane32_swap(next_bits[ks][1], next_bits[ks][3], false, false);
            xf[ks] = __builtin_bit_cast(bf16x8, u32x4{first_pair[0], second_pair[0], first_pair[1], second_pair[1]});
        }
        if (tile0 + TILE * 4 < end) fetch_token_row(next_bits, row_of(tile0 + TILE * 4), tile0 + TILE * 4 + lq < tokens, g);
        f32x16 acc[BLOCKS];
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[b][i] = 0.f;
        }
        bf16x8 ring[AHEAD];
        unrolled<0, AHEAD>([&](auto tag) { ring[decltype(tag)::value] = weight_fragment(tag); });
        unrolled<0, KSTEPS * BLOCKS>([&](auto tag) {
            constexpr int I = decltype(tag)::value;
            acc[I % BLOCKS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[I % AHEAD], xf[I / BLOCKS], acc[I % BLOCKS], 0, 0, 0);
            if constexpr (I + AHEAD < KSTEPS * BLOCKS) {
                ring[I % AHEAD] = weight_fragment(std::integral_constant<int, I + AHEAD>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        // lane holds token lq and columns 32*b + 8*(i/4) + 4*g + i%4
#pragma unroll
        for (int b = 0; b < BLOCKS; b += 2) {
            store_block_pair(acc, b, stage, y + head * strides.y_head, strides.y_token, tile0, tokens, lane);
        }
    }
}

// out = o_latent W_UV^T
__global__ __launch_bounds__(THREADS) void mla_unabsorb_output_kernel(bf16_t* __restrict__ y,
                                                                      const bf16_t* __restrict__ x,
                                                                      const bf16_t* __restrict__ weight,
                                                                      long long tokens, long long tokens_per_workgroup,
                                                                      Strides strides) {
    constexpr int KSTEPS = RANK / 16;      // 32
    constexpr int BLOCKS = HEAD / 32;      // 4 output column blocks = the weight's four row tiles
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = tid / 64;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int head = blockIdx.y;
    stage_weight(lds, weight + head * strides.w_head, tid);
    unsigned char* stage = lds + WEIGHT_BYTES + wave * STAGE_BYTES;
    __syncthreads();

    auto weight_fragment = [&](auto tag) {
        constexpr int I = decltype(tag)::value;   // k-step I / BLOCKS, output block (weight row tile) I % BLOCKS
        constexpr int KS = I / BLOCKS;
        constexpr int BLOCK = I % BLOCKS;
        return *reinterpret_cast<const bf16x8*>(lds + BLOCK * TILE_BYTES + lq * PITCH + 32 * KS + 16 * g);
    };

    const long long first = (long long)blockIdx.x * tokens_per_workgroup;
    const long long end = min(first + tokens_per_workgroup, tokens);
    const bf16_t* x_head = x + head * strides.x_head;
    auto row_of = [&](long long tile0) { return x_head + min(tile0 + lq, tokens - 1) * strides.x_token; };
    u32x4 next_bits[KSTEPS];
    fetch_token_row(next_bits, row_of(first + TILE * wave), first + TILE * wave + lq < tokens, g);
    for (long long tile0 = first + TILE * wave; tile0 < end; tile0 += TILE * 4) {
        bf16x8 xf[KSTEPS];
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) xf[ks] = __builtin_bit_cast(bf16x8, next_bits[ks]);
        if (tile0 + TILE * 4 < end) fetch_token_row(next_bits, row_of(tile0 + TILE * 4), tile0 + TILE * 4 + lq < tokens, g);
        f32x16 acc[BLOCKS];
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[b][i] = 0.f;
        }
        bf16x8 ring[AHEAD];
        unrolled<0, AHEAD>([&](auto tag) { ring[decltype(tag)::value] = weight_fragment(tag); });
        unrolled<0, KSTEPS * BLOCKS>([&](auto tag) {
            constexpr int I = decltype(tag)::value;
            acc[I % BLOCKS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[I % AHEAD], xf[I / BLOCKS], acc[I % BLOCKS], 0, 0, 0);
            if constexpr (I + AHEAD < KSTEPS * BLOCKS) {
                ring[I % AHEAD] = weight_fragment(std::integral_constant<int, I + AHEAD>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        // lane holds token lq and columns 32*b + 8*(i/4) + 4*g + i%4
#pragma unroll
        for (int b = 0; b < BLOCKS; b += 2) {
            store_block_pair(acc, b, stage, y + head * strides.y_head, strides.y_token, tile0, tokens, lane);
        }
    }
}

// ---- few tokens ---------------------------------------------------------------------
// A decode step has a handful of tokens per head: the kernels above would put a head on one compute unit, which then
// waits for 128 KB of weight before its first product.  Here a workgroup takes a quarter of a head's weight and 32
// tokens, and every load of a thread is in flight at once: one round trip to memory, eight MFMAs a wave.  16 tokens of
// 16 heads: absorb 7.6 -> 3.2 us, un-absorb 6.6 -> 3.7.
//
// Every 32 tokens fetch the weight again, so the kernels for more tokens win once (token tiles) x heads is large.  Absorb by
// quarters, below, against few tokens: equal up to 128 tiles, 6.2 / 7.5 us at 256 (128 tokens of 64 heads), 9.1 / 12.8 at 512.  One
// tile a head fetches it once either way: 7 tokens of 140 heads 8.3 / 4.1, of 500 18.2 / 12.1, 32 of 256 11.7 / 9.3; two tiles, of
// which four waves leave two idle there: 33 of 70 heads 6.0 / 5.2, 64 of 128 7.8 / 7.5, 33 of 250 (500 tiles) 11.9 / 12.9.  Un-absorb, whose weight rows come as 32 bytes of 32 rows an instruction, at 128 tiles 5.1-5.8 against 6.7-9.7 us
// (16 tokens of 128 heads, 128 of 32), at 256 tiles 10.2-12.8 against 8.1-9.8.
constexpr long long ABSORB_FEW_TILES = 128;
constexpr long long UNABSORB_FEW_TILES = 128;

constexpr int SLICE = RANK / 4;                    // output columns of an absorb workgroup
constexpr int SLICE_PITCH = 2 * SLICE + 16;        // bytes; 16 modulo 256 as above
constexpr int SLICE_BYTES = HEAD * SLICE_PITCH;
constexpr int FEW_LDS_BYTES = SLICE_BYTES + TILE * SLICE_PITCH;

// q_latent = q_nope W_UK: blockIdx.x = 4 * head + quarter of the columns, blockIdx.y = 32 tokens; a wave per 32 columns
__global__ __launch_bounds__(THREADS) void mla_absorb_query_few_kernel(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
                                                                       const bf16_t* __restrict__ weight, long long tokens,
                                                                       Strides strides) {
    constexpr int KSTEPS = HEAD / 16;
    constexpr int PIECES = HEAD * SLICE / 8 / THREADS;   // 16-byte pieces of the weight slice per thread
    __shared__ __attribute__((aligned(16))) unsigned char lds[FEW_LDS_BYTES];
    const int tid = threadIdx.x;
    const int wave = tid / 64;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int head = blockIdx.x / 4;
    const int column0 = blockIdx.x % 4 * SLICE;
    const long long tile0 = (long long)blockIdx.y * TILE;

    u32x4 rows[KSTEPS], pieces[PIECES];
    const bf16_t* x_head = x + head * strides.x_head;
    fetch_token_row(rows, x_head + min(tile0 + lq, tokens - 1) * strides.x_token, tile0 + lq < tokens, g);
    const bf16_t* slice = weight + head * strides.w_head + column0;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const int piece = tid + j * THREADS;
        pieces[j] = *reinterpret_cast<const u32x4*>(slice + piece / (SLICE / 8) * RANK + 8 * (piece % (SLICE / 8)));
    }
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const int piece = tid + j * THREADS;
        *reinterpret_cast<u32x4*>(lds + piece / (SLICE / 8) * SLICE_PITCH + 16 * (piece % (SLICE / 8))) = pieces[j];
    }
    __syncthreads();

    // operands as in mla_absorb_query_kernel
    const int s = lane % 16;
    const int half = (lane / 16) % 2;
    const unsigned char* at = lds + (4 * g + s / 4) * SLICE_PITCH + 32 * half + 8 * (s % 4) + 64 * wave;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        const auto first_pair = __builtin_amdgcn_permlane32_swap(rows[ks][0], rows[ks][2], false, false);
        const auto second_pair = __builtin_amdgcn_permlane32_swap(rows[ks][1], rows[ks][3], false, false);
        const bf16x8 xf = __builtin_bit_cast(bf16x8, u32x4{first_pair[0], second_pair[0], first_pair[1], second_pair[1]});
        const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(at + 16 * ks * SLICE_PITCH));
        const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(at + (16 * ks + 8) * SLICE_PITCH));
        const bf16x8 wf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf, acc, 0, 0, 0);
    }
    // lane holds token lq and columns 32*wave + 8*i4 + 4*g .. +3: rows of 256 bytes through LDS
    unsigned char* out_rows = lds + SLICE_BYTES;
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
        u32x2 packed;
        packed.x = pack_bf16(acc[4 * i4 + 0], acc[4 * i4 + 1]);
        packed.y = pack_bf16(acc[4 * i4 + 2], acc[4 * i4 + 3]);
        *reinterpret_cast<u32x2*>(out_rows + lq * SLICE_PITCH + 64 * wave + 16 * i4 + 8 * g) = packed;
    }
    __syncthreads();
    for (int piece = tid; piece < TILE * SLICE / 8; piece += THREADS) {
        const int row = piece / (SLICE / 8);
        const int chunk = piece % (SLICE / 8);
        if (tile0 + row < tokens) {
            *reinterpret_cast<u32x4*>(y + head * strides.y_head + (tile0 + row) * strides.y_token + column0 + 8 * chunk) =
                *reinterpret_cast<const u32x4*>(out_rows + row * SLICE_PITCH + 16 * chunk);
        }
    }
}

// out = o_latent W_UV^T: blockIdx.x = 4 * head + 32 of the weight's rows, blockIdx.y = 32 tokens; each wave contracts a
// quarter of the latent columns, weight rows straight from memory, and the quarters are added in order
__global__ __launch_bounds__(THREADS) void mla_unabsorb_output_few_kernel(bf16_t* __restrict__ y,
                                                                          const bf16_t* __restrict__ x,
                                                                          const bf16_t* __restrict__ weight,
                                                                          long long tokens, Strides strides) {
    constexpr int WAVES = THREADS / 64;
    constexpr int COLUMNS = RANK / WAVES;
    constexpr int KSTEPS = COLUMNS / 16;
    constexpr int SUM_PITCH = TILE + 4;   // floats per token
    __shared__ __attribute__((aligned(16))) float sums[WAVES][TILE * SUM_PITCH];
    const int tid = threadIdx.x;
    const int wave = tid / 64;
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int head = blockIdx.x / 4;
    const int row0 = blockIdx.x % 4 * TILE;
    const long long tile0 = (long long)blockIdx.y * TILE;

    u32x4 rows[KSTEPS], weights[KSTEPS];
    fetch_token_row(weights, weight + head * strides.w_head + (row0 + lq) * RANK + COLUMNS * wave, true, g);
    fetch_token_row(rows, x + head * strides.x_head + min(tile0 + lq, tokens - 1) * strides.x_token + COLUMNS * wave,
                    tile0 + lq < tokens, g);
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, weights[ks]),
                                                      __builtin_bit_cast(bf16x8, rows[ks]), acc, 0, 0, 0);
    }
    // lane holds token lq and weight rows 8*i4 + 4*g .. +3
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
        *reinterpret_cast<f32x4*>(&sums[wave][lq * SUM_PITCH + 8 * i4 + 4 * g]) =
            f32x4{acc[4 * i4], acc[4 * i4 + 1], acc[4 * i4 + 2], acc[4 * i4 + 3]};
    }
    __syncthreads();
    const int token = tid / 8;
    const int column = 4 * (tid % 8);
    f32x4 sum = *reinterpret_cast<const f32x4*>(&sums[0][token * SUM_PITCH + column]);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += *reinterpret_cast<const f32x4*>(&sums[w][token * SUM_PITCH + column]);
    if (tile0 + token < tokens) {
        u32x2 packed;
        packed.x = pack_bf16(sum[0], sum[1]);
        packed.y = pack_bf16(sum[2], sum[3]);
        *reinterpret_cast<u32x2*>(y + head * strides.y_head + (tile0 + token) * strides.y_token + row0 + column) = packed;
    }
}

// ---- more tokens, results that the memory-side cache takes -----------------------------
// q_latent = q_nope W_UK by quarters of the columns: a wave holds the quarter's weight in 128 registers and takes every
// fourth token tile, and two workgroups share a compute unit, so that one's loads and stores go on while the other
// multiplies or fetches its 32 KB of weight (mla_absorb_query_kernel keeps 128 KB in LDS, one workgroup of four waves
// per compute unit, which fetches first and then streams).  blockIdx.x = (chunk of the tokens, head, quarter); the
// quarters of a head, which read the same rows, go to one XCD.  Bound by the bytes written: into the
// results of the call before, 1024 tokens x 128 heads 40.0 -> 32.1 us (168 MB of rows in and out, 5.2 TB/s), 1000 x 64 24.2 -> 19.0,
// 1000 x 16 12.4 -> 8.6, 250 x 64 12.8 -> 8.6; into results of their own 42.9 -> 43.3 (3.9 TB/s), 25.6 -> 24.0, 13.4 -> 9.1, 13.5 -> 9.1.
// Rows written as four times 256 bytes by workgroups of their own are slower once they go to memory.  Whole rows / quarters
// into results of their own: 144 MB (1100 x 128) 46.8 / 46.6, 157 MB 46.8 / 49.9, 168 MB 48.7 / 51.9, 197 MB 54.4 / 59.3; into those
// of the call before 157 MB 43.7 / 36.1, 197 MB 51.1 / 42.8, 223 MB 59.7 / 68.1, 268 MB 72.4 / 84.1.  From 45 MB on calls of
// their own are 0 to 10 % slower by quarters (2594 x 34 32.7 / 36.9; 5777 x 11 23.6 / 28.5), but not between the other operators of
// a layer, absorb, forward and un-absorb: 512 x 128 107.9 / 103.2, 2500 x 32 289.6 / 282.6, 2000 x 64 367.8 / 364.2, 750 x 128 177.0 / 178.1.
// Up to 128 tokens of so many heads that a workgroup of whole rows a head is a nearly full round, quarters are two rounds:
// 33 x 250 10.5 / 12.4, 128 x 200 14.9 / 15.5.
constexpr long long SLICE_RESULT_BYTES = 144LL << 20;
constexpr int XCDS = 8;

__global__ __launch_bounds__(THREADS, 2) void mla_absorb_query_slice_kernel(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
                                                                            const bf16_t* __restrict__ weight,
                                                                            long long tokens, long long tokens_per_workgroup,
                                                                            int heads, Strides strides) {
    constexpr int KSTEPS = HEAD / 16;
    constexpr int BLOCKS = SLICE / 32;
    constexpr int PIECES = HEAD * SLICE / 8 / THREADS;   // 16-byte pieces of the weight slice per thread
    static_assert(4 * TILE * SLICE_PITCH == SLICE_BYTES, "the waves' output rows take the place of the weight");
    __shared__ __attribute__((aligned(16))) unsigned char lds[SLICE_BYTES];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    // groups of eight (chunk, head) one behind the other in blockIdx.x, the last of them filled up
    const unsigned quarter = blockIdx.x / XCDS % 4;
    const unsigned item = blockIdx.x / XCDS / 4 * XCDS + blockIdx.x % XCDS;
    if (item / heads * tokens_per_workgroup >= tokens) return;
    const int head = item % heads;
    const long long chunk = item / heads;
    const int column0 = quarter * SLICE;
    const long long first = chunk * tokens_per_workgroup + TILE * wave;
    const long long end = min((chunk + 1) * tokens_per_workgroup, tokens);
    const bf16_t* x_head = x + head * strides.x_head;
    auto row_of = [&](long long tile0) { return x_head + min(tile0 + lq, tokens - 1) * strides.x_token; };

    u32x4 next_bits[KSTEPS], pieces[PIECES];
    const bf16_t* slice = weight + head * strides.w_head + column0;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const int piece = tid + j * THREADS;
        pieces[j] = *reinterpret_cast<const u32x4*>(slice + piece / (SLICE / 8) * RANK + 8 * (piece % (SLICE / 8)));
    }
    // rows past the end repeat the last one
    fetch_token_row(next_bits, row_of(first), true, g);
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const int piece = tid + j * THREADS;
        *reinterpret_cast<u32x4*>(lds + piece / (SLICE / 8) * SLICE_PITCH + 16 * (piece % (SLICE / 8))) = pieces[j];
    }
    __syncthreads();
    // operands as in mla_absorb_query_kernel
    const int s = lane % 16;
    const unsigned char* at = lds + (4 * g + s / 4) * SLICE_PITCH + 32 * (lane / 16 % 2) + 8 * (s % 4);
    bf16x8 weights[KSTEPS][BLOCKS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            const unsigned char* here = at + 16 * ks * SLICE_PITCH + 64 * b;
            const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)here);
            const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(here + 8 * SLICE_PITCH));
            weights[ks][b] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
    __syncthreads();

    unsigned char* out_rows = lds + wave * TILE * SLICE_PITCH;
    bf16_t* y_head = y + head * strides.y_head + column0;
    for (long long tile0 = first; tile0 < end; tile0 += 4 * TILE) {
        bf16x8 xf[KSTEPS];
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            const auto first_pair = __builtin_amdgcn_permlane32_swap(next_bits[ks][0], next_bits[ks][2], false, false);
            const auto second_pair = __builtin_amdgcn_permlane32_swap(next_bits[ks][1], next_bits[ks][3], false, false);
            xf[ks] = __builtin_bit_cast(bf16x8, u32x4{first_pair[0], second_pair[0], first_pair[1], second_pair[1]});
        }
        if (tile0 + 4 * TILE < end) fetch_token_row(next_bits, row_of(tile0 + 4 * TILE), true, g);
#pragma unroll
        for (int pair = 0; pair < BLOCKS; pair += 2) {
            f32x16 acc[2];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(weights[ks][pair], xf[ks], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(weights[ks][pair + 1], xf[ks], acc[1], 0, 0, 0);
            }
            // lane holds token lq and columns 32*block + 8*i4 + 4*g .. +3
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    *reinterpret_cast<u32x2*>(out_rows + lq * SLICE_PITCH + 64 * (pair + b) + 16 * i4 + 8 * g) =
                        u32x2{pack_bf16(acc[b][4 * i4 + 0], acc[b][4 * i4 + 1]), pack_bf16(acc[b][4 * i4 + 2], acc[b][4 * i4 + 3])};
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's LDS writes have landed
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int row = 4 * j + lane / 16;   // 256 bytes of four rows an instruction
            const u32x4 bits = *reinterpret_cast<const u32x4*>(out_rows + row * SLICE_PITCH + 16 * (lane % 16));
            if (tile0 + row < end) {
                *reinterpret_cast<u32x4*>(y_head + (tile0 + row) * strides.y_token + 8 * (lane % 16)) = bits;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);   // the reads are done before the next tile's rows take their place
        __builtin_amdgcn_wave_barrier();
    }
}

// out = o_latent W_UV^T as a stream of token tiles: a wave holds 32 of the head's 128 weight rows in 128 registers, the four
// waves of a workgroup read each tile of 32 tokens from LDS, whole rows of 1 KB brought there by global_load_lds two tiles
// ahead, a workgroup a compute unit (its LDS admits a second one, for what does not come out even).  Workgroup index =
// chunk * heads + head.  Bound by the rows read.  mla_unabsorb_output_kernel, each of whose waves fetches a token's row 32
// bytes at a time and keeps 128 KB of weight in LDS, -> here, us, inputs that are not in the caches: 1024 tokens x 128 heads
// 41.1 -> 33.9 (185 MB, 5.5 TB/s), 4096 x 128 135 -> 125, 512 x 128 26.2 -> 19.9, 300 x 128 22.4 -> 14.5, 200 x 300 36 -> 27,
// 1000 x 64 25.9 -> 20.1, 1000 x 16 10.9 -> 9.5, 700 x 8 9.9 -> 7.6, 4000 x 8 13.2 / 13.3.  Three or four tiles ahead: 34.3 / 34.5,
// 122 / 123, 20.7 / 21.1, 15.5 / 16.2, 31 / 32, 20.7 / 21.4.
constexpr int STREAM_TILE_BYTES = TILE * 2 * RANK;           // 32 KB
constexpr int STREAM_SLOTS = 2;
constexpr int STREAM_OUT_AT = STREAM_SLOTS * STREAM_TILE_BYTES;
constexpr int STREAM_OUT_PITCH = 2 * HEAD + 16;
constexpr int STREAM_LDS_BYTES = STREAM_OUT_AT + TILE * STREAM_OUT_PITCH;
static_assert(2 * STREAM_LDS_BYTES <= 160 * 1024, "two workgroups fit a compute unit");

// BYPASS: rows that do not all survive in the caches behind the forward that wrote them are read around them.  Forward and
// un-absorb, us, as usual / so: 600 tokens x 128 heads (79 MB) 108.5 / 109.2, 1200 x 64 (79) 149.2 / 150.1, 660 x 128 (87)
// 123.2 / 122.5, 4 x 340 x 64 (89) 99.3 / 99.8, 700 x 128 (92) 133.9 / 131.0, 16 x 90 x 64 (94) 95.2 / 89.1, 768 x 128 (101) 151.3 / 145.9,
// 3200 x 32 (105) 371.6 / 364.9, 1024 x 128 (134) 223.9 / 223.2, 2048 x 128 683 / 678.  4096 x 128 alone 125.5 / 117.6.
constexpr long long BYPASS_BYTES = 84LL << 20;

// Up to so many heads an XCD takes a run of indices, that is all heads of its tokens.  Dealt one by one, with 4, 8 or 16 heads an XCD
// has the same one or two heads of all tokens, 1 KB of every 4 or 8.  us, whole weights in LDS / dealt / runs: 4000 tokens x 4 heads
// 10.2 / 11.4 / 9.1, 8000 x 8 25.5 / 26.1 / 22.3, 16000 x 8 42.1 / 41.3 / 33.3, 2000 x 16 15.6 / 16.9 / 14.1, 8192 x 16 41.9 / 43.8 /
// 34.0.  More heads share their weights in an L2 when dealt: 1000 x 24 13.3 / 11.3 / 11.6, 1000 x 48 23.7 / 17.6 / 18.3, 300 x 64 12.4 /
// 10.3 / 12.0, 4096 x 128 135.7 / 117.8 / 126.3; 1000 x 32 equal, 4096 x 32 43.5 / 38.0 / 35.2.
constexpr int RUN_HEADS = 16;

template <bool BYPASS>
__global__ __launch_bounds__(THREADS, 2) void mla_unabsorb_output_stream_kernel(bf16_t* __restrict__ y,
                                                                                const bf16_t* __restrict__ x,
                                                                                const bf16_t* __restrict__ weight,
                                                                                long long tokens,
                                                                                long long tokens_per_workgroup, int heads,
                                                                                Strides strides) {
    constexpr int KSTEPS = RANK / 16;
    constexpr int ROWS = TILE / (THREADS / 64);    // of a tile that a wave requests, one an instruction
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const unsigned index = heads <= RUN_HEADS ? index_math::run_index(blockIdx.x, gridDim.x) : blockIdx.x;
    const int head = index % (unsigned)heads;
    const long long first = index / (unsigned)heads * tokens_per_workgroup;
    const int tiles = (int)((min(tokens_per_workgroup, tokens - first) + TILE - 1) / TILE);
    const bf16_t* x_head = x + head * strides.x_head;
    const unsigned lds_base = lds_offset_of(lds);
    auto request = [&](int tile) {
        const long long token0 = first + (long long)tile * TILE;
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int row = ROWS * wave + i;
            // rows past the end repeat the last one, nothing of theirs is stored
            const bf16_t* source = x_head + min(token0 + row, tokens - 1) * strides.x_token;
            const unsigned chunk = 16u * (unsigned)(lane ^ index_math::tile_swizzle<2 * RANK>(row));
            const unsigned target = lds_base + tile % STREAM_SLOTS * STREAM_TILE_BYTES + row * 2 * RANK;
            if constexpr (BYPASS) direct_load_16_offset_streaming(source, chunk, target);
            else direct_load_16_offset(source, chunk, target);
        }
    };
    u32x4 weights[KSTEPS];
    fetch_token_row(weights, weight + head * strides.w_head + (TILE * wave + lq) * RANK, true, g);
    for (int tile = 0; tile < min(tiles, STREAM_SLOTS); ++tile) request(tile);
    TileReads<2 * RANK> reads;
    reads.init(lane);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" : "+v"(weights[ks]));   // here, not at every use
    for (int tile = 0; tile < tiles; ++tile) {
        // The tile has landed; the requests of the next one, the youngest of this wave, may be on their way.
        if (tile + 1 < tiles) wait_vector_memory<ROWS>(); else wait_vector_memory<0>();
        workgroup_barrier();
        unsigned at[TileReads<2 * RANK>::NAT];
        rebase(at, reads.natural, tile % STREAM_SLOTS * STREAM_TILE_BYTES);
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
        bf16x8 ring[AHEAD];
        unrolled<0, AHEAD>([&](auto tag) { ring[decltype(tag)::value] = natural_fragment<2 * RANK, 0, decltype(tag)::value>(lds, at); });
        unrolled<0, KSTEPS>([&](auto tag) {
            constexpr int I = decltype(tag)::value;
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, weights[I]), ring[I % AHEAD], acc, 0, 0, 0);
            if constexpr (I + AHEAD < KSTEPS) ring[I % AHEAD] = natural_fragment<2 * RANK, 0, I + AHEAD>(lds, at);
            __builtin_amdgcn_sched_barrier(0);
        });
        // lane holds token lq and columns 32*wave + 8*i4 + 4*g .. +3: rows of 256 bytes through LDS
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            *reinterpret_cast<u32x2*>(lds + STREAM_OUT_AT + lq * STREAM_OUT_PITCH + 64 * wave + 16 * i4 + 8 * g) =
                u32x2{pack_bf16(acc[4 * i4 + 0], acc[4 * i4 + 1]), pack_bf16(acc[4 * i4 + 2], acc[4 * i4 + 3])};
        }
        workgroup_barrier();   // the rows are there, and everybody has read the tile
        const long long token0 = first + (long long)tile * TILE;
        bf16_t* y_tile = y + head * strides.y_head + token0 * strides.y_token;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = 8 * wave + 4 * j + lane / 16;   // 256 bytes of four rows an instruction
            const u32x4 bits = *reinterpret_cast<const u32x4*>(lds + STREAM_OUT_AT + row * STREAM_OUT_PITCH + 16 * (lane % 16));
            if (token0 + row < tokens) *reinterpret_cast<u32x4*>(y_tile + row * strides.y_token + 8 * (lane % 16)) = bits;
        }
        // behind the stores: the wait above then counts these requests alone
        if (tile + STREAM_SLOTS < tiles) request(tile + STREAM_SLOTS);
    }
}

void check(bool condition, const char* message) {
    if (!condition) throw std::invalid_argument(message);
}

int compute_units() {
    return hip_common::compute_units_of_current_device();
}

bool rows_apart(const bf16_t* y, const bf16_t* x, long long tokens, int heads, const Strides& strides, int x_width, int y_width) {
    const long long offset = ((long long)reinterpret_cast<uintptr_t>(y) - (long long)reinterpret_cast<uintptr_t>(x)) / 2;
    return index_math::rows_apart({strides.x_token, strides.x_head, x_width}, {strides.y_token, strides.y_head, y_width}, offset,
                                  tokens, heads);
}

template <typename Kernel>
void launch_few(Kernel kernel, bf16_t* y, const bf16_t* x, const bf16_t* weight, long long tokens, int heads,
                const Strides& strides, hipStream_t stream) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(4 * heads), (unsigned)((tokens + TILE - 1) / TILE)), dim3(THREADS), 0, stream, y,
                       x, weight, tokens, strides);
    HIP_CHECK(hipGetLastError());
}

// Chunks that fill one to four rounds of two workgroups per compute unit, and of these the shortest schedule: rounds
// times the cost of a workgroup, which fetches its quarter of the weight in the time of some 128 tokens.
void launch_slices(bf16_t* y, const bf16_t* x, const bf16_t* weight, long long tokens, int heads, const Strides& strides,
                   hipStream_t stream) {
    constexpr long long STAGING_TOKENS = 4 * TILE;
    constexpr long long GRANULE = 4 * TILE;
    const long long slots = 2LL * std::max(1, compute_units());
    long long per_workgroup = 0, best = -1;
    for (long long rounds = 1; rounds <= 4; ++rounds) {
        const long long chunks = std::max(1LL, rounds * slots / (4LL * heads));
        const long long per_chunk = ((tokens + chunks - 1) / chunks + GRANULE - 1) / GRANULE * GRANULE;
        const long long workgroups = 4LL * heads * ((tokens + per_chunk - 1) / per_chunk);
        const long long cost = (workgroups + slots - 1) / slots * (STAGING_TOKENS + per_chunk);
        if (best < 0 || cost < best) {
            best = cost;
            per_workgroup = per_chunk;
        }
    }
    const long long chunks = (tokens + per_workgroup - 1) / per_workgroup;
    const long long grid = 4 * XCDS * ((chunks * heads + XCDS - 1) / XCDS);
    check(grid <= 0x7fffffffLL, "MLA projection: more tokens than the grid allows");
    hipLaunchKernelGGL(mla_absorb_query_slice_kernel, dim3((unsigned)grid), dim3(THREADS), 0, stream, y, x, weight, tokens,
                       per_workgroup, heads, strides);
    HIP_CHECK(hipGetLastError());
}

// The tokens of a head are cut into chunks, one workgroup each, multiples of `granule` tokens; every
// workgroup fetches the head's weight first, which costs it about as long as 128 tokens.  The number of chunks is
// the one with the shortest schedule: rounds of workgroups over the compute units times the cost of a workgroup
// (whole weights in LDS, 4096 tokens x 128 heads on 256 compute units: two chunks, one round, 138 / 171 us against 145 / 178
// us with four; un-absorb as a stream, 1024 x 128: 256 workgroups 33.5 us, 128 45.5, 384 37.3, 512 36.0, 768 40.3).
long long tokens_per_workgroup(long long tokens, int heads, long long granule) {
    constexpr long long STAGING_TOKENS = 4 * TILE;
    const long long units = std::max(1, compute_units());
    const long long most = (tokens + granule - 1) / granule;
    const long long limit = std::min(most, std::max(1LL, (4 * units + heads - 1) / heads));
    long long chunks = 1, best = -1;
    for (long long candidate = 1; candidate <= limit; ++candidate) {
        const long long per_chunk = ((tokens + candidate - 1) / candidate + granule - 1) / granule * granule;
        const long long workgroups = heads * ((tokens + per_chunk - 1) / per_chunk);
        const long long cost = (workgroups + units - 1) / units * (STAGING_TOKENS + per_chunk);
        if (best < 0 || cost < best) {
            best = cost;
            chunks = candidate;
        }
    }
    return ((tokens + chunks - 1) / chunks + granule - 1) / granule * granule;
}

// Whole weights in LDS: chunks are multiples of the 128 tokens four waves take.
template <typename Kernel>
void launch_whole(Kernel kernel, bf16_t* y, const bf16_t* x, const bf16_t* weight, long long tokens, int heads,
                  const Strides& strides, hipStream_t stream) {
    const long long per_workgroup = tokens_per_workgroup(tokens, heads, 4 * TILE);
    const long long grid = (tokens + per_workgroup - 1) / per_workgroup;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid, (unsigned)heads), dim3(THREADS), LDS_BYTES, stream, y, x, weight,
                       tokens, per_workgroup, strides);
    HIP_CHECK(hipGetLastError());
}

template <bool BYPASS>
void launch_stream(bf16_t* y, const bf16_t* x, const bf16_t* weight, long long tokens, int heads, const Strides& strides,
                   hipStream_t stream) {
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_unabsorb_output_stream_kernel<BYPASS>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, STREAM_LDS_BYTES));
    });
    const long long per_workgroup = tokens_per_workgroup(tokens, heads, TILE);
    const long long grid = (tokens + per_workgroup - 1) / per_workgroup * heads;
    check(grid <= 0x7fffffffLL, "MLA projection: more tokens than the grid allows");
    hipLaunchKernelGGL(mla_unabsorb_output_stream_kernel<BYPASS>, dim3((unsigned)grid), dim3(THREADS), STREAM_LDS_BYTES, stream,
                       y, x, weight, tokens, per_workgroup, heads, strides);
    HIP_CHECK(hipGetLastError());
}

void validate(const void* y, const void* x, const void* weight, long long tokens, int heads, const Strides& s,
              int x_width, int y_width) {
    check(tokens > 0 && heads > 0, "MLA projection: tokens and heads must be positive");
    check(y != nullptr && x != nullptr && weight != nullptr, "MLA projection: null tensor");
    check(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(y) % 16 == 0,
          "MLA projection: tensors must be aligned to 16 bytes");
    check(s.x_token % 8 == 0 && s.x_head % 8 == 0 && s.w_head % 8 == 0 && s.y_token % 8 == 0 && s.y_head % 8 == 0,
          "MLA projection: strides must be multiples of 8 elements (rows aligned to 16 bytes)");
    check(s.x_head >= x_width && s.y_head >= y_width && s.x_token >= s.x_head * (heads - 1) + x_width &&
              s.y_token >= s.y_head * (heads - 1) + y_width && s.w_head >= (long long)HEAD * RANK,
          "MLA projection: strides smaller than the rows they separate");
}

}  // namespace

void mla_absorb_query_dispatch(bf16_t* query_latent, const bf16_t* query_nope, const bf16_t* weight, long long tokens,
                               int heads, long long query_nope_token_stride, long long query_nope_head_stride,
                               long long query_latent_token_stride, long long query_latent_head_stride,
                               long long weight_head_stride, hipStream_t stream) {
    const Strides strides = {query_nope_token_stride, query_nope_head_stride, query_latent_token_stride,
                             query_latent_head_stride, weight_head_stride};
    validate(query_latent, query_nope, weight, tokens, heads, strides, HEAD, RANK);
    check(heads <= 65535, "MLA projection: more heads than the grid allows");
    const long long tiles = (tokens + TILE - 1) / TILE;
    const bool apart = rows_apart(query_latent, query_nope, tokens, heads, strides, HEAD, RANK);
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_absorb_query_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES));
    });
    const long long units = compute_units();
    const bool full_round = tokens <= 4 * TILE && heads <= units && 4LL * heads > 3 * units;   // whole rows, a workgroup a head
    if (apart && (tiles == 1 || tiles * heads <= (tiles == 2 ? 2 : 1) * ABSORB_FEW_TILES)) {
        launch_few(mla_absorb_query_few_kernel, query_latent, query_nope, weight, tokens, heads, strides, stream);
    } else if (!apart || full_round || tokens * heads * (2LL * RANK) > SLICE_RESULT_BYTES) {
        launch_whole(mla_absorb_query_kernel, query_latent, query_nope, weight, tokens, heads, strides, stream);
    } else {
        launch_slices(query_latent, query_nope, weight, tokens, heads, strides, stream);
    }
}

void mla_unabsorb_output_dispatch(bf16_t* output, const bf16_t* output_latent, const bf16_t* weight, long long tokens,
                                  int heads, long long output_latent_token_stride, long long output_latent_head_stride,
                                  long long output_token_stride, long long output_head_stride,
                                  long long weight_head_stride, hipStream_t stream) {
    const Strides strides = {output_latent_token_stride, output_latent_head_stride, output_token_stride,
                             output_head_stride, weight_head_stride};
    validate(output, output_latent, weight, tokens, heads, strides, RANK, HEAD);
    check(heads <= 65535, "MLA projection: more heads than the grid allows");
    const long long tiles = (tokens + TILE - 1) / TILE;
    const bool apart = rows_apart(output, output_latent, tokens, heads, strides, RANK, HEAD);
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_unabsorb_output_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES));
    });
    if (apart && tiles * heads <= UNABSORB_FEW_TILES) {
        launch_few(mla_unabsorb_output_few_kernel, output, output_latent, weight, tokens, heads, strides, stream);
        return;
    }
    if (apart) {
        const bool bypass = tokens * heads * (2LL * RANK) >= BYPASS_BYTES;
        (bypass ? launch_stream<true> : launch_stream<false>)(output, output_latent, weight, tokens, heads, strides, stream);
        return;
    }
    launch_whole(mla_unabsorb_output_kernel, output, output_latent, weight, tokens, heads, strides, stream);
}

}  // namespace dscuda
