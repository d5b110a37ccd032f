// Row-major swizzled LDS tiles of bf16 rows: the global -> LDS requests that fill one and the reads of MFMA operand
// fragments out of it (index_math::TileRequestMath, TileReadMath).  A tile is stored once and read both ways: 16-byte
// row reads where the contraction runs along the columns, transposing reads where it runs along the rows.
#pragma once

#include "hip_common.h"
#include "index_math.h"

namespace dscuda {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* transposing_read_pointer;

// One wave's share of the global_load_lds requests of a [ROWS][ROW_BYTES] tile that
// WAVES waves fetch together; the offsets are those of index_math::TileRequestMath.
// Full tiles take the fast form (a per-lane base per residue, computed once, plus
// compile-time constants); at a ragged end rows past `row_limit` repeat that row
// (general form).
template <int ROW_BYTES, int WAVES, int ROWS = 64>
struct TileRequests {
    using Math = index_math::TileRequestMath<ROW_BYTES, WAVES, ROWS>;
    static constexpr int LOADS = Math::LOADS;
    static constexpr int PERIOD = Math::PERIOD;
    unsigned base[PERIOD];

    __device__ __forceinline__ void init(unsigned row_stride, int wave, int lane) {
#pragma unroll
        for (int r = 0; r < PERIOD; ++r) base[r] = Math::base_of(r, lane, row_stride, wave);
    }
    // `tile` = address of the tile's first row (uniform)
    __device__ __forceinline__ void request(const unsigned char* tile, unsigned row_stride, int row_limit,
                                            unsigned lds_target, int wave) const {
        if (row_limit >= ROWS - 1) {
            const unsigned char* rows = tile + (size_t)Math::rows_before(0, wave) * row_stride;
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                direct_load_16_offset(rows + (size_t)Math::rows_before(i, 0) * row_stride,
                                      Math::lane_part(base[i % PERIOD], i), lds_target + (wave * LOADS + i) * 1024);
            }
        } else {
            const int lane = fresh_lane_id();
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                direct_load_16_offset(tile, Math::offset_of(wave * LOADS + i, lane, row_stride, row_limit),
                                      lds_target + (wave * LOADS + i) * 1024);
            }
        }
    }
    // The same for a row stride whose tile may span more than 32 bits of address, a 64-bit address per lane and load:
    // for tiles that are loaded once.
    static __device__ __forceinline__ void request_far(const unsigned char* tile, size_t row_stride, int row_limit,
                                                       unsigned lds_target, int wave) {
        const int lane = fresh_lane_id();
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int load = wave * LOADS + i;
            direct_load_16(tile + (size_t)min(Math::row_of(load, lane), row_limit) * row_stride + 16 * Math::chunk_of(load, lane),
                           lds_target + load * 1024);
        }
    }
};

// Per-lane byte offsets of the fragment reads of a row-major swizzled tile
// (index_math::TileReadMath); a user adds the (run-time) tile base to the per-lane
// values once per tile.
template <int ROW_BYTES>
struct TileReads {
    using Math = index_math::TileReadMath<ROW_BYTES>;
    static constexpr int NAT = Math::NAT;
    static constexpr int TR = Math::TR;
    unsigned natural[NAT];
    unsigned transposed[2][TR];

    __device__ __forceinline__ void init(int lane) {
#pragma unroll
        for (int i = 0; i < NAT; ++i) natural[i] = Math::natural(i, lane);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < TR; ++i) transposed[h][i] = Math::transposed(h, i, lane);
        }
    }
};

// `at` = TileReads::natural plus the tile's LDS offset; rows ROW0 + lane%32, k-step KS
template <int ROW_BYTES, int ROW0, int KS>
__device__ __forceinline__ bf16x8 natural_fragment(const unsigned char* lds, const unsigned (&at)[TileReads<ROW_BYTES>::NAT]) {
    using Math = index_math::TileReadMath<ROW_BYTES>;
    return *reinterpret_cast<const bf16x8*>(lds + at[KS % Math::NAT] + Math::natural_constant(ROW0, KS));
}

// `at` = TileReads::transposed plus the tile's LDS offset; 16 rows from ROW0, column block BLOCK
template <int ROW_BYTES, int ROW0, int BLOCK>
__device__ __forceinline__ bf16x8 transposed_fragment(const unsigned char* lds,
                                                      const unsigned (&at)[2][TileReads<ROW_BYTES>::TR]) {
    using Math = index_math::TileReadMath<ROW_BYTES>;
    constexpr int CONSTANT = Math::transposed_constant(ROW0, BLOCK);
    const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (transposing_read_pointer)(lds + at[0][BLOCK % Math::TR] + CONSTANT));
    const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (transposing_read_pointer)(lds + at[1][BLOCK % Math::TR] + CONSTANT));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
}

// at = reads + offset, as values the optimiser cannot take apart again: the
// fragment reads then keep the form (per-lane register) + (immediate) instead of
// one address computation per read.
__device__ __forceinline__ unsigned opaque(unsigned value) {
    asm volatile("" : "+v"(value));
    return value;
}
template <int N>
__device__ __forceinline__ void rebase(unsigned (&at)[N], const unsigned (&reads)[N], unsigned offset) {
#pragma unroll
    for (int i = 0; i < N; ++i) at[i] = opaque(reads[i] + offset);
}
template <int N>
__device__ __forceinline__ void rebase(unsigned (&at)[2][N], const unsigned (&reads)[2][N], unsigned offset) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < N; ++i) at[h][i] = opaque(reads[h][i] + offset);
    }
}

}  // namespace
}  // namespace dscuda
