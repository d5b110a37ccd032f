// Query gradients of the absorbed MLA backward from dS that the key-gradient launch has kept:
// dQ [rows, 576] = dS [rows, keys] [latent | rope], a plain causal product.
//
// mla_absorbed_query_gradient_kernel (mla_absorbed.hip) forms the scores and dP a second time, 1088 of its 1664
// multiplications per (row, key) pair; with dS in memory (index_math::KeptGradients, T * rows bytes and a little)
// this launch carries the other 576 and reads two bytes a pair instead.
//
// 2048 tokens x 128 heads: 815 us of query gradients there, 358 here, for 77 us more in the key gradients, whose score
// waves store the 0.55 GB (1236 -> 1313); 2 x 592 x 16 35 -> 24.
//
// A workgroup of eight waves owns 64 * GROUP rows and walks the 32-key tiles they see, all of them through LDS stages
// of [32 keys][512] + [32 keys][64] + dS.  Wave (r, v) = (w / 4, w % 4): row tiles GROUP * r .., latent column blocks
// 4v .. 4v + 3 of each of them and one of the rope blocks.  Bound by the key tiles a compute unit draws from its L2
// (36 KB a step, some 21 bytes a cycle against 1152 matrix cycles at GROUP = 2), hence 128 rows wherever that leaves
// workgroups enough; 192 rows need more registers than there are.  With few rows a workgroup takes half of the columns
// (PARTS = 2, 18 KB of keys a step and compute unit).
// The fragments are read a few products ahead, at GROUP = 2 with a tile's requests spread among the products. The backward in us
// with requests and fragments in front of the products instead, -> here (gradient rows with ordinary stores): 1000 tokens x 64
// heads 251 / 252, 2048 x 16 247 -> 245, 4096 x 32 1577 -> 1566, 2048 x 128 1679 -> 1664. 256 rows and half of the columns a
// workgroup, the halves side by side on an XCD, draw as many bytes and are not faster, here / there, both with rows
// past the caches: 1000 x 64 235 / 248, 2048 x 16 244 / 249, 4096 x 8 465 / 477, 1024 x 128 486 / 498, 2048 x 128 1658 / 1683;
// 8 x 300 x 32 157 / 156.
#include "attn_kernels.h"
#include "hip_common.h"
#include "index_math.h"
#include "lds_tiles.h"

#include <cstdint>

namespace dscuda {
namespace {

constexpr int RANK = 512;
constexpr int ROPE = 64;
constexpr int TILE = 32;
constexpr int THREADS = 512;

template <int GROUP, int PARTS>
struct ProductLayout {
    static_assert(PARTS == 1 || GROUP == 1, "halves of the columns are for few rows");
    static constexpr int ROWS = 64 * GROUP;
    static constexpr int ROW_TILES = 2 * GROUP;
    static constexpr int WIDE_ROW = 2 * RANK / PARTS;
    static constexpr int NARROW_ROW = 2 * ROPE;
    static constexpr int ROPE_AT = TILE * WIDE_ROW;
    static constexpr int DS_AT = ROPE_AT + TILE * NARROW_ROW;
    static constexpr int STAGE_BYTES = DS_AT + ROW_TILES * index_math::KeptGradients::BLOCK_BYTES;
    static constexpr int STAGES = GROUP == 1 ? 4 : 3;
    static constexpr int OUT_ROPE = WIDE_ROW;                            // of a staged gradient row
    static constexpr int OUT_PITCH = WIDE_ROW + 2 * ROPE / PARTS + 16;
    static constexpr int OUT_BYTES = ROWS * OUT_PITCH;
    static constexpr int LDS_BYTES = STAGES * STAGE_BYTES > OUT_BYTES ? STAGES * STAGE_BYTES : OUT_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a compute unit");
};

template <int GROUP, int PARTS>
__global__ __launch_bounds__(THREADS) void mla_absorbed_query_product_kernel(
    bf16_t* __restrict__ query_latent_gradient, bf16_t* __restrict__ query_rope_gradient,
    const unsigned char* __restrict__ kept_gradients, const bf16_t* __restrict__ kv_latent,
    const bf16_t* __restrict__ key_rope, int batch_size, int sequence_length, int heads, int key_tiles, int row_blocks) {
    using L = ProductLayout<GROUP, PARTS>;
    using Wide = index_math::TileReadMath<L::WIDE_ROW>;
    using Narrow = index_math::TileReadMath<L::NARROW_ROW>;
    constexpr int LATENT_BLOCKS = RANK / TILE / 4 / PARTS;   // 32-column blocks of a wave
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int lane = tid % 64;
    const int lq = lane % 32;
    const int g = lane / 32;
    const int T = sequence_length;
    const long long rows = (long long)T * heads;
    const int column_part = blockIdx.x % PARTS;
    const int batch = blockIdx.x / PARTS % batch_size;
    const int row_block = row_blocks - 1 - blockIdx.x / PARTS / batch_size;   // latest rows (most keys) first
    const long long row0 = (long long)row_block * L::ROWS;
    const long long batch_row0 = (long long)batch * rows;
    const unsigned char* latent = reinterpret_cast<const unsigned char*>(kv_latent + (size_t)batch * T * RANK) + column_part * L::WIDE_ROW;
    const unsigned char* rope = reinterpret_cast<const unsigned char*>(key_rope + (size_t)batch * T * ROPE);
    const int tiles = (int)((min(row0 + L::ROWS, rows) - 1) / heads) / TILE + 1;   // key tiles the rows see
    const index_math::KeptGradients kept = index_math::kept_gradients(T, heads, key_tiles);
    const unsigned char* kept_batch = kept_gradients + (size_t)batch * kept.bytes();
    const int first_row_tile = row_block * L::ROW_TILES;

    const int v = wave % 4;
    const int wave_row_tile = GROUP * (wave / 4);   // of the workgroup's
    const int rope_tile = GROUP == 1 ? 0 : v / 2;   // whose rope block the wave sums; GROUP = 1: not every wave has one
    const int rope_block = PARTS == 1 ? v % 2 : column_part;
    const bool sums_rope = GROUP > 1 || v < 2 / PARTS;

    // A wave requests key rows 4*wave .. +3 of the wide tile (1 KB an instruction), waves 0 .. 3 also eight rows of the narrow one, and 1 KB,
    // half a row tile, of dS: every wave at GROUP = 2, waves 4 .. 7 at GROUP = 1.  Keys past the end repeat the last
    // one (their dS is zero), row tiles past the end repeat the last one (their results are not stored), and a tile
    // that does not see the keys yet may read what precedes its blocks and is left out below.
    const unsigned lds_base = lds_offset_of(lds);
    const int ds_part = GROUP == 1 ? wave - 4 : wave;
    const int ds_row_tile = min(first_row_tile + max(ds_part, 0) / 2, kept.visits.row_tiles - 1);
    // request I (0 .. REQUESTS - 1) of a tile
    constexpr int WIDE_REQUESTS = 4 / PARTS;
    constexpr int REQUESTS = WIDE_REQUESTS + 2;
    auto request = [&](int tile, auto tag) {
        constexpr int I = decltype(tag)::value;
        const unsigned target = lds_base + tile % L::STAGES * L::STAGE_BYTES;
        if constexpr (I < WIDE_REQUESTS) {
            const int last = min(T - tile * TILE, TILE) - 1;
            const int first = 4 * wave + PARTS * I;
            const int key = first + lane / (64 / PARTS);
            const int chunk = lane % (64 / PARTS) ^ index_math::tile_swizzle<L::WIDE_ROW>(key);
            direct_load_16_offset(latent + (size_t)tile * TILE * (2 * RANK), (unsigned)(min(key, last) * (2 * RANK) + 16 * chunk),
                                  target + first * L::WIDE_ROW);
        } else if constexpr (I == WIDE_REQUESTS) {
            if (wave < 4) {
                const int last = min(T - tile * TILE, TILE) - 1;
                const int key = 8 * wave + lane / 8;
                direct_load_16_offset(rope + (size_t)tile * TILE * L::NARROW_ROW,
                                      (unsigned)(min(key, last) * L::NARROW_ROW +
                                                 16 * ((lane % 8) ^ index_math::tile_swizzle<L::NARROW_ROW>(key))),
                                      target + L::ROPE_AT + 8 * wave * L::NARROW_ROW);
            }
        } else if (GROUP > 1 || wave >= 4) {
            direct_load_16_offset_streaming(kept_batch + kept.at(tile, ds_row_tile) + 1024 * (ds_part % 2), 16u * (unsigned)lane,
                                            target + L::DS_AT + 1024 * ds_part);
        }
    };
    auto request_tile = [&](int tile) {
        unrolled<0, REQUESTS>([&](auto tag) { request(tile, tag); });
    };
    // all but the newest `tiles_in_flight` tiles of the wave's requests have arrived
    auto wait_for_all_but = [&](auto tiles_in_flight) {
        constexpr int N = decltype(tiles_in_flight)::value;
        if (GROUP > 1 && wave < 4) wait_vector_memory<REQUESTS * N>(); else wait_vector_memory<(REQUESTS - 1) * N>();
    };
    constexpr int AHEAD = L::STAGES - 1;
    for (int tile = 0; tile < min(tiles, AHEAD); ++tile) request_tile(tile);

    unsigned wide_at[2][LATENT_BLOCKS], narrow_at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < LATENT_BLOCKS; ++j) {
            const int block = LATENT_BLOCKS * v + j;
            wide_at[h][j] = Wide::transposed(h, block % Wide::TR, lane) + 64 * Wide::TR * (block / Wide::TR);
        }
        narrow_at[h] = L::ROPE_AT + Narrow::transposed(h, rope_block, lane);
    }
    // dS as it was kept: key k of a block in bytes 64k .., the transposing read takes four keys of 16 rows
    const unsigned ds_at = L::DS_AT + wave_row_tile * index_math::KeptGradients::BLOCK_BYTES +
                           64 * (4 * g + lane % 16 / 4) + 16 * (lane % 4) + 8 * (lane / 16 % 2);
    f32x16 sum[GROUP][LATENT_BLOCKS], rope_sum;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        rope_sum[i] = 0.f;
#pragma unroll
        for (int t = 0; t < GROUP; ++t) {
#pragma unroll
            for (int j = 0; j < LATENT_BLOCKS; ++j) sum[t][j][i] = 0.f;
        }
    }
    // One key tile; the wave's row tiles from FIRST on see it.  Those before are left out, not multiplied by zeros: a key
    // that is not finite would reach rows of earlier tokens.
    auto step = [&](int tile, auto first_tag) {
        constexpr int FIRST = decltype(first_tag)::value;
        const int behind = min(tiles - 1 - tile, AHEAD - 1);   // tiles that may stay in flight
        if (behind == 0) {
            wait_for_all_but(std::integral_constant<int, 0>{});
        } else if (AHEAD == 2 || behind == 1) {
            wait_for_all_but(std::integral_constant<int, 1>{});
        } else {
            wait_for_all_but(std::integral_constant<int, 2>{});
        }
        workgroup_barrier();   // the tile is there, and the stage of the tile before has been read
        const bool more = tile + AHEAD < tiles;
        // Few rows: the requests, a step's longest part, go first (1000 tokens x 8 heads 104.3 us, among the products 107.4).
        constexpr bool SPREAD = GROUP == 2 && FIRST < GROUP;
        if (!SPREAD && more) request_tile(tile + AHEAD);
        if constexpr (FIRST < GROUP) {
            // one stream of products, its fragments read RING column blocks ahead
            const unsigned char* stage = lds + tile % L::STAGES * L::STAGE_BYTES;
            auto fragment = [&](unsigned low_at, unsigned high_at) {
                const s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(stage + low_at));
                const s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((transposing_read_pointer)(stage + high_at));
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
            };
            constexpr int COUNT = 2 * LATENT_BLOCKS;   // column blocks of two 16-key steps
            constexpr int RING = LATENT_BLOCKS < 3 ? LATENT_BLOCKS : 3;
            bf16x8 ds[2][GROUP], ring[RING], narrow[2];
            auto read_ds = [&](int n) {
#pragma unroll
                for (int t = FIRST; t < GROUP; ++t) {
                    const unsigned at = ds_at + t * index_math::KeptGradients::BLOCK_BYTES + 1024 * n;
                    ds[n][t] = fragment(at, at + 512);
                }
            };
            auto read_columns = [&](auto tag) {
                constexpr int I = decltype(tag)::value;
                constexpr int N = I / LATENT_BLOCKS, J = I % LATENT_BLOCKS;
                ring[I % RING] = fragment(wide_at[0][J] + 16 * N * L::WIDE_ROW, wide_at[1][J] + 16 * N * L::WIDE_ROW);
            };
            const bool own_rope = sums_rope && rope_tile >= FIRST;
            read_ds(0);
            unrolled<0, RING>(read_columns);
            unrolled<0, COUNT>([&](auto tag) {
                constexpr int I = decltype(tag)::value;
                constexpr int N = I / LATENT_BLOCKS, J = I % LATENT_BLOCKS;
#pragma unroll
                for (int t = FIRST; t < GROUP; ++t) {
                    sum[t][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[I % RING], ds[N][t], sum[t][J], 0, 0, 0);
                }
                if constexpr (I == LATENT_BLOCKS - RING) read_ds(1);
                if constexpr (I + RING < COUNT) read_columns(std::integral_constant<int, I + RING>{});
                if constexpr (J == LATENT_BLOCKS - 2 + LATENT_BLOCKS % 2) {
                    if (own_rope) narrow[N] = fragment(narrow_at[0] + 16 * N * L::NARROW_ROW, narrow_at[1] + 16 * N * L::NARROW_ROW);
                }
                if (SPREAD && more) {
                    unrolled<I * REQUESTS / COUNT, (I + 1) * REQUESTS / COUNT>([&](auto piece) { request(tile + AHEAD, piece); });
                }
                if constexpr (J == LATENT_BLOCKS - 1) {
                    if (own_rope) {
                        bf16x8 own = ds[N][FIRST];
                        if (GROUP > 1 && rope_tile == 1) own = ds[N][GROUP - 1];
                        rope_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(narrow[N], own, rope_sum, 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    };
    // key tile t is seen from row 32 * t * heads on, the first row of row tile t * heads
    const int wave_tile = first_row_tile + wave_row_tile;
    const int seen_by_all = min(wave_tile / heads + 1, tiles);
    int tile = 0;
    for (; tile < seen_by_all; ++tile) step(tile, std::integral_constant<int, 0>{});
    if constexpr (GROUP == 2) {
        const int seen_by_second = min((wave_tile + 1) / heads + 1, tiles);
        for (; tile < seen_by_second; ++tile) step(tile, std::integral_constant<int, 1>{});
    }
    for (; tile < tiles; ++tile) step(tile, std::integral_constant<int, GROUP>{});

    // A lane holds row lq of its row tiles and columns 32*block + 8*(i/4) + 4*g + i%4: rows through LDS, so that a store
    // instruction writes whole lines
    workgroup_barrier();
    auto stage_block = [&](const f32x16& values, int row_tile, int byte) {
        unsigned char* staged = lds + (TILE * row_tile + lq) * L::OUT_PITCH + byte + 8 * g;
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            *reinterpret_cast<u32x2*>(staged + 16 * i4) =
                u32x2{pack_bf16(values[4 * i4 + 0], values[4 * i4 + 1]), pack_bf16(values[4 * i4 + 2], values[4 * i4 + 3])};
        }
    };
#pragma unroll
    for (int t = 0; t < GROUP; ++t) {
#pragma unroll
        for (int j = 0; j < LATENT_BLOCKS; ++j) stage_block(sum[t][j], wave_row_tile + t, 2 * TILE * (LATENT_BLOCKS * v + j));
    }
    if (sums_rope) stage_block(rope_sum, wave_row_tile + rope_tile, L::OUT_ROPE + (PARTS == 1 ? 2 * TILE * rope_block : 0));
    workgroup_barrier();
    const int valid_rows = (int)min((long long)L::ROWS, rows - row0);
    constexpr int LANES = 64 / PARTS;   // of a row
    for (int out_row = PARTS * wave + lane / LANES; out_row < valid_rows; out_row += PARTS * THREADS / 64) {
        const size_t target = batch_row0 + row0 + out_row;
        const int part = lane % LANES;
        const unsigned char* staged = lds + out_row * L::OUT_PITCH + 16 * part;
        // (past the caches, backward and then a product that reads the rows, us, this / that: 300 tokens x 128 heads 122 / 125, 512 x 128
        // 208 / 207, 1024 x 128 532 / 532, 4096 x 32 1593 / 1609, 3000 x 128 3492 / 3501, 1000 x 64 272 / 269, 40 x 85 x 64 335 / 340)
        *reinterpret_cast<u32x4*>(query_latent_gradient + target * RANK + column_part * (RANK / PARTS) + 8 * part) =
            *reinterpret_cast<const u32x4*>(staged);
        if (part < ROPE / 8 / PARTS) {
            *reinterpret_cast<u32x4*>(query_rope_gradient + target * ROPE + column_part * (ROPE / PARTS) + 8 * part) =
                *reinterpret_cast<const u32x4*>(staged + L::OUT_ROPE);
        }
    }
}

template <int GROUP, int PARTS>
void launch(bf16_t* query_latent_gradient, bf16_t* query_rope_gradient, const unsigned char* kept_gradients,
            const bf16_t* kv_latent, const bf16_t* key_rope, int batch_size, int sequence_length, int heads, int key_tiles,
            hipStream_t stream) {
    using L = ProductLayout<GROUP, PARTS>;
    static hip_common::OncePerDevice prepared;
    prepared.run([] {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mla_absorbed_query_product_kernel<GROUP, PARTS>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, L::LDS_BYTES));
    });
    const long long rows = (long long)sequence_length * heads;
    const long long row_blocks = (rows + L::ROWS - 1) / L::ROWS;
    hipLaunchKernelGGL((mla_absorbed_query_product_kernel<GROUP, PARTS>), dim3((unsigned)(row_blocks * batch_size * PARTS)), dim3(THREADS),
                       L::LDS_BYTES, stream, query_latent_gradient, query_rope_gradient, kept_gradients, kv_latent, key_rope,
                       batch_size, sequence_length, heads, key_tiles, (int)row_blocks);
    HIP_CHECK(hipGetLastError());
}

}  // namespace

void mla_absorbed_query_product_launch(bf16_t* query_latent_gradient, bf16_t* query_rope_gradient,
                                       const unsigned char* kept_gradients, const bf16_t* kv_latent,
                                       const bf16_t* key_rope, int batch_size, int sequence_length, int heads,
                                       int key_tiles, hipStream_t stream) {
    // 128 rows a workgroup where that is a workgroup per compute unit. The whole backward in us, 64 / 128 rows: 148 workgroups of
    // 128 98 / 103, 226 82 / 81, 282 349 / 350, 304 118 / 114, 512 235 / 228, 1500 1995 / 1895; 33 81 / 87;
    // not for elements of at most 64 rows: 568 x 1 x 1 30.9 / 33.9, 1079 x 8 x 7 91 / 97.
    // Workgroups of 64 rows and half the columns where whole rows are no workgroup per compute unit, halves / whole rows: 38 workgroups
    // of 64 rows 45 / 49, 63 63 / 68, 128 106 / 118, 220 (2010 x 7) 130 / 143, 159 (3 x 279 x 12) 49 / 51; but where the halves are
    // more than one round of them, short walks pay for a second start: 165 x 1 x 1 17.0 / 14.7, 57 x 21 x 11 32.5 / 30.1,
    // 14 x 73 x 12 40.4 / 38.2, 47 x 133 x 1 30.7 / 29.6, 3 x 182 x 20 45.9 / 44.9; 3 x 204 x 14 41.2 / 42.0.
    constexpr int SHORT_TOKENS = 192;
    const long long rows = (long long)sequence_length * heads;
    const int units = hip_common::compute_units_of_current_device();
    auto start = [&](auto launch_form) {
        launch_form(query_latent_gradient, query_rope_gradient, kept_gradients, kv_latent, key_rope, batch_size, sequence_length,
                    heads, key_tiles, stream);
    };
    const long long workgroups = (rows + 63) / 64 * batch_size;   // of 64 rows
    if (rows > 64 && (rows + 127) / 128 * batch_size >= units) {
        start(launch<2, 1>);
    } else if (workgroups > units || (2 * workgroups > units && sequence_length <= SHORT_TOKENS)) {
        start(launch<1, 1>);
    } else {
        start(launch<1, 2>);
    }
}

}  // namespace dscuda
