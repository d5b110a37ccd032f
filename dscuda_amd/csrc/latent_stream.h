// The shared 576-wide latent key stream in units of 32 keys: where a unit lies in memory (paged, contiguous, or
// latent and rope parts in tensors of their own), the global -> LDS requests that fetch it, and the fragment reads
// of a unit in LDS.  Used by the absorbed decode and prefill-forward kernels.
#pragma once

#include "hip_common.h"
#include "index_math.h"

namespace dscuda {
namespace {

constexpr int RANK = 512;
constexpr int ROPE = 64;
constexpr int WIDTH = RANK + ROPE;
constexpr int BN = 64;                      // keys per tile, the grain of the decode work list
constexpr int CHUNKS = WIDTH / 8;           // 72 16-byte chunks per key row
constexpr int ROW_BYTES = CHUNKS * 16;      // 1152

constexpr int UNIT = 32;
constexpr int UNIT_BYTES = UNIT * ROW_BYTES;              // 36 KB
constexpr int UNIT_SLOTS = 4;
constexpr int LOAD_WAVES = 4;                             // waves that share the requests of a unit
constexpr int UNIT_LOADS = UNIT * CHUNKS / (64 * LOAD_WAVES);   // 9 wave instructions of 1 KB per wave and unit
static_assert(UNIT_LOADS * 64 * LOAD_WAVES == UNIT * CHUNKS, "unit loads must divide evenly");

__device__ __forceinline__ int swizzle_of_row(int row) {
    return index_math::tile_swizzle<ROW_BYTES>(row);
}

__device__ __forceinline__ int tiles_of(int length) {
    return (max(length, 0) + BN - 1) / BN;
}

struct KeyStream {
    const bf16_t* latent;      // token t at latent + t*latent_stride, 512 wide
    const bf16_t* rope;        // token t at rope + t*rope_stride, 64 wide
    size_t latent_stride;
    size_t rope_stride;
    const int* block_table;    // nullptr: tokens are stored contiguously
    int page_size;
};

struct UnitSource {
    const bf16_t* base;      // first row of the unit (contiguous form; split form: of its latent part)
    const bf16_t* rope_base; // split form: first row of the unit's rope part
    unsigned lds_base;       // LDS byte offset of this wave's 9 KB of the unit's slot
    int key0;
    int row_limit;           // rows above it repeat it (>= 0: the unit holds a visible token)
    bool contiguous;         // the unit is one run of rows: no paging, or pages that hold whole units
    bool split;              // no paging, latent and rope parts in tensors of their own, offsets that fit 32 bits
    bool full;               // all 32 rows are visible tokens: the per-lane offsets are the same for every such unit
    bool enabled;
};

// Hands out the sources of consecutive units of one sequence.  The decode cache is packed
// (576-wide rows), so only paging decides the form.  When pages hold whole units, the ids of
// 64 consecutive pages of the sequence sit in one register (lane l: page first_page + l) and a
// unit finds its page with one lane read: a scalar load per unit would have its wait drain the
// LDS queue as well, in the middle of the fragment stream.
struct UnitCursor {
    int unit;                // the unit handed out next
    int page;                // its page (index into the sequence's block table) ...
    int within;              // ... and its place inside that page, in units
    int units_per_page;
    int first_page;          // page whose id lane 0 of `ids` holds
    int last_page;           // last page of the sequence with a visible token: no entry past it is read
    int ids;
    bool paged;
    bool contiguous;
    bool split;

    // Waits for the ids on the spot (the empty asm statement is their first use): a wait left to the
    // first lane read would sit on the path of every step and wait for the unit requests as well.
    __device__ __forceinline__ void load_ids(const KeyStream& keys, int from) {
        first_page = from;
        ids = keys.block_table[min(from + fresh_lane_id(), last_page)];
        asm volatile("" : "+v"(ids));
    }

    __device__ __forceinline__ void init(const KeyStream& keys, int first_unit, int last_token) {
        paged = keys.block_table != nullptr;
        contiguous = !paged || (keys.page_size % UNIT == 0);
        split = false;
        unit = __builtin_amdgcn_readfirstlane(first_unit);
        page = within = units_per_page = first_page = last_page = ids = 0;
        if (paged && contiguous) {
            units_per_page = __builtin_amdgcn_readfirstlane(keys.page_size / UNIT);
            page = __builtin_amdgcn_readfirstlane(first_unit / units_per_page);
            within = __builtin_amdgcn_readfirstlane(first_unit - page * units_per_page);
            last_page = __builtin_amdgcn_readfirstlane(last_token / keys.page_size);
            load_ids(keys, page);
        }
    }

    // Pages that do not hold whole units: every key finds its own page when the unit is requested.
    __device__ __forceinline__ void init_key_by_key(int first_unit) {
        paged = true;
        contiguous = split = false;
        unit = __builtin_amdgcn_readfirstlane(first_unit);
        page = within = units_per_page = first_page = last_page = ids = 0;
    }

    __device__ __forceinline__ UnitSource next(unsigned char* lds, const KeyStream& keys, int last_token, int wave,
                                               int unit_end) {
        UnitSource source;
        source.contiguous = contiguous;
        source.split = split;
        source.enabled = unit < unit_end;
        source.key0 = unit * UNIT;
        source.row_limit = last_token - source.key0;
        source.full = source.row_limit >= UNIT - 1;
        source.lds_base = __builtin_amdgcn_readfirstlane(lds_offset_of(lds) + ((unsigned)unit % UNIT_SLOTS) * UNIT_BYTES +
                                                         wave * (UNIT_LOADS * 1024));
        source.base = keys.latent;
        source.rope_base = keys.rope;
        if (split) {
            source.base = keys.latent + (size_t)source.key0 * keys.latent_stride;
            source.rope_base = keys.rope + (size_t)source.key0 * keys.rope_stride;
        }
        if (source.enabled && contiguous) {
            long long physical = source.key0;
            if (paged) {
                // enabled: the unit holds a visible token, so page <= last_page
                if (page - first_page >= 64) load_ids(keys, page);
                const int id = __builtin_amdgcn_readlane(ids, page - first_page);
                physical = (long long)id * keys.page_size + within * UNIT;
            }
            source.base = keys.latent + physical * WIDTH;
        }
        ++unit;
        if (paged && contiguous && ++within == units_per_page) {
            within = 0;
            ++page;
        }
        return source;
    }
};

// Per-lane offsets of the nine loads of a full unit (no row past the end of the sequence).
struct FullUnitOffsets {
    unsigned of[UNIT_LOADS];

    __device__ __forceinline__ void init(int wave, int lane) {
#pragma unroll
        for (int i = 0; i < UNIT_LOADS; ++i) {
            of[i] = index_math::contiguous_load_offset<ROW_BYTES, UNIT / 4>(wave, i, lane, UNIT - 1);
        }
    }
};

// Load number i (0..8) of a contiguous unit; i is a constant after unrolling.
__device__ __forceinline__ void issue_unit_load(const UnitSource& source, const FullUnitOffsets& offsets, int wave, int i,
                                                int lane) {
    const unsigned offset = source.full
        ? offsets.of[i]
        : index_math::contiguous_load_offset<ROW_BYTES, UNIT / 4>(wave, i, lane, source.row_limit);
    direct_load_16_offset_streaming(source.base, offset, source.lds_base + i * 1024);   // each head group reads the cache once
}

// Load I of a unit whose latent and rope parts lie in tensors of their own, unpaged (`split`): a wave instruction
// covers at most two rows of the unit (compile-time boundary), and a lane's 16 bytes come from the one tensor or the
// other.  Row strides stay below 2^24 elements (the caller saw to that).
template <int I>
__device__ __forceinline__ void issue_split_load(const UnitSource& source, const KeyStream& keys, int wave, int lane) {
    constexpr int FIRST_ROW = (64 * I) / CHUNKS;                 // of the wave's eight rows: the row of lane 0
    constexpr int BOUNDARY = CHUNKS * (FIRST_ROW + 1) - 64 * I;   // first lane of the next row (64 or more: none)
    // what depends on the row is the same for all lanes of a row: two candidates, wave-uniform
    const int row = (UNIT / 4) * wave + FIRST_ROW;
    const int swizzle[2] = {swizzle_of_row(row), swizzle_of_row(row + 1)};
    const unsigned row_here[2] = {(unsigned)min(row, source.row_limit), (unsigned)min(row + 1, source.row_limit)};
    const bool second = BOUNDARY < 64 && lane >= BOUNDARY;
    const int position = lane + (64 * I - CHUNKS * FIRST_ROW) - (second ? CHUNKS : 0);
    const int chunk = position ^ (second ? swizzle[1] : swizzle[0]);
    const bool rope = chunk >= RANK / 8;
    // bytes from the first row of the unit's part in the lane's tensor (the bases of the source hold key0 * stride)
    const unsigned row_bytes = __umul24(second ? row_here[1] : row_here[0],
                                        rope ? 2u * (unsigned)keys.rope_stride : 2u * (unsigned)keys.latent_stride);
    const unsigned bytes = row_bytes + 16u * (unsigned)chunk - (rope ? 2u * RANK : 0u);
    const unsigned char* part = reinterpret_cast<const unsigned char*>(rope ? source.rope_base : source.base);
    direct_load_16(part + bytes, source.lds_base + I * 1024);
}

// All nine loads of a unit whose rows are found one by one: a page lookup per lane, or strides beyond those of `split`.
__device__ __forceinline__ void issue_unit_key_by_key(const UnitSource& source, const KeyStream& keys, bool paged, int wave) {
    if (!source.enabled) return;
    const int lane = fresh_lane_id();
#pragma unroll 1
    for (int i = 0; i < UNIT_LOADS; ++i) {
        const int slot = 64 * i + lane;
        const int row = (UNIT / 4) * wave + slot / CHUNKS;
        const int chunk = (slot % CHUNKS) ^ swizzle_of_row(row);
        const int token = source.key0 + min(row, source.row_limit);
        long long physical = token;
        if (paged) {
            const int page = keys.block_table[token / keys.page_size];
            physical = (long long)page * keys.page_size + token % keys.page_size;
        }
        const bf16_t* address = chunk < RANK / 8 ? keys.latent + physical * keys.latent_stride + 8 * chunk
                                                 : keys.rope + physical * keys.rope_stride + 8 * (chunk - RANK / 8);
        direct_load_16(address, source.lds_base + i * 1024);
    }
}

// All nine loads of a unit at once, of any form.
__device__ __forceinline__ void issue_unit(const UnitSource& source, const FullUnitOffsets& offsets, const KeyStream& keys,
                                           int wave) {
    if (!source.enabled) return;
    const int lane = fresh_lane_id();
    if (source.contiguous) {
#pragma unroll
        for (int i = 0; i < UNIT_LOADS; ++i) issue_unit_load(source, offsets, wave, i, lane);
        return;
    }
    if (source.split) {
        unrolled<0, UNIT_LOADS>([&](auto tag) { issue_split_load<decltype(tag)::value>(source, keys, wave, lane); });
        return;
    }
    issue_unit_key_by_key(source, keys, keys.block_table != nullptr, wave);
}

// Per-lane byte offsets of the fragment reads inside a unit (rows 0..31 of 1152 bytes).
// K operand: row lane%32, 16-byte chunk 2*ks + g at position (2*ks + g) ^ f(row); the XOR
// only mixes the low three bits, so four offsets plus (ks/4)*128 reach every k-step.
// V^T operand through transposing reads: in a block of 16 lanes, lane s points at row
// 4*g + s/4 (+8 for the second read), columns 4*(s%4)..+3 of the 16-column group
// 16*(block%2); bit 2 of f moves a row's data by one 64-byte column block, which two
// offsets per read (even / odd column block) turn back into immediates.
struct UnitReads {
    unsigned k[4];
    unsigned v_first[2];
    unsigned v_second[2];

    __device__ __forceinline__ void init(int lane) {
        const int lq = lane % 32;
        const int g = lane / 32;
        const int swz = swizzle_of_row(lq);
#pragma unroll
        for (int j = 0; j < 4; ++j) k[j] = lq * ROW_BYTES + ((2 * j + g) ^ swz) * 16;
        const int s16 = lane % 16;
        const int block = lane / 16;
        const int row1 = 4 * g + s16 / 4;
        const int f1 = swizzle_of_row(row1);
        const int chunk_low = (2 * (block % 2) + (s16 % 4) / 2) ^ (f1 & 3);
        const int flip = 64 * ((row1 >> 1) & 1);
        const int lane1 = row1 * ROW_BYTES + chunk_low * 16 + 8 * (s16 & 1);
        const int lane2 = (row1 + 8) * ROW_BYTES + (chunk_low ^ 1) * 16 + 8 * (s16 & 1);
        v_first[0] = lane1 + flip;
        v_first[1] = lane1 - flip;
        v_second[0] = lane2 + flip;
        v_second[1] = lane2 - flip;
    }
};

typedef short unit_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) unit_s16x4* unit_tr_pointer;

template <int KS>
__device__ __forceinline__ bf16x8 unit_key_fragment(const unsigned char* unit, const UnitReads& reads) {
    return *reinterpret_cast<const bf16x8*>(unit + reads.k[KS % 4] + (KS / 4) * 128);
}

// 16-key step N (0, 1) of the unit, column block D (0..15)
template <int N, int D>
__device__ __forceinline__ bf16x8 unit_value_fragment(const unsigned char* unit, const UnitReads& reads) {
    constexpr int CONSTANT = N * 16 * ROW_BYTES + D * 64;
    const unit_s16x4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((unit_tr_pointer)(unit + reads.v_first[D % 2] + CONSTANT));
    const unit_s16x4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((unit_tr_pointer)(unit + reads.v_second[D % 2] + CONSTANT));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
}

// ---- decode: a workgroup's range of the work list -----------------------------------------------------------------

using index_math::PLAN_HEADER;
using index_math::PLAN_MODE;
using index_math::PLAN_OVERHEAD;
using index_math::PLAN_PARTS;
using index_math::PLAN_RANGES;
using index_math::PLAN_TOTAL;
using index_math::PLAN_WHOLE;
using index_math::PLAN_WIDE_PARTS;
using index_math::PLAN_WORKGROUPS;

constexpr int SELF_PLAN_BATCH = 256;   // sequences a workgroup turns into a plan by itself

struct DecodeRange {
    const int* prefix;   // positions before each sequence, in memory (the caller's plan) or in LDS
    int overhead;
    int begin, end;      // positions of this workgroup's range; begin >= end: nothing to do
    int sequence;        // first sequence that reaches past `begin`
    bool wide;           // parts of cut sequences are kept in fp32
    bool local;          // prefix and lengths lie in LDS
};

// How a call cuts its list (index_math::DecodeLayout).
struct DecodeCut {
    int workgroups;
    int whole_sequences;
    int reference_ranges;
    int wide_ranges;
};

__device__ __forceinline__ int plan_mode(const DecodeCut& cut, bool wide) {
    return cut.whole_sequences ? PLAN_WHOLE : wide ? PLAN_WIDE_PARTS : PLAN_PARTS;
}

// The ranges `total` positions are cut into, and whether with fp32 parts.  Called by all threads of a workgroup;
// `prefix`: positions before each of the batch's sequences, visible to all of them; `fewest`: at most the positions of any
// sequence that has some.  A run of as many tiles as the longest range has positions holds a boundary: where that settles
// it for the shortest sequence, no sequence is looked at (64-bit divisions and a barrier, 0.7 us of a call).
__device__ __forceinline__ int choose_ranges(const DecodeCut& cut, const int* prefix, int batch_size, int total, int fewest,
                                             int overhead, int tid, int threads, bool& wide) {
    wide = false;
    if (cut.reference_ranges > 0 && total > 0) {
        const int reference = index_math::ranges_of(total, cut.reference_ranges);
        if (fewest - overhead - 1 < (total + reference - 1) / reference) {
            int all_cut = 1;
            for (int s = tid; s < batch_size; s += threads) {
                const int before = prefix[s], positions = prefix[s + 1] - before;
                if (positions > 0 && !index_math::sequence_is_cut(total, reference, before, positions, overhead)) all_cut = 0;
            }
            if (__syncthreads_and(all_cut) == 0) {
                wide = cut.wide_ranges > 0;
                return wide ? index_math::ranges_of(total, cut.wide_ranges) : reference;
            }
        }
    }
    return index_math::ranges_of(total, cut.workgroups);
}

__device__ __forceinline__ int wave_min(int value) {
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) value = min(value, __shfl_xor(value, offset));
    return value;
}

// Sum over the lanes up to this one.
__device__ __forceinline__ int wave_prefix_sum(int value) {
    auto add = [&](auto control, auto rows) {
        value += __builtin_amdgcn_update_dpp(0, value, decltype(control)::value, decltype(rows)::value, 0xf, false);
    };
    using All = std::integral_constant<int, 0xf>;
    add(std::integral_constant<int, 0x111>{}, All{});   // row_shr 1, 2, 4, 8: within 16 lanes
    add(std::integral_constant<int, 0x112>{}, All{});
    add(std::integral_constant<int, 0x114>{}, All{});
    add(std::integral_constant<int, 0x118>{}, All{});
    add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});   // row_bcast 15, 31
    add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    return value;
}

// decode_range for at most 64 sequences: every wave scans the batch in its own registers, lane = sequence, without a
// barrier or a search in LDS, and the plan of a caller comes in one round trip with the lengths.  Stamps of a workgroup's
// start: 3.5 us with the scan over a workgroup of 256, 1.0 so (of which a round trip to memory is 0.7).
__device__ __forceinline__ DecodeRange small_decode_range(int* plan, const int* cache_lengths, int batch_size, bool own_plan,
                                                          bool recut, const DecodeCut& cut, int* own_prefix, int* own_lengths,
                                                          int tid, int workgroup, bool leave_plan) {
    DecodeRange range;
    const int lane = tid % 64;
    const int length = cache_lengths[min(lane, batch_size - 1)];
    int before, after, total, ranges;
    bool whole_sequences;
    if (own_plan) {
        whole_sequences = cut.whole_sequences != 0;
        range.overhead = whole_sequences ? 0 : index_math::SEGMENT_OVERHEAD;
        const int positions = lane < batch_size ? index_math::positions_of(tiles_of(length), range.overhead) : 0;
        after = wave_prefix_sum(positions);
        before = after - positions;
        total = __builtin_amdgcn_readlane(after, 63);
        ranges = index_math::ranges_of(total, cut.workgroups);
        range.wide = false;
        if (cut.reference_ranges > 0 && total > 0) {   // as choose_ranges
            const int reference = index_math::ranges_of(total, cut.reference_ranges);
            const bool uncut = positions > 0 && !index_math::sequence_is_cut(total, reference, before, positions, range.overhead);
            if (__builtin_amdgcn_ballot_w64(uncut) != 0) {
                range.wide = cut.wide_ranges > 0;
                ranges = range.wide ? index_math::ranges_of(total, cut.wide_ranges) : reference;
            }
        }
        if (leave_plan && tid < 64) {
            if (lane == 0) {
                plan[PLAN_TOTAL] = total;
                plan[PLAN_WORKGROUPS] = cut.workgroups;
                plan[PLAN_OVERHEAD] = range.overhead;
                plan[PLAN_MODE] = plan_mode(cut, range.wide);
                plan[PLAN_RANGES] = ranges;
                plan[index_math::plan_prefix_at()] = 0;
            }
            if (lane < batch_size) plan[index_math::plan_prefix_at() + lane + 1] = after;
        }
    } else {
        const int* prefix = plan + index_math::plan_prefix_at();
        before = prefix[min(lane, batch_size)];
        after = prefix[min(lane + 1, batch_size)];
        total = __builtin_amdgcn_readfirstlane(plan[PLAN_TOTAL]);
        range.overhead = __builtin_amdgcn_readfirstlane(plan[PLAN_OVERHEAD]);
        const int mode = __builtin_amdgcn_readfirstlane(plan[PLAN_MODE]);
        ranges = __builtin_amdgcn_readfirstlane(plan[PLAN_RANGES]);
        whole_sequences = mode == PLAN_WHOLE;
        range.wide = mode == PLAN_WIDE_PARTS;
        if (recut) ranges = index_math::ranges_of(total, cut.workgroups);
    }
    // the same from every wave, which reads what it wrote
    own_prefix[lane] = before;
    own_prefix[lane + 1] = after;
    own_lengths[lane] = length;
    range.prefix = own_prefix;
    range.local = true;
    range.sequence = 0;
    if (whole_sequences) {
        range.begin = __builtin_amdgcn_readlane(before, workgroup);
        range.end = __builtin_amdgcn_readlane(after, workgroup);
        range.sequence = workgroup;
        return range;
    }
    range.begin = range.end = 0;
    if (workgroup >= ranges) return range;
    range.begin = __builtin_amdgcn_readfirstlane(index_math::range_begin_of(total, ranges, workgroup));
    range.end = __builtin_amdgcn_readfirstlane(index_math::range_begin_of(total, ranges, workgroup + 1));
    // sequences that end before the range
    range.sequence = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < batch_size && after <= range.begin));
    return range;
}

// The plan comes from memory (own_plan false: the caller's, or one mla_decode_plan_kernel has just built), or,
// for a batch that one workgroup scans in one go, is worked out here by every workgroup for itself, which saves the
// call a kernel launch; `leave_plan`: this workgroup then also writes what the merge kernel reads of it.  `recut`: the
// plan in memory was built for other ranges; its positions hold, the ranges are those of `cut`.  Called by
// all threads of a workgroup of at least SELF_PLAN_BATCH threads; the three arrays (own_wave_totals: two ints per 64
// sequences) are in LDS.
__device__ __forceinline__ DecodeRange decode_range(int* plan, const int* cache_lengths, int batch_size, bool own_plan,
                                                    bool recut, const DecodeCut& cut, int* own_prefix, int* own_lengths,
                                                    int* own_wave_totals, int tid, int threads, int workgroup, bool leave_plan) {
    if (batch_size <= 64) {
        return small_decode_range(plan, cache_lengths, batch_size, own_plan, recut, cut, own_prefix, own_lengths, tid, workgroup,
                                  leave_plan);
    }
    DecodeRange range;
    range.local = own_plan;
    int total, ranges;
    bool whole_sequences;
    if (own_plan) {
        whole_sequences = cut.whole_sequences != 0;
        range.overhead = whole_sequences ? 0 : index_math::SEGMENT_OVERHEAD;
        int value = 0;
        if (tid < SELF_PLAN_BATCH) {
            const int own_length = tid < batch_size ? cache_lengths[tid] : 0;
            own_lengths[tid] = own_length;
            value = tid < batch_size ? index_math::positions_of(tiles_of(own_length), range.overhead) : 0;
            const int fewest = cut.reference_ranges > 0 ? wave_min(value > 0 ? value : 0x7fffffff) : 0;
#pragma unroll
            for (int offset = 1; offset < 64; offset <<= 1) {
                const int other = __shfl_up(value, offset);
                if (tid % 64 >= offset) value += other;
            }
            if (tid % 64 == 63) {
                own_wave_totals[tid / 64] = value;
                own_wave_totals[SELF_PLAN_BATCH / 64 + tid / 64] = fewest;
            }
            if (tid == 0) own_prefix[0] = 0;
        }
        __syncthreads();
        if (tid < batch_size) {
            int before = 0;
#pragma unroll
            for (int w = 0; w < SELF_PLAN_BATCH / 64; ++w) {
                if (w < tid / 64) before += own_wave_totals[w];
            }
            own_prefix[tid + 1] = before + value;
        }
        __syncthreads();
        // what comes out of LDS is the same in every lane, which the compiler cannot know
        total = __builtin_amdgcn_readfirstlane(own_prefix[batch_size]);
        int fewest = own_wave_totals[SELF_PLAN_BATCH / 64];
#pragma unroll
        for (int w = 1; w < SELF_PLAN_BATCH / 64; ++w) fewest = min(fewest, own_wave_totals[SELF_PLAN_BATCH / 64 + w]);
        fewest = __builtin_amdgcn_readfirstlane(fewest);
        ranges = choose_ranges(cut, own_prefix, batch_size, total, fewest, range.overhead, tid, threads, range.wide);
        range.prefix = own_prefix;
        if (leave_plan) {
            if (tid == 0) {
                plan[PLAN_TOTAL] = total;
                plan[PLAN_WORKGROUPS] = cut.workgroups;
                plan[PLAN_OVERHEAD] = range.overhead;
                plan[PLAN_MODE] = plan_mode(cut, range.wide);
                plan[PLAN_RANGES] = ranges;
            }
            index_math::leave_prefix(plan, own_prefix, batch_size, tid, threads);
        }
    } else {
        total = plan[PLAN_TOTAL];
        range.overhead = plan[PLAN_OVERHEAD];
        whole_sequences = plan[PLAN_MODE] == PLAN_WHOLE;
        range.wide = plan[PLAN_MODE] == PLAN_WIDE_PARTS;
        ranges = recut ? index_math::ranges_of(total, cut.workgroups) : plan[PLAN_RANGES];
        range.prefix = plan + index_math::plan_prefix_at();
    }

    range.sequence = 0;
    if (whole_sequences) {
        range.begin = __builtin_amdgcn_readfirstlane(range.prefix[workgroup]);
        range.end = __builtin_amdgcn_readfirstlane(range.prefix[workgroup + 1]);
    } else {
        range.begin = range.end = 0;
        if (workgroup >= ranges) return range;
        range.begin = index_math::range_begin_of(total, ranges, workgroup);
        range.end = index_math::range_begin_of(total, ranges, workgroup + 1);
    }
    if (range.begin >= range.end) return range;
    if (own_plan && !whole_sequences) {
        int low = 0, high = batch_size;
        while (low < high) {
            const int mid = (low + high) / 2;
            if (__builtin_amdgcn_readfirstlane(range.prefix[mid + 1]) <= range.begin) low = mid + 1; else high = mid;
        }
        range.sequence = low;
    } else if (own_plan) {
        range.sequence = workgroup;
    } else if (recut) {
        for (int first = 0; first < batch_size; first += 64) {   // sequences that end before the range
            const int s = first + tid % 64;
            range.sequence += __builtin_popcountll(__ballot(s < batch_size && range.prefix[min(s, batch_size - 1) + 1] <= range.begin));
        }
    } else {
        range.sequence = plan[index_math::plan_first_sequence_at(batch_size) + workgroup];
    }
    return range;
}

}  // namespace
}  // namespace dscuda
