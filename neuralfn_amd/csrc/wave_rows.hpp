// Pieces shared by the wave-per-row decode kernels (gemv_dot.hip, gemv_q6.hip):
// fixed-order wave reductions on DPP, the activation load with its fused
// prologue, and the cursor that walks a wave's (row, slice) pairs.
#pragma once

#include "common.hpp"

namespace nfn {

template <int CTRL>
__device__ __forceinline__ int dpp_move(int value) {
    return __builtin_amdgcn_update_dpp(0, value, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float value) {
    return __builtin_bit_cast(float, dpp_move<CTRL>(__builtin_bit_cast(int, value)));
}

constexpr int kQuadXor1 = 0xB1;     // quad_perm [1,0,3,2]
constexpr int kQuadXor2 = 0x4E;     // quad_perm [2,3,0,1]
constexpr int kHalfMirror = 0x141;  // lane k <-> 7-k within 8 lanes
constexpr int kRowMirror = 0x140;   // lane k <-> 15-k within 16 lanes

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Largest of the wave's values, all of them non-negative: such floats order
// like their bit patterns, so the reduction runs on unsigned integers (one
// instruction per step with the lane exchange folded in).  Butterfly within
// rows of 16 lanes, then row 0 -> 1 and 2 -> 3, then lane 31 -> rows 2 and 3:
// lane 63 holds the result.
__device__ __forceinline__ float wave_max(float value) {
    std::uint32_t v = __float_as_uint(value);
    v = max(v, static_cast<std::uint32_t>(dpp_move<kQuadXor1>(static_cast<int>(v))));
    v = max(v, static_cast<std::uint32_t>(dpp_move<kQuadXor2>(static_cast<int>(v))));
    v = max(v, static_cast<std::uint32_t>(dpp_move<kHalfMirror>(static_cast<int>(v))));
    v = max(v, static_cast<std::uint32_t>(dpp_move<kRowMirror>(static_cast<int>(v))));
    constexpr int kRowBroadcast15 = 0x142, kRowBroadcast31 = 0x143;
    v = max(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(
                   static_cast<int>(v), static_cast<int>(v), kRowBroadcast15, 0xA, 0xF, false)));
    v = max(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(
                   static_cast<int>(v), static_cast<int>(v), kRowBroadcast31, 0xC, 0xF, false)));
    return __uint_as_float(static_cast<std::uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(v), 63)));
}

// Sum over the wave in a fixed order; the total is returned in every lane.
__device__ __forceinline__ float wave_total(float v) {
    v += dpp_move<kQuadXor1>(v);
    v += dpp_move<kQuadXor2>(v);
    v += dpp_move<kHalfMirror>(v);
    v += dpp_move<kRowMirror>(v);
    // (row 0 + row 1) + (row 2 + row 3)
    auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    rows = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
}

__device__ __forceinline__ std::uint32_t perm(std::uint32_t hi, std::uint32_t lo, std::uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

constexpr float kCodeRange = 32512.0f;  // 127*256: the high byte stays in [-127, 127]

// Four activations of one lane as 16-bit fixed-point codes, code = x * 32512 /
// (largest magnitude among the wave's 256 values), rounded to nearest even and
// split into two int8 planes: code = 256*hi + lo with lo in [-128, 127].
struct ActivationCodes {
    std::uint32_t hi, lo;  // four bytes each, value order
    int sum;               // of this lane's four codes
    float maximum;         // the wave's largest magnitude; scale = maximum / 32512
};

__device__ __forceinline__ float code_factor(float maximum) {
    return maximum > 1.0e-30f ? kCodeRange * __builtin_amdgcn_rcpf(maximum) : 0.0f;
}
__device__ __forceinline__ void encode_quad(float4 x, float factor, std::uint32_t& hi, std::uint32_t& lo) {
    // 1.5*2^23 + 128: the low 16 bits of the sum's bit pattern are
    // round-to-nearest-even(x*factor) + 128 in two's complement.
    constexpr float kMagic = 12582912.0f + 128.0f;
    const std::uint32_t u0 = __float_as_uint(fmaf(x.x, factor, kMagic));
    const std::uint32_t u1 = __float_as_uint(fmaf(x.y, factor, kMagic));
    const std::uint32_t u2 = __float_as_uint(fmaf(x.z, factor, kMagic));
    const std::uint32_t u3 = __float_as_uint(fmaf(x.w, factor, kMagic));
    // code + 128 = 256*hi + (lo + 128): hi is byte 1, lo is byte 0 with its top bit flipped
    const std::uint32_t p01 = perm(u1, u0, 0x05010400u);  // [u0.b0, u1.b0, u0.b1, u1.b1]
    const std::uint32_t p23 = perm(u3, u2, 0x05010400u);
    lo = perm(p23, p01, 0x05040100u) ^ 0x80808080u;
    hi = perm(p23, p01, 0x07060302u);
}

__device__ __forceinline__ ActivationCodes encode_activations(float4 x) {
    const float local = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
    ActivationCodes codes;
    codes.maximum = wave_max(local);
    encode_quad(x, code_factor(codes.maximum), codes.hi, codes.lo);
    codes.sum = (__builtin_amdgcn_sdot4(static_cast<int>(codes.hi), 0x01010101, 0, false) << 8) +
        __builtin_amdgcn_sdot4(static_cast<int>(codes.lo), 0x01010101, 0, false);
    return codes;
}

// Activation record of one (token, 256-value block) in a caller's workspace:
// what a later launch needs to skip the quantization.  [0,256) high plane,
// [256,512) low plane (value order), [512,544) eight int32 sums of the codes
// per 32 values, [544] the scale, [548] the block's largest magnitude.
constexpr int kActRecord = 576;
constexpr int kRecordSums = 512;
constexpr int kRecordScale = 544;
constexpr int kRecordMaximum = 548;

// The four values of lane `column % 256 / 4` of block `column / 256` as the
// kernels' quantizers take them: floats with the prologue applied, or for
// kRecords the raw (high word, low word, maximum) of the stored record.
template <int P>
__device__ __forceinline__ float4 load_activations(const float* __restrict__ first,
                                                   const float* __restrict__ second,
                                                   std::int64_t column) {
    if constexpr (P == kRecords) {
        const std::uint8_t* record =
            reinterpret_cast<const std::uint8_t*>(first) + (column >> 8) * kActRecord;
        const int offset = static_cast<int>(column & 255);  // 4 * lane
        float4 raw;
        raw.x = *reinterpret_cast<const float*>(record + offset);
        raw.y = *reinterpret_cast<const float*>(record + 256 + offset);
        raw.z = *reinterpret_cast<const float*>(record + kRecordMaximum);
        raw.w = 0.0f;
        return raw;
    }
    float4 x = *reinterpret_cast<const float4*>(first + column);
    if constexpr (P == kGated || P == kSwiGlu) {
        const float4 y = *reinterpret_cast<const float4*>(second + column);
        x.x = apply_prologue<P>(x.x, y.x);
        x.y = apply_prologue<P>(x.y, y.y);
        x.z = apply_prologue<P>(x.z, y.z);
        x.w = apply_prologue<P>(x.w, y.w);
    }
    return x;
}

// First input of the pass that starts at token `token0`.
template <int P>
__device__ __forceinline__ const float* pass_input(const float* first, int token0, int input_dim) {
    if constexpr (P == kRecords) {
        return reinterpret_cast<const float*>(reinterpret_cast<const std::uint8_t*>(first) +
                                              static_cast<std::int64_t>(token0) * (input_dim >> 8) * kActRecord);
    } else {
        return first + static_cast<std::int64_t>(token0) * input_dim;
    }
}

// Codes of what load_activations<P> returned.
template <int P>
__device__ __forceinline__ ActivationCodes activation_codes(float4 loaded) {
    if constexpr (P == kRecords) {
        ActivationCodes codes;
        codes.hi = __float_as_uint(loaded.x);
        codes.lo = __float_as_uint(loaded.y);
        codes.maximum = loaded.z;
        codes.sum = (__builtin_amdgcn_sdot4(static_cast<int>(codes.hi), 0x01010101, 0, false) << 8) +
            __builtin_amdgcn_sdot4(static_cast<int>(codes.lo), 0x01010101, 0, false);
        return codes;
    } else {
        return encode_activations(loaded);
    }
}

// Writes the record of one block (four values per lane) for a later launch.
__device__ __forceinline__ void store_record(std::uint8_t* record, int lane,
                                             const ActivationCodes& codes) {
    int sum = codes.sum;  // over the 8 lanes of a 32-value group
    sum += dpp_move<kQuadXor1>(sum);
    sum += dpp_move<kQuadXor2>(sum);
    sum += dpp_move<kHalfMirror>(sum);
    *reinterpret_cast<std::uint32_t*>(record + lane * 4) = codes.hi;
    *reinterpret_cast<std::uint32_t*>(record + 256 + lane * 4) = codes.lo;
    if ((lane & 7) == 0) *reinterpret_cast<int*>(record + kRecordSums + (lane >> 3) * 4) = sum;
    if (lane == 0) {
        *reinterpret_cast<float*>(record + kRecordScale) = codes.maximum * (1.0f / kCodeRange);
        *reinterpret_cast<float*>(record + kRecordMaximum) = codes.maximum;
    }
}

// Token of activation record `record` (records run token by token, `blocks`
// per token), of T tokens at most: no division on the way to the first loads.
template <int T>
__device__ __forceinline__ int token_of_record(int record, int blocks) {
    int token = 0;
#pragma unroll
    for (int t = 1; t < T; ++t) token += record >= t * blocks ? 1 : 0;
    return token;
}

// ---- several records at once by a wave: the one-row kernels' quantizer.  LANES lanes to a record (16 or 32): lane c of
// them holds its words LANES k + c of four values, k = 0..64 / LANES (each load reads 16 LANES bytes in a row a record).
// What bounds it is instructions, since every workgroup quantizes the whole row for itself: a record a wave and pass, as
// encode_activations has it, takes 60 of them a record, this 25 (of 16 lanes), for the same codes, sums and maximum.
// Thirty-two lanes where sixteen would leave half of the waves without a record (rows of up to 4,096 columns).
// With the rows' bookkeeping at compile time (gemv_dot.hip), us: two rows of 6,656 columns into 4,608 of Q4_K 9.5 -> 8.3,
// one of 16,384 into 6,656 of Q4_K 15.8 -> 14.7, of Q5_K 19.0 -> 17.9, of Q8_0 25.5 -> 24.7.
constexpr int records_of_group(int lanes) { return kWave / lanes; }

template <int P, int LANES>
struct RecordQuads {
    static constexpr int kQuads = 64 / LANES;
    float4 quad[kQuads];
    float4 other[P == kGated || P == kSwiGlu ? kQuads : 1];  // the prologue's second operand
};
template <int LANES>
struct QuadCodes {
    std::uint32_t hi[64 / LANES], lo[64 / LANES];  // four bytes each, value order
    int sum[64 / LANES];                           // of a quad's four codes
    float maximum;                                 // the record's largest magnitude
};

// The lane's record of group `group`; from the number of records on there is none.
template <int LANES>
__device__ __forceinline__ int record_of_lane(int group, int lane) {
    return records_of_group(LANES) * group + lane / LANES;
}

// ... its values as they lie in memory (records past the last repeat it).
template <int T, int P, int LANES>
__device__ __forceinline__ void request_records(RecordQuads<P, LANES>& x, const float* __restrict__ first,
                                                const float* __restrict__ second, int group, int records, int blocks,
                                                int input_dim, int lane) {
    const int record = min(record_of_lane<LANES>(group, lane), records - 1);
    const int token = token_of_record<T>(record, blocks);
    const std::int64_t column =
        static_cast<std::int64_t>(token) * input_dim + (record - token * blocks) * 256 + 4 * (lane % LANES);
#pragma unroll
    for (int k = 0; k < x.kQuads; ++k) {
        x.quad[k] = load_activations<P == kRecords ? kRecords : kPlain>(first, second, column + 4 * LANES * k);
    }
    if constexpr (P == kGated || P == kSwiGlu) {
#pragma unroll
        for (int k = 0; k < x.kQuads; ++k) x.other[k] = *reinterpret_cast<const float4*>(second + column + 4 * LANES * k);
    }
}

// For a wave that has no record of a group it has requested: without a use on every path the compiler moves the
// requests to the one that has it, behind the weights' requests.
template <int P, int LANES>
__device__ __forceinline__ void drop_records(const RecordQuads<P, LANES>& x) {
#pragma unroll
    for (int k = 0; k < x.kQuads; ++k) {
        asm volatile("" : : "v"(x.quad[k].x), "v"(x.quad[k].y), "v"(x.quad[k].z), "v"(x.quad[k].w));
        if constexpr (P == kGated || P == kSwiGlu) {
            asm volatile("" : : "v"(x.other[k].x), "v"(x.other[k].y), "v"(x.other[k].z), "v"(x.other[k].w));
        }
    }
}

template <int P, int LANES>
__device__ __forceinline__ QuadCodes<LANES> quad_codes(const RecordQuads<P, LANES>& x) {
    static_assert(LANES == 16 || LANES == 32, "a row or two of lanes");
    constexpr int kQuads = 64 / LANES;
    QuadCodes<LANES> codes;
    if constexpr (P == kRecords) {
#pragma unroll
        for (int k = 0; k < kQuads; ++k) {
            codes.hi[k] = __float_as_uint(x.quad[k].x);
            codes.lo[k] = __float_as_uint(x.quad[k].y);
        }
        codes.maximum = x.quad[0].z;
    } else {
        float4 values[kQuads];
        std::uint32_t largest = 0;  // (wave_max's order of magnitudes)
#pragma unroll
        for (int k = 0; k < kQuads; ++k) {
            float4 q = x.quad[k];
            if constexpr (P == kGated || P == kSwiGlu) {
                q.x = apply_prologue<P>(q.x, x.other[k].x);
                q.y = apply_prologue<P>(q.y, x.other[k].y);
                q.z = apply_prologue<P>(q.z, x.other[k].z);
                q.w = apply_prologue<P>(q.w, x.other[k].w);
            }
            values[k] = q;
            largest = max(largest, __float_as_uint(fmaxf(fmaxf(fabsf(q.x), fabsf(q.y)), fmaxf(fabsf(q.z), fabsf(q.w)))));
        }
        largest = max(largest, static_cast<std::uint32_t>(dpp_move<kQuadXor1>(static_cast<int>(largest))));
        largest = max(largest, static_cast<std::uint32_t>(dpp_move<kQuadXor2>(static_cast<int>(largest))));
        largest = max(largest, static_cast<std::uint32_t>(dpp_move<kHalfMirror>(static_cast<int>(largest))));
        largest = max(largest, static_cast<std::uint32_t>(dpp_move<kRowMirror>(static_cast<int>(largest))));
        if constexpr (LANES == 32) {
            const auto rows = __builtin_amdgcn_permlane16_swap(largest, largest, false, false);
            largest = max(rows[0], rows[1]);
        }
        codes.maximum = __uint_as_float(largest);
        const float inverse = code_factor(codes.maximum);
#pragma unroll
        for (int k = 0; k < kQuads; ++k) encode_quad(values[k], inverse, codes.hi[k], codes.lo[k]);
    }
#pragma unroll
    for (int k = 0; k < kQuads; ++k) {
        codes.sum[k] = (__builtin_amdgcn_sdot4(static_cast<int>(codes.hi[k]), 0x01010101, 0, false) << 8) +
            __builtin_amdgcn_sdot4(static_cast<int>(codes.lo[k]), 0x01010101, 0, false);
    }
    return codes;
}

// The sum over the lane's four (eight) neighbours of the record: of sixteen (32) values in a row.
__device__ __forceinline__ int sum_of_sixteen(int sum) {
    sum += dpp_move<kQuadXor1>(sum);
    return sum + dpp_move<kQuadXor2>(sum);
}
__device__ __forceinline__ int sum_of_thirty_two(int sum) {
    sum = sum_of_sixteen(sum);
    return sum + dpp_move<kHalfMirror>(sum);
}

// store_record from such lanes; `c` = lane % LANES.
template <int LANES>
__device__ __forceinline__ void store_record_quads(std::uint8_t* record, int c, const QuadCodes<LANES>& codes) {
#pragma unroll
    for (int k = 0; k < 64 / LANES; ++k) {
        const int word = LANES * k + c;
        *reinterpret_cast<std::uint32_t*>(record + 4 * word) = codes.hi[k];
        *reinterpret_cast<std::uint32_t*>(record + 256 + 4 * word) = codes.lo[k];
        const int sum = sum_of_thirty_two(codes.sum[k]);
        if ((c & 7) == 0) *reinterpret_cast<int*>(record + kRecordSums + (word >> 3) * 4) = sum;
    }
    if (c == 0) {
        *reinterpret_cast<float*>(record + kRecordScale) = codes.maximum * (1.0f / kCodeRange);
        *reinterpret_cast<float*>(record + kRecordMaximum) = codes.maximum;
    }
}

typedef const __attribute__((address_space(1))) std::uint8_t* GlobalBytes;

// Four 48-bit device addresses in three 64-bit words.
struct PackedPointers {
    std::uint64_t a, b, c;
};
constexpr std::uint64_t kAddressMask = (std::uint64_t(1) << 48) - 1;
inline PackedPointers pack_pointers(const void* const p[4]) {
    std::uint64_t v[4];
    for (int i = 0; i < 4; ++i) v[i] = reinterpret_cast<std::uint64_t>(p[i]) & kAddressMask;
    PackedPointers packed;
    packed.a = v[0] | (v[1] << 48);
    packed.b = (v[1] >> 16) | (v[2] << 32);
    packed.c = (v[2] >> 32) | (v[3] << 16);
    return packed;
}
__device__ __forceinline__ GlobalBytes unpack_pointer(std::uint64_t a, std::uint64_t b,
                                                      std::uint64_t c, int index) {
    const std::uint64_t p0 = a & kAddressMask;
    const std::uint64_t p1 = (a >> 48) | ((b & 0xffffffffull) << 16);
    const std::uint64_t p2 = (b >> 32) | ((c & 0xffffull) << 32);
    const std::uint64_t p3 = c >> 16;
    std::uint64_t p = p0;
    p = index == 1 ? p1 : p;
    p = index == 2 ? p2 : p;
    p = index == 3 ? p3 : p;
    return reinterpret_cast<GlobalBytes>(p);
}

// Projection `index` of the set, chosen with scalar selects from fields that
// were all read with static offsets: a dynamically indexed read of the kernel
// arguments is a dependent scalar load, and its first touch of a cache line
// costs a trip to memory in the middle of the kernel.
__device__ __forceinline__ Projection pick(const ProjectionSet& set, int index) {
    Projection p = set.op[0];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        const bool take = index == k;
        p.data = take ? set.op[k].data : p.data;
        p.output = take ? set.op[k].output : p.output;
        p.output_dim = take ? set.op[k].output_dim : p.output_dim;
        p.row_stride = take ? set.op[k].row_stride : p.row_stride;
        p.first_tile = take ? set.op[k].first_tile : p.first_tile;
    }
    return p;
}

// Walks the (row, iteration) pairs of one wave without divisions: everything
// here is uniform and lives in scalar registers.
struct PairCursor {
    int op;                   // projection index
    Projection current;       // its fields
    std::int64_t local_row;   // row inside that projection
    int iteration;            // which 64-unit slice of the row
    const std::uint8_t* row;  // first byte of the row

    __device__ __forceinline__ void start(const ProjectionSet& set, int global_row) {
        op = 0;
#pragma unroll
        for (int index = 1; index < 4; ++index) {
            if (index < set.count && global_row >= static_cast<int>(set.op[index].first_tile)) op = index;
        }
        current = pick(set, op);
        local_row = global_row - static_cast<int>(current.first_tile);
        iteration = 0;
        row = current.data + local_row * current.row_stride;
    }
    __device__ __forceinline__ void advance(const ProjectionSet& set, int iterations) {
        if (++iteration < iterations) return;
        iteration = 0;
        ++local_row;
        row += current.row_stride;
        if (local_row == current.output_dim && op + 1 < set.count) {
            ++op;
            current = pick(set, op);
            local_row = 0;
            row = current.data;
        }
    }
};

// The rows of one wave.  The launch deals its rows out evenly twice: over the
// workgroups (the first `longer_groups` take one more than `rows_per_group`),
// so that every compute unit streams the same number of bytes, and inside a
// workgroup over its waves (the first few take one more; they sit on different
// SIMDs).  Each wave gets a contiguous range.  No division: the quotients come
// from the host and the wave count is a power of two.
struct WaveRows {
    int begin, count;
};
template <int WAVES>
__device__ __forceinline__ WaveRows wave_rows(int group, int wave, int rows_per_group,
                                              int longer_groups) {
    static_assert((WAVES & (WAVES - 1)) == 0, "waves per workgroup must be a power of two");
    const int group_begin = group * rows_per_group + min(group, longer_groups);
    const int group_rows = rows_per_group + (group < longer_groups ? 1 : 0);
    const int base = group_rows / WAVES;
    const int extra = group_rows % WAVES;
    WaveRows rows;
    rows.begin = group_begin + wave * base + min(wave, extra);
    rows.count = base + (wave < extra ? 1 : 0);
    return rows;
}

// How many tiles of up to `whole` rows of a set's first `count` projections a workgroup takes where every unit has one, and
// the fewest rows a tile, `fewest` at least, with which no workgroup takes more.
struct EvenTiles {
    std::int64_t each;
    int rows;
};
inline EvenTiles even_tiles(const ProjectionSet& set, int count, int whole, int fewest) {
    const std::int64_t units = compute_units();
    const auto tiles_of = [&](int rows) {
        std::int64_t tiles = 0;
        for (int index = 0; index < count; ++index) tiles += (set.op[index].output_dim + rows - 1) / rows;
        return tiles;
    };
    EvenTiles even{(tiles_of(whole) + units - 1) / units, whole};
    int low = fewest;
    while (low < even.rows) {  // fewer rows make no fewer tiles
        const int middle = (low + even.rows) / 2;
        if (tiles_of(middle) <= even.each * units) {
            even.rows = middle;
        } else {
            low = middle + 1;
        }
    }
    return even;
}

// Workgroups of a wave-per-row decode launch.  Small launches are bound by
// fixed costs: waves start at a limited rate and every workgroup quantizes the
// whole activation vector, so one workgroup per compute unit (all resident at
// once, equally loaded) is fastest until a wave would own more than about three
// rows; from there the grid grows to up to four workgroups per unit, which a
// large weight stream needs to keep enough loads in flight.
inline std::int64_t decode_groups(std::int64_t rows, int waves_per_group, int most_per_unit = 4) {
    const std::int64_t units = compute_units();
    std::int64_t per_unit = rows / (units * waves_per_group * 3);
    if (per_unit < 1) per_unit = 1;
    if (per_unit > most_per_unit) per_unit = most_per_unit;
    std::int64_t groups = units * per_unit;
    const std::int64_t useful = (rows + waves_per_group - 1) / waves_per_group;  // a row per wave
    return groups < useful ? groups : useful;
}

}  // namespace nfn
