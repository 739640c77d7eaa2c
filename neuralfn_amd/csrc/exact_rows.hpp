// Exact float dot products of packed weight rows with one to three input rows: device code shared
// by the generic linear (linear_rows.hip) and the one-row lm_head of the formats without a
// streaming kernel of their own (lm_head.hip).
//
// The decoded weight d * sc * q - d_min * m is one fused multiply-add: d * sc and d_min * m are
// exact in float (at most 19 bits), and so is d * sc * q (at most 24), so that the fused form
// rounds where the CPU engine's two products and a subtraction round
// (neuralfn/csrc/native_gpt2/resident_glimmer.cpp:542-616).  A code byte becomes a float in one
// instruction: 2.25 vector instructions a weight before the products with the input rows.  Formats
// without a minimum multiply signed codes, exactly: with the offset of the codes in a fused form an
// infinite scale would give infinity less infinity where the weight is infinite.
//
// The input rows lie in LDS, 64 columns (a unit) at a pitch of 68 floats: a lane owns whole units,
// and neighbouring lanes' 16-byte reads then fall into distinct banks.  A wave takes two weight
// rows at a time, so that an input value read from LDS serves both, and requests a pair's packed
// bytes one turn ahead.
#pragma once

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "q6_words.hpp"
#include "wave_rows.hpp"

namespace nfn {

typedef float exact_f32x4 __attribute__((ext_vector_type(4)));
typedef std::uint32_t exact_u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef std::uint32_t exact_u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int kExactPitch = 68;  // floats from one unit to the next in LDS
constexpr int kExactWaves = 8;
constexpr int kExactPair = 2;    // weight rows a wave takes at a time

// LDS bytes of `rows` input rows
constexpr std::int64_t exact_rows_lds(std::int64_t rows, std::int64_t input_dim) {
    return rows * ((input_dim + 63) / 64) * kExactPitch * 4;
}

// What a lane holds of one unit of a weight row.  values<I>(): columns 4 I .. 4 I + 3 of it.
template <std::uint32_t ENC>
struct ExactUnit;

__device__ __forceinline__ float code_byte(std::uint32_t word, int index) {
    return static_cast<float>((word >> (8 * index)) & 255u);
}

template <std::uint32_t ENC>
struct ExactUnitOfQ4KOrQ5K {
    exact_u32x4_a4 header, codes[2], fifth[2];
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit) {
        const std::uint8_t* block = row + (unit >> 2) * static_cast<int>(block_bytes(ENC));
        const std::uint8_t* source = block + (ENC == kEncQ5K ? 48 : 16) + (unit & 3) * 32;
        header = *reinterpret_cast<const exact_u32x4_a4*>(block);
        codes[0] = *reinterpret_cast<const exact_u32x4_a4*>(source);
        codes[1] = *reinterpret_cast<const exact_u32x4_a4*>(source + 16);
        if constexpr (ENC == kEncQ5K) {
            fifth[0] = *reinterpret_cast<const exact_u32x4_a4*>(block + 16);
            fifth[1] = *reinterpret_cast<const exact_u32x4_a4*>(block + 32);
        }
    }
    // scales and minimums of the unit's two sub-blocks (k_scale_min's indexing, without a branch)
    float scale[2], offset[2];
    int group;
    __device__ __forceinline__ void prepare(int unit) {
        group = unit & 3;
        const float d = half_bits_to_float(header[0] & 0xffffu), dmin = half_bits_to_float(header[0] >> 16);
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            const int sub = 2 * group + step, shift = 8 * (sub & 3), upper = -(sub >> 2);
            const int y = static_cast<int>(header[1] >> shift), z = static_cast<int>(header[2] >> shift);
            const int w = static_cast<int>(header[3] >> shift);
            const int sc = ((y & 63) & ~upper) | (((w & 15) | (((y >> 6) & 3) << 4)) & upper);
            const int m = ((z & 63) & ~upper) | ((((w >> 4) & 15) | (((z >> 6) & 3) << 4)) & upper);
            scale[step] = d * static_cast<float>(sc);
            offset[step] = -(dmin * static_cast<float>(m));
        }
    }
    template <int I>
    __device__ __forceinline__ exact_f32x4 values() const {
        constexpr int kStep = I / 8, kWord = I % 8;
        std::uint32_t q = (codes[kWord / 4][kWord % 4] >> (4 * kStep)) & 0x0f0f0f0fu;
        if constexpr (ENC == kEncQ5K) {
            q |= ((fifth[kWord / 4][kWord % 4] >> (2 * group + kStep)) & 0x01010101u) << 4;
        }
        exact_f32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = fmaf(scale[kStep], code_byte(q, j), offset[kStep]);
        return w;
    }
};
template <>
struct ExactUnit<kEncQ4K> : ExactUnitOfQ4KOrQ5K<kEncQ4K> {};
template <>
struct ExactUnit<kEncQ5K> : ExactUnitOfQ4KOrQ5K<kEncQ5K> {};

template <>
struct ExactUnit<kEncQ6K> {
    // Every other block of a row starts two bytes past a word, and sixteen bytes from there take the address
    // unit four times as long as from a word: pieces are requested from the word at or before them and moved up
    // in prepare().  One row of 2,048 / 6,656 / 8,192 -> 6,656 12.6 / 19.4 / 19.7 -> 9.3 / 17.2 / 18.6 us, three rows
    // of 4,096 17.5 -> 16.6; two of 8,192, bound by the vector ALU, 23.8 -> 24.0.
    exact_u32x4_a4 low[4], high[2];
    std::uint32_t behind_low, behind_high, shift;
    std::uint32_t codes_of_scale, d;
    float scale[4];
    int upper;
    __device__ __forceinline__ void load(const std::uint8_t* tensor, const std::uint8_t* row, int unit) {
        const std::uint8_t* block = row + (unit >> 2) * 210;
        shift = q6_past_word(reinterpret_cast<std::uintptr_t>(tensor), reinterpret_cast<std::uintptr_t>(block));
        const std::uint8_t* lower = block - shift + ((unit >> 1) & 1) * 64;
        const std::uint8_t* top = block - shift + 128 + ((unit >> 1) & 1) * 32;
#pragma unroll
        for (int piece = 0; piece < 4; ++piece) {
            low[piece] = *reinterpret_cast<const exact_u32x4_a4*>(lower + 16 * piece);
        }
        high[0] = *reinterpret_cast<const exact_u32x4_a4*>(top);
        high[1] = *reinterpret_cast<const exact_u32x4_a4*>(top + 16);
        behind_low = *reinterpret_cast<const std::uint32_t*>(lower + 64);
        behind_high = *reinterpret_cast<const std::uint32_t*>(top + 32);
        typedef std::uint32_t u32_a2 __attribute__((aligned(2)));
        codes_of_scale = *reinterpret_cast<const u32_a2*>(block + 192 + 4 * (unit & 3));
        d = *reinterpret_cast<const std::uint16_t*>(block + 208);
    }
    __device__ __forceinline__ void prepare(int unit) {
        upper = (unit & 1) * 4;  // quarters 2 and 3 of the half block: high nibbles, high-bit pairs 2 and 3
#pragma unroll
        for (int word = 0; word < 16; ++word) {
            const std::uint32_t behind = word < 15 ? low[(word + 1) / 4][(word + 1) % 4] : behind_low;
            low[word / 4][word % 4] = __builtin_amdgcn_alignbyte(behind, low[word / 4][word % 4], shift);
        }
#pragma unroll
        for (int word = 0; word < 8; ++word) {
            const std::uint32_t behind = word < 7 ? high[(word + 1) / 4][(word + 1) % 4] : behind_high;
            high[word / 4][word % 4] = __builtin_amdgcn_alignbyte(behind, high[word / 4][word % 4], shift);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            scale[k] = half_bits_to_float(d) * 0.25f * static_cast<float>(static_cast<std::int8_t>(codes_of_scale >> (8 * k)));
        }
    }
    template <int I>
    __device__ __forceinline__ exact_f32x4 values() const {
        constexpr int kStep = I / 8, kWord = I % 8;
        // in every byte 4 (q - 32): the nibble in bits 2 to 5, the high bits above, their sign flipped
        const std::uint32_t lower = low[2 * kStep + kWord / 4][kWord % 4], above = high[kWord / 4][kWord % 4];
        const std::uint32_t q = (__builtin_rotateright32(lower, upper - 2) & 0x3c3c3c3cu) |
            (__builtin_rotateright32(above, upper + 2 * kStep - 6) & 0xc0c0c0c0u);
        const float factor = scale[2 * kStep + kWord / 4];
        exact_f32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = factor * static_cast<float>(static_cast<std::int8_t>((q ^ 0x80808080u) >> (8 * j)));
        return w;
    }
};

template <>
struct ExactUnit<kEncQ8_0> {
    // two 34-byte blocks: 17 words, the codes of the first block half a word off
    std::uint32_t words[17];
    float scale[2];
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit) {
        const std::uint8_t* source = row + unit * 68;
#pragma unroll
        for (int piece = 0; piece < 4; ++piece) {
            const exact_u32x4_a2 four = *reinterpret_cast<const exact_u32x4_a2*>(source + 16 * piece);
#pragma unroll
            for (int j = 0; j < 4; ++j) words[4 * piece + j] = four[j];
        }
        typedef std::uint32_t u32_a2 __attribute__((aligned(2)));
        words[16] = *reinterpret_cast<const u32_a2*>(source + 64);
    }
    __device__ __forceinline__ void prepare(int) {
        scale[0] = half_bits_to_float(words[0] & 0xffffu);
        scale[1] = half_bits_to_float(words[8] >> 16);
    }
    template <int I>
    __device__ __forceinline__ exact_f32x4 values() const {
        constexpr int kStep = I / 8, kWord = I % 8;
        float code[4];
        signed_bytes(kStep == 0 ? __builtin_amdgcn_alignbyte(words[kWord + 1], words[kWord], 2) : words[9 + kWord], code);
        exact_f32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = scale[kStep] * code[j];
        return w;
    }
};

template <std::uint32_t ENC>
constexpr bool kExactRowsFormat = ENC == kEncQ4K || ENC == kEncQ5K || ENC == kEncQ6K || ENC == kEncQ8_0;

// The workgroup's copy of the input rows: [row][unit][kExactPitch].  PARTLY: the first `there` exist.
template <int R, bool PARTLY = false>
__device__ __forceinline__ void exact_rows_stage(const float* __restrict__ input, std::int64_t input_dim,
                                                 float* staged, int there = R) {
    const int units = static_cast<int>(input_dim >> 6);
    for (int index = threadIdx.x; index < R * units * 16; index += kExactWaves * kWave) {
        const int row = index / (units * 16), piece = index % (units * 16);
        typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
        const exact_f32x4 x = *reinterpret_cast<const f32x4_a4*>(input + (PARTLY ? min(row, there - 1) : row) * input_dim + 4 * piece);
        *reinterpret_cast<exact_f32x4*>(staged + (row * units + (piece >> 4)) * kExactPitch + 4 * (piece & 15)) = x;
    }
    __syncthreads();
}

template <typename F, int... I>
__device__ __forceinline__ void for_each_piece(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

// Lanes of both halves: lanes 0 to 31 return the sum of `a` over l and l + 32, the others that of `b`.
// (The instruction swaps the upper half of its first operand with the lower half of its second.)
__device__ __forceinline__ double fold_halves(double a, double b) {
    const std::uint64_t x = __builtin_bit_cast(std::uint64_t, a), y = __builtin_bit_cast(std::uint64_t, b);
    const auto low = __builtin_amdgcn_permlane32_swap(static_cast<std::uint32_t>(x), static_cast<std::uint32_t>(y), false, false);
    const auto high = __builtin_amdgcn_permlane32_swap(static_cast<std::uint32_t>(x >> 32), static_cast<std::uint32_t>(y >> 32),
                                                       false, false);
    return __builtin_bit_cast(double, low[0] | static_cast<std::uint64_t>(high[0]) << 32) +
        __builtin_bit_cast(double, low[1] | static_cast<std::uint64_t>(high[1]) << 32);
}
// ... of neighbouring rows of sixteen lanes: rows 0 and 2 return `a` over their pair of rows, rows 1 and 3 `b`.
__device__ __forceinline__ double fold_rows(double a, double b) {
    const std::uint64_t x = __builtin_bit_cast(std::uint64_t, a), y = __builtin_bit_cast(std::uint64_t, b);
    const auto low = __builtin_amdgcn_permlane16_swap(static_cast<std::uint32_t>(x), static_cast<std::uint32_t>(y), false, false);
    const auto high = __builtin_amdgcn_permlane16_swap(static_cast<std::uint32_t>(x >> 32), static_cast<std::uint32_t>(y >> 32),
                                                       false, false);
    return __builtin_bit_cast(double, low[0] | static_cast<std::uint64_t>(high[0]) << 32) +
        __builtin_bit_cast(double, low[1] | static_cast<std::uint64_t>(high[1]) << 32);
}
template <int CTRL>
__device__ __forceinline__ double dpp_add(double value) {
    const std::uint64_t x = __builtin_bit_cast(std::uint64_t, value);
    const std::uint32_t low = static_cast<std::uint32_t>(dpp_move<CTRL>(static_cast<int>(x)));
    const std::uint32_t high = static_cast<std::uint32_t>(dpp_move<CTRL>(static_cast<int>(x >> 32)));
    return value + __builtin_bit_cast(double, low | static_cast<std::uint64_t>(high) << 32);
}

// The wave's sums of R values each for two weight rows, in every lane, rounded once: four values at a time are
// folded into the four rows of sixteen lanes, which costs a third of a butterfly for each.
template <int R>
__device__ __forceinline__ void wave_sums(const double (&values)[kExactPair][R], float (&totals)[kExactPair][R]) {
    static_assert(kExactPair == 2);
    const auto within_row = [](double value) {
        value = dpp_add<kQuadXor1>(value);
        value = dpp_add<kQuadXor2>(value);
        value = dpp_add<kHalfMirror>(value);
        return static_cast<float>(dpp_add<kRowMirror>(value));
    };
#pragma unroll
    for (int r = 0; r < R; r += 2) {
        const double first = fold_halves(values[0][r], values[1][r]);
        const bool two = r + 1 < R;
        const double second = two ? fold_halves(values[0][two ? r + 1 : r], values[1][two ? r + 1 : r]) : first;
        const float folded = within_row(fold_rows(first, second));
        totals[0][r] = lane_value(folded, 0);
        totals[1][r] = lane_value(folded, 32);
        if (two) {
            totals[0][two ? r + 1 : r] = lane_value(folded, 16);
            totals[1][two ? r + 1 : r] = lane_value(folded, 48);
        }
    }
}

// Calls take(row, sums) for the weight rows `first`, `first + step`, ... below `output_dim`, two at a
// time (rows 2 p and 2 p + 1); sums[r]: this wave's total for input row r, in every lane.  A row's
// sum does not depend on the launch: lane l adds the units l, l + span, ... in rising order and the lanes
// meet in doubles.  Every fourth column is added in a chain of its own; of Q8_0 sixteen columns are added in two
// chains of eight and go to one of two sums in turn, for 12 % more additions (4,352 columns, three rows 11.0 -> 11.9 us).
// Rounding against float64 at 4,096 / 8,192 columns: 7.7e-8 / 1.02e-7 (Q4_K, Q5_K), 7.4e-8 / 9.7e-8 (Q6_K), 6.8e-8 / 7.4e-8
// (Q8_0); on the matrix-core kernel, which more rows run on, 1.2e-7 / 1.4e-7, 8.7e-8 / 1.1e-7 and 7.4e-8 / 8.9e-8.  (Two
// chains a lane and a float butterfly: 1.2e-7 / 1.6e-7, and 1 % slower.)
template <std::uint32_t ENC, int R, typename Take>
__device__ __forceinline__ void exact_rows_walk(const std::uint8_t* __restrict__ data, std::int64_t row_stride,
                                                std::int64_t output_dim, std::int64_t input_dim,
                                                const float* staged, std::int64_t first_pair, std::int64_t pair_step,
                                                std::int64_t end_pair, Take&& take) {
    const int lane = threadIdx.x & 63;
    const int units = static_cast<int>(input_dim >> 6);
    const int turns = (units + 63) / 64;
    // A last turn of eight lanes or fewer takes twice as long as one of twelve or more (4,608 columns, one row 8.2 us,
    // 4,864 6.5): it gets sixteen units at least.
    constexpr int kLeastUnits = 16;
    const int span = turns > 1 && units - 64 * (turns - 1) < kLeastUnits ? (units - kLeastUnits + turns - 2) / (turns - 1) : 64;
    if (first_pair >= end_pair) return;
    ExactUnit<ENC> now[kExactPair], next[kExactPair];
    auto load = [&](ExactUnit<ENC> (&into)[kExactPair], std::int64_t pair, int turn) {
        const int unit = min(lane + span * turn, units - 1);
#pragma unroll
        for (int k = 0; k < kExactPair; ++k) {
            const std::uint8_t* row = data + min(pair * kExactPair + k, output_dim - 1) * row_stride;
            if constexpr (ENC == kEncQ6K) {
                into[k].load(data, row, unit);
            } else {
                into[k].load(row, unit);
            }
        }
    };
    load(now, first_pair, 0);
    for (std::int64_t pair = first_pair; pair < end_pair; pair += pair_step) {
        constexpr bool kShort = ENC == kEncQ8_0;
        constexpr int kSums = kShort ? 2 : 4;
        float sums[kExactPair][R][kSums] = {};
        for (int turn = 0; turn < turns; ++turn) {
            const bool more = turn + 1 < turns;
            // (unconditional: behind the last pair its own bytes are read again)
            load(next, more ? pair : pair + pair_step < end_pair ? pair + pair_step : pair, more ? turn + 1 : 0);
            const int unit = lane + span * turn;
            if (lane < span && unit < units) {
#pragma unroll
                for (int k = 0; k < kExactPair; ++k) now[k].prepare(unit);
                const float* x = staged + unit * kExactPitch;
                float chains[kExactPair][R][2];  // (Q8_0)
                const auto four = [&](auto index) {
                    constexpr int kI = decltype(index)::value;
                    exact_f32x4 w[kExactPair];
#pragma unroll
                    for (int k = 0; k < kExactPair; ++k) w[k] = now[k].template values<kI>();
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const exact_f32x4 v =
                            *reinterpret_cast<const exact_f32x4*>(x + r * units * kExactPitch + 4 * kI);
#pragma unroll
                        for (int k = 0; k < kExactPair; ++k) {
                            float (&chain)[2] = chains[k][r];
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                if constexpr (!kShort) {
                                    sums[k][r][j] = fmaf(v[j], w[k][j], sums[k][r][j]);
                                } else {
                                    chain[j & 1] = kI % 4 == 0 && j < 2 ? v[j] * w[k][j] : fmaf(v[j], w[k][j], chain[j & 1]);
                                }
                            }
                            if constexpr (kShort && kI % 4 == 3) sums[k][r][kI / 4 & 1] += chain[0] + chain[1];
                        }
                    }
                };
                for_each_piece(four, std::make_integer_sequence<int, 16>{});
            }
#pragma unroll
            for (int k = 0; k < kExactPair; ++k) now[k] = next[k];
        }
        double both[kExactPair][R];
        float totals[kExactPair][R];
#pragma unroll
        for (int k = 0; k < kExactPair; ++k) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                both[k][r] = static_cast<double>(sums[k][r][0]) + static_cast<double>(sums[k][r][1]);
                if constexpr (!kShort) both[k][r] += static_cast<double>(sums[k][r][2]) + static_cast<double>(sums[k][r][3]);
            }
        }
        wave_sums<R>(both, totals);
#pragma unroll
        for (int k = 0; k < kExactPair; ++k) {
            const std::int64_t row = pair * kExactPair + k;
            if (row < output_dim) take(row, totals[k]);
        }
    }
}

}  // namespace nfn
