// The exact tier on the bf16 matrix cores: many input rows of one projection, float in, float
// out, every weight at its decoded value.
//
// A float times 2^24 is the sum of three bf16 numbers (24 significant bits cut into 8 + 8 + 8 by
// truncation; the last bit of the smallest float becomes 2^-125, which bf16 holds as a normal
// number, so that nothing is left over down to zero), and the integer code of a packed weight is
// one bf16 number (at most eight significant bits).  Sums carry the factor to the end.
// v_mfma_f32_32x32x16_bf16 multiplies bf16 exactly and adds in float, so three of them per code give
// the product of the float activations with the codes, at a sixteenth of the cycles of the float
// instruction each: 3/16 of v_mfma_f32_32x32x2_f32's time.  A sub-block's scale d * sc is exact in
// float (11 + 6 or 7 bits) and multiplies the sub-block's sums on their way into the accumulators; the
// minimum's part d_min * m times the sub-block's sum of activations goes in by one float matrix
// instruction per 64 columns.  A one-hot input row returns the dequantized weight bit for bit:
// d * sc * q is exact, the subtraction of d_min * m is the one rounding that the decode has.  Float
// weights are cut into three terms as well (eight products of the nine: the one left out is below
// 2^-32 of the product), bf16 weights are one term.
//
// A workgroup's waves share one tile and cut K between them; their sums meet in LDS at the end, in
// a fixed order.  Two forms:
//   linear_exact_small_kernel, a tile of 32 MT x 32 NT, each wave streaming its own weights straight
//   into registers and its own activations through LDS, where they lie cut (no barrier in the loop): what a
//   problem of a few tiles needs (38 rows x 332 outputs are 22 of 32 x 32 for 256 compute units), there is no
//   long walk over K;
//   linear_exact_kernel, a tile of 32 MT input rows x 128 weight rows for two waves (64 weight rows
//   each) in each of four K groups.  The two cut the activations of a step of 32 columns between
//   them and hand the terms over in LDS.
// What bounded both is the vector cache: a load instruction that reads 16 bytes from each of 32 rows
// looks up 32 lines for 1 KB, and a unit pulls some 20 GB/s that way.  The small form loads its activations
// eight lanes a row instead, eight rows an instruction, and so loads and cuts only the rows that are there (by
// eights: 8, 16 or 32), which every tile of weight rows does again: 4,096 -> 6,656 at 5 / 16 / 25 / 64 rows Q4_K
// 15.2 / 17.4 / 19.6 / 28.7 -> 12.2 / 15.1 / 18.1 / 28.4 us, Q5_K 16.8 / 19.7 / 22.2 / 34.0 -> 13.7 / 16.3 /
// 20.0 / 30.8, Q6_K 21.8 / 24.1 / 27.6 / 46.6 -> 15.4 / 18 / 20 / 35.9, Q8_0 24.2 / 28.2 / 31.0 / 45.9 ->
// 12.9 / 15 / 16.5 / 26.2, bf16 20.4 / 23.9 / 27.1 / 38.4 -> 18.1 / 21.1 / 23.2 / 31.5, F32 32.4 / 33.5 / 35.7 /
// 55.9 -> 28.4 / 31.2 / 33.1 / 51.6, at 200 rows 135 -> 114.  (Its buffer loads of activations as global ones take
// registers that Q5_K does not have: 25 rows 20.0 -> 24.3.  Weights requested behind the next step's activations:
// Q8_0 2 % faster, F32 of 64 rows 46.6 -> 55.0.)  What is left is the cut and the decode (16 waves'
// vector instructions, 4 to 10 us) and for Q8_0, bf16 and F32 the look-ups of their weights.  The large form
// (a look-up in 72 % of the cycles, the matrix cores busy in 26 %) loads its weights with
// neighbouring lanes on neighbouring pieces of a row and turns them in LDS, each wave its own, and the two
// waves of a group wait for each other alone instead of for the workgroup.  4,096 -> 6,656 at 100 / 200 /
// 512 rows, loads as the lanes use them -> through LDS -> and with waits in pairs: Q8_0 73 / 84 / 165 -> 41 /
// 60 / 118 -> 38 / 55 / 108 us; Q5_K 61 / 83 / 165 -> 54 / 76 / 151 -> 43 / 65 / 127 (with sums of
// activations by DPP instead of LDS permutes); Q4_K 49 / 70 / 138 -> 46 / 72 / 142 -> 40 / 62 / 121; Q6_K 87 /
// 105 / 208 -> 77 / 97 / 192 -> 58 / 76 / 151 (scales requested a step later, out of the registers' way);
// bf16 58 / 67 / 131 -> 45 / 55 / 108 -> 39 / 50 / 98 (both halves of a line at once).  What is left of the
// 55 us (200 rows of Q8_0) in parts, each by leaving it out: cutting 8, weights' loads 8, decode 5, scaling 3,
// matrix instructions 21: two waves a SIMD overlap them in part.  (Sums of all tiles meeting in LDS at
// once instead of tile by tile: no difference.  Requests two steps ahead instead of one, and the matrix
// instructions of a step before its other work instead of between it: neither.)  The 64 x 128 form of Q6_K
// keeps six registers that do not change in its loop in scratch (28 bytes a lane), read outside of it; the
// others none.
// Measured at 4,096 -> 6,656, against the vector kernel (16 rows) and the float matrix instruction (200,
// 512 rows) before: Q4_K 134 -> 15 us at 16 rows, 203 -> 62 at 200, 311 -> 121 at 512; Q8_0 368 -> 23,
// 180 -> 55, 279 -> 108; F32 406 -> 31, 172 -> 114, 271 -> 217.
//
// The entry point, nfn_native_tile_linear_packed_weight_float32_v1, has no workspace argument
// (neuralfn/csrc/native_train/tile_ops.h:614-620; reference kernel
// neuralfn/csrc/tile_cuda/kernels.cu:26943-26983), so nothing is converted ahead of the launch.
// Weight layouts and decode: neuralfn/csrc/native_gpt2/resident_glimmer.cpp:542-616.
#include "common.hpp"
#include "kernels.hpp"
#include "q6_words.hpp"

#include <algorithm>

namespace nfn {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef std::uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef std::uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef std::uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// The factor that floats are cut with: without it the third term of an activation below 2^-110
// would fall under 2^-133, the smallest bf16 number, and lose bits (relative error 5e-5 at 1e-36).
// Sums of ordinary numbers keep their bits.  It costs the small forms up to 5 % (4 rows of Q4_K,
// 5,120 -> 178: 15.2 -> 15.9 us) and the large ones little (200 rows of Q8_0 81.5 -> 81.8).  Float weights
// are cut with it too.
constexpr float kLift = 0x1p24f;
template <std::uint32_t ENC>
constexpr float kLower = ENC == kEncF32 ? 0x1p-48f : 0x1p-24f;  // ... and taken out of the sums

__device__ __forceinline__ bf16x8 as_bf16(u32x4 words) { return __builtin_bit_cast(bf16x8, words); }

// the upper halves of two floats, `low` in the lower half: two bf16 numbers by truncation
__device__ __forceinline__ std::uint32_t upper_halves(float low, float high) {
    return __builtin_amdgcn_perm(__float_as_uint(high), __float_as_uint(low), 0x07060302u);
}

// Two of the eight values of a fragment, times kLift: word `pair` of its three terms.
__device__ __forceinline__ void cut_pair(float x0, float x1, std::uint32_t& a, std::uint32_t& b, std::uint32_t& c) {
    const float l0 = x0 * kLift, l1 = x1 * kLift;
    a = upper_halves(l0, l1);
    const float y0 = fmaf(x0, kLift, -__uint_as_float(__float_as_uint(l0) & 0xffff0000u));
    const float y1 = fmaf(x1, kLift, -__uint_as_float(__float_as_uint(l1) & 0xffff0000u));
    b = upper_halves(y0, y1);
    const float z0 = y0 - __uint_as_float(__float_as_uint(y0) & 0xffff0000u);
    const float z1 = y1 - __uint_as_float(__float_as_uint(y1) & 0xffff0000u);
    c = upper_halves(z0, z1);
}

// Eight floats, times kLift, as three bf16 fragments whose sum they are.
struct Terms {
    bf16x8 first, second, third;
};
__device__ __forceinline__ Terms cut(const float (&x)[8]) {
    u32x4 a, b, c;
#pragma unroll
    for (int pair = 0; pair < 4; ++pair) {
        std::uint32_t wa, wb, wc;
        cut_pair(x[2 * pair], x[2 * pair + 1], wa, wb, wc);
        a[pair] = wa;
        b[pair] = wb;
        c[pair] = wc;
    }
    return Terms{as_bf16(a), as_bf16(b), as_bf16(c)};
}

__device__ __forceinline__ float sum_of(const float (&x)[8]) {
    return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
}

// four code bytes (0..255) less `offset` as four bf16 numbers
__device__ __forceinline__ void codes_to_bf16(std::uint32_t bytes, float offset, std::uint32_t& low,
                                              std::uint32_t& high) {
    const float q0 = static_cast<float>(bytes & 255u) - offset;
    const float q1 = static_cast<float>((bytes >> 8) & 255u) - offset;
    const float q2 = static_cast<float>((bytes >> 16) & 255u) - offset;
    const float q3 = static_cast<float>(bytes >> 24) - offset;
    low = upper_halves(q0, q1);
    high = upper_halves(q2, q3);
}
// ... signed ones: one instruction a code.  200 rows 4,096 -> 6,656 Q8_0 89 -> 85 us; Q6_K, whose codes
// would take two more instructions to become signed bytes, gains 4 % in the large form and loses 5 % in
// the small one and keeps the offset.
__device__ __forceinline__ void signed_codes_to_bf16(std::uint32_t bytes, std::uint32_t& low, std::uint32_t& high) {
    float q[4];
    signed_bytes(bytes, q);
    low = upper_halves(q[0], q[1]);
    high = upper_halves(q[2], q[3]);
}

// -----------------------------------------------------------------------------------------------
// What a lane holds of one weight row for 64 columns (a unit: two steps of 32).  The lane's
// columns of a step: kWide formats 16 half + 8 chunk + j, the others 16 chunk + 8 half + j
// (half = lane / 32, chunk = 0 or 1, j = 0..7); the matrix instruction does not care which
// column carries which k index as long as both operands agree, and 16 neighbouring code bytes
// are one load.  Q6_K has a scale per 16 columns, which a chunk's instructions must not mix.
//   load(row, unit, half); arrange(), once, when the bytes are there; words(step, chunk, word, ..):
//   four codes as bf16; scale(step, chunk); minimum(step): d_min * m
// Every load looks up a cache line for each of its lanes, however few bytes it brings, and those
// look-ups bound the kernels: the two lanes of a row (half 0 and 1, 32 lanes apart) therefore
// fetch different pieces, 16 bytes wherever a piece has them, and trade words in arrange().  Q6_K
// takes five loads a unit instead of nine, Q8_0 three instead of four.
// Sixteen bytes that start two past a word keep the address unit four times as long as sixteen that start at one (a
// wave's load of 32 rows 55 ns a compute unit, aligned 15; of two words twice, of one word or less as long as ever),
// and half of Q6_K's and of Q8_0's pieces do.  The small form asks for the words that hold a piece and moves them
// up by two bytes: 4,096 / 6,400 -> 1,700 of Q6_K, 4 rows 17.0 / 39.1 -> 13.4 / 21.8 us, 32 rows 22.4 / 46.1 -> 18.9 /
// 30.5; of Q8_0 17.4 / 20.2 -> 10.6 / 14.3 and 21.9 / 27.6 -> 15.7 / 22.4; 64 rows -> 6,656 of Q6_K 40.8 / 76.6 ->
// 35.9 / 53.9.  (Q6_K rows of an odd number of blocks begin past a word by turns, so that every load was a slow one.)
// -----------------------------------------------------------------------------------------------
// first: the lower 32 lanes' `a` and `b` (in the lower and the upper lanes), second: the upper lanes'
struct Traded {
    std::uint32_t first, second;
};
__device__ __forceinline__ Traded trade(std::uint32_t a, std::uint32_t b) {
    const auto both = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return Traded{both[0], both[1]};
}
// another lane's value, by a pattern within sixteen lanes
template <int PATTERN>
__device__ __forceinline__ float of_lane(float value) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(value), PATTERN, 0xf, 0xf, true));
}
template <std::uint32_t ENC>
struct Unit;

template <std::uint32_t ENC>
struct UnitOfQ4KOrQ5K {
    static constexpr bool kWide = true, kScaled = true, kMinimum = true, kScalePerChunk = false;
    u32x4_a4 header, codes, fifth;
    int group;
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit, int half) {
        const std::uint8_t* block = row + (unit >> 2) * static_cast<int>(block_bytes(ENC));
        group = unit & 3;
        header = *reinterpret_cast<const u32x4_a4*>(block);
        codes = *reinterpret_cast<const u32x4_a4*>(block + (ENC == kEncQ5K ? 48 : 16) + group * 32 + half * 16);
        if constexpr (ENC == kEncQ5K) fifth = *reinterpret_cast<const u32x4_a4*>(block + 16 + half * 16);
    }
    __device__ __forceinline__ void arrange() {
        if constexpr (ENC == kEncQ5K) {
            // the unit's two bits of every byte, all four words in one (three registers a unit less)
            std::uint32_t bits = fifth[0] >> (2 * group) & 0x03030303u;
#pragma unroll
            for (int word = 1; word < 4; ++word) bits |= (fifth[word] >> (2 * group) & 0x03030303u) << (2 * word);
            fifth[0] = bits;
        }
    }
    __device__ __forceinline__ void words(int step, int chunk, int word, std::uint32_t& low, std::uint32_t& high) const {
        std::uint32_t q = (codes[2 * chunk + word] >> (4 * step)) & 0x0f0f0f0fu;
        if constexpr (ENC == kEncQ5K) {
            const int bit = 2 * (2 * chunk + word) + step;  // (constant where it is used)
            q |= ((bit < 4 ? fifth[0] << (4 - bit) : fifth[0] >> (bit - 4)) & 0x10101010u);
        }
        codes_to_bf16(q, 0.0f, low, high);
    }
    // scale and minimum bytes of sub-block 2 group + step (k_scale_min's indexing, without a branch)
    __device__ __forceinline__ float scale(int step, int) const {
        const int sub = 2 * group + step, shift = 8 * (sub & 3), upper = -(sub >> 2);
        const int y = static_cast<int>(header[1] >> shift), w = static_cast<int>(header[3] >> shift);
        const int code = ((y & 63) & ~upper) | (((w & 15) | (((y >> 6) & 3) << 4)) & upper);
        return half_bits_to_float(header[0] & 0xffffu) * static_cast<float>(code);
    }
    __device__ __forceinline__ float minimum(int step) const {
        const int sub = 2 * group + step, shift = 8 * (sub & 3), upper = -(sub >> 2);
        const int z = static_cast<int>(header[2] >> shift), w = static_cast<int>(header[3] >> shift);
        const int code = ((z & 63) & ~upper) | ((((w >> 4) & 15) | (((z >> 6) & 3) << 4)) & upper);
        return half_bits_to_float(header[0] >> 16) * static_cast<float>(code);
    }
};
template <>
struct Unit<kEncQ4K> : UnitOfQ4KOrQ5K<kEncQ4K> {};
template <>
struct Unit<kEncQ5K> : UnitOfQ4KOrQ5K<kEncQ5K> {};

template <>
struct Unit<kEncQ6K> {
    static constexpr bool kWide = false, kScaled = true, kMinimum = false, kScalePerChunk = true;
    // as loaded: the 16 columns of chunk `half`, from the word at or before the first (every other block of a row
    // starts two bytes past a word); aligned: the columns; arranged: words 0 and 1 the lane's columns of chunk 0, words 2 and 3 those of chunk 1
    u32x4_a4 low[2], high;  // low: [step]
    std::uint32_t beyond;   // the word behind the lower bits (half 0), the upper ones (half 1)
    std::uint32_t scales;   // the unit's four sub-scales, (step, chunk) at byte 2 step + chunk
    std::uint32_t d;        // in the upper half
    int upper;
    __device__ __forceinline__ static std::uint32_t past_word(const std::uint8_t* tensor, const std::uint8_t* row, int unit) {
        return q6_past_word(reinterpret_cast<std::uintptr_t>(tensor), reinterpret_cast<std::uintptr_t>(row) + 2u * (unit >> 2));
    }
    __device__ __forceinline__ void load(const std::uint8_t* tensor, const std::uint8_t* row, int unit, int half) {
        typedef std::uint32_t u32_a2 __attribute__((aligned(2)));
        const std::uint8_t* block = row + (unit >> 2) * 210;
        const int half_block = (unit >> 1) & 1;
        upper = unit & 1;  // quarters 2 and 3 of the half block: high nibbles, high-bit pairs 2 and 3
        const std::uint8_t* word = block - past_word(tensor, row, unit);
        low[0] = *reinterpret_cast<const u32x4_a4*>(word + half_block * 64 + 16 * half);
        low[1] = *reinterpret_cast<const u32x4_a4*>(word + half_block * 64 + 32 + 16 * half);
        high = *reinterpret_cast<const u32x4_a4*>(word + 128 + half_block * 32 + 16 * half);
        beyond = *reinterpret_cast<const std::uint32_t*>(word + (half != 0 ? 160 + 32 * half_block : 64 + 64 * half_block));
        scales = *reinterpret_cast<const u32_a2*>(block + (half != 0 ? 192 + 4 * (unit & 3) : 206));
    }
    __device__ __forceinline__ void align(const std::uint8_t* tensor, const std::uint8_t* row, int unit) {
        const std::uint32_t shift = past_word(tensor, row, unit);
        if (__ballot(shift != 0) == 0) return;
        // each piece's following word lies in the other lane of the row or, behind the last, in `beyond`
        const bool second = (threadIdx.x & 32) != 0;
        const Traded a = trade(low[0][0], low[1][0]), b = trade(low[1][0], beyond), c = trade(high[0], high[0]);
        const std::uint32_t behind[3] = {second ? a.first : a.second, second ? b.first : b.second,
                                         second ? beyond : c.second};
#pragma unroll
        for (int word = 0; word < 4; ++word) {
            low[0][word] = __builtin_amdgcn_alignbyte(word < 3 ? low[0][word + 1] : behind[0], low[0][word], shift);
            low[1][word] = __builtin_amdgcn_alignbyte(word < 3 ? low[1][word + 1] : behind[1], low[1][word], shift);
            high[word] = __builtin_amdgcn_alignbyte(word < 3 ? high[word + 1] : behind[2], high[word], shift);
        }
    }
    __device__ __forceinline__ void arrange() {
#pragma unroll
        for (int word = 0; word < 2; ++word) {
#pragma unroll
            for (int step = 0; step < 2; ++step) {
                const Traded t = trade(low[step][word], low[step][word + 2]);
                low[step][word] = t.first;
                low[step][word + 2] = t.second;
            }
            const Traded t = trade(high[word], high[word + 2]);
            high[word] = t.first;
            high[word + 2] = t.second;
        }
        const Traded t = trade(scales, scales);
        d = t.first;
        scales = t.second;
    }
    __device__ __forceinline__ void words(int step, int chunk, int word, std::uint32_t& even, std::uint32_t& odd) const {
        const std::uint32_t q = ((low[step][2 * chunk + word] >> (4 * upper)) & 0x0f0f0f0fu) |
            (((high[2 * chunk + word] >> (4 * upper + 2 * step)) & 0x03030303u) << 4);
        codes_to_bf16(q, 32.0f, even, odd);
    }
    __device__ __forceinline__ float scale(int step, int chunk) const {
        const int code = static_cast<std::int8_t>(scales >> (8 * (2 * step + chunk)));
        return half_bits_to_float(d >> 16) * static_cast<float>(code);
    }
    __device__ __forceinline__ float minimum(int) const { return 0.0f; }
};

template <>
struct Unit<kEncQ8_0> {
    static constexpr bool kWide = true, kScaled = true, kMinimum = false, kScalePerChunk = false;
    u32x4_a2 codes[2];
    std::uint32_t d[2];  // as loaded: [0] the scale of block `half`; of a pair: [0] the word behind it
    // Rows of whole units: a pair of blocks is 68 bytes, whole words where the tensor begins at one.
    __device__ __forceinline__ void load_pair(const std::uint8_t* row, int unit, int half) {
        const std::uint8_t* pair = row + 68 * unit;
        codes[0] = *reinterpret_cast<const u32x4_a2*>(pair + 16 * half);
        codes[1] = *reinterpret_cast<const u32x4_a2*>(pair + 32 + 16 * half);
        typedef std::uint32_t u32_a2 __attribute__((aligned(2)));
        d[0] = *reinterpret_cast<const u32_a2*>(pair + 64);
    }
    // The lane has words 4 half .. 4 half + 3 and 8 + 4 half .. 11 + 4 half of the pair's seventeen.  The first
    // block's codes begin in the middle of word 0, the second one's are words 9 to 16, behind its scale.
    __device__ __forceinline__ void arrange_pair() {
        const bool second = (threadIdx.x & 32) != 0;
        const Traded a = trade(codes[0][0], codes[1][0]), b = trade(codes[1][0], codes[1][0]);
        const std::uint32_t behind0 = second ? a.first : a.second, behind1 = second ? d[0] : b.second;
        const std::uint32_t scales = (codes[0][0] & 0xffffu) | (codes[1][0] & 0xffff0000u);  // (of the lower lanes)
        const Traded t = trade(scales, scales);
        d[0] = t.first & 0xffffu;
        d[1] = t.first >> 16;
#pragma unroll
        for (int word = 0; word < 4; ++word) {
            codes[0][word] = __builtin_amdgcn_alignbyte(word < 3 ? codes[0][word + 1] : behind0, codes[0][word], 2);
            codes[1][word] = word < 3 ? codes[1][word + 1] : behind1;
        }
    }
    // (`steps`: the row's 32-column blocks; a row of an odd number of them reads its last one twice)
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit, int half, int steps) {
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            const std::uint8_t* block = row + min(2 * unit + step, steps - 1) * 34;
            codes[step] = *reinterpret_cast<const u32x4_a2*>(block + 2 + 16 * half);
        }
        d[0] = *reinterpret_cast<const std::uint16_t*>(row + min(2 * unit + half, steps - 1) * 34);
    }
    __device__ __forceinline__ void arrange() {
        const Traded t = trade(d[0], d[0]);
        d[0] = t.first;
        d[1] = t.second;
    }
    __device__ __forceinline__ void words(int step, int chunk, int word, std::uint32_t& even, std::uint32_t& odd) const {
        signed_codes_to_bf16(codes[step][2 * chunk + word], even, odd);
    }
    __device__ __forceinline__ float scale(int step, int) const { return half_bits_to_float(d[step]); }
    __device__ __forceinline__ float minimum(int) const { return 0.0f; }
};

template <>
struct Unit<kEncBF16> {
    static constexpr bool kWide = true, kScaled = false, kMinimum = false, kScalePerChunk = false;
    u32x4_a2 values[2][2];
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit, int half, int steps) {
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            const std::uint8_t* source = row + min(2 * unit + step, steps - 1) * 64 + 32 * half;
            values[step][0] = *reinterpret_cast<const u32x4_a2*>(source);
            values[step][1] = *reinterpret_cast<const u32x4_a2*>(source + 16);
        }
    }
    __device__ __forceinline__ void arrange() {}
    __device__ __forceinline__ void words(int step, int chunk, int word, std::uint32_t& low, std::uint32_t& high) const {
        low = values[step][chunk][2 * word];
        high = values[step][chunk][2 * word + 1];
    }
    __device__ __forceinline__ float scale(int, int) const { return 1.0f; }
};

template <>
struct Unit<kEncF32> {
    static constexpr bool kWide = true, kScaled = false, kMinimum = false;
    f32x4_a4 values[2][2][2];  // [step][chunk][piece]
    __device__ __forceinline__ void load_step(const std::uint8_t* row, int unit, int half, int steps, int step) {
        const auto* source = reinterpret_cast<const float*>(row) + min(2 * unit + step, steps - 1) * 32 + 16 * half;
#pragma unroll
        for (int piece = 0; piece < 4; ++piece) {
            values[step][piece >> 1][piece & 1] = *reinterpret_cast<const f32x4_a4*>(source + 4 * piece);
        }
    }
    __device__ __forceinline__ void load(const std::uint8_t* row, int unit, int half, int steps) {
#pragma unroll
        for (int step = 0; step < 2; ++step) load_step(row, unit, half, steps, step);
    }
    __device__ __forceinline__ void arrange() {}
    __device__ __forceinline__ Terms terms(int step, int chunk) const {
        float eight[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) eight[j] = values[step][chunk][j >> 2][j & 3];
        return cut(eight);
    }
};

// the codes of one chunk
template <std::uint32_t ENC>
__device__ __forceinline__ bf16x8 fragment_of(const Unit<ENC>& unit, int step, int chunk) {
    u32x4 out;
#pragma unroll
    for (int word = 0; word < 2; ++word) {
        std::uint32_t low, high;
        unit.words(step, chunk, word, low, high);
        out[2 * word] = low;
        out[2 * word + 1] = high;
    }
    return as_bf16(out);
}

template <std::uint32_t ENC>
constexpr bool kWholeBlocks = ENC == kEncQ4K || ENC == kEncQ5K || ENC == kEncQ6K;

__device__ __forceinline__ f32x16 product(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// the small terms first
__device__ __forceinline__ f32x16 product(const Terms& a, bf16x8 b, f32x16 c) {
    return product(a.first, b, product(a.second, b, product(a.third, b, c)));
}
__device__ __forceinline__ f32x16 product(const Terms& a, const Terms& b, f32x16 c) {
    c = product(a.second, b.third, product(a.third, b.second, c));
    c = product(a.second, b.second, product(a.first, b.third, product(a.third, b.first, c)));
    return product(a.first, b.first, product(a.second, b.first, product(a.first, b.second, c)));
}

// One step of 32 columns of one wave: 32 MT input rows (their terms in `a`) by 32 weight rows.
template <std::uint32_t ENC, int MT>
__device__ __forceinline__ void multiply(f32x16 (&acc)[MT], const Terms (&a)[MT][2], const Unit<ENC>& unit, int step) {
    using Slice = Unit<ENC>;
    if constexpr (!Slice::kScaled && MT == 1) {
        // A step's sums by themselves, then one addition: the eight (F32) or three products of a chunk
        // round at the size of a step's sum, not of the row's (relative error at 16 rows of 4,096
        // columns 2.4e-7 -> 1.3e-7 and 1.2e-7 -> 8.3e-8, with the tree below; the vector kernel's 1.6e-7 and 8.4e-8).
        f32x16 sums = f32x16{};
        if constexpr (ENC == kEncF32) {
#pragma unroll
            for (int chunk = 0; chunk < 2; ++chunk) sums = product(a[0][chunk], unit.terms(step, chunk), sums);
        } else {
            const bf16x8 b0 = fragment_of<ENC>(unit, step, 0), b1 = fragment_of<ENC>(unit, step, 1);
            sums = product(a[0][1].third, b1, product(a[0][0].third, b0, sums));
            sums = product(a[0][1].second, b1, product(a[0][0].second, b0, sums));
            sums = product(a[0][1].first, b1, product(a[0][0].first, b0, sums));
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][r] += sums[r];
    } else if constexpr (!Slice::kScaled) {
#pragma unroll
        for (int chunk = 0; chunk < 2; ++chunk) {
            if constexpr (ENC == kEncF32) {
                const Terms b = unit.terms(step, chunk);
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[m] = product(a[m][chunk], b, acc[m]);
            } else {
                const bf16x8 b = fragment_of<ENC>(unit, step, chunk);
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[m] = product(a[m][chunk], b, acc[m]);
            }
        }
    } else if constexpr (Slice::kScalePerChunk) {
#pragma unroll
        for (int chunk = 0; chunk < 2; ++chunk) {
            const bf16x8 b = fragment_of<ENC>(unit, step, chunk);
            const float scale = unit.scale(step, chunk);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const f32x16 sums = product(a[m][chunk], b, f32x16{});
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[m][r] = fmaf(scale, sums[r], acc[m][r]);
            }
        }
    } else {
        const bf16x8 b0 = fragment_of<ENC>(unit, step, 0), b1 = fragment_of<ENC>(unit, step, 1);
        const float scale = unit.scale(step, 0);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x16 sums = product(a[m][0].third, b0, f32x16{});
            sums = product(a[m][1].third, b1, sums);
            sums = product(a[m][0].second, b0, sums);
            sums = product(a[m][1].second, b1, sums);
            sums = product(a[m][0].first, b0, sums);
            sums = product(a[m][1].first, b1, sums);
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][r] = fmaf(scale, sums[r], acc[m][r]);
        }
    }
}

template <std::uint32_t ENC>
__device__ __forceinline__ void load_unit(Unit<ENC>& into, const std::uint8_t* tensor, const std::uint8_t* row, int unit,
                                          int half, int steps) {
    if constexpr (ENC == kEncQ6K) {
        into.load(tensor, row, unit, half);
    } else if constexpr (kWholeBlocks<ENC>) {
        into.load(row, unit, half);
    } else {
        into.load(row, unit, half, steps);
    }
}

// 32 columns of one weight row, decoded as the dequantize entry point does; infinite scales too.
template <std::uint32_t ENC>
struct DecodedPiece {
    u32x4_a2 codes[ENC == kEncF32 ? 8 : ENC == kEncBF16 ? 4 : 2], fifth[2];
    float scale[2], offset;
    int shift, high_shift;
    __device__ __forceinline__ void load(const std::uint8_t* row, int piece) {
        if constexpr (ENC == kEncF32 || ENC == kEncBF16) {
            constexpr int kLoads = ENC == kEncF32 ? 8 : 4;
#pragma unroll
            for (int k = 0; k < kLoads; ++k) {
                codes[k] = *reinterpret_cast<const u32x4_a2*>(row + (static_cast<std::int64_t>(piece) * kLoads + k) * 16);
            }
        } else if constexpr (ENC == kEncQ8_0) {
            const std::uint8_t* block = row + static_cast<std::int64_t>(piece) * 34;
            scale[0] = load_half(block);
            codes[0] = *reinterpret_cast<const u32x4_a2*>(block + 2);
            codes[1] = *reinterpret_cast<const u32x4_a2*>(block + 18);
        } else if constexpr (ENC == kEncQ6K) {
            const std::uint8_t* block = row + (piece >> 3) * 210;
            const int half = (piece >> 2) & 1, quarter = piece & 3;
            const float d = load_half(block + 208);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                codes[k] = *reinterpret_cast<const u32x4_a2*>(block + half * 64 + (quarter & 1) * 32 + 16 * k);
                fifth[k] = *reinterpret_cast<const u32x4_a2*>(block + 128 + half * 32 + 16 * k);
                scale[k] = d * static_cast<float>(static_cast<std::int8_t>(block[192 + half * 8 + quarter * 2 + k]));
            }
            shift = 4 * (quarter >> 1);
            high_shift = 2 * quarter;
        } else {
            const std::uint8_t* block = row + (piece >> 3) * static_cast<int>(block_bytes(ENC));
            int sc, m;
            k_scale_min(block + 4, piece & 7, &sc, &m);
            scale[0] = load_half(block) * static_cast<float>(sc);
            offset = load_half(block + 2) * static_cast<float>(m);
            const std::uint8_t* source = block + (ENC == kEncQ5K ? 48 : 16) + ((piece >> 1) & 3) * 32;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                codes[k] = *reinterpret_cast<const u32x4_a2*>(source + 16 * k);
                if constexpr (ENC == kEncQ5K) fifth[k] = *reinterpret_cast<const u32x4_a2*>(block + 16 + 16 * k);
            }
            shift = 4 * (piece & 1);
            high_shift = piece & 7;
        }
    }
    // columns 4 quad .. 4 quad + 3
    __device__ __forceinline__ void decode(int quad, float (&w)[4]) const {
        if constexpr (ENC == kEncF32) {
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = __uint_as_float(codes[quad][j]);
        } else if constexpr (ENC == kEncBF16) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const std::uint32_t two = codes[quad >> 1][2 * (quad & 1) + (j >> 1)];
                w[j] = __uint_as_float(j & 1 ? two & 0xffff0000u : two << 16);
            }
        } else {
            const std::uint32_t word = codes[quad >> 2][quad & 3];
            const std::uint32_t high = ENC == kEncQ5K || ENC == kEncQ6K ? fifth[quad >> 2][quad & 3] : 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (ENC == kEncQ8_0) {
                    w[j] = scale[0] * static_cast<float>(static_cast<std::int8_t>(word >> (8 * j)));
                } else if constexpr (ENC == kEncQ6K) {
                    const int q = static_cast<int>((word >> (shift + 8 * j) & 15u) | (high >> (high_shift + 8 * j) & 3u) << 4);
                    w[j] = scale[quad >> 2] * static_cast<float>(q - 32);
                } else {
                    int q = static_cast<int>(word >> (shift + 8 * j) & 15u);
                    if constexpr (ENC == kEncQ5K) q |= static_cast<int>(high >> (high_shift + 8 * j) & 1u) << 4;
                    w[j] = scale[0] * static_cast<float>(q) - offset;
                }
            }
        }
    }
};

// The sums of a tile's waves meet, 32 x 32 outputs at a time: register r of lane l is row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.  GROUPS sets of sums, set g in meeting[g]; the
// workgroup's wave `wave` of WAVES adds up and stores its registers' worth.  Sums that are not
// finite are left for take_again: a bit a lane, the word of the pass's part p in `again` of lane
// pass * 16 / WAVES + p.
template <std::uint32_t ENC, int GROUPS, int WAVES>
__device__ __forceinline__ void add_up_and_store(const float (*meeting)[16 * kWave], int pass, std::uint64_t& again,
                                                 int wave, int lane, const float* bias, float* output,
                                                 std::int64_t rows, std::int64_t output_dim, std::int64_t row0,
                                                 std::int64_t column) {
#pragma unroll
    for (int part = 0; part < 16 / WAVES; ++part) {
        const int r = part * WAVES + wave;
        float sums[GROUPS];  // (added in a balanced tree, which rounds less than one after another)
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) sums[g] = meeting[g][r * kWave + lane];
#pragma unroll
        for (int width = GROUPS / 2; width > 0; width /= 2) {
#pragma unroll
            for (int g = 0; g < width; ++g) sums[g] += sums[g + width];
        }
        const float total = sums[0] * kLower<ENC>;
        const std::int64_t row = row0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const bool exists = row < rows && column < output_dim, finite = isfinite(total);
        if (exists && finite) output[row * output_dim + column] = total + (bias != nullptr ? bias[column] : 0.0f);
        const std::uint64_t left = __ballot(exists && !finite);
        again = lane == pass * (16 / WAVES) + part ? left : again;
    }
}

// One output from the decoded weights and the activations as they are.  The lanes of a wave take
// different outputs; it ends early when all of them are NaN, which they stay.
template <std::uint32_t ENC>
__device__ __forceinline__ float decoded_dot(const std::uint8_t* row, const float* x, std::int64_t input_dim) {
    float even = 0.0f, odd = 0.0f;
    const auto take = [&](const float (&w)[4], const float* at) {
        const f32x4_a4 v = *reinterpret_cast<const f32x4_a4*>(at);
        even = fmaf(v[0], w[0], even);
        odd = fmaf(v[1], w[1], odd);
        even = fmaf(v[2], w[2], even);
        odd = fmaf(v[3], w[3], odd);
    };
    const int pieces = static_cast<int>(input_dim / 32);
#pragma unroll 1
    for (int piece = 0; piece < pieces; ++piece) {
        DecodedPiece<ENC> weights;
        weights.load(row, piece);
#pragma unroll
        for (int quad = 0; quad < 8; ++quad) {
            float w[4];
            weights.decode(quad, w);
            take(w, x + 32 * static_cast<std::int64_t>(piece) + 4 * quad);
        }
        if (__ballot(!isnan(even + odd)) == 0) break;
    }
    return even + odd;
}

// The outputs that a wave left in `again`, taken from the decoded weights: infinity less its own upper
// half is NaN where the product with the weight is infinite, and the lifted products leave the float
// range (activations above some 2^90 with codes, products above 2^80 with float weights) before those
// with the weights do.  MT: as in the kernels below.
// 4,096 -> 6,656 at 200 rows (Q8_0 / Q4_K, 60 / 68 us from Python): with a NaN in one row 62 / 72 us, in
// every row 100 / 91; an infinity or activations of 3e37 in one row 181 / 225, in every row 3.6 / 3.4 ms
// (a byte and a weight at a time: 1.1 / 1.9 ms for one row of either kind, 29 / 64 for all).
template <std::uint32_t ENC, int MT, int WAVES>
__device__ __forceinline__ void take_again(std::uint64_t again, int wave, const std::uint8_t* data,
                                           std::int64_t row_stride, const float* input, std::int64_t input_dim,
                                           const float* bias, float* output, std::int64_t output_dim,
                                           std::int64_t row0, std::int64_t col0) {
    const int lane = threadIdx.x & 63;
    for (std::uint64_t holders = __ballot(again != 0); holders != 0; holders &= holders - 1) {
        const int index = __builtin_ctzll(holders);
        const std::uint32_t low = __builtin_amdgcn_readlane(static_cast<std::uint32_t>(again), index);
        const std::uint32_t high = __builtin_amdgcn_readlane(static_cast<std::uint32_t>(again >> 32), index);
        if (((lane < 32 ? low : high) >> (lane & 31) & 1) != 0) {
            const int pass = index / (16 / WAVES), r = index % (16 / WAVES) * WAVES + wave;
            const std::int64_t row = row0 + 32 * (pass % MT) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            const std::int64_t column = col0 + 32 * (pass / MT) + (lane & 31);
            const float total = decoded_dot<ENC>(data + column * row_stride, input + row * input_dim, input_dim);
            output[row * output_dim + column] = total + (bias != nullptr ? bias[column] : 0.0f);
        }
    }
}

// The same as a function of its own: the small forms keep the registers and the schedule that their
// loop has by itself (4 rows of Q6_K, 5,120 -> 178: 23.3 -> 21.8 us).  The large forms, whose loops need
// every register, would lose some to the call.
template <std::uint32_t ENC, int MT, int WAVES>
__device__ __attribute__((noinline)) void take_again_apart(std::uint64_t again, int wave, const std::uint8_t* data,
                                                           std::int64_t row_stride, const float* input,
                                                           std::int64_t input_dim, const float* bias, float* output,
                                                           std::int64_t output_dim, std::int64_t row0,
                                                           std::int64_t col0) {
    take_again<ENC, MT, WAVES>(again, wave, data, row_stride, input, input_dim, bias, output, output_dim, row0, col0);
}

// Where a lane writes in LDS what others of its wave read.  LDS takes a wave's operations in order; this keeps
// the compiler to it, which sees one lane's addresses only: it cannot tell that the lane itself reads
// elsewhere.  (Fences around the writes, which nothing may pass: Q6_K up to 23 % slower, four rows of Q5_K 7.)
__device__ __forceinline__ std::uint32_t for_others(std::uint32_t place) {
    asm("" : "+v"(place));
    return place;
}

// A wave's activations of one step in LDS, [term][row tile][octet of columns][row] of 16 bytes; the rows
// of an octet change places by its number, so that four lanes with a row's octets and lanes with
// neighbouring rows of one find distinct banks.
template <int MT>
constexpr int kOwnTerms = 3 * MT * 4 * 512;
template <int MT, int NT, int WAVES>
constexpr int kSmallLds = WAVES * (kOwnTerms<MT> + 4 * 32 * MT * 4);

// WAVES waves share a tile of 32 MT input rows x 32 NT weight rows, of which the first 8 ITEMS of each
// 32 exist (the products of the others are not stored).  ITEMS = 0: each lane loads and cuts what it
// multiplies, which spares a short walk over K the way through LDS.
// PAIRS: Q8_0 rows of whole units.
template <std::uint32_t ENC, int MT, int NT, int WAVES, int ITEMS, bool PAIRS>
__global__ __launch_bounds__(WAVES * kWave, WAVES >= 16 ? 4 : 2) void linear_exact_small_kernel(
    const std::uint8_t* __restrict__ data, std::int64_t row_stride, const float* __restrict__ input,
    const float* __restrict__ bias, float* __restrict__ output, std::int64_t rows, std::int64_t input_dim,
    std::int64_t output_dim, int row_tiles) {
    using Slice = Unit<ENC>;
    extern __shared__ __attribute__((aligned(16))) std::uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inner = lane & 31, half = lane >> 5;
    const std::int64_t row0 = static_cast<std::int64_t>(blockIdx.x % row_tiles) * (32 * MT);
    const std::int64_t col0 = static_cast<std::int64_t>(blockIdx.x / row_tiles) * (32 * NT);
    // Rows past the end read the last one again; their results are not stored.
    const std::uint8_t* w_row[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) w_row[n] = data + min(col0 + 32 * n + inner, output_dim - 1) * row_stride;
    const int steps = static_cast<int>(input_dim / 32);
    const int units = (steps + 1) / 2;
    const int first_unit = units * wave / WAVES, end_unit = units * (wave + 1) / WAVES;
    const int last_step = min(2 * end_unit, steps) - 1;

    f32x16 acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = f32x16{};
    }
    // Cutter: quad lane % 8 of the rows 8 item + lane / 8; a load instruction reads whole lines.
    float* const sums = reinterpret_cast<float*>(lds + WAVES * kOwnTerms<MT>) + wave * 4 * 32 * MT;  // [step % 4][row]
    const int quad = lane & 7;
    // Rows past the end: the last one again.  Q6_K has no registers for every item's place (five ended up in
    // scratch): there they lie past the buffer's end, and a load has zeros for them from nowhere.
    constexpr bool kSpare = ENC == kEncQ6K;
    const std::int64_t tile_rows = min(rows - row0, std::int64_t(32 * MT));
    const __amdgpu_buffer_rsrc_t x_tile = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(input + row0 * input_dim), 0, kSpare ? static_cast<int>(tile_rows * input_dim * 4) : -1, 0x00020000);
    // (ITEMS = 0: columns 16 half + 8 chunk (kWide), 8 half + 16 chunk of row `inner`)
    const float* const x_row = input + min(row0 + inner, rows - 1) * input_dim + (Slice::kWide ? 16 : 8) * half;
    const int last_row = static_cast<int>(tile_rows - 1);
    constexpr int kLoads = ITEMS == 0 ? 4 : ITEMS;
    const std::uint32_t eight_rows = 32 * static_cast<std::uint32_t>(input_dim);
    std::uint32_t x_from[kSpare ? 1 : MT][kSpare ? 1 : kLoads];
#pragma unroll
    for (int m = 0; m < (kSpare ? 1 : MT); ++m) {
#pragma unroll
        for (int item = 0; item < (kSpare ? 1 : kLoads); ++item) {
            const int row = 32 * m + 8 * item + (lane >> 3);
            x_from[m][item] = 4 * (static_cast<std::uint32_t>(kSpare ? row : min(row, last_row)) *
                                       static_cast<std::uint32_t>(input_dim) + 4 * quad);
        }
    }
    f32x4_a4 x[MT][kLoads];  // of the step behind the one in LDS
    const auto load_inputs = [&](int step) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int item = 0; item < kLoads; ++item) {
                if constexpr (ITEMS == 0) {
                    constexpr int kNext = Slice::kWide ? 8 : 16;
                    x[m][item] = *reinterpret_cast<const f32x4_a4*>(
                        x_row + static_cast<std::int64_t>(min(step, last_step)) * 32 + kNext * (item >> 1) + 4 * (item & 1));
                } else {
                    x[m][item] = __builtin_bit_cast(f32x4_a4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                  x_tile,
                                                                  kSpare ? x_from[0][0] + (4 * m + item) * eight_rows
                                                                         : x_from[kSpare ? 0 : m][kSpare ? 0 : item],
                                                                  min(step, last_step) * 128, 0));
                }
            }
        }
    };
    const int octet = quad >> 1;
    // (eight rows on: 128 bytes, in the other order where the octet changes that bit)
    const std::uint32_t target =
        for_others(wave * kOwnTerms<MT> + octet * 512 + ((lane >> 3) ^ (4 * octet)) * 16 + (quad & 1) * 8);
    const std::uint32_t sum_target = for_others(lane >> 3);
    const auto cut_inputs = [&](int step) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int item = 0; item < ITEMS; ++item) {
                const f32x4_a4 v = x[m][item];
                std::uint32_t a0, b0, c0, a1, b1, c1;
                cut_pair(v[0], v[1], a0, b0, c0);
                cut_pair(v[2], v[3], a1, b1, c1);
                std::uint8_t* const to = lds + (target ^ (item * 128)) + m * 2048;
                *reinterpret_cast<uint2*>(to) = make_uint2(a0, a1);
                *reinterpret_cast<uint2*>(to + MT * 2048) = make_uint2(b0, b1);
                *reinterpret_cast<uint2*>(to + 2 * MT * 2048) = make_uint2(c0, c1);
                if constexpr (Slice::kMinimum) {
                    float total = ((v[0] + v[1]) + (v[2] + v[3])) * kLift;
                    total += of_lane<0xb1>(total);   // lane ^ 1
                    total += of_lane<0x4e>(total);   // lane ^ 2
                    total += of_lane<0x141>(total);  // the row's other four lanes (mirrored; all eight store the same sum)
                    sums[(step & 3) * 32 * MT + 32 * m + 8 * item + sum_target] = total;
                }
            }
        }
    };
    // Multiplier: octets 2 half + chunk (kWide) or 2 chunk + half of row `inner`
    const int from = Slice::kWide ? 2 * half : half;
    const std::uint32_t fragments = wave * kOwnTerms<MT> + from * 512 + (inner ^ (4 * from)) * 16;
    constexpr std::uint32_t kOther = Slice::kWide ? 512 + 4 * 16 : 1024 + 8 * 16;  // the bits that chunk 1 changes
    if (first_unit < end_unit) {
        // (2 x 2 tiles leave no registers for a second unit of float weights: a step's, as they are used up)
        constexpr bool kAhead = MT * NT < 4;
        Slice now[NT], next[NT];
        const auto load_weights = [&](Slice& into, const std::uint8_t* row, int unit) {
            if constexpr (PAIRS) {
                into.load_pair(row, unit, half);
            } else {
                load_unit<ENC>(into, data, row, unit, half, steps);
            }
        };
#pragma unroll
        for (int n = 0; n < NT; ++n) load_weights(now[n], w_row[n], first_unit);
        load_inputs(2 * first_unit);
        if constexpr (ITEMS > 0) {
            cut_inputs(2 * first_unit);
            load_inputs(2 * first_unit + 1);
        }
        for (int unit = first_unit; unit < end_unit; ++unit) {
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                if constexpr (ENC == kEncQ6K) now[n].align(data, w_row[n], unit);
                if constexpr (PAIRS) {
                    now[n].arrange_pair();
                } else {
                    now[n].arrange();
                }
            }
            if constexpr (kAhead) {
#pragma unroll
                for (int n = 0; n < NT; ++n) load_weights(next[n], w_row[n], min(unit + 1, end_unit - 1));
            }
            float partial[2];  // (ITEMS == 0: the lane's half of its row's sums)
#pragma unroll
            for (int step = 0; step < 2; ++step) {
                if (!kWholeBlocks<ENC> && 2 * unit + step > last_step) break;  // (uniform: a row's odd last block)
                const auto read = [&](int m, int chunk) {
                    const std::uint8_t* const at = lds + (fragments ^ (chunk * kOther)) + m * 2048;
                    return Terms{*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + MT * 2048),
                                 *reinterpret_cast<const bf16x8*>(at + 2 * MT * 2048)};
                };
                // (the cut behind the reads of what it overwrites: LDS keeps a wave's order)
                // (of 32 rows the one past a wave's end is worth leaving out: 25 rows of Q4_K, 2,304 -> 8,000
                // 15.2 -> 13.7 us; of fewer the branch costs as much)
                const auto cut_next = [&] {
                    if (ITEMS < 4 || ENC == kEncQ6K || step == 0 || unit + 1 < end_unit) cut_inputs(2 * unit + step + 1);
                    load_inputs(2 * unit + step + 2);
                };
                if constexpr (ITEMS == 0) {
                    Terms a[1][2];
                    partial[step] = 0.0f;
#pragma unroll
                    for (int chunk = 0; chunk < 2; ++chunk) {
                        float eight[8];
#pragma unroll
                        for (int j = 0; j < 8; ++j) eight[j] = x[0][2 * chunk + (j >> 2)][j & 3];
                        a[0][chunk] = cut(eight);
                        if constexpr (Slice::kMinimum) partial[step] += sum_of(eight) * kLift;
                    }
                    load_inputs(2 * unit + step + 1);
#pragma unroll
                    for (int n = 0; n < NT; ++n) multiply<ENC, 1>(acc[n], a, now[n], step);
                } else if constexpr (MT == 1) {
                    const Terms a[1][2] = {{read(0, 0), read(0, 1)}};
                    cut_next();
#pragma unroll
                    for (int n = 0; n < NT; ++n) multiply<ENC, 1>(acc[n], a, now[n], step);
                } else {
                    static_assert(MT == 1 || ENC == kEncF32, "no registers for both chunks' fragments");
#pragma unroll
                    for (int chunk = 0; chunk < 2; ++chunk) {
                        Terms a[MT];
#pragma unroll
                        for (int m = 0; m < MT; ++m) a[m] = read(m, chunk);
#pragma unroll
                        for (int n = 0; n < NT; ++n) {
                            const Terms b = now[n].terms(step, chunk);
#pragma unroll
                            for (int m = 0; m < MT; ++m) acc[n][m] = product(a[m], b, acc[n][m]);
                        }
                    }
                    if constexpr (!kAhead) {
#pragma unroll
                        for (int n = 0; n < NT; ++n) now[n].load_step(w_row[n], min(unit + 1, end_unit - 1), half, steps, step);
                    }
                    cut_next();
                }
            }
            if constexpr (Slice::kMinimum) {
                // k index = half: the lower lanes bring step 0's sums and minimums, the upper ones
                // step 1's
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    float total;
                    if constexpr (ITEMS == 0) {
                        total = (half != 0 ? partial[1] : partial[0]) + __shfl_xor(half != 0 ? partial[0] : partial[1], 32);
                    } else {
                        total = sums[((2 * unit + half) & 3) * 32 * MT + 32 * m + inner];
                    }
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        const float least = -(half != 0 ? now[n].minimum(1) : now[n].minimum(0));
                        acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x2f32(total, least, acc[n][m], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int n = 0; n < NT; ++n) now[n] = kAhead ? next[n] : now[n];
        }
    }
    if constexpr (ITEMS > 0) __syncthreads();
    float(*meeting)[16 * kWave] = reinterpret_cast<float(*)[16 * kWave]>(lds);
    std::uint64_t again = 0;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (n + m > 0) __syncthreads();
#pragma unroll
            for (int r = 0; r < 16; ++r) meeting[wave][r * kWave + lane] = acc[n][m][r];
            __syncthreads();
            add_up_and_store<ENC, WAVES, WAVES>(meeting, n * MT + m, again, wave, lane, bias, output, rows, output_dim,
                                                row0 + 32 * m, col0 + 32 * n + inner);
        }
    }
    if (__ballot(again != 0) != 0) {
        take_again_apart<ENC, MT, WAVES>(again, wave, data, row_stride, input, input_dim, bias, output, output_dim, row0,
                                         col0);
    }
}

// -- the large form --------------------------------------------------------------------------------

constexpr int kGroups = 4;                      // K groups of a workgroup
constexpr int kPartners = 2;                    // waves of a K group, 64 weight rows each
constexpr int kLargeWaves = kGroups * kPartners;
constexpr int kOctetBytes = 32 * 16 + 32;       // eight columns of 32 rows, as bf16; the padding keeps the
                                                // writes of four lanes that share a row in distinct banks
constexpr int kTermBytes = 4 * kOctetBytes;     // one term of 32 rows x 32 columns
template <int MT>
constexpr int kStepBytes = 3 * MT * kTermBytes;  // one step of a K group: [term][row tile][octet][row]
template <int MT>
constexpr int kSumBytes = 4 * 32 * MT * 4;       // sums of the activations, [step % 4][row]
template <int MT>
constexpr int kGroupBytes = 2 * kStepBytes<MT> + kSumBytes<MT>;

// A wave's 64 weight rows on their way: pieces of 16 bytes, neighbouring lanes on neighbouring pieces of
// a row, wait in registers and lie in LDS for one unit (bf16: one step).  A row's pieces are one or two runs:
// the first kFirst of them, then kSecond, each run of all rows an area of its own, row by row.
template <std::uint32_t ENC>
struct Staged {
    static constexpr int kFirst = ENC == kEncQ4K ? 1 : ENC == kEncQ5K ? 3 : ENC == kEncQ8_0 ? 5 : 4;
    static constexpr int kSecond = ENC == kEncQ8_0 || ENC == kEncBF16 ? 0 : 2;
    static constexpr int kPieces = kFirst + kSecond;
    static constexpr int kBytes = 64 * 16 * kPieces;
    // bf16: a unit is a line a row, requested as a whole (lines come to the vector cache as such, and
    // do not stay there for a second request), and lies in LDS a step at a time
    static constexpr int kParts = ENC == kEncBF16 ? 2 : 1;
    u32x4_a2 held[kParts][kPieces];
    std::uint32_t scales[2];   // Q6_K: of the rows `inner` and 32 + inner, as Unit loads them
    std::uint32_t from[kPieces], scales_from[2];
    std::uint8_t* first;       // where the lane's pieces go
    std::uint8_t* second;
    const std::uint8_t* tile;  // the wave's first row

    __device__ __forceinline__ Staged(const std::uint8_t* data, std::int64_t row_stride, std::int64_t col0,
                                      std::int64_t output_dim, std::uint8_t* lds, int lane) {
        const std::int64_t row0 = min(col0, output_dim - 1);
        const int last = static_cast<int>(min(output_dim - 1 - row0, std::int64_t(63)));  // (rows past the end: the last one again)
        const auto bytes = [&](int row) { return static_cast<std::uint32_t>(min(row, last)) * static_cast<std::uint32_t>(row_stride); };
        tile = data + row0 * row_stride;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int lanes = i < kFirst ? kFirst : kSecond, index = (i < kFirst ? i : i - kFirst) * kWave + lane;
            const int row = index / lanes, piece = index % lanes;
            // (Q8_0, two blocks of 34 bytes: the codes of the second one as two pieces of their own)
            from[i] = bytes(row) + 16 * piece - (ENC == kEncQ8_0 && piece >= 2 ? 12 : 0);
        }
        if constexpr (ENC == kEncQ6K) {
#pragma unroll
            for (int n = 0; n < 2; ++n) scales_from[n] = bytes(32 * n + (lane & 31));
        }
        // runs of four and of two pieces would put every fourth or eighth row on the same banks
        first = lds + for_others(kFirst == 4 ? (lane ^ (lane >> 4)) * 16 : lane * 16);
        second = lds + kFirst * 1024 + for_others((lane ^ (lane >> 4 & 1)) * 16);
    }
    __device__ __forceinline__ void load(int unit) {
        const std::uint8_t* one = tile;
        const std::uint8_t* two = tile;
        if constexpr (ENC == kEncQ8_0) {
            one += unit * 68;
        } else if constexpr (ENC == kEncBF16) {
            one += unit * 128;
        } else {
            one += (unit >> 2) * static_cast<int>(block_bytes(ENC));
            two = one + (ENC == kEncQ4K ? 16 + 32 * (unit & 3) : ENC == kEncQ5K ? 48 + 32 * (unit & 3) : 128 + 16 * (unit & 2));
            if constexpr (ENC == kEncQ6K) one += 32 * (unit & 2);
        }
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
#pragma unroll
            for (int part = 0; part < kParts; ++part) {
                held[part][i] = *reinterpret_cast<const u32x4_a2*>((i < kFirst ? one : two) + (from[i] + 64 * part));
            }
        }
    }
    // (Q6_K) straight into registers, when those of the unit before are taken
    __device__ __forceinline__ void load_scales(int unit, int half) {
        typedef std::uint32_t u32_a2 __attribute__((aligned(2)));
        const std::uint8_t* block = tile + (unit >> 2) * 210;
        const int place = half != 0 ? 192 + 4 * (unit & 3) : 206;
#pragma unroll
        for (int n = 0; n < 2; ++n) scales[n] = *reinterpret_cast<const u32_a2*>(block + (scales_from[n] + place));
    }
    __device__ __forceinline__ void store(int part, int piece) const {
        std::uint8_t* const target = piece < kFirst ? first + piece * 1024 : second + (piece - kFirst) * 1024;
        *reinterpret_cast<u32x4*>(target) = held[part][piece];
    }
};

// ... and back: a lane's words of row 32 n + inner
template <std::uint32_t ENC>
struct Taken {
    Unit<ENC> unit;
    std::uint32_t tail;
    __device__ __forceinline__ void take(const std::uint8_t* lds, const Staged<ENC>& staged, int n, int at, int step, int lane) {
        const int inner = lane & 31, half = lane >> 5;
        const auto piece = [&](int offset) { return *reinterpret_cast<const u32x4*>(lds + offset); };
        if constexpr (ENC == kEncQ8_0) {
            const int row = (32 * n + inner) * 80;
            if (step == 0) {
                unit.codes[0] = piece(row + 16 * half);
                tail = *reinterpret_cast<const std::uint32_t*>(lds + row + 16 + 28 * half);
            } else {
                unit.codes[1] = piece(row + 48 + 16 * half);
            }
        } else if constexpr (ENC == kEncBF16) {
            const int row = (32 * n + inner) * 64, turn = inner >> 2 & 3;
            unit.values[step][0] = piece(row + 16 * ((2 * half) ^ turn));
            unit.values[step][1] = piece(row + 16 * ((2 * half + 1) ^ turn));
        } else if (step == 0) {
            const int second = 1024 * Staged<ENC>::kFirst + (32 * n + inner) * 32 + 16 * (half ^ (inner >> 3 & 1));
            if constexpr (ENC == kEncQ6K) {
                const int row = (32 * n + inner) * 64, turn = inner >> 2 & 3;
                unit.upper = at & 1;
                unit.low[0] = piece(row + 16 * (half ^ turn));
                unit.low[1] = piece(row + 16 * ((2 + half) ^ turn));
                unit.high = piece(second);
                unit.scales = staged.scales[n];
            } else {
                const int row = (32 * n + inner) * 16 * Staged<ENC>::kFirst;
                unit.group = at & 3;
                unit.header = piece(row);
                if constexpr (ENC == kEncQ5K) unit.fifth = piece(row + 16 + 16 * half);
                unit.codes = piece(second);
            }
        }
    }
    // once, when the words are there
    __device__ __forceinline__ void arrange(int step, int half) {
        if constexpr (ENC == kEncQ8_0) {
            // the first block's codes begin at byte 2; behind the upper lanes' lies the second block's scale
            if (step != 0) return;
            unit.d[0] = half != 0 ? tail >> 16 : unit.codes[0][0];
            unit.d[0] &= 0xffffu;
#pragma unroll
            for (int word = 0; word < 4; ++word) {
                unit.codes[0][word] = __builtin_amdgcn_alignbyte(word < 3 ? unit.codes[0][word + 1] : tail, unit.codes[0][word], 2);
            }
            unit.arrange();
        } else if (step == 0) {
            unit.arrange();
        }
    }
};

template <std::uint32_t ENC, int MT>
__global__ __launch_bounds__(kLargeWaves * kWave, 2) void linear_exact_kernel(
    const std::uint8_t* __restrict__ data, std::int64_t row_stride, const float* __restrict__ input,
    const float* __restrict__ bias, float* __restrict__ output, std::int64_t rows, std::int64_t input_dim,
    std::int64_t output_dim, int row_tiles) {
    using Slice = Unit<ENC>;
    extern __shared__ __attribute__((aligned(16))) std::uint8_t lds[];
    constexpr int kItems = 2 * MT;  // quads (four columns of a row) that a lane cuts per step
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = wave / kPartners, partner = wave % kPartners;
    const int inner = lane & 31, half = lane >> 5;
    // row tiles next to each other share their weight rows, which come from L2 for all but one
    const std::int64_t row0 = static_cast<std::int64_t>(blockIdx.x % row_tiles) * (32 * MT);
    const std::int64_t col0 = static_cast<std::int64_t>(blockIdx.x / row_tiles) * (64 * kPartners) + 64 * partner;
    const int steps = static_cast<int>(input_dim / 32);
    const int units = (steps + 1) / 2;
    const int first_unit = units * group / kGroups, end_unit = units * (group + 1) / kGroups;

    // cutter's role: quad lane % 8 of the rows 8 (2 item + partner) + lane / 8: a load instruction
    // reads whole 128-byte lines of eight rows
    std::uint8_t* const own = lds + group * kGroupBytes<MT>;
    float* const sums = reinterpret_cast<float*>(own + 2 * kStepBytes<MT>);
    const int quad = lane & 7;
    // (a buffer load takes a register for the row and a scalar for the step; 64-bit addresses took eight
    // registers and an addition a load: 200 rows of Q8_0 81.8 -> 79.6 us, of Q5_K 86 -> 80)
    const __amdgpu_buffer_rsrc_t x_tile = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(input + row0 * input_dim), 0, 0xffffffff, 0x00020000);
    std::uint32_t x_row[kItems];  // bytes from the tile's first row
#pragma unroll
    for (int item = 0; item < kItems; ++item) {
        const int row = min(8 * (2 * item + partner) + (lane >> 3), static_cast<int>(min(rows - 1 - row0, std::int64_t(64))));
        x_row[item] = 4 * (static_cast<std::uint32_t>(row) * static_cast<std::uint32_t>(input_dim) + 4 * quad);
    }
    const int target = (quad >> 1) * kOctetBytes + (8 * partner + (lane >> 3)) * 16 + (quad & 1) * 8;
    f32x4_a4 x[kItems];
    const auto load_input = [&](int item, int step) {
        x[item] = __builtin_bit_cast(
            f32x4_a4, __builtin_amdgcn_raw_buffer_load_b128(x_tile, x_row[item], min(step, steps - 1) * 128, 0));
    };
    const auto cut_input = [&](int item, int step) {
        std::uint32_t a0, b0, c0, a1, b1, c1;
        cut_pair(x[item][0], x[item][1], a0, b0, c0);
        cut_pair(x[item][2], x[item][3], a1, b1, c1);
        std::uint8_t* const stage = own + (step & 1) * kStepBytes<MT> + (item >> 1) * kTermBytes + target + (item & 1) * 256;
        *reinterpret_cast<uint2*>(stage) = make_uint2(c0, c1);
        *reinterpret_cast<uint2*>(stage + MT * kTermBytes) = make_uint2(b0, b1);
        *reinterpret_cast<uint2*>(stage + 2 * MT * kTermBytes) = make_uint2(a0, a1);
        if constexpr (Slice::kMinimum) {
            float total = ((x[item][0] + x[item][1]) + (x[item][2] + x[item][3])) * kLift;
            total += of_lane<0xb1>(total);   // lane ^ 1
            total += of_lane<0x4e>(total);   // lane ^ 2
            total += of_lane<0x141>(total);  // the row's other four lanes (mirrored; all eight store the same sum)
            sums[(step & 3) * 32 * MT + 8 * (2 * item + partner) + (lane >> 3)] = total;
        }
    };
    // multiplier's role: the lane's fragment of a term, octets 2 half + chunk (wide) or 2 chunk + half.
    // Fragments in the order in which they are used: the small terms first, chunk by chunk where a
    // scale belongs to a chunk.
    constexpr int kHalfOctets = Slice::kWide ? 2 : 1, kChunkOctets = Slice::kWide ? 1 : 2;
    constexpr int kUses = 6, kSum = Slice::kScalePerChunk ? 3 : 6;  // products of a tile, of one scale
    const auto chunk_of = [](int use) { return Slice::kScalePerChunk ? use / 3 : use & 1; };
    const auto term_of = [](int use) { return Slice::kScalePerChunk ? use % 3 : use >> 1; };
    const std::uint8_t* const fragments = own + half * kHalfOctets * kOctetBytes + inner * 16;
    const auto read_fragment = [&](int use, int m, int step) {
        return *reinterpret_cast<const bf16x8*>(fragments + (step & 1) * kStepBytes<MT> + term_of(use) * MT * kTermBytes +
                                                m * kTermBytes + chunk_of(use) * kChunkOctets * kOctetBytes);
    };

    using Stage = Staged<ENC>;
    std::uint8_t* const stage = lds + kGroups * kGroupBytes<MT> + wave * Stage::kBytes;
    Stage weights(data, row_stride, col0, output_dim, stage, lane);
    Taken<ENC> taken[2];
    f32x16 acc[2][MT];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = f32x16{};
    }
    bf16x8 a[kUses];
    u32x4 b[2][2];  // [n][chunk]: codes; those of n = 0 are decoded a step ahead, those of n = 1 under the first tile
    float scale[2][2], scale_before[2];
    const auto load_weights = [&](int unit) { weights.load(min(unit, end_unit - 1)); };
    const auto decode_piece = [&](int n, int step, int piece) {
        Taken<ENC>& source = taken[n];
        if (piece == 0) source.arrange(step, half);
        const int chunk = piece >> 1, word = piece & 1;
        std::uint32_t low, high;
        source.unit.words(step, chunk, word, low, high);
        b[n][chunk][2 * word] = low;
        b[n][chunk][2 * word + 1] = high;
        if (word == 1) scale[n][chunk] = source.unit.scale(step, chunk);
    };
    if (first_unit < end_unit) {
        load_weights(first_unit);
#pragma unroll
        for (int item = 0; item < kItems; ++item) load_input(item, 2 * first_unit);
#pragma unroll
        for (int item = 0; item < kItems; ++item) {
            cut_input(item, 2 * first_unit);
            load_input(item, 2 * first_unit + 1);
        }
#pragma unroll
        for (int piece = 0; piece < Stage::kPieces; ++piece) weights.store(0, piece);
        if constexpr (ENC == kEncQ6K) weights.load_scales(first_unit, half);
        taken[0].take(stage, weights, 0, first_unit, 0, lane);
        taken[1].take(stage, weights, 1, first_unit, 0, lane);
        if constexpr (Stage::kParts == 1) load_weights(first_unit + 1);
#pragma unroll
        for (int piece = 0; piece < 4; ++piece) decode_piece(0, 0, piece);
    }
    // Each wave says which step's terms it has handed over; its partner waits for that alone.  (The two
    // take the same steps, and either says so before it waits: each wait ends.)
    // (a word a lane: 64 writes of one word would take turns)
    std::uint32_t* const handed = reinterpret_cast<std::uint32_t*>(lds + kGroups * kGroupBytes<MT> + kLargeWaves * Stage::kBytes);
    handed[wave * kWave + lane] = 2 * first_unit;
    __syncthreads();
    if (first_unit < end_unit) {
#pragma unroll
        for (int use = 0; use < kUses; ++use) a[use] = read_fragment(use, 0, 2 * first_unit);
    }

    const auto partners_step = [&] {
        return __hip_atomic_load(&handed[(wave ^ 1) * kWave], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const std::uint32_t partners_word = static_cast<std::uint32_t>(reinterpret_cast<std::uintptr_t>(
        (__attribute__((address_space(3))) std::uint32_t*)(handed + (wave ^ 1) * kWave)));
    // (in assembly: with a branch that the compiler sees, its registers no longer do)
    const auto wait_for_partner = [&](std::uint32_t seen, int step) {
        std::uint32_t word, place = partners_word;
        int value = static_cast<int>(__builtin_amdgcn_readfirstlane(seen));
        __asm__ volatile(
            "s_cmp_lt_i32 %0, %3\n\t"
            "s_cbranch_scc0 .Lhanded%=\n"
            ".Lwait%=:\n\t"
            "ds_read_b32 %1, %2\n\t"
            "s_waitcnt lgkmcnt(0)\n\t"
            "v_readfirstlane_b32 %0, %1\n\t"
            "s_cmp_lt_i32 %0, %3\n\t"
            "s_cbranch_scc1 .Lwait%=\n"
            ".Lhanded%=:"
            : "+s"(value), "=&v"(word)
            : "v"(place), "s"(step)
            : "scc", "memory");
    };
    // One unit, two steps.
    const auto pass = [&](int unit) {
        float least[2] = {};
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            const int at = 2 * unit + step;
            // A step is 12 MT slots of one matrix instruction each, fenced against reordering: what
            // stands between two of them is issued in their shadow (32 cycles, eight vector
            // instructions).  The waves of a unit run in step, so that nothing else would overlap.
            // Slots bring: the scaling of the sums before; the next step's activations cut and
            // handed over (before the last tile, whose slots read the next step's fragments) and
            // their successors requested; codes.
            constexpr int kSlots = 12 * MT, kHandOver = kSlots - kUses, kPerPiece = MT == 1 ? 2 : 4;
            constexpr int kHandOut = (kItems - 1) * kPerPiece;  // the last piece of activations is cut
            f32x16 partial[2];
            std::uint32_t seen = 0;
#pragma unroll
            for (int slot = 0; slot < kSlots; ++slot) {
                const int tile = slot / kUses, use = slot % kUses, m = tile >> 1, n = tile & 1;
                const int sum = slot / kSum;  // sums since the step's start; partial[sum & 1]
                __builtin_amdgcn_sched_barrier(0);
                if (slot == kHandOver) {
                    wait_for_partner(seen, at + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (Slice::kScaled) {
                    partial[sum & 1] = product(a[use], as_bf16(b[n][chunk_of(use)]),
                                               slot % kSum == 0 ? f32x16{} : partial[sum & 1]);
                    if (sum > 0 && slot % kSum >= 1 && slot % kSum <= 2) {
                        const int before = sum - 1, at_tile = before * kSum / kUses;
                        const float factor = slot >= kHandOver && (at_tile & 1) == 0 ? scale_before[Slice::kScalePerChunk ? before & 1 : 0]
                                                                   : scale[at_tile & 1][Slice::kScalePerChunk ? before & 1 : 0];
#pragma unroll
                        for (int r = 8 * (slot % kSum - 1); r < 8 * (slot % kSum); ++r) {
                            acc[at_tile & 1][at_tile >> 1][r] =
                                fmaf(factor, partial[before & 1][r], acc[at_tile & 1][at_tile >> 1][r]);
                        }
                    }
                } else {
                    acc[n][m] = product(a[use], as_bf16(b[n][chunk_of(use)]), acc[n][m]);
                }
                if (n == 1) a[use] = m + 1 < MT ? read_fragment(use, m + 1, at) : read_fragment(use, 0, at + 1);
                if (slot % kPerPiece == 0 && slot / kPerPiece < kItems) {
                    cut_input(slot / kPerPiece, at + 1);
                    load_input(slot / kPerPiece, at + 2);
                }
                if (slot < 4) decode_piece(1, step, slot);
                // What the next step (packed formats: the next unit) needs goes to where the wave's reads
                // are behind it: LDS keeps a wave's order.  bf16's next unit, requested in this one, as late
                // as its readers allow.
                constexpr int kStores = (Stage::kPieces + 1) / 2;
                const int first_store = Stage::kParts == 2 && step == 1 ? kHandOver - 1 - kStores : 0;
                if ((Stage::kParts == 2 || step == 1) && slot >= first_store && slot < first_store + kStores) {
                    const int piece = 2 * (slot - first_store);
                    weights.store(Stage::kParts == 2 ? 1 - step : 0, piece);
                    if (piece + 1 < Stage::kPieces) weights.store(Stage::kParts == 2 ? 1 - step : 0, piece + 1);
                }
                if (slot == 4) {
                    if constexpr (Slice::kMinimum) {
#pragma unroll
                        for (int k = 0; k < 2 && step == 1; ++k) least[k] = -(half != 0 ? taken[k].unit.minimum(1) : taken[k].unit.minimum(0));
                    }
                    if (step == (Stage::kParts == 2 ? 0 : 1)) load_weights(unit + (Stage::kParts == 2 ? 1 : 2));
                }
                if (ENC == kEncQ6K && slot == 5 && step == 0) weights.load_scales(min(unit + 1, end_unit - 1), half);
                if (slot == kHandOut) {
                    // (LDS takes a wave's operations in order: the terms, and the reads of what the partner will
                    // overwrite next, are ahead of this)
                    __asm__ volatile("" ::: "memory");
                    __hip_atomic_store(&handed[wave * kWave + lane], at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __asm__ volatile("" ::: "memory");
                }
                if (slot == kHandOver - 2) seen = partners_step();
                if (slot == kHandOver - 1) taken[0].take(stage, weights, 0, unit + step, 1 - step, lane);
                if (slot == kHandOver + 4) taken[1].take(stage, weights, 1, unit + step, 1 - step, lane);
                if (slot == kHandOver) {  // (the last sums of n = 0 are scaled below, with the old factors)
                    scale_before[0] = scale[0][0];
                    scale_before[1] = scale[0][1];
                }
                if (slot > kHandOver && slot <= kHandOver + 4) {
                    decode_piece(0, 1 - step, slot - kHandOver - 1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (Slice::kScaled) {  // the last sums
                const float factor = scale[1][Slice::kScalePerChunk ? 1 : 0];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[1][MT - 1][r] = fmaf(factor, partial[(kSlots / kSum - 1) & 1][r], acc[1][MT - 1][r]);
                }
            }
            if constexpr (Slice::kMinimum) {
                // k index = half: the lower lanes bring step 0's sums and minimums, the upper step 1's
#pragma unroll
                for (int m = 0; m < MT && step == 1; ++m) {
                    const float total = sums[((2 * unit + half) & 3) * 32 * MT + 32 * m + inner];
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x2f32(total, least[n], acc[n][m], 0, 0, 0);
                    }
                }
            }
        }
    };
    for (int unit = first_unit; unit < end_unit; ++unit) pass(unit);
    __syncthreads();

    // meeting[group] of either partner's 32 x 32 outputs: partner p's sets lie behind each other
    float(*meeting)[16 * kWave] = reinterpret_cast<float(*)[16 * kWave]>(lds);
    std::uint64_t again = 0;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (n + m > 0) __syncthreads();
#pragma unroll
            for (int r = 0; r < 16; ++r) meeting[partner * kGroups + group][r * kWave + lane] = acc[n][m][r];
            __syncthreads();
            add_up_and_store<ENC, kGroups, kGroups>(meeting + partner * kGroups, n * MT + m, again, group, lane, bias,
                                                    output, rows, output_dim, row0 + 32 * m, col0 + 32 * n + inner);
        }
    }
    if (__ballot(again != 0) != 0) {
        take_again<ENC, MT, kGroups>(again, group, data, row_stride, input, input_dim, bias, output, output_dim, row0, col0);
    }
}

template <std::uint32_t ENC, int MT>
void launch_large(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                  hipStream_t stream) {
    const std::int64_t row_tiles = (rows + 32 * MT - 1) / (32 * MT);
    const std::int64_t column_tiles = (weight.output_dim + 64 * kPartners - 1) / (64 * kPartners);
    constexpr int kLds = kGroups * kGroupBytes<MT> + kLargeWaves * (Staged<ENC>::kBytes + 4 * kWave);
    static_assert(kLds <= 160 * 1024 && kLds >= kLargeWaves * 16 * kWave * 4, "the waves' sums meet in the same memory");
    allow_large_lds<linear_exact_kernel<ENC, MT>>();
    hipLaunchKernelGGL((linear_exact_kernel<ENC, MT>), dim3(static_cast<unsigned>(row_tiles * column_tiles)),
                       dim3(kLargeWaves * kWave), kLds, stream, weight.data, weight.row_stride_bytes, input,
                       bias, output, rows, weight.input_dim, weight.output_dim, static_cast<int>(row_tiles));
}

template <std::uint32_t ENC, int MT, int NT, int WAVES, int ITEMS>
void launch_small_form(const Descriptor& weight, const float* input, const float* bias, float* output,
                       std::int64_t rows, hipStream_t stream) {
    const std::int64_t row_tiles = (rows + 32 * MT - 1) / (32 * MT);
    const std::int64_t column_tiles = (weight.output_dim + 32 * NT - 1) / (32 * NT);
    constexpr int kLds = ITEMS == 0 ? WAVES * 16 * kWave * 4 : kSmallLds<MT, NT, WAVES>;
    static_assert(kLds >= WAVES * 16 * kWave * 4, "the waves' sums meet in the same memory");
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(row_tiles * column_tiles)), dim3(WAVES * kWave), kLds, stream,
                           weight.data, weight.row_stride_bytes, input, bias, output, rows, weight.input_dim,
                           weight.output_dim, static_cast<int>(row_tiles));
    };
    if constexpr (ENC == kEncQ8_0) {
        if (weight.input_dim % 64 == 0) {
            allow_large_lds<linear_exact_small_kernel<ENC, MT, NT, WAVES, ITEMS, true>>();
            return launch(linear_exact_small_kernel<ENC, MT, NT, WAVES, ITEMS, true>);
        }
    }
    allow_large_lds<linear_exact_small_kernel<ENC, MT, NT, WAVES, ITEMS, false>>();
    launch(linear_exact_small_kernel<ENC, MT, NT, WAVES, ITEMS, false>);
}

template <std::uint32_t ENC, int MT, int NT, int WAVES>
void launch_small(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                  hipStream_t stream) {
    if constexpr (WAVES == 16 && kWholeBlocks<ENC>) {
        // Short walks, the same bits with or without the way through LDS.  Q6_K from 1,155 shapes of 7 to 64 rows, 512 to 3,072
        // columns and 64 to 6,656 outputs, geometric means of the time through LDS over the time without: up to 8 rows 0.95 to
        // 0.97 at 512 to 1,024 columns; 9 to 16 rows 1.03 to 1.05 there, 0.94 to 0.96 at 1,280; 17 to 20 rows 1.17 to 1.21 there,
        // 1.01 to 1.07 at 1,280 to 2,560, 0.97 to 0.99 at 2,816; more rows 1.04 to 1.21 up to 1,024, 1.00 to 1.05 up to 1,536,
        // 0.95 to 1.02 at 1,792.  Q4_K and Q5_K: 25 rows of Q4_K 2,560 -> 8,000 14.3 and 13.7 us, 3,072 -> 2,000 12.9 and
        // 13.4, and 2,048 -> 300 9.1 and 10.3.
        const bool wide = (weight.output_dim + 31) / 32 * 3 > compute_units();
        const std::int64_t q6_columns = rows <= 8 ? 0 : rows <= 16 ? 1024 : rows <= 20 ? 2560 : 1536;
        if (ENC == kEncQ6K ? weight.input_dim <= q6_columns : rows > 16 && weight.input_dim <= 2560 && wide) {
            return launch_small_form<ENC, MT, NT, WAVES, 0>(weight, input, bias, output, rows, stream);
        }
    }
    if constexpr (MT == 1) {
        if (rows <= 8) return launch_small_form<ENC, MT, NT, WAVES, 1>(weight, input, bias, output, rows, stream);
        if (rows <= 16) return launch_small_form<ENC, MT, NT, WAVES, 2>(weight, input, bias, output, rows, stream);
    }
    launch_small_form<ENC, MT, NT, WAVES, 4>(weight, input, bias, output, rows, stream);
}

// What a round of the larger tiles costs in rounds of 32 x 32: 32 x 64, 32 x 128 and 64 x 128 (F32:
// 64 x 32 and 64 x 64).  They choose how many waves share K, and with that how a sum rounds: 16
// (32 x 32 tiles), eight (32 x 64) or four (the tiles of 128 columns; F32: eight, then four).  From a sweep
// of 484 shapes an encoding (4..512 rows, 64..8,192 outputs, 2,048..8,192 columns) before the tiles of
// 128 columns loaded whole lines.  Those would win more shapes of Q4_K and Q5_K since (257 to 512 rows into
// 4,128 to 8,192 outputs: 1.5, 1.9 and 3.3 lose 0.01 % to the fastest form on average, these 0.6 %,
// at most 20), with sums of half the waves: 2.6e-7 of the result (rms) instead of 2.4e-7 at 4,096 columns,
// 3.3e-7 instead of 3.0e-7 at 8,192.  F32's 1.35 and 1.65 would gain 0.2 % with 3.4e-7 instead of 1.3e-7.
template <std::uint32_t ENC>
constexpr double kRounds[3] = {1.45, 2.1, 2.6};  // Q6_K, Q8_0
template <>
constexpr double kRounds<kEncQ4K>[3] = {1.4, 2.5, 3.9};
template <>
constexpr double kRounds<kEncQ5K>[3] = {1.35, 2.5, 3.6};
template <>
constexpr double kRounds<kEncBF16>[3] = {1.5, 2.0, 2.4};
template <>
constexpr double kRounds<kEncF32>[3] = {1.6, 2.1, 0.0};
// A round of 64 x 128 in rounds of 32 x 128, whose sums are the same: from 242 shapes an encoding with
// the tiles as they are (Q8_0 with 1.24: 0.3 % slower on average, 7 % at most).
template <std::uint32_t ENC>
constexpr double kTaller = 1.24;  // Q6_K, bf16
template <>
constexpr double kTaller<kEncQ4K> = 1.74;
template <>
constexpr double kTaller<kEncQ5K> = 1.74;
template <>
constexpr double kTaller<kEncQ8_0> = 1.65;

template <std::uint32_t ENC>
void launch_for(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                hipStream_t stream) {
    // A round of tiles, one workgroup a unit, takes as long however many of its rows are real: the
    // form with the cheapest rounds takes the call.
    const std::int64_t units = compute_units();
    const auto rounds = [&](std::int64_t height, std::int64_t width) {
        const std::int64_t tiles = (rows + height - 1) / height * ((weight.output_dim + width - 1) / width);
        return static_cast<double>((tiles + units - 1) / units);
    };
    const double cost_small = rounds(32, 32);
    if constexpr (ENC == kEncF32) {
        const double cost_high = kRounds<ENC>[0] * rounds(64, 32), cost_square = kRounds<ENC>[1] * rounds(64, 64);
        if (cost_square <= cost_high && cost_square <= cost_small) {
            launch_small<ENC, 2, 2, 4>(weight, input, bias, output, rows, stream);
        } else if (cost_high <= cost_small) {
            launch_small<ENC, 2, 1, 4>(weight, input, bias, output, rows, stream);
        } else {
            launch_small<ENC, 1, 1, 8>(weight, input, bias, output, rows, stream);
        }
    } else {
        const bool whole = weight.input_dim % 64 == 0;
        const double cost_wide = kRounds<ENC>[0] * rounds(32, 64);
        const double low = rounds(32, 128), high = rounds(64, 128);
        const double cost_large = whole ? std::min(kRounds<ENC>[1] * low, kRounds<ENC>[2] * high) : 1e30;
        if (cost_large <= cost_wide && cost_large <= cost_small) {
            if (kTaller<ENC> * high <= low) {
                launch_large<ENC, 2>(weight, input, bias, output, rows, stream);
            } else {
                launch_large<ENC, 1>(weight, input, bias, output, rows, stream);
            }
        } else if (cost_wide <= cost_small) {
            launch_small<ENC, 1, 2, 8>(weight, input, bias, output, rows, stream);
        } else {
            launch_small<ENC, 1, 1, 16>(weight, input, bias, output, rows, stream);
        }
    }
}

}  // namespace

bool linear_exact_supports(const Descriptor& weight, std::int64_t rows) {
    const std::int64_t tiles = ((rows + 31) / 32) * ((weight.output_dim + 31) / 32);
    return rows > 0 && weight.input_dim > 0 && weight.input_dim % 32 == 0 && block_bytes(weight.encoding) != 0 &&
           weight.input_dim <= (std::int64_t(1) << 23) &&  // a tile's rows within 32-bit offsets
           tiles < (std::int64_t(1) << 31);
}

void launch_linear_exact(const Descriptor& weight, const float* input, const float* bias, float* output,
                         std::int64_t rows, hipStream_t stream) {
    switch (weight.encoding) {
        case kEncQ4K: launch_for<kEncQ4K>(weight, input, bias, output, rows, stream); break;
        case kEncQ5K: launch_for<kEncQ5K>(weight, input, bias, output, rows, stream); break;
        case kEncQ6K: launch_for<kEncQ6K>(weight, input, bias, output, rows, stream); break;
        case kEncQ8_0: launch_for<kEncQ8_0>(weight, input, bias, output, rows, stream); break;
        case kEncBF16: launch_for<kEncBF16>(weight, input, bias, output, rows, stream); break;
        default: launch_for<kEncF32>(weight, input, bias, output, rows, stream); break;
    }
}

}  // namespace nfn
