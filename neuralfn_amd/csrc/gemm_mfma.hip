// Prefill dequant-GEMM on the fp16 matrix cores:
//   Y[M, N] = X[M, K] * W[N, K]^T,  W packed (Q4_K / Q5_K / Q6_K / Q8_0).
//
// A workgroup of 8 or 4 waves owns a 512 or 256 x 128 tile of Y; wave w owns rows
// 64w .. 64w+63 and all 128 columns, and walks K in steps of 64 with 32
// v_mfma_f32_32x32x16_f16 per step and float accumulators.  (128-row tiles: four waves, half
// the rows and instructions a wave; up to 32 rows have a kernel of their own below.)
//
// Activations never touch LDS.  A pre-pass converts them to fp16 once per call
// and stores them in matrix-core operand order: for every block of 32 rows and
// every K chunk of 16 the 1 KB that one operand fragment needs is contiguous,
// lane l's 16 bytes (row l%32, the 8 values of K half l/32) at offset 16*l.
// The main loop loads fragments with one fully coalesced 16-byte load per lane
// straight into the registers the matrix instruction reads, one step ahead.
// The pre-pass also scales every row by a power of two so that its largest
// magnitude lands in [2^14, 2^15); the epilogue multiplies the row's results
// by the inverse, so neither large nor tiny activations leave the fp16 range.
//
// Weights go through LDS: per step every thread turns 32 (eight waves: 16) weights of the
// 128 x 64 slice (two runs of 16: of one row for Q4_K and Q5_K, 16 packed bytes;
// of two rows for Q6_K and Q8_0) into fp16 in registers with packed
// fp16 arithmetic (code bytes become 1024+q by a byte permute, then
// (x-1024)*(d*sc) - dmin*m as one packed fused multiply-add) and writes them
// to a double-buffered stage; the packed bytes are read from HBM once per tile
// column and never exist dequantized in memory.  LDS writes run at about half
// the rate of reads on this chip, which is why only the smaller operand is
// staged.  Stage rows are padded to 144 bytes so that the 16-byte fragment
// reads of 16 lanes hit distinct banks.
//
// A step is written as 16 phases of two matrix instructions each, fenced
// against reordering, so that the dequantization, the LDS traffic and the
// global loads of later steps are issued in the shadow of the matrix
// instructions; weight fragments are read one K chunk ahead, packed bytes are
// loaded three steps before they are decoded (Q6_K: two; where the registers allow
// it a whole block together, a block ahead).  Consecutive workgroups walk M first:
// with 8 XCDs picking workgroups round robin each XCD keeps one or two 256-row
// slices of X in its L2 while the packed weights stream through.
//
// The reference has no kernel of this kind: its small-batch path stops at 16
// rows (neuralfn/csrc/tile_cuda/glimmer_k_mmq.cu:1326-1328) and more rows run
// the float kernel neuralfn/csrc/tile_cuda/kernels.cu:1398-1525.  Weight
// layouts and decode: neuralfn/csrc/native_gpt2/resident_glimmer.cpp:542-616.
#include "common.hpp"
#include "f16_decode.hpp"
#include "gemm_mfma.hpp"

#include <algorithm>

namespace nfn {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kBM = 256;
constexpr int kBN = 128;
constexpr int kBK = 64;
constexpr int kThreads = 256;
constexpr int kMaxProjections = 4;  // of one call
constexpr int kLowRows = 32;    // rows up to which every wave takes all of them
constexpr int kLowShares = 8;   // K shares of theirs at most
constexpr int kMaxShares = 4;   // K shares of a split launch at most that plan() gives (shares_with_room: eight)
constexpr int kLeastCutTiles = 16;  // column tiles and
constexpr int kMostCutRows = 1024;  // rows up to which shares_with_room() looks for more
constexpr int kRowBytes = 144;  // 64 fp16 + 16 bytes of padding
constexpr int kStageBytes = kBN * kRowBytes;
constexpr int kFragmentBytes = 1024;  // 32 rows x 16 K values of fp16 in operand order

struct __attribute__((packed, aligned(2))) Chunk16 {
    std::uint32_t v[4];
};
struct __attribute__((packed, aligned(2))) Chunk8 {
    std::uint32_t v[2];
};
struct __attribute__((packed, aligned(2))) Chunk4 {
    std::uint32_t v;
};

// ---------------------------------------------------------------------------
// activations: fp32 -> row-scaled fp16 in operand order, whole 256-row tiles
// (rows past the end are zeros), in one launch that reads the input once.
// ---------------------------------------------------------------------------

// A lane owns groups of eight
// consecutive columns (one 16-byte piece of the fp16 copy each); rows of up to
// 8,192 columns stay in the lane's registers between the search for the row's
// largest magnitude and the conversion, wider rows are read again (from L2).
// The row's scale is the power of two that brings that magnitude into
// [2^14, 2^15); zero, subnormal, infinite or NaN maxima keep scale 1; padding
// rows get inverse 0 and zeros.
// The workgroups that fill one 32-row block of the operand-order copy (8, 16 or 32: four, two
// rows or one each) are the ones a round-robin placement over the eight XCDs puts on the same
// XCD (workgroup w lands on XCD w % 8), so that the 16-byte pieces they
// scatter into the same cache lines merge in one L2 before going to memory.
// Rows of up to 8,192 columns take four waves each, for the loads in flight of a short prompt
// (6,656 columns, a wave a row: 17 rows 7.6 -> 4.5 us, 333 rows 8.6 -> 6.2, 4,096 rows 52 -> 45),
// wider ones two (four: 1,024 rows of 16,384 23.0 -> 23.8).
// SPLIT waves share a row (each takes a contiguous part of its columns and they exchange
// their maxima through LDS): rows of up to 16,384 columns still fit the registers.
template <int HELD, int SPLIT>  // HELD: 8-column groups a lane keeps in registers; 0 = read the row twice
__global__ __launch_bounds__(256) void prepare_activations_kernel(
    const float* __restrict__ input, std::uint8_t* __restrict__ output,
    float* __restrict__ inverse_scale, std::int64_t rows, std::int64_t width) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const std::int64_t group_index = blockIdx.x;
    const std::int64_t xcd = group_index & 7;
    const std::int64_t turn = group_index >> 3;
    constexpr int kRowsPerGroup = 4 / SPLIT;
    constexpr int kGroupsPerBlock = 32 / kRowsPerGroup;  // workgroups that fill a 32-row block
    const std::int64_t block_index = (turn / kGroupsPerBlock) * 8 + xcd;  // 32-row block of the copy
    const int r = static_cast<int>(turn % kGroupsPerBlock) * kRowsPerGroup + wave / SPLIT;  // row inside it
    const int part = wave % SPLIT;  // which part of the row's columns this wave takes
    const std::int64_t row = block_index * 32 + r;
    const bool live = row < rows;
    const float* source = input + (live ? row : 0) * width;
    const std::int64_t all_groups = width / 8;
    const std::int64_t part_groups = (all_groups + SPLIT - 1) / SPLIT;
    const std::int64_t first_group = part * part_groups;
    const std::int64_t groups = min(all_groups, first_group + part_groups);  // end of this wave's groups

    float4 held_x[HELD > 0 ? HELD : 1], held_y[HELD > 0 ? HELD : 1];
    float largest = 0.0f;
    if constexpr (HELD > 0) {
#pragma unroll
        for (int j = 0; j < HELD; ++j) {
            const std::int64_t g = first_group + lane + 64 * j;
            held_x[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            held_y[j] = held_x[j];
            if (live && g < groups) {
                held_x[j] = *reinterpret_cast<const float4*>(source + g * 8);
                held_y[j] = *reinterpret_cast<const float4*>(source + g * 8 + 4);
            }
        }
#pragma unroll
        for (int j = 0; j < HELD; ++j) {
            const float4 x = held_x[j], y = held_y[j];
            largest = fmaxf(largest, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
            largest = fmaxf(largest, fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
        }
    } else {
        for (std::int64_t g = first_group + lane; live && g < groups; g += 64) {
            const float4 x = *reinterpret_cast<const float4*>(source + g * 8);
            const float4 y = *reinterpret_cast<const float4*>(source + g * 8 + 4);
            largest = fmaxf(largest, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
            largest = fmaxf(largest, fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
        }
    }
    // NaN never wins fmaxf: a row with NaN keeps the largest finite magnitude, as before
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        largest = fmaxf(largest, __shfl_xor(largest, offset));
    }
    if constexpr (SPLIT > 1) {
        __shared__ float maxima[4];
        if (lane == 0) maxima[wave] = largest;
        __syncthreads();
        const int first_wave = wave - part;
#pragma unroll
        for (int k = 0; k < SPLIT; ++k) largest = fmaxf(largest, maxima[first_wave + k]);
    }
    const std::uint32_t exponent = (__float_as_uint(largest) >> 23) & 0xffu;
    const bool usable = exponent >= 16u && exponent <= 254u;
    const float factor = !live ? 0.0f
        : usable ? __uint_as_float((127u + 14u + 127u - exponent) << 23) : 1.0f;
    if (lane == 0 && part == 0) {
        inverse_scale[row] = !live ? 0.0f : usable ? __uint_as_float((exponent - 14u) << 23) : 1.0f;
    }

    std::uint8_t* block = output + block_index * (width / 16) * kFragmentBytes;
    auto store = [&](std::int64_t g, float4 x, float4 y) {
        const f16x2 h0 = {static_cast<_Float16>(x.x * factor), static_cast<_Float16>(x.y * factor)};
        const f16x2 h1 = {static_cast<_Float16>(x.z * factor), static_cast<_Float16>(x.w * factor)};
        const f16x2 h2 = {static_cast<_Float16>(y.x * factor), static_cast<_Float16>(y.y * factor)};
        const f16x2 h3 = {static_cast<_Float16>(y.z * factor), static_cast<_Float16>(y.w * factor)};
        std::uint8_t* target = block + (g >> 1) * kFragmentBytes + ((g & 1) * 32 + r) * 16;
        *reinterpret_cast<u32x4*>(target) = u32x4{bits_of(h0), bits_of(h1), bits_of(h2), bits_of(h3)};
    };
    if constexpr (HELD > 0) {
#pragma unroll
        for (int j = 0; j < HELD; ++j) {
            const std::int64_t g = first_group + lane + 64 * j;
            if (g < groups) store(g, held_x[j], held_y[j]);
        }
    } else {
        for (std::int64_t g = first_group + lane; g < groups; g += 64) {
            float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f), y = x;
            if (live) {
                x = *reinterpret_cast<const float4*>(source + g * 8);
                y = *reinterpret_cast<const float4*>(source + g * 8 + 4);
            }
            store(g, x, y);
        }
    }
}

// ---------------------------------------------------------------------------
// What one thread holds of the packed weights: 32 weights of a K step, in two runs of 16.
//   Q4_K, Q5_K: positions 16*part .. 16*part+15 of both 32-value groups of the step, of one row;
//               two neighbouring lanes share a row.  Q5_K's fifth bits, which serve the whole block,
//               come with the block's header (2,048 rows of gate and up 863 -> 836 us).
//   Q6_K, Q8_0: the step's columns 16*part .. 16*part+15 of two rows, 64 apart; four neighbouring
//               lanes share a row.  A Q6_K slice serves the two steps of a half block, whose
//               codes share their bytes.
// A load instruction looks up every cache line that its lanes touch, and with a row a lane
// (64 lines for 1 KB, more where the pieces straddle lines) those look-ups, not the matrix
// instructions, bounded Q6_K: three such loads a step, 2,048 x 16,384 -> 6,656 in 764 us where
// Q4_K took 467.  Lanes that share a row share its lines: 556 (Q6_K), Q8_0 687 -> 542, Q5_K 507 ->
// 490, Q4_K 461; 17 rows 98 -> 66 us (Q6_K), 86 -> 64 (Q8_0).
// Decoding is cut into pieces of
// at most eight vector instructions so that each fits behind one matrix
// instruction: prepare_bits() and prepare_scales() derive the fp16 scale
// constants; group_a<I>() / group_b<I>() decode code word I into positions
// 4I..4I+3 of the first / second run (two packed fp16 pairs).
// ---------------------------------------------------------------------------
struct WeightRows {
    const std::uint8_t *first, *second;  // (second: Q6_K and Q8_0)
};
template <std::uint32_t ENC>
struct PackedSlice;
// what all K steps of one 256-value block share; loaded once per block
template <std::uint32_t ENC>
struct BlockHeader;

template <>
struct BlockHeader<kEncQ4K> {
    u32x4 words;  // d, dmin and the twelve scale bytes
    __device__ __forceinline__ void load(const std::uint8_t* row, int block, int part) {
        words = *reinterpret_cast<const u32x4*>(row + block * 144);
    }
};

template <>
struct PackedSlice<kEncQ4K> {
    u32x4 codes;
    KBlockScales c;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        codes = *reinterpret_cast<const u32x4*>(rows.first + block * 144 + 16 + pair * 32 + part * 16);
    }
    __device__ __forceinline__ void prepare_bits(const BlockHeader<kEncQ4K>& header, int pair, int) {
        c.bits(header.words, pair);
    }
    __device__ __forceinline__ void prepare_scales(const BlockHeader<kEncQ4K>& header) {
        c.scales(header.words);
    }
    template <int I>
    __device__ __forceinline__ void group_a(std::uint32_t (&out)[2]) const {
        scale_bytes(codes[I] & 0x0f0f0f0fu, splat(-1024.0f), c.scale_a, c.shift_a, out[0], out[1]);
    }
    template <int I>
    __device__ __forceinline__ void group_b(std::uint32_t (&out)[2]) const {
        scale_bytes((codes[I] >> 4) & 0x0f0f0f0fu, splat(-1024.0f), c.scale_b, c.shift_b, out[0],
                    out[1]);
    }
};

template <>
struct BlockHeader<kEncQ5K> {
    u32x4 words;  // d, dmin and the twelve scale bytes
    u32x4 high;   // the fifth bits of the lane's positions, two for each of the block's steps
    __device__ __forceinline__ void load(const std::uint8_t* row, int block, int part) {
        words = *reinterpret_cast<const u32x4*>(row + block * 176);
        high = *reinterpret_cast<const u32x4*>(row + block * 176 + 16 + part * 16);
    }
};

template <>
struct PackedSlice<kEncQ5K> {
    u32x4 codes;
    KBlockScales c;
    u32x4 high;
    int high_shift;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        codes = *reinterpret_cast<const u32x4*>(rows.first + block * 176 + 48 + pair * 32 + part * 16);
    }
    __device__ __forceinline__ void prepare_bits(const BlockHeader<kEncQ5K>& header, int pair, int) {
        c.bits(header.words, pair);
        high = header.high;
        high_shift = 2 * pair;  // bit 2*pair: first group, bit 2*pair+1: second
    }
    __device__ __forceinline__ void prepare_scales(const BlockHeader<kEncQ5K>& header) {
        c.scales(header.words);
    }
    template <int I>
    __device__ __forceinline__ void group_a(std::uint32_t (&out)[2]) const {
        const std::uint32_t bits = high[I] >> high_shift;
        const std::uint32_t q = (codes[I] & 0x0f0f0f0fu) | ((bits & 0x01010101u) << 4);
        scale_bytes(q, splat(-1024.0f), c.scale_a, c.shift_a, out[0], out[1]);
    }
    template <int I>
    __device__ __forceinline__ void group_b(std::uint32_t (&out)[2]) const {
        const std::uint32_t bits = high[I] >> high_shift;
        const std::uint32_t q = ((codes[I] >> 4) & 0x0f0f0f0fu) | ((bits & 0x02020202u) << 3);
        scale_bytes(q, splat(-1024.0f), c.scale_b, c.shift_b, out[0], out[1]);
    }
};

template <>
struct BlockHeader<kEncQ6K> {  // the scales come with the slice
    __device__ __forceinline__ void load(const std::uint8_t*, int, int) {}
};

template <>
struct PackedSlice<kEncQ6K> {
    // a K step of 64 is two quarters (32 values each) of one half of the block: quarters (0,1) or
    // (2,3), the low or the high nibbles of the half's 64 bytes; `pair` = 2 * half + (quarters 2,3 ? 1 : 0)
    u32x4 low_a, high_a, low_b, high_b;
    std::uint32_t scales_a[2], scales_b[2], d_a, d_b;  // the half's eight sub-scales; [0]: quarters 0,1
    f16x2 scale_a, scale_b;
    int upper, high_shift, sa, sb;
    __device__ __forceinline__ static void load_row(const std::uint8_t* p, int half, int part, u32x4& low, u32x4& high,
                                                    std::uint32_t (&scales)[2], std::uint32_t& d) {
        const Chunk16 l = *reinterpret_cast<const Chunk16*>(p + half * 64 + part * 16);
        const Chunk16 h = *reinterpret_cast<const Chunk16*>(p + 128 + half * 32 + (part & 1) * 16);
        const Chunk8 sc = *reinterpret_cast<const Chunk8*>(p + 192 + half * 8);
        low = u32x4{l.v[0], l.v[1], l.v[2], l.v[3]};
        high = u32x4{h.v[0], h.v[1], h.v[2], h.v[3]};
        scales[0] = sc.v[0];
        scales[1] = sc.v[1];
        d = *reinterpret_cast<const std::uint16_t*>(p + 208);
    }
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        load_row(rows.first + block * 210, pair >> 1, part, low_a, high_a, scales_a, d_a);
        load_row(rows.second + block * 210, pair >> 1, part, low_b, high_b, scales_b, d_b);
    }
    __device__ __forceinline__ void prepare_bits(const BlockHeader<kEncQ6K>&, int pair, int part) {
        // sub-scale of the run: 2*quarter + position/16 = 4 * (pair & 1) + part of the half's eight
        sa = static_cast<std::int8_t>((scales_a[pair & 1] >> (8 * part)) & 0xffu);
        sb = static_cast<std::int8_t>((scales_b[pair & 1] >> (8 * part)) & 0xffu);
        upper = (pair & 1) * 4;                   // quarters 2,3: high nibbles,
        high_shift = upper + 2 * (part >> 1);     // bit pairs 2 and 3 of the high bits
    }
    __device__ __forceinline__ void prepare_scales(const BlockHeader<kEncQ6K>&) {
        scale_a = splat(half_bits_to_float(d_a) * static_cast<float>(sa));
        scale_b = splat(half_bits_to_float(d_b) * static_cast<float>(sb));
    }
    // bias: 1024 + the format's offset of 32
    template <int I>
    __device__ __forceinline__ void group_a(std::uint32_t (&out)[2]) const {
        const std::uint32_t q = ((low_a[I] >> upper) & 0x0f0f0f0fu) | (((high_a[I] >> high_shift) & 0x03030303u) << 4);
        scale_bytes(q, splat(-1056.0f), scale_a, splat(0.0f), out[0], out[1]);
    }
    template <int I>
    __device__ __forceinline__ void group_b(std::uint32_t (&out)[2]) const {
        const std::uint32_t q = ((low_b[I] >> upper) & 0x0f0f0f0fu) | (((high_b[I] >> high_shift) & 0x03030303u) << 4);
        scale_bytes(q, splat(-1056.0f), scale_b, splat(0.0f), out[0], out[1]);
    }
};

template <>
struct BlockHeader<kEncQ8_0> {  // the scales sit next to the codes
    __device__ __forceinline__ void load(const std::uint8_t*, int, int) {}
};

template <>
struct PackedSlice<kEncQ8_0> {
    // a K step of 64 is two 34-byte blocks; `pair` counts K steps inside 256 values
    u32x4 codes_a, codes_b;
    std::uint32_t behind_a, behind_b;
    f16x2 scale_a, scale_b;
    // The two are seventeen words: the first one's codes start in the middle of word 0, the second one's
    // scale is the upper half of word 8.  Four lanes take words 0..3, 4..7, 9..12 and 13..16, and word 4
    // or 8 beside them: from where the first one's codes begin, two bytes past a word, sixteen bytes take the
    // address unit four times as long.  Loaded as they lie -> from words, us: 17 rows of 6,656 into Q, K, V and gate 39.7 ->
    // 33.7, 32 of gate and up 4,096 -> 11,264 64.5 -> 57.8, 100 of Q, K, V and gate 47.4 -> 42.7, 333 of down 11,264 ->
    // 5,632 103 -> 93, 1,400 of it 282 -> 254.  (Q6_K's pieces, of which half begin past a word, the same way: three to
    // eight more instructions a piece for as many loads, 17 to 2,048 rows 0 to 5 % slower.)
    __device__ __forceinline__ static void load_row(const std::uint8_t* p, int part, u32x4& codes, std::uint32_t& behind) {
        const Chunk16 c = *reinterpret_cast<const Chunk16*>(p + part * 16 + (part >> 1) * 4);
        codes = u32x4{c.v[0], c.v[1], c.v[2], c.v[3]};
        behind = reinterpret_cast<const Chunk4*>(p + (part == 0 ? 16 : 32))->v;
    }
    __device__ __forceinline__ static void arrange_row(int part, u32x4& codes, std::uint32_t behind, f16x2& scale) {
        // (of the first lane, for the first two)
        const std::uint32_t first = __builtin_amdgcn_update_dpp(0, static_cast<int>(codes[0]), 0xe0, 0xf, 0xf, true);
        scale = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(behind, first, part < 2 ? 0x01000100u : 0x07060706u));
        const std::uint32_t shift = part < 2 ? 2 : 0;
#pragma unroll
        for (int word = 0; word < 4; ++word) {
            codes[word] = __builtin_amdgcn_alignbyte(word < 3 ? codes[word + 1] : behind, codes[word], shift);
        }
    }
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        const int offset = (block * 4 + pair) * 68;
        load_row(rows.first + offset, part, codes_a, behind_a);
        load_row(rows.second + offset, part, codes_b, behind_b);
    }
    __device__ __forceinline__ void prepare_bits(const BlockHeader<kEncQ8_0>&, int, int part) {
        arrange_row(part, codes_a, behind_a, scale_a);
        arrange_row(part, codes_b, behind_b, scale_b);
    }
    __device__ __forceinline__ void prepare_scales(const BlockHeader<kEncQ8_0>&) {}
    // flipping the sign bit turns the int8 code q into the byte q+128: bias 1024+128
    template <int I>
    __device__ __forceinline__ void group_a(std::uint32_t (&out)[2]) const {
        scale_bytes(codes_a[I] ^ 0x80808080u, splat(-1152.0f), scale_a, splat(0.0f), out[0], out[1]);
    }
    template <int I>
    __device__ __forceinline__ void group_b(std::uint32_t (&out)[2]) const {
        scale_bytes(codes_b[I] ^ 0x80808080u, splat(-1152.0f), scale_b, splat(0.0f), out[0], out[1]);
    }
};

// The same with every lane's codes loaded from where they begin, two bytes past a word for half the lanes, for
// the tiles of 256 rows, which have no register left for the words' way (six in scratch: 200 rows of gate and up
// 4,096 -> 11,264 80 -> 92 us).
struct CodesAsTheyLie {
    // a K step of 64 is two 34-byte blocks; `pair` counts K steps inside 256 values
    u32x4 codes_a, codes_b;
    std::uint32_t d_a, d_b;
    f16x2 scale_a, scale_b;
    __device__ __forceinline__ static void load_row(const std::uint8_t* p, int part, u32x4& codes, std::uint32_t& d) {
        const Chunk16 c = *reinterpret_cast<const Chunk16*>(p + 2 + (part & 1) * 16);
        codes = u32x4{c.v[0], c.v[1], c.v[2], c.v[3]};
        d = *reinterpret_cast<const std::uint16_t*>(p);
    }
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        const int offset = (block * 8 + pair * 2 + (part >> 1)) * 34;
        load_row(rows.first + offset, part, codes_a, d_a);
        load_row(rows.second + offset, part, codes_b, d_b);
    }
    __device__ __forceinline__ void prepare_bits(const BlockHeader<kEncQ8_0>&, int, int) {}
    __device__ __forceinline__ void prepare_scales(const BlockHeader<kEncQ8_0>&) {
        const _Float16 a = __builtin_bit_cast(_Float16, static_cast<std::uint16_t>(d_a));
        const _Float16 b = __builtin_bit_cast(_Float16, static_cast<std::uint16_t>(d_b));
        scale_a = f16x2{a, a};
        scale_b = f16x2{b, b};
    }
    // flipping the sign bit turns the int8 code q into the byte q+128: bias 1024+128
    template <int I>
    __device__ __forceinline__ void group_a(std::uint32_t (&out)[2]) const {
        scale_bytes(codes_a[I] ^ 0x80808080u, splat(-1152.0f), scale_a, splat(0.0f), out[0], out[1]);
    }
    template <int I>
    __device__ __forceinline__ void group_b(std::uint32_t (&out)[2]) const {
        scale_bytes(codes_b[I] ^ 0x80808080u, splat(-1152.0f), scale_b, splat(0.0f), out[0], out[1]);
    }
};

// The same with eight waves a workgroup: 16 weights of a K step a thread, four lanes a row.
//   Q4_K, Q5_K: positions 8*part .. 8*part+7 of both 32-value groups of the step
//   Q6_K, Q8_0: the step's columns 16*part .. 16*part+15
// decode<I>() gives four of them, I = 0, 1 the first 16 bytes that the thread writes.
template <std::uint32_t ENC>
struct PackedRun;
template <std::uint32_t ENC>
struct RunHeader;

template <>
struct RunHeader<kEncQ4K> : BlockHeader<kEncQ4K> {};
template <>
struct RunHeader<kEncQ6K> : BlockHeader<kEncQ6K> {};
template <>
struct RunHeader<kEncQ8_0> : BlockHeader<kEncQ8_0> {};
template <>
struct RunHeader<kEncQ5K> {
    u32x4 words;
    std::uint32_t high[2];
    __device__ __forceinline__ void load(const std::uint8_t* row, int block, int part) {
        words = *reinterpret_cast<const u32x4*>(row + block * 176);
        const uint2 bits = *reinterpret_cast<const uint2*>(row + block * 176 + 16 + part * 8);
        high[0] = bits.x;
        high[1] = bits.y;
    }
};

template <>
struct PackedRun<kEncQ4K> {
    std::uint32_t codes[2];
    KBlockScales c;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        const uint2 both = *reinterpret_cast<const uint2*>(rows.first + block * 144 + 16 + pair * 32 + part * 8);
        codes[0] = both.x;
        codes[1] = both.y;
    }
    __device__ __forceinline__ void prepare_bits(const RunHeader<kEncQ4K>& header, int pair, int) {
        c.bits(header.words, pair);
    }
    __device__ __forceinline__ void prepare_scales(const RunHeader<kEncQ4K>& header) { c.scales(header.words); }
    template <int I>
    __device__ __forceinline__ void decode(std::uint32_t (&out)[2]) const {
        if constexpr (I < 2) {
            scale_bytes(codes[I] & 0x0f0f0f0fu, splat(-1024.0f), c.scale_a, c.shift_a, out[0], out[1]);
        } else {
            scale_bytes((codes[I - 2] >> 4) & 0x0f0f0f0fu, splat(-1024.0f), c.scale_b, c.shift_b, out[0], out[1]);
        }
    }
};

template <>
struct PackedRun<kEncQ5K> {
    std::uint32_t codes[2], high[2];
    KBlockScales c;
    int high_shift;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        const uint2 both = *reinterpret_cast<const uint2*>(rows.first + block * 176 + 48 + pair * 32 + part * 8);
        codes[0] = both.x;
        codes[1] = both.y;
    }
    __device__ __forceinline__ void prepare_bits(const RunHeader<kEncQ5K>& header, int pair, int) {
        c.bits(header.words, pair);
        high[0] = header.high[0];
        high[1] = header.high[1];
        high_shift = 2 * pair;
    }
    __device__ __forceinline__ void prepare_scales(const RunHeader<kEncQ5K>& header) { c.scales(header.words); }
    template <int I>
    __device__ __forceinline__ void decode(std::uint32_t (&out)[2]) const {
        const std::uint32_t bits = high[I & 1] >> high_shift;
        if constexpr (I < 2) {
            const std::uint32_t q = (codes[I] & 0x0f0f0f0fu) | ((bits & 0x01010101u) << 4);
            scale_bytes(q, splat(-1024.0f), c.scale_a, c.shift_a, out[0], out[1]);
        } else {
            const std::uint32_t q = ((codes[I - 2] >> 4) & 0x0f0f0f0fu) | ((bits & 0x02020202u) << 3);
            scale_bytes(q, splat(-1024.0f), c.scale_b, c.shift_b, out[0], out[1]);
        }
    }
};

template <>
struct PackedRun<kEncQ6K> {
    u32x4 low, high;
    std::uint32_t scales[2], d;
    f16x2 scale;
    int upper, high_shift, sub_scale;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        PackedSlice<kEncQ6K>::load_row(rows.first + block * 210, pair >> 1, part, low, high, scales, d);
    }
    __device__ __forceinline__ void prepare_bits(const RunHeader<kEncQ6K>&, int pair, int part) {
        sub_scale = static_cast<std::int8_t>((scales[pair & 1] >> (8 * part)) & 0xffu);
        upper = (pair & 1) * 4;
        high_shift = upper + 2 * (part >> 1);
    }
    __device__ __forceinline__ void prepare_scales(const RunHeader<kEncQ6K>&) {
        scale = splat(half_bits_to_float(d) * static_cast<float>(sub_scale));
    }
    template <int I>
    __device__ __forceinline__ void decode(std::uint32_t (&out)[2]) const {
        const std::uint32_t q = ((low[I] >> upper) & 0x0f0f0f0fu) | (((high[I] >> high_shift) & 0x03030303u) << 4);
        scale_bytes(q, splat(-1056.0f), scale, splat(0.0f), out[0], out[1]);
    }
};

template <>
struct PackedRun<kEncQ8_0> {
    u32x4 codes;
    std::uint32_t behind;
    f16x2 scale;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int pair, int part) {
        PackedSlice<kEncQ8_0>::load_row(rows.first + (block * 4 + pair) * 68, part, codes, behind);
    }
    __device__ __forceinline__ void prepare_bits(const RunHeader<kEncQ8_0>&, int, int part) {
        PackedSlice<kEncQ8_0>::arrange_row(part, codes, behind, scale);
    }
    __device__ __forceinline__ void prepare_scales(const RunHeader<kEncQ8_0>&) {}
    template <int I>
    __device__ __forceinline__ void decode(std::uint32_t (&out)[2]) const {
        scale_bytes(codes[I] ^ 0x80808080u, splat(-1152.0f), scale, splat(0.0f), out[0], out[1]);
    }
};

// what a thread holds and decodes with WAVES waves a workgroup and RB 32-row blocks a wave
template <std::uint32_t ENC, int RB, int WAVES>
struct Held {
    using Slice = PackedSlice<ENC>;
    using Header = BlockHeader<ENC>;
};
template <std::uint32_t ENC, int RB>
struct Held<ENC, RB, 8> {
    using Slice = PackedRun<ENC>;
    using Header = RunHeader<ENC>;
};
template <>
struct Held<kEncQ8_0, 2, 4> {
    using Slice = CodesAsTheyLie;
    using Header = BlockHeader<kEncQ8_0>;
};
template <int I>
__device__ __forceinline__ void decode(const CodesAsTheyLie& slice, std::uint32_t (&out)[2]) {
    if constexpr (I < 4) {
        slice.template group_a<I>(out);
    } else {
        slice.template group_b<I - 4>(out);
    }
}
template <int I, std::uint32_t ENC>
__device__ __forceinline__ void decode(const PackedSlice<ENC>& slice, std::uint32_t (&out)[2]) {
    if constexpr (I < 4) {
        slice.template group_a<I>(out);
    } else {
        slice.template group_b<I - 4>(out);
    }
}
template <int I, std::uint32_t ENC>
__device__ __forceinline__ void decode(const PackedRun<ENC>& run, std::uint32_t (&out)[2]) {
    run.template decode<I>(out);
}

// lanes that share a weight row
template <std::uint32_t ENC>
constexpr int kParts = ENC == kEncQ4K || ENC == kEncQ5K ? 2 : 4;
// a slice serves two steps
template <std::uint32_t ENC>
constexpr bool kHalfBlocks = ENC == kEncQ6K;
// from the first run of 16 to the second, in the stage
template <std::uint32_t ENC>
constexpr int kSecondRun = kParts<ENC> == 2 ? 64 : 64 * kRowBytes;
// eight waves: from a thread's first 16 bytes to the others
template <std::uint32_t ENC>
constexpr int kRunSecond = ENC == kEncQ4K || ENC == kEncQ5K ? 64 : 16;

// What a lane wrote to LDS is seen by the wave's other lanes, and no access moves across (no instruction of its own).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The activation fragments of one K step for one wave: row blocks 0 and 1,
// K chunks 0..3, in named registers (an array here ends up in scratch memory).
struct ActivationSlice {
    f16x8 r0k0, r0k1, r0k2, r0k3, r1k0, r1k1, r1k2, r1k3;
};

// the four weight fragments (column blocks) of one K chunk of 16
struct WeightFragments {
    f16x8 c0, c1, c2, c3;
};

#define NFN_FENCE() __builtin_amdgcn_sched_barrier(0)
#define NFN_MFMA(A, B, C) C = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B, C, 0, 0, 0)
#define NFN_READ_WEIGHTS(base, column_block, chunk) \
    (*reinterpret_cast<const f16x8*>((base) + (column_block) * 32 * kRowBytes + (chunk) * 32))
#define NFN_LOAD_ACTIVATIONS(base, row_block, chunk) \
    (*reinterpret_cast<const f16x8*>((base) + (row_block) * row_block_bytes + (chunk) * kFragmentBytes))
#define NFN_WRITE16(target, x, y, z, w) *reinterpret_cast<u32x4*>(target) = u32x4{x, y, z, w}
#define NFN_WRITE8(target, pair) *reinterpret_cast<uint2*>(target) = make_uint2((pair)[0], (pair)[1])

// One matrix instruction with the statements issued in its shadow.  A wave
// issues in order and stalls at a matrix instruction while the previous one
// occupies the pipe (32 cycles), so only what stands between two of them
// overlaps: about seven vector instructions fit.
#define NFN_SLOT(A, W, C, ...) \
    __VA_ARGS__;               \
    NFN_MFMA(A, W, C);         \
    NFN_FENCE();

// One K step for one wave: 32 slots.  A row block 0 fragment is last used in
// the fourth slot of its chunk, a row block 1 fragment in the eighth; each is
// refilled with the fragment of the next step right after.
//   a_now:    activation fragments of this step
//   current:  weight fragments of K chunk 0 of this step (read at the end of
//             the previous one); on return they hold chunk 0 of the next step
//   b_next:   packed weights of the next step: dequantized into the other
//             stage with the scales in `header`, then refilled with the packed
//             bytes of `fetch_step`
template <std::uint32_t ENC, int RB, int WAVES, bool REFILL>
__device__ __forceinline__ void k_step(
    v16f (&acc)[RB][4], ActivationSlice& a_now, WeightFragments& current,
    const std::uint8_t* b_read, const std::uint8_t* b_read_next, std::uint8_t* b_write,
    typename Held<ENC, RB, WAVES>::Slice& b_next, const typename Held<ENC, RB, WAVES>::Header& header, int decode_pair,
    int b_part, const std::uint8_t* a_fetch, std::int64_t row_block_bytes, const WeightRows& b_global,
    int fetch_step) {
    WeightFragments ahead;
    std::uint32_t w[2], v[2];

    if constexpr (RB == 1) {
        // One row block per wave: 16 slots carry the same side work.
        NFN_SLOT(a_now.r0k0, current.c0, acc[0][0], b_next.prepare_bits(header, decode_pair, b_part))
        NFN_SLOT(a_now.r0k0, current.c1, acc[0][1], b_next.prepare_scales(header);
                 ahead.c0 = NFN_READ_WEIGHTS(b_read, 0, 1))
        NFN_SLOT(a_now.r0k0, current.c2, acc[0][2], b_next.template group_a<0>(w);
                 ahead.c1 = NFN_READ_WEIGHTS(b_read, 1, 1))
        NFN_SLOT(a_now.r0k0, current.c3, acc[0][3], b_next.template group_a<1>(v);
                 NFN_WRITE16(b_write, w[0], w[1], v[0], v[1]); ahead.c2 = NFN_READ_WEIGHTS(b_read, 2, 1);
                 ahead.c3 = NFN_READ_WEIGHTS(b_read, 3, 1))
        NFN_SLOT(a_now.r0k1, ahead.c0, acc[0][0], b_next.template group_a<2>(w);
                 current.c0 = NFN_READ_WEIGHTS(b_read, 0, 2);
                 a_now.r0k0 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 0))
        NFN_SLOT(a_now.r0k1, ahead.c1, acc[0][1], b_next.template group_a<3>(v);
                 NFN_WRITE16(b_write + 16, w[0], w[1], v[0], v[1]); current.c1 = NFN_READ_WEIGHTS(b_read, 1, 2))
        NFN_SLOT(a_now.r0k1, ahead.c2, acc[0][2], b_next.template group_b<0>(w);
                 current.c2 = NFN_READ_WEIGHTS(b_read, 2, 2))
        NFN_SLOT(a_now.r0k1, ahead.c3, acc[0][3], b_next.template group_b<1>(v);
                 NFN_WRITE16(b_write + kSecondRun<ENC>, w[0], w[1], v[0], v[1]); current.c3 = NFN_READ_WEIGHTS(b_read, 3, 2))
        NFN_SLOT(a_now.r0k2, current.c0, acc[0][0], b_next.template group_b<2>(w);
                 ahead.c0 = NFN_READ_WEIGHTS(b_read, 0, 3);
                 a_now.r0k1 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 1))
        NFN_SLOT(a_now.r0k2, current.c1, acc[0][1], b_next.template group_b<3>(v);
                 NFN_WRITE16(b_write + kSecondRun<ENC> + 16, w[0], w[1], v[0], v[1]); ahead.c1 = NFN_READ_WEIGHTS(b_read, 1, 3))
        NFN_SLOT(a_now.r0k2, current.c2, acc[0][2], ahead.c2 = NFN_READ_WEIGHTS(b_read, 2, 3))
        NFN_SLOT(a_now.r0k2, current.c3, acc[0][3], ahead.c3 = NFN_READ_WEIGHTS(b_read, 3, 3))
        __syncthreads();
        NFN_SLOT(a_now.r0k3, ahead.c0, acc[0][0], current.c0 = NFN_READ_WEIGHTS(b_read_next, 0, 0);
                 a_now.r0k2 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 2))
        NFN_SLOT(a_now.r0k3, ahead.c1, acc[0][1], current.c1 = NFN_READ_WEIGHTS(b_read_next, 1, 0))
        NFN_SLOT(a_now.r0k3, ahead.c2, acc[0][2], current.c2 = NFN_READ_WEIGHTS(b_read_next, 2, 0))
        NFN_SLOT(a_now.r0k3, ahead.c3, acc[0][3], current.c3 = NFN_READ_WEIGHTS(b_read_next, 3, 0))
        a_now.r0k3 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 3);
        NFN_FENCE();
        if constexpr (REFILL) b_next.load(b_global, fetch_step >> 2, fetch_step & 3, b_part);
        NFN_FENCE();
        return;
    } else {
    // K chunk 0: read chunk 1, decode; every decoded run of eight values is written to the other
    // stage at once (16 bytes), which keeps few registers live
    constexpr int kSecond = WAVES == 8 ? kRunSecond<ENC> : 16;  // of the second 16 bytes
    NFN_SLOT(a_now.r0k0, current.c0, acc[0][0], b_next.prepare_bits(header, decode_pair, b_part))
    NFN_SLOT(a_now.r0k0, current.c1, acc[0][1], b_next.prepare_scales(header);
             ahead.c0 = NFN_READ_WEIGHTS(b_read, 0, 1))
    NFN_SLOT(a_now.r0k0, current.c2, acc[0][2], decode<0>(b_next, w);
             ahead.c1 = NFN_READ_WEIGHTS(b_read, 1, 1))
    NFN_SLOT(a_now.r0k0, current.c3, acc[0][3], decode<1>(b_next, v);
             NFN_WRITE16(b_write, w[0], w[1], v[0], v[1]))
    NFN_SLOT(a_now.r1k0, current.c0, acc[1][0], decode<2>(b_next, w);
             ahead.c2 = NFN_READ_WEIGHTS(b_read, 2, 1);
             a_now.r0k0 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 0))
    NFN_SLOT(a_now.r1k0, current.c1, acc[1][1], decode<3>(b_next, v);
             NFN_WRITE16(b_write + kSecond, w[0], w[1], v[0], v[1]))
    NFN_SLOT(a_now.r1k0, current.c2, acc[1][2], if constexpr (WAVES == 4) decode<4>(b_next, w);
             ahead.c3 = NFN_READ_WEIGHTS(b_read, 3, 1))
    NFN_SLOT(a_now.r1k0, current.c3, acc[1][3], if constexpr (WAVES == 4) {
                 decode<5>(b_next, v);
                 NFN_WRITE16(b_write + kSecondRun<ENC>, w[0], w[1], v[0], v[1]);
             })
    // K chunk 1: read chunk 2, finish decoding
    NFN_SLOT(a_now.r0k1, ahead.c0, acc[0][0], if constexpr (WAVES == 4) decode<6>(b_next, w);
             current.c0 = NFN_READ_WEIGHTS(b_read, 0, 2);
             a_now.r1k0 = NFN_LOAD_ACTIVATIONS(a_fetch, 1, 0))
    NFN_SLOT(a_now.r0k1, ahead.c1, acc[0][1], if constexpr (WAVES == 4) {
                 decode<7>(b_next, v);
                 NFN_WRITE16(b_write + kSecondRun<ENC> + 16, w[0], w[1], v[0], v[1]);
             })
    NFN_SLOT(a_now.r0k1, ahead.c2, acc[0][2], current.c1 = NFN_READ_WEIGHTS(b_read, 1, 2))
    NFN_SLOT(a_now.r0k1, ahead.c3, acc[0][3], (void)0)
    NFN_SLOT(a_now.r1k1, ahead.c0, acc[1][0], current.c2 = NFN_READ_WEIGHTS(b_read, 2, 2);
             a_now.r0k1 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 1))
    NFN_SLOT(a_now.r1k1, ahead.c1, acc[1][1], (void)0)
    NFN_SLOT(a_now.r1k1, ahead.c2, acc[1][2], current.c3 = NFN_READ_WEIGHTS(b_read, 3, 2))
    NFN_SLOT(a_now.r1k1, ahead.c3, acc[1][3], (void)0)
    // K chunk 2: read chunk 3
    NFN_SLOT(a_now.r0k2, current.c0, acc[0][0], ahead.c0 = NFN_READ_WEIGHTS(b_read, 0, 3);
             a_now.r1k1 = NFN_LOAD_ACTIVATIONS(a_fetch, 1, 1))
    NFN_SLOT(a_now.r0k2, current.c1, acc[0][1], (void)0)
    NFN_SLOT(a_now.r0k2, current.c2, acc[0][2], ahead.c1 = NFN_READ_WEIGHTS(b_read, 1, 3))
    NFN_SLOT(a_now.r0k2, current.c3, acc[0][3], (void)0)
    NFN_SLOT(a_now.r1k2, current.c0, acc[1][0], ahead.c2 = NFN_READ_WEIGHTS(b_read, 2, 3);
             a_now.r0k2 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 2))
    NFN_SLOT(a_now.r1k2, current.c1, acc[1][1], (void)0)
    NFN_SLOT(a_now.r1k2, current.c2, acc[1][2], ahead.c3 = NFN_READ_WEIGHTS(b_read, 3, 3))
    NFN_SLOT(a_now.r1k2, current.c3, acc[1][3], (void)0)

    // every wave has written its part of the other stage and read the last
    // fragments of this one: after the barrier the other stage may be read and
    // this one overwritten
    __syncthreads();

    // K chunk 3: read chunk 0 of the next step; the packed bytes are loaded
    // last: the waits of the step that decodes them count on this order
    NFN_SLOT(a_now.r0k3, ahead.c0, acc[0][0], current.c0 = NFN_READ_WEIGHTS(b_read_next, 0, 0);
             a_now.r1k2 = NFN_LOAD_ACTIVATIONS(a_fetch, 1, 2))
    NFN_SLOT(a_now.r0k3, ahead.c1, acc[0][1], (void)0)
    NFN_SLOT(a_now.r0k3, ahead.c2, acc[0][2], current.c1 = NFN_READ_WEIGHTS(b_read_next, 1, 0))
    NFN_SLOT(a_now.r0k3, ahead.c3, acc[0][3], (void)0)
    NFN_SLOT(a_now.r1k3, ahead.c0, acc[1][0], current.c2 = NFN_READ_WEIGHTS(b_read_next, 2, 0);
             a_now.r0k3 = NFN_LOAD_ACTIVATIONS(a_fetch, 0, 3))
    NFN_SLOT(a_now.r1k3, ahead.c1, acc[1][1], (void)0)
    NFN_SLOT(a_now.r1k3, ahead.c2, acc[1][2], current.c3 = NFN_READ_WEIGHTS(b_read_next, 3, 0))
    NFN_SLOT(a_now.r1k3, ahead.c3, acc[1][3], (void)0)
    a_now.r1k3 = NFN_LOAD_ACTIVATIONS(a_fetch, 1, 3);
    NFN_FENCE();
    if constexpr (REFILL) b_next.load(b_global, fetch_step >> 2, fetch_step & 3, b_part);
    NFN_FENCE();
    }
}

// bytes of 256 packed values
template <std::uint32_t ENC>
constexpr int kBlockBytes = ENC == kEncQ4K ? 144 : ENC == kEncQ5K ? 176 : ENC == kEncQ6K ? 210 : 272;

// Workgroups per compute unit (= waves per SIMD): as many as the registers
// allow; while one wave waits at the barrier or for LDS, another keeps the
// matrix pipe busy.  With 256-row tiles the Q6_K decode holds too much live
// state for two (of 22 registers in scratch memory with two).
template <std::uint32_t ENC, int RB, int WAVES>
constexpr int kWavesPerSimd = WAVES == 8 ? 2 : ENC == kEncQ6K ? RB == 1 ? 2 : 1 : RB == 1 && ENC == kEncQ4K ? 3 : 2;

// The packed bytes of a block of a lane's rows.
template <std::uint32_t ENC, int RB, int WAVES>
struct Slices {
    typename Held<ENC, RB, WAVES>::Slice b0, b1, b2, b3;  // of its four steps; Q6_K: b0 the first half, b1 the second
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int part) {
        b0.load(rows, block, 0, part);
        b1.load(rows, block, kHalfBlocks<ENC> ? 2 : 1, part);
        if constexpr (!kHalfBlocks<ENC>) {
            b2.load(rows, block, 2, part);
            b3.load(rows, block, 3, part);
        }
    }
};
// Where the registers allow a second set, a block's packed bytes are requested together, one block
// ahead: the steps' pieces of a row lie in the same cache lines, which do not stay in the vector
// cache from one step to the next (4,096 rows of gate and up, Q4_K: 1,577 -> 1,533 us; 100 rows of
// Q5_K 92 -> 88).  Q6_K, whose slices serve two steps, gains nothing by it, and Q8_0, whose block of a
// row is more than two lines, loses: 100 rows of O 55 -> 69 us.
template <std::uint32_t ENC, int RB, int WAVES>
constexpr bool kWholeBlocks = (ENC == kEncQ4K && RB == 2) || (ENC == kEncQ5K && RB == 1);

// The projections of one launch: one encoding, one input.
struct GemmGroup {
    const std::uint8_t* weights[kMaxProjections];
    float* output[kMaxProjections];    // share 0
    float* partials[kMaxProjections];  // the other shares, one copy of the output each
    std::int64_t output_dim[kMaxProjections];
    std::int64_t row_stride;
    int shares[kMaxProjections];
};

// ... as the kernels take them.  Workgroup numbers run through the projections, inside each through its K
// shares, inside each through its tiles.  Where the projections behind the first begin is among the leading
// arguments, which lie in registers when a wave starts, so that what a workgroup needs to know of its own is
// one request to the argument block.  Picked from arrays by branches it was eight, one behind the other, and the
// first bytes of the weights were asked for 1.2 us after a workgroup's start instead of 0.8.
struct GemmSlot {
    const std::uint8_t* weights;
    float* output;
    float* partials;
    std::int64_t output_dim;
    int first;  // workgroup number
    int tiles;
    int shares;
    std::uint32_t by_tiles, by_shares;  // what `divided` divides by the two with
    int pad[3];
};
static_assert(sizeof(GemmSlot) == 64, "a slot begins at a multiple of 64 bytes");
struct GemmSlots {
    GemmSlot slot[kMaxProjections];
};
static_assert(kMaxProjections == 4, "three starts among the kernels' leading arguments");

// n / d for n < 2^31 by the host's inverse of d: the product's upper half is the quotient or one less, because
// the inverse falls short of 2^32 / d by at most one.
inline std::uint32_t inverse_of(int d) { return 0xffffffffu / static_cast<std::uint32_t>(d); }
__device__ __forceinline__ int divided(int n, int d, std::uint32_t inverse) {
    const int quotient = static_cast<int>(__umulhi(static_cast<std::uint32_t>(n), inverse));
    return n - quotient * d >= d ? quotient + 1 : quotient;
}

// this workgroup's projection, share and tile, and the blocks of 256 columns that its share has
struct GroupPlace {
    const std::uint8_t* weights;
    float *output, *partials;
    std::int64_t output_dim;
    int share, tile, first_block, end_block;
};
// (a macro: a reference to a kernel's argument makes the compiler copy it to scratch memory)
#define NFN_PLACE(place, slots)                                                                             \
    GroupPlace place;                                                                                       \
    {                                                                                                       \
        const int number = static_cast<int>(blockIdx.x);                                                    \
        int index = number >= first1 ? 1 : 0;                                                               \
        index = number >= first2 ? 2 : index;                                                               \
        index = number >= first3 ? 3 : index;                                                               \
        const GemmSlot& mine = slots.slot[index];                                                           \
        place.weights = mine.weights;                                                                       \
        place.output = mine.output;                                                                         \
        place.partials = mine.partials;                                                                     \
        asm volatile("" : "+s"(place.partials)); /* (requested with the others, in every share) */          \
        place.output_dim = mine.output_dim;                                                                 \
        const int tiles = mine.tiles, shares = mine.shares, whole = number - mine.first;                    \
        const std::uint32_t by_shares = mine.by_shares;                                                     \
        place.share = divided(whole, tiles, mine.by_tiles);                                                 \
        place.tile = whole - place.share * tiles;                                                           \
        place.first_block = divided(total_blocks * place.share, shares, by_shares);                         \
        place.end_block = divided(total_blocks * (place.share + 1), shares, by_shares);                     \
    }

// RB: 32-row blocks per wave; the workgroup's tile is 32 * RB * WAVES rows by 128 columns.
template <std::uint32_t ENC, int RB, int WAVES>
__global__ __launch_bounds__(WAVES * kWave)
__attribute__((amdgpu_waves_per_eu(kWavesPerSimd<ENC, RB, WAVES>, kWavesPerSimd<ENC, RB, WAVES>))) void gemm_f16_kernel(
    const std::uint8_t* __restrict__ activations, const float* __restrict__ inverse_scale, std::int64_t row_stride,
    std::int64_t rows, int total_blocks, int m_tiles, std::uint32_t by_m_tiles, int first1, int first2, int first3,
    GemmSlots slots) {
    extern __shared__ __attribute__((aligned(16))) std::uint8_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // rows 64*wave .. +63 of the tile
    NFN_PLACE(place, slots)
    const std::uint8_t* weights = place.weights;
    float* output = place.output;
    const std::int64_t output_dim = place.output_dim;
    const int share = place.share;
    const int n_tile = divided(place.tile, m_tiles, by_m_tiles);
    const int m_tile = place.tile - n_tile * m_tiles;
    using Slice = typename Held<ENC, RB, WAVES>::Slice;
    using Header = typename Held<ENC, RB, WAVES>::Header;
    constexpr int kTileRows = 32 * RB * WAVES;
    const std::int64_t m0 = static_cast<std::int64_t>(m_tile) * kTileRows;
    const std::int64_t n0 = static_cast<std::int64_t>(n_tile) * kBN;
    // which share of the K dimension (whole 256-value blocks) this workgroup sums; each share
    // writes its own copy of the output
    const int first_block = place.first_block;
    const int steps = (place.end_block - first_block) * 4;  // a positive multiple of 4
    const int last = steps - 1;
    if (share > 0) output = place.partials + (share - 1) * rows * output_dim;

    // activations: fragment (row block, K chunk) is 1 KB, a row block's chunks are consecutive
    const std::int64_t row_block_bytes = static_cast<std::int64_t>(total_blocks) * 16 * kFragmentBytes;
    // (a tile of 512 rows can reach past the rows the copy is padded to: its last waves take blocks
    // that are there and store nothing)
    int row_block = static_cast<int>(m0 / 32) + wave * RB;
    if constexpr (WAVES == 8) row_block = min(row_block, static_cast<int>((rows + kBM - 1) / kBM * (kBM / 32)) - RB);
    const std::uint8_t* a_global = activations + row_block * row_block_bytes +
        static_cast<std::int64_t>(first_block) * 16 * kFragmentBytes + lane * 16;
    constexpr int kStepBytes = (kBK / 16) * kFragmentBytes;
    // weights: thread -> (row, which run of 16).  Eight consecutive lanes write their 16-byte
    // pieces into distinct banks: with stage rows of 36 words and runs of 8, rows k and k + 1
    // times four runs do, and so do rows k, k + 1, k + 4, k + 5 times two.
    constexpr int kLanes = WAVES == 8 ? 4 : kParts<ENC>;
    const int b_part = tid & (kLanes - 1);
    const int b_turn = tid / kLanes;
    const int b_row = kLanes == 4 ? b_turn : (b_turn & ~6) | ((b_turn & 2) << 1) | ((b_turn & 4) >> 1);
    const std::int64_t b_skip = static_cast<std::int64_t>(first_block) * kBlockBytes<ENC>;
    WeightRows b_global;
    b_global.first = weights + min(n0 + b_row, output_dim - 1) * row_stride + b_skip;
    b_global.second = weights + min(n0 + b_row + 64, output_dim - 1) * row_stride + b_skip;  // (four waves)
    const int b_target = b_row * kRowBytes + b_part * (WAVES == 8 && kRunSecond<ENC> == 64 ? 16 : 32);

    v16f acc[RB][4];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }

    // Activation fragments come from L2 (the other workgroups of this XCD read
    // the same rows): one slice, each fragment refilled right after its last use
    // with the same fragment of the next step, which leaves the load one step
    // to land.  Packed weights come from HBM or the memory-side cache: four
    // slices, each refilled right after it is decoded with the bytes of four
    // steps later (slice j holds the steps congruent to j modulo 4), which
    // gives their loads three steps.
    // The header of a 256-value block is loaded once, three or more steps
    // before the first of its four steps is decoded.
    ActivationSlice a_now;
    constexpr bool kWhole = kWholeBlocks<ENC, RB, WAVES>;
    Slices<ENC, RB, WAVES> set0, set1;  // (set1: whole blocks only; the sets swap roles like the headers)
    Header header_even, header_odd;  // blocks 0, 2, 4 ... and 1, 3, 5 ...
    const int last_block = (steps >> 2) - 1;
    header_even.load(b_global.first, 0, b_part);
    header_odd.load(b_global.first, min(1, last_block), b_part);
    set0.load(b_global, 0, b_part);
    a_now.r0k0 = NFN_LOAD_ACTIVATIONS(a_global, 0, 0);
    a_now.r0k1 = NFN_LOAD_ACTIVATIONS(a_global, 0, 1);
    a_now.r0k2 = NFN_LOAD_ACTIVATIONS(a_global, 0, 2);
    a_now.r0k3 = NFN_LOAD_ACTIVATIONS(a_global, 0, 3);
    if constexpr (RB == 2) {
        a_now.r1k0 = NFN_LOAD_ACTIVATIONS(a_global, 1, 0);
        a_now.r1k1 = NFN_LOAD_ACTIVATIONS(a_global, 1, 1);
        a_now.r1k2 = NFN_LOAD_ACTIVATIONS(a_global, 1, 2);
        a_now.r1k3 = NFN_LOAD_ACTIVATIONS(a_global, 1, 3);
    }
    {
        std::uint32_t wa[4][2], wb[4][2];
        set0.b0.prepare_bits(header_even, 0, b_part);
        set0.b0.prepare_scales(header_even);
        decode<0>(set0.b0, wa[0]);
        decode<1>(set0.b0, wa[1]);
        decode<2>(set0.b0, wa[2]);
        decode<3>(set0.b0, wa[3]);
        if constexpr (WAVES == 4) {
            decode<4>(set0.b0, wb[0]);
            decode<5>(set0.b0, wb[1]);
            decode<6>(set0.b0, wb[2]);
            decode<7>(set0.b0, wb[3]);
        }
        std::uint8_t* target = lds + b_target;
        NFN_WRITE16(target, wa[0][0], wa[0][1], wa[1][0], wa[1][1]);
        NFN_WRITE16(target + (WAVES == 8 ? kRunSecond<ENC> : 16), wa[2][0], wa[2][1], wa[3][0], wa[3][1]);
        if constexpr (WAVES == 4) {
            NFN_WRITE16(target + kSecondRun<ENC>, wb[0][0], wb[0][1], wb[1][0], wb[1][1]);
            NFN_WRITE16(target + kSecondRun<ENC> + 16, wb[2][0], wb[2][1], wb[3][0], wb[3][1]);
        }
    }
    if constexpr (!kHalfBlocks<ENC> && !kWhole) set0.b0.load(b_global, min(1, last_block), 0, b_part);  // step 4, or step 0 again
    __syncthreads();

    const int operand = (lane & 31) * kRowBytes + (lane >> 5) * 16;
    const std::uint8_t* b_read0 = lds + operand;
    const std::uint8_t* b_read1 = b_read0 + kStageBytes;
    std::uint8_t* b_write0 = lds + b_target;
    std::uint8_t* b_write1 = b_write0 + kStageBytes;
    WeightFragments current;
    current.c0 = NFN_READ_WEIGHTS(b_read0, 0, 0);
    current.c1 = NFN_READ_WEIGHTS(b_read0, 1, 0);
    current.c2 = NFN_READ_WEIGHTS(b_read0, 2, 0);
    current.c3 = NFN_READ_WEIGHTS(b_read0, 3, 0);
    // Enter the loop with no load in flight: the waits inside the loop are then
    // derived from the loop's own issue order alone, not from whatever order
    // the set-up code above was scheduled in.
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    NFN_FENCE();
    const auto activations_of = [&](int step) {
        return a_global + static_cast<std::int64_t>(min(step, last)) * kStepBytes;
    };
    // Four steps: one 256-value block.  Step s computes from stage s%2 while
    // step s+1 is decoded into the other stage; the decoded slice then loads
    // step s+5 and the activation slice step s+1.  `now` holds the scales of
    // this block, `next` those of the following one (needed by the fourth step,
    // which decodes the first step of that block).
    // (Whole blocks: the next block goes to the other set at the start instead.
    // Q6_K: b0 holds a block's first half, which the first and, of the next block, the fourth step
    // decode, b1 the second.)
    auto block_of_four = [&](int step, const Header& now, const Header& next, Slices<ENC, RB, WAVES>& mine,
                             Slices<ENC, RB, WAVES>& other) {
        constexpr bool kHalves = kHalfBlocks<ENC>;
        constexpr int kAhead = kHalves ? 3 : 4;  // from the step that is decoded to the one that is fetched
        Slices<ENC, RB, WAVES>& after = kWhole ? other : mine;
        if constexpr (kWhole) {
            const int block = min((step >> 2) + 1, last_block);
            other.load(b_global, block, b_part);
            NFN_FENCE();
        }
        Slice &second = kHalves ? mine.b0 : mine.b1, &third = kHalves ? mine.b1 : mine.b2, &fourth = kHalves ? mine.b1 : mine.b3;
        k_step<ENC, RB, WAVES, !kWhole>(acc, a_now, current, b_read0, b_read1, b_write1, second, now, 1, b_part,
                    activations_of(step + 1), row_block_bytes, b_global, min(step + 1 + kAhead, last));
        k_step<ENC, RB, WAVES, !kHalves && !kWhole>(acc, a_now, current, b_read1, b_read0, b_write0, third, now, 2, b_part,
                    activations_of(step + 2), row_block_bytes, b_global, min(step + 2 + kAhead, last));
        k_step<ENC, RB, WAVES, !kWhole>(acc, a_now, current, b_read0, b_read1, b_write1, fourth, now, 3, b_part,
                    activations_of(step + 3), row_block_bytes, b_global, min(step + 3 + kAhead, last));
        k_step<ENC, RB, WAVES, !kHalves && !kWhole>(acc, a_now, current, b_read1, b_read0, b_write0, after.b0, next, 0, b_part,
                    activations_of(step + 4), row_block_bytes, b_global, min(step + 4 + kAhead, last));
    };
    // The two header register sets swap roles every block; the loop body is two
    // blocks so that no copy (and no wait for the load that feeds it) is needed.
    // An odd block count runs its first block ahead of the loop.  The loop has
    // its only exit at the end: values loaded for later steps are then live
    // around the back edge and the loads stay where they are written.
    int block = 0;
    if ((last_block & 1) == 0) {
        block_of_four(0, header_even, header_odd, set0, set1);
        if constexpr (kWhole) set0 = set1;
        header_even.load(b_global.first, min(2, last_block), b_part);
        NFN_FENCE();
        const Header second = header_odd;
        header_odd = header_even;
        header_even = second;
        block = 1;
    }
    while (block < last_block) {
        block_of_four(block * 4, header_even, header_odd, set0, set1);
        header_even.load(b_global.first, min(block + 2, last_block), b_part);
        NFN_FENCE();
        block_of_four(block * 4 + 4, header_odd, header_even, kWhole ? set1 : set0, kWhole ? set0 : set1);
        header_odd.load(b_global.first, min(block + 3, last_block), b_part);
        NFN_FENCE();
        block += 2;
    }

    // D register r of lane l is row 8*(r/4) + 4*(l/32) + r%4, column l%32.  A store of it as it lies is 128 bytes of
    // two rows; a wave turns it in its part of the stages into whole rows of the tile and stores 512 bytes of each at
    // once (256 where the output's rows do not begin at 16 bytes).  Workgroups that start together end together, and
    // what they then have to write is megabytes: 1,316 rows of 2,048 -> 7,680 (Q5_K), 40 MB, spent 10 to 15 of 62 us
    // here with the stores as the results lie, and now take 58; 1,148 rows of 2,048 -> 4,864 (Q8_0) 46.0 -> 40.7, 250
    // rows of 3,328 into Q, K, V and gate (Q4_K) 42.8 -> 36.9, 36 rows of 2,048 -> 6,144 (Q6_K) 31.4 -> 28.0; a launch
    // of one long round (2,048 rows of 16,384 -> 6,656, 433) gains nothing.
    const int end_lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));  // (no register held for it)
    const int column = end_lane & 31;
    const int half = end_lane >> 5;
    constexpr int kPitch = kBN + 8;               // floats: rows that lie four apart begin in different banks
    constexpr int kTurned = WAVES == 8 ? 8 : 16;  // rows at a time
    static_assert(kTurned * kPitch * 4 * WAVES <= 2 * kStageBytes, "the waves' parts fit the stages");
    const bool wide = output_dim % 4 == 0 && reinterpret_cast<std::uintptr_t>(output) % 16 == 0;
    __syncthreads();
    float* const turned = reinterpret_cast<float*>(lds) + wave * (kTurned * kPitch);
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const std::int64_t first_row = m0 + wave * (32 * RB) + i * 32;
        const float* const scales = inverse_scale + (WAVES == 8 ? row_block * 32 + i * 32 : first_row) + 4 * half;
#pragma unroll
        for (int part = 0; part < 32 / kTurned; ++part) {
#pragma unroll
            for (int r = part * kTurned / 2; r < (part + 1) * kTurned / 2; ++r) {
                const float inverse = scales[8 * (r >> 2) + (r & 3)];
                const int row = 4 * half + 8 * (r >> 2) + (r & 3) - part * kTurned;
#pragma unroll
                for (int j = 0; j < 4; ++j) turned[row * kPitch + j * 32 + column] = acc[i][j][r] * inverse;
            }
            wave_sync();
            const std::int64_t m = first_row + part * kTurned;
            if (wide) {
                const std::int64_t n = n0 + 4 * column;
#pragma unroll
                for (int t = 0; t < kTurned; t += 2) {
                    const v4f four = *reinterpret_cast<const v4f*>(turned + (t + half) * kPitch + 4 * column);
                    if (m + t + half < rows && n < output_dim) {
                        *reinterpret_cast<v4f*>(output + (m + t + half) * output_dim + n) = four;
                    }
                }
            } else {
                const std::int64_t n = n0 + end_lane;
#pragma unroll
                for (int t = 0; t < kTurned; ++t) {
                    const float first = turned[t * kPitch + end_lane], second = turned[t * kPitch + end_lane + 64];
                    if (m + t < rows && n < output_dim) output[(m + t) * output_dim + n] = first;
                    if (m + t < rows && n + 64 < output_dim) output[(m + t) * output_dim + n + 64] = second;
                }
            }
            wave_sync();
        }
    }
}

// ---------------------------------------------------------------------------
// Up to 32 rows: a wave owns 32 columns and all rows of the same 128-column tile, so that a decoded
// weight fragment is read from LDS by one wave instead of four and by the wave that wrote it: no
// barrier, a quarter of the LDS reads, no matrix instructions for rows that are not there.  What
// bounds it: 17 rows of gate and up (Q4_K) take 40 us with the vector caches looking up a line in 68 % of
// the cycles, the vector ALU busy in half of them and a quarter of the waves' time in waits; the
// packed bytes and the fragments from L2 are requested a block and four steps ahead, and few
// tiles leave units without work: K is cut into up to eight shares.  17 rows, width 6,656, against 128-row tiles: Q, K, V and gate 41 -> 32 us for Q4_K, 50 -> 41
// for Q6_K; O (4,096 wide) 43 -> 21 and 52 -> 25; gate and up 68 -> 54 and 85 -> 68; down 56 -> 39
// and 66 -> 49; Q8_0 50 -> 47, 52 -> 32, 86 -> 84, 64 -> 60.
// ---------------------------------------------------------------------------
struct LowActivations {
    f16x8 chunk[4];
};

// from the first run of 16 to the second: 16 rows apart where four lanes share a row
template <std::uint32_t ENC>
constexpr int kLowSecondRun = kParts<ENC> == 2 ? 64 : 16 * kRowBytes;

// One K step of one wave: multiplies the step in `stage` and decodes the next one into `next_stage`.
template <std::uint32_t ENC>
__device__ __forceinline__ void low_step(v16f& acc, LowActivations& a, const std::uint8_t* stage,
                                         std::uint8_t* next_stage, PackedSlice<ENC>& b_next,
                                         const BlockHeader<ENC>& header, int decode_pair, int b_part,
                                         const std::uint8_t* a_fetch) {
    wave_sync();
    f16x8 weights[4];
#pragma unroll
    for (int chunk = 0; chunk < 4; ++chunk) weights[chunk] = *reinterpret_cast<const f16x8*>(stage + chunk * 32);
    wave_sync();
    std::uint32_t w[2], v[2];
    b_next.prepare_bits(header, decode_pair, b_part);
    b_next.prepare_scales(header);
    b_next.template group_a<0>(w);
    b_next.template group_a<1>(v);
    NFN_WRITE16(next_stage, w[0], w[1], v[0], v[1]);
    b_next.template group_a<2>(w);
    b_next.template group_a<3>(v);
    NFN_WRITE16(next_stage + 16, w[0], w[1], v[0], v[1]);
    b_next.template group_b<0>(w);
    b_next.template group_b<1>(v);
    NFN_WRITE16(next_stage + kLowSecondRun<ENC>, w[0], w[1], v[0], v[1]);
    b_next.template group_b<2>(w);
    b_next.template group_b<3>(v);
    NFN_WRITE16(next_stage + kLowSecondRun<ENC> + 16, w[0], w[1], v[0], v[1]);
#pragma unroll
    for (int chunk = 0; chunk < 4; ++chunk) NFN_MFMA(a.chunk[chunk], weights[chunk], acc);
    NFN_FENCE();
#pragma unroll
    for (int chunk = 0; chunk < 4; ++chunk) {
        a.chunk[chunk] = *reinterpret_cast<const f16x8*>(a_fetch + chunk * kFragmentBytes);
    }
    NFN_FENCE();
}

template <std::uint32_t ENC>
struct LowBlock {
    BlockHeader<ENC> header;
    Slices<ENC, 1, 4> slices;
    __device__ __forceinline__ void load(const WeightRows& rows, int block, int part) {
        header.load(rows.first, block, part);
        slices.load(rows, block, part);
    }
};

template <std::uint32_t ENC>
__global__ __launch_bounds__(kThreads, 2) void gemm_f16_low_kernel(
    const std::uint8_t* __restrict__ activations, const float* __restrict__ inverse_scale, std::int64_t row_stride,
    std::int64_t rows, int total_blocks, int first1, int first2, int first3, GemmSlots slots) {
    extern __shared__ __attribute__((aligned(16))) std::uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    NFN_PLACE(place, slots)
    const std::int64_t output_dim = place.output_dim;
    const std::int64_t n0 = static_cast<std::int64_t>(place.tile) * kBN + 32 * wave;
    const int first_block = place.first_block;
    const int steps = (place.end_block - first_block) * 4;
    const int last = steps - 1;
    const int last_block = (steps >> 2) - 1;
    float* const output = place.share > 0 ? place.partials + (place.share - 1) * rows * output_dim : place.output;

    constexpr int kStepBytes = (kBK / 16) * kFragmentBytes;
    const std::uint8_t* a_global =
        activations + static_cast<std::int64_t>(first_block) * 16 * kFragmentBytes + lane * 16;
    const auto activations_of = [&](int step) {
        return a_global + static_cast<std::int64_t>(min(step, last)) * kStepBytes;
    };
    // (the rows of a lane inside the wave's 32: the same bank pattern as above)
    const int b_part = lane & (kParts<ENC> - 1);
    const int b_turn = lane / kParts<ENC>;
    const int b_row = kParts<ENC> == 4 ? b_turn : (b_turn & ~6) | ((b_turn & 2) << 1) | ((b_turn & 4) >> 1);
    const std::int64_t b_skip = static_cast<std::int64_t>(first_block) * kBlockBytes<ENC>;
    WeightRows b_global;
    b_global.first = place.weights + min(n0 + b_row, output_dim - 1) * row_stride + b_skip;
    b_global.second = place.weights + min(n0 + b_row + 16, output_dim - 1) * row_stride + b_skip;

    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    LowActivations a0, a1, a2, a3;
    LowBlock<ENC> even, odd;  // blocks 0, 2, 4 ... and 1, 3, 5 ...
    even.load(b_global, 0, b_part);
    const auto load_activations = [&](LowActivations& a, int step) {
#pragma unroll
        for (int chunk = 0; chunk < 4; ++chunk) {
            a.chunk[chunk] = *reinterpret_cast<const f16x8*>(activations_of(step) + chunk * kFragmentBytes);
        }
    };
    load_activations(a0, 0);
    load_activations(a1, 1);
    load_activations(a2, 2);
    load_activations(a3, 3);

    std::uint8_t* const mine = lds + wave * 32 * kRowBytes;
    std::uint8_t* const write0 = mine + b_row * kRowBytes + b_part * 32;
    std::uint8_t* const write1 = write0 + kStageBytes;
    const std::uint8_t* const read0 = mine + (lane & 31) * kRowBytes + (lane >> 5) * 16;
    const std::uint8_t* const read1 = read0 + kStageBytes;
    {
        std::uint32_t wa[4][2], wb[4][2];
        even.slices.b0.prepare_bits(even.header, 0, b_part);
        even.slices.b0.prepare_scales(even.header);
        even.slices.b0.template group_a<0>(wa[0]);
        even.slices.b0.template group_a<1>(wa[1]);
        even.slices.b0.template group_a<2>(wa[2]);
        even.slices.b0.template group_a<3>(wa[3]);
        even.slices.b0.template group_b<0>(wb[0]);
        even.slices.b0.template group_b<1>(wb[1]);
        even.slices.b0.template group_b<2>(wb[2]);
        even.slices.b0.template group_b<3>(wb[3]);
        NFN_WRITE16(write0, wa[0][0], wa[0][1], wa[1][0], wa[1][1]);
        NFN_WRITE16(write0 + 16, wa[2][0], wa[2][1], wa[3][0], wa[3][1]);
        NFN_WRITE16(write0 + kLowSecondRun<ENC>, wb[0][0], wb[0][1], wb[1][0], wb[1][1]);
        NFN_WRITE16(write0 + kLowSecondRun<ENC> + 16, wb[2][0], wb[2][1], wb[3][0], wb[3][1]);
    }

    // four steps, one block: `now` is decoded from its second step on and the first of `next`
    const auto block_of_four = [&](int block, LowBlock<ENC>& now, LowBlock<ENC>& next) {
        constexpr bool kHalves = kHalfBlocks<ENC>;
        const int step = 4 * block;
        next.load(b_global, min(block + 1, last_block), b_part);
        NFN_FENCE();
        low_step<ENC>(acc, a0, read0, write1, kHalves ? now.slices.b0 : now.slices.b1, now.header, 1, b_part,
                          activations_of(step + 4));
        low_step<ENC>(acc, a1, read1, write0, kHalves ? now.slices.b1 : now.slices.b2, now.header, 2, b_part, activations_of(step + 5));
        low_step<ENC>(acc, a2, read0, write1, kHalves ? now.slices.b1 : now.slices.b3, now.header, 3, b_part,
                          activations_of(step + 6));
        low_step<ENC>(acc, a3, read1, write0, next.slices.b0, next.header, 0, b_part, activations_of(step + 7));
    };
    for (int block = 0; block <= last_block; block += 2) {
        block_of_four(block, even, odd);
        if (block < last_block) block_of_four(block + 1, odd, even);
    }

    const std::int64_t n = n0 + (lane & 31);
    const int row_base = (lane >> 5) * 4;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = row_base + 8 * (r >> 2) + (r & 3);
        if (row < rows && n < output_dim) output[row * output_dim + n] = acc[r] * inverse_scale[row];
    }
}

// Sum of the K shares: output[i] = share 0 (in place) + share 1 + ..., in that order;
// blockIdx.y: the projection.
struct ShareSums {
    float* output[kMaxProjections];
    const float* partials[kMaxProjections];
    std::int64_t count[kMaxProjections];
    int shares[kMaxProjections];
};
// PER outputs a thread, all of whose loads are under way together: one where the workgroups are few
// anyway, four beyond (333 rows of 16,384 -> 6,656 in four shares 11.4 -> 8.7 us).
template <int PER>
__global__ __launch_bounds__(256) void sum_shares_kernel(ShareSums sums) {
    float* output = sums.output[0];
    const float* partials = sums.partials[0];
    std::int64_t count = sums.count[0];
    int shares = sums.shares[0];
#pragma unroll
    for (int i = 1; i < kMaxProjections; ++i) {
        if (static_cast<int>(blockIdx.y) == i) {
            output = sums.output[i];
            partials = sums.partials[i];
            count = sums.count[i];
            shares = sums.shares[i];
        }
    }
    for (std::int64_t base = static_cast<std::int64_t>(blockIdx.x) * (256 * PER) + threadIdx.x; base < count;
         base += static_cast<std::int64_t>(gridDim.x) * (256 * PER)) {
        float total[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) total[k] = output[min(base + 256 * k, count - 1)];
#pragma unroll 8 / PER
        for (int share = 1; share < shares; ++share) {
#pragma unroll
            for (int k = 0; k < PER; ++k) total[k] += partials[(share - 1) * count + min(base + 256 * k, count - 1)];
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            if (base + 256 * k < count) output[base + 256 * k] = total[k];
        }
    }
}

// Tile height and K shares of a launch, from a sweep over both on this chip.
// 256-row tiles reuse each weight fragment twice as often and win whenever
// they give every compute unit a workgroup.  A smaller problem splits K over
// several workgroups per tile (at least twelve 256-value blocks each, at most
// four shares) until the grid fills the units' two (256-row tiles) or three
// (128-row tiles) workgroup slots; the shares are summed by a second launch in
// a fixed order.  256-row tiles stay the better choice as long as two shares or
// more fit; at most 128 rows take 128-row tiles.
// Narrow projections (an eighth of the units' count in 256-row tiles at most) take
// 128-row tiles and shares of six blocks or more.
// A K too short to split takes 256-row tiles from half a workgroup a unit on: 4,096 -> 6,656, 700
// rows (156 tiles) 82 -> 75 us for Q5_K and 94 -> 79 for Q6_K, 1,024 rows 87 -> 75; 512 rows (104
// tiles) would lose, 56 -> 62.
// The projections of one call run in one launch an encoding, each with the shares that it has by
// itself, so that few workgroups of one do not wait for those of another: 17 rows into Q, K, V and
// the gate of width 6,656 took 107 us (Q5_K) one after another and take 44, 333 rows 170 and 84.
// Up to 32 rows run on the kernel that cuts the columns among the waves, with shares of three blocks
// or more, at most eight, until there are two workgroups a unit.  (Two 32-row blocks a wave, for up
// to 64 rows: 128-row tiles are as fast or faster where the tiles are many, 64 rows of gate and up
// 81 us (Q4_K) and 203 (Q8_0) against 78 and 93 at 65.)
// (A call of more than 32 rows with room for it may cut further: shares_with_room.)
// (The heights here are those that the shares are cut for.  The launch takes the one that costs
// least with these shares, see tile_height; a sum does not depend on it.)
struct Plan {
    int tile_rows;  // 256 and 128 (two 32-row blocks a wave or one), 32 (all rows in every wave)
    int shares;
};

Plan plan(std::uint32_t encoding, std::int64_t rows, std::int64_t output_dim, std::int64_t input_dim,
          std::int64_t units) {
    const std::int64_t n_tiles = (output_dim + kBN - 1) / kBN;
    if (rows <= kLowRows) {
        std::int64_t shares = 2 * units / n_tiles;
        const std::int64_t most = (input_dim >> 8) / 3;
        if (shares > most) shares = most;
        if (shares > kLowShares) shares = kLowShares;
        if (shares < 1) shares = 1;
        return Plan{kLowRows, static_cast<int>(shares)};
    }
    const std::int64_t tall_tiles = (rows + 255) / 256 * n_tiles;
    if (tall_tiles >= units) return Plan{256, 1};
    std::int64_t longest = (input_dim >> 8) / 12;  // shares that still get twelve blocks each
    if (longest > kMaxShares) longest = kMaxShares;
    if (tall_tiles * 8 <= units) {
        // A narrow projection (a few tiles for the whole chip, e.g. 256 outputs): what it
        // takes is the length of one workgroup's walk over K, so the shares may be as short
        // as six blocks and the tiles are the small ones (1,024 x 6,656 -> 256: 53 -> 34 us).
        std::int64_t shortest = (input_dim >> 8) / 6;
        if (shortest > kMaxShares) shortest = kMaxShares;
        if (shortest < 1) shortest = 1;
        const std::int64_t tiles = (rows + 127) / 128 * n_tiles;
        std::int64_t shares = units * 3 / tiles;
        if (shares > shortest) shares = shortest;
        if (shares < 1) shares = 1;
        return Plan{128, static_cast<int>(shares)};
    }
    if (rows > 128) {
        std::int64_t shares = 2 * units / tall_tiles;
        if (shares > longest) shares = longest;
        if (shares >= 2) return Plan{256, static_cast<int>(shares)};
        if (2 * tall_tiles >= units) return Plan{256, 1};
    }
    const std::int64_t tiles = (rows + 127) / 128 * n_tiles;
    std::int64_t shares = units * (encoding == kEncQ6K ? 2 : 3) / tiles;
    if (shares > longest) shares = longest;
    if (shares < 1) shares = 1;
    return Plan{128, static_cast<int>(shares)};
}

template <std::uint32_t ENC, int RB, int WAVES>
void launch_tiles(const GemmGroup& group, int count, const std::uint8_t* activations, const float* inverse_scale,
                  std::int64_t rows, std::int64_t input_dim, hipStream_t stream) {
    const int m_tiles = static_cast<int>((rows + 32 * RB * WAVES - 1) / (32 * RB * WAVES));
    GemmSlots slots{};
    int workgroups = 0, first[kMaxProjections];
    for (int i = 0; i < kMaxProjections; ++i) {
        first[i] = i < count ? workgroups : 0x7fffffff;
        if (i >= count) continue;
        const int tiles = m_tiles * static_cast<int>((group.output_dim[i] + kBN - 1) / kBN);
        slots.slot[i] = GemmSlot{group.weights[i], group.output[i], group.partials[i], group.output_dim[i],
                                 workgroups, tiles, group.shares[i], inverse_of(tiles), inverse_of(group.shares[i]), {}};
        workgroups += tiles * group.shares[i];
    }
    const int blocks = static_cast<int>(input_dim >> 8);
    if (rows > kLowRows) {
        hipLaunchKernelGGL((gemm_f16_kernel<ENC, RB, WAVES>), dim3(static_cast<unsigned>(workgroups)), dim3(WAVES * kWave),
                           2 * kStageBytes, stream, activations, inverse_scale, group.row_stride, rows, blocks, m_tiles,
                           inverse_of(m_tiles), first[1], first[2], first[3], slots);
    } else {
        hipLaunchKernelGGL(gemm_f16_low_kernel<ENC>, dim3(static_cast<unsigned>(workgroups)), dim3(kThreads),
                           2 * kStageBytes, stream, activations, inverse_scale, group.row_stride, rows, blocks, first[1],
                           first[2], first[3], slots);
    }
}

// What a workgroup takes for 256 columns of K, in us, where one, two or three of the tile's height
// share a compute unit and all units are at work (0: so many do not fit).
struct TileCost {
    int rows;
    double block[3];
};
template <std::uint32_t ENC>
constexpr TileCost kTileCosts[3] = {{512, {6.9, 0, 0}}, {256, {4.1, 7.4, 0}}, {128, {2.7, 4.5, 6.6}}};
template <>
constexpr TileCost kTileCosts<kEncQ5K>[3] = {{512, {6.6, 0, 0}}, {256, {4.0, 7.2, 0}}, {128, {2.9, 4.5, 0}}};
template <>
constexpr TileCost kTileCosts<kEncQ6K>[3] = {{512, {7.0, 0, 0}}, {256, {4.6, 0, 0}}, {128, {3.2, 5.3, 0}}};
template <>
constexpr TileCost kTileCosts<kEncQ8_0>[3] = {{512, {6.8, 0, 0}}, {256, {4.1, 8.0, 0}}, {128, {3.1, 5.75, 0}}};

// What so many workgroups take for 256 columns each, round behind round, in us.
template <typename Int>
double rounds_of(const TileCost& tile, Int workgroups, Int units) {
    const int places = tile.block[2] > 0 ? 3 : tile.block[1] > 0 ? 2 : 1;
    const Int full = workgroups / (units * places), rest = workgroups - full * units * places;
    double rounds = static_cast<double>(full) * tile.block[places - 1];
    if (rest > 0) {
        const int last = static_cast<int>((rest + units - 1) / units);
        const double at_work = static_cast<double>(rest) / static_cast<double>(units * last);
        const double clock = 1.0 + 0.35 * (at_work - 1.0);
        rounds += tile.block[last - 1] * (clock > 0.75 ? clock : 0.75);
    }
    return rounds;
}

// The tile height of a launch of more than 32 rows.  The workgroups go to the units in rounds of as
// many as fit; the last one may leave places or whole units empty, and a chip at work in part runs
// at a higher clock, down to three quarters of the time.  The figures are fitted to 160 to 3,000
// rows into Q, K, V and gate, O, gate and up, and down at one to four shares: the times are met to
// 5 %, and the height chosen costs 0.2 % more than the best one on average.  At widths they are not
// fitted to (2,048 to 13,824 columns into 4,096 to 28,672 outputs, 48 to 4,096 rows, 448 calls) 0.2 % too,
// 13 at most: 1,537 rows of 13,824 -> 5,120 of Q4_K run on 128 rows in 349 us, and would on 512 in 310.
// Eight waves on 512 rows decode a weight for twice the rows, and Q6_K's registers then allow two
// waves a SIMD instead of one: 2,048 rows of 16,384 -> 6,656 474 -> 441 us (Q4_K), 486 -> 446 (Q5_K),
// 561 -> 466 (Q6_K), 548 -> 465 (Q8_0); 4,096 rows of gate and up 1,524 -> 1,467, 1,588 -> 1,501,
// 1,837 -> 1,517, 1,743 -> 1,527 (one chip, runs in turn; faster ones take a tenth less on either side).  Lower tiles where 512 rows leave too many units idle: 160 rows of gate
// and up 108 us in tiles of 256 rows (128: 124, 512: 163), of O 47 in tiles of 128 (58, 85).
//
// ... and what the launch costs at that height, in us: `blocks` of 256 columns that a workgroup walks on
// average, `extra` blocks' time for its start and end.
struct TileChoice {
    int rows;
    double cost;
};
TileChoice cheapest_tile(const TileCost (&tiles_of)[3], const std::int64_t* output_dims, const int* shares, int count,
                         std::int64_t rows, std::int64_t input_dim, double extra, std::int64_t units) {
    TileChoice best{0, 0};
    for (const TileCost& tile : tiles_of) {
        const std::int64_t m_tiles = (rows + tile.rows - 1) / tile.rows;
        std::int64_t workgroups = 0, tiles = 0;
        for (int i = 0; i < count; ++i) {
            const std::int64_t here = m_tiles * ((output_dims[i] + kBN - 1) / kBN);
            tiles += here;
            workgroups += here * shares[i];
        }
        const double rounds = rounds_of(tile, workgroups, units);
        const double blocks = static_cast<double>(input_dim >> 8) * static_cast<double>(tiles) / static_cast<double>(workgroups);
        const double cost = (blocks + extra) * rounds;
        if (best.rows == 0 || cost < best.cost) best = TileChoice{tile.rows, cost};
    }
    return best;
}

template <std::uint32_t ENC>
int tile_height(const GemmGroup& group, int count, std::int64_t rows, std::int64_t input_dim) {
    return cheapest_tile(kTileCosts<ENC>, group.output_dim, group.shares, count, rows, input_dim, 0.2, compute_units()).rows;
}

// K shares beyond those of plan(), where the workspace has room for them (gemm_f16_workspace_bytes asks for
// it): plan() leaves a share twelve blocks, which leaves most of the chip idle at a K of a few thousand
// columns into few tiles (35 rows of 4,096 -> 5,376: 42 workgroups on 256 units).  By the tiles' costs and
// the sums' (a launch, 3 us, and 0.4 us a MB of partial outputs), shares are added if they save a
// fifteenth of the call by itself and cost no more where two to two and a half such projections share a
// launch: a projection has the same shares, and with them the same bits, whatever runs beside it.
// Without the second condition 859 single calls (48 to 1,400 rows, 2,048 to 16,384 columns into 256 to
// 16,384 outputs) take 14 % less than plan()'s on average, but Q, K, V and gate of 2,304 columns and 218
// rows 33 -> 45 us.  With it, of 45 calls of 33 to 1,024 rows five gain (35 rows of 4,096 -> 5,376, Q4_K, 43.4 ->
// 23.4 us; 55 of 11,776 -> 5,376, Q8_0, 54.8 -> 39.3; 33 of 16,640 -> 2,048, Q6_K, 75.7 -> 61.4) and none
// loses.  Projections of fewer than 2,048 outputs (K and V) keep plan()'s: beside others their shares are
// not what a launch waits for.  One table of costs (Q4_K's) for all encodings, so that the workspace
// query, which knows none, need not ask for four.
int shares_with_room(const Plan& least, std::int64_t rows, std::int64_t output_dim, std::int64_t input_dim,
                     std::int64_t units) {
    const std::int64_t n_tiles = (output_dim + kBN - 1) / kBN;
    if (rows <= kLowRows || rows > kMostCutRows || n_tiles < kLeastCutTiles) return least.shares;
    if ((rows + 255) / 256 * n_tiles >= units) return least.shares;
    // (the same for every count up to the next multiple of 128: what gemm_f16_workspace_bytes relies on; and
    // from here on every number of tiles and workgroups is a small one)
    const int counted = static_cast<int>((rows + 127) / 128 * 128), wide = static_cast<int>(n_tiles);
    const double blocks = static_cast<double>(input_dim >> 8);
    const auto sums = [&](int shares, int quarters) {
        return shares == 1 ? 0.0 : 3.0 + 1.6e-6 * static_cast<double>((shares + 1) * counted) * (quarters * wide * kBN / 4);
    };
    const auto cost = [&](int shares, int quarters) {
        double least_walk = 0;
        for (const TileCost& tile : kTileCosts<kEncQ4K>) {
            const int tiles = (counted + tile.rows - 1) / tile.rows * ((quarters * wide + 3) / 4);
            const double walk = rounds_of(tile, tiles * shares, static_cast<int>(units));
            if (least_walk == 0 || walk < least_walk) least_walk = walk;
        }
        return blocks / shares * least_walk + sums(shares, quarters);
    };
    // What the blocks take with every place of every unit at work: no cut gets below it.
    double fullest = 0;
    for (const TileCost& tile : kTileCosts<kEncQ4K>) {
        double block = tile.block[0];
        for (int places = 2; places <= 3; ++places) {
            if (tile.block[places - 1] > 0) block = std::min(block, tile.block[places - 1] / places);
        }
        const double here = block * ((counted + tile.rows - 1) / tile.rows * wide);
        if (fullest == 0 || here < fullest) fullest = here;
    }
    fullest *= blocks / static_cast<double>(units);
    // quarters of the outputs: alone, with another, ...  (The host pays for this in every call and several
    // times in a query, so what saves too little by itself, or cannot, goes no further, and the unit count is asked
    // once: queries of 333 rows of 6,656 into Q, K, V and gate / of 1,000 rows of 4,096 -> 6,656 5.2 / 4.9 -> 0.4 /
    // 0.9 us, without any further shares 2.5 / 0.8.)
    constexpr int kBeside[4] = {4, 8, 9, 10};
    constexpr double kSaved = 0.94;
    double least_cost[4] = {cost(least.shares, kBeside[0])};
    int best = least.shares;
    double best_saved = 1.0;
    for (const int shares : {2, 3, 4, 6, 8}) {
        if (shares <= least.shares) continue;
        if (2 * shares > (input_dim >> 8) || fullest + sums(shares, kBeside[0]) >= kSaved * least_cost[0]) break;
        double saved = cost(shares, kBeside[0]) / least_cost[0];
        bool pays = saved < kSaved;
        for (int i = 1; i < 4 && pays; ++i) {
            if (least_cost[i] == 0) least_cost[i] = cost(least.shares, kBeside[i]);
            const double here = cost(shares, kBeside[i]) / least_cost[i];
            pays = here < 1.0;
            saved *= here;
        }
        if (pays && saved < best_saved) {
            best = shares;
            best_saved = saved;
        }
    }
    return best;
}

// One launch for `count` projections of one encoding and, if any of them splits K, one for the sums.
template <std::uint32_t ENC>
void launch_group(const GemmGroup& group, int count, const std::uint8_t* activations,
                  const float* inverse_scale, std::int64_t rows, std::int64_t input_dim, hipStream_t stream) {
    const int height = rows <= kLowRows ? 128 : tile_height<ENC>(group, count, rows, input_dim);
    if (height == 512) {
        launch_tiles<ENC, 2, 8>(group, count, activations, inverse_scale, rows, input_dim, stream);
    } else if (height == 256) {
        launch_tiles<ENC, 2, 4>(group, count, activations, inverse_scale, rows, input_dim, stream);
    } else {
        launch_tiles<ENC, 1, 4>(group, count, activations, inverse_scale, rows, input_dim, stream);
    }
    ShareSums sums{};
    int split = 0;
    std::int64_t most = 0;
    for (int i = 0; i < count; ++i) {
        if (group.shares[i] == 1) continue;
        sums.output[split] = group.output[i];
        sums.partials[split] = group.partials[i];
        sums.count[split] = rows * group.output_dim[i];
        sums.shares[split] = group.shares[i];
        if (sums.count[split] > most) most = sums.count[split];
        ++split;
    }
    if (split > 0) {
        const bool few = most <= 256 * 1024;
        const std::int64_t blocks = (most + (few ? 255 : 1023)) / (few ? 256 : 1024);
        const dim3 grid(static_cast<unsigned>(blocks < 4096 ? blocks : 4096), split);
        if (few) {
            hipLaunchKernelGGL(sum_shares_kernel<1>, grid, dim3(256), 0, stream, sums);
        } else {
            hipLaunchKernelGGL(sum_shares_kernel<4>, grid, dim3(256), 0, stream, sums);
        }
    }
}

std::int64_t padded_rows(std::int64_t rows) { return (rows + kBM - 1) / kBM * kBM; }

// fp16 activations in whole 256-row tiles, then the inverse scale of every row (8 bytes a row
// are kept for it: the size is part of what callers were told to allocate)
std::int64_t activation_bytes(std::int64_t rows, std::int64_t input_dim) {
    return (padded_rows(rows) * input_dim * 2 + padded_rows(rows) * 8 + 255) & ~std::int64_t(255);
}

// The largest of needed(count) over the row counts up to `rows`, of projections of `narrowest` outputs
// and more: short chunks split K further than longer ones and can take more memory.  What a plan
// gives stays the same from one multiple of 128 rows to the next, so that only those can be largest,
// and from a tile a unit on nothing is split.  at_most(count): no less than needed() of that count and of every
// smaller one, so that the small counts need no choice of shares.
template <typename F, typename G>
std::int64_t largest_up_to(std::int64_t rows, std::int64_t narrowest, std::int64_t units, F&& needed, G&& at_most) {
    std::int64_t largest = needed(rows);
    const std::int64_t n_tiles = (narrowest + kBN - 1) / kBN;
    // the last count below `rows` whose tiles of 256 rows are fewer than the units
    const std::int64_t split_rows = (units - 1) / n_tiles * 256, below = (rows - 1) / 128 * 128;
    for (std::int64_t count = std::min(split_rows, below); count > 0; count -= 128) {
        if (at_most(count) <= largest) return largest;
        largest = std::max(largest, needed(count));
    }
    if (kLowRows < rows && at_most(kLowRows) > largest) largest = std::max(largest, needed(kLowRows));
    return largest;
}

// floats of a projection's shares behind the first
std::int64_t partial_floats(int shares, std::int64_t rows, std::int64_t output_dim) {
    return (shares - 1) * rows * output_dim;
}

std::int64_t required_bytes(std::int64_t rows, std::int64_t input_dim, std::int64_t output_dim, int shares) {
    return activation_bytes(rows, input_dim) + (shares > 1 ? shares * rows * output_dim * 4 : 0) + 256;
}

// ... of the shares that a call with room for them takes, whatever the encoding (plan() gives Q4_K the most,
// and with as many or more the other encodings take none that it does not); *required: required_bytes().
std::int64_t most_partial_floats(std::int64_t rows, std::int64_t output_dim, std::int64_t input_dim, std::int64_t units,
                                 std::int64_t* required) {
    const Plan q4 = plan(kEncQ4K, rows, output_dim, input_dim, units), q6 = plan(kEncQ6K, rows, output_dim, input_dim, units);
    *required = required_bytes(rows, input_dim, output_dim, q4.shares);
    int most = shares_with_room(q4, rows, output_dim, input_dim, units);
    if (q6.shares != q4.shares) most = std::max(most, shares_with_room(q6, rows, output_dim, input_dim, units));
    return partial_floats(most, rows, output_dim);
}

// The launches of a call whose workspace has `room` floats behind the activations: each takes projections of
// one encoding whose partial outputs find room beside each other.  launch(indexes, count, shares): the
// projections of a launch; shares[i]: of projection i.  (The plan's shares where there is no room for more.)
template <typename F>
void for_each_launch(const std::uint32_t* encodings, const std::int64_t* output_dims, int count, std::int64_t rows,
                     std::int64_t input_dim, std::int64_t room, F&& launch) {
    const std::int64_t units = compute_units();
    int shares[kMaxProjections];
    std::int64_t floats[kMaxProjections];
    for (int i = 0; i < count; ++i) {
        int same = 0;
        while (encodings[same] != encodings[i] || output_dims[same] != output_dims[i]) ++same;
        if (same < i) {
            shares[i] = shares[same];
            floats[i] = floats[same];
            continue;
        }
        const Plan least = plan(encodings[i], rows, output_dims[i], input_dim, units);
        shares[i] = shares_with_room(least, rows, output_dims[i], input_dim, units);
        floats[i] = partial_floats(shares[i], rows, output_dims[i]);
        if (floats[i] > room) {
            shares[i] = least.shares;
            floats[i] = partial_floats(shares[i], rows, output_dims[i]);
        }
    }
    bool done[kMaxProjections] = {};
    for (int start = 0; start < count; ++start) {
        if (done[start]) continue;
        int members[kMaxProjections], found = 0;
        std::int64_t used = 0;
        for (int i = start; i < count; ++i) {
            if (done[i] || encodings[i] != encodings[start] || (i != start && used + floats[i] > room)) continue;
            done[i] = true;
            members[found++] = i;
            used += floats[i];
        }
        launch(members, found, shares);
    }
}

}  // namespace

std::int64_t gemm_f16_required_bytes(std::int64_t rows, std::int64_t input_dim, std::int64_t output_dim) {
    // the activations, then one copy of the output per K share of a split
    // launch (the encoding with the most shares bounds the others)
    return required_bytes(rows, input_dim, output_dim, plan(kEncQ4K, rows, output_dim, input_dim, compute_units()).shares);
}

std::int64_t gemm_f16_workspace_bytes(std::int64_t rows, std::int64_t input_dim, std::int64_t output_dim) {
    return gemm_f16_multi_workspace_bytes(rows, input_dim, &output_dim, 1);
}

void gemm_f16_plan(std::uint32_t encoding, std::int64_t rows, std::int64_t input_dim,
                   std::int64_t output_dim, int* tile_rows, int* k_shares) {
    const Plan chosen = plan(encoding, rows, output_dim, input_dim, compute_units());
    *tile_rows = chosen.tile_rows;
    *k_shares = chosen.shares;
}

void gemm_f16_launches(std::uint32_t encoding, std::int64_t rows, std::int64_t input_dim,
                       const std::int64_t* output_dims, int count, std::int64_t workspace_bytes, int* tile_rows,
                       int* k_shares) {
    const std::uint32_t encodings[kMaxProjections] = {encoding, encoding, encoding, encoding};
    const std::int64_t room = (workspace_bytes - activation_bytes(rows, input_dim)) / 4;
    for_each_launch(encodings, output_dims, count, rows, input_dim, room,
                    [&](const int* members, int found, const int* shares) {
        GemmGroup group{};
        for (int m = 0; m < found; ++m) {
            group.output_dim[m] = output_dims[members[m]];
            group.shares[m] = shares[members[m]];
        }
        int height = kLowRows;
        if (rows > kLowRows) {
            switch (encoding) {
                case kEncQ4K: height = tile_height<kEncQ4K>(group, found, rows, input_dim); break;
                case kEncQ5K: height = tile_height<kEncQ5K>(group, found, rows, input_dim); break;
                case kEncQ6K: height = tile_height<kEncQ6K>(group, found, rows, input_dim); break;
                default: height = tile_height<kEncQ8_0>(group, found, rows, input_dim); break;
            }
        }
        for (int m = 0; m < found; ++m) {
            tile_rows[members[m]] = height;
            k_shares[members[m]] = shares[members[m]];
        }
    });
}

bool gemm_f16_supports(std::uint32_t encoding, std::int64_t input_dim) {
    return (encoding == kEncQ4K || encoding == kEncQ5K || encoding == kEncQ6K ||
            encoding == kEncQ8_0) && input_dim % 256 == 0;
}

void convert_gemm_activations(const float* input, std::int64_t rows, std::int64_t input_dim,
                              void* workspace, hipStream_t stream) {
    std::uint8_t* activations = static_cast<std::uint8_t*>(workspace);
    float* inverse_scale = reinterpret_cast<float*>(activations + padded_rows(rows) * input_dim * 2);
    const std::int64_t groups = input_dim / 8;
    const unsigned wave_a_row = static_cast<unsigned>(padded_rows(rows) / 4);  // workgroups of four rows
    if (groups <= 4 * 64 * 2) {
        hipLaunchKernelGGL((prepare_activations_kernel<2, 4>), dim3(4 * wave_a_row), dim3(256), 0, stream,
                           input, activations, inverse_scale, rows, input_dim);
    } else if (groups <= 4 * 64 * 4) {
        hipLaunchKernelGGL((prepare_activations_kernel<4, 4>), dim3(4 * wave_a_row), dim3(256), 0, stream,
                           input, activations, inverse_scale, rows, input_dim);
    } else if (groups <= 2 * 64 * 16) {
        hipLaunchKernelGGL((prepare_activations_kernel<16, 2>), dim3(2 * wave_a_row), dim3(256), 0,
                           stream, input, activations, inverse_scale, rows, input_dim);
    } else {
        hipLaunchKernelGGL((prepare_activations_kernel<0, 1>), dim3(wave_a_row), dim3(256), 0, stream,
                           input, activations, inverse_scale, rows, input_dim);
    }
}

std::int64_t gemm_f16_multi_workspace_bytes(std::int64_t rows, std::int64_t input_dim, const std::int64_t* output_dims,
                                            int count) {
    std::int64_t narrowest = output_dims[0], outputs = 0;
    for (int i = 0; i < count; ++i) {
        if (output_dims[i] < narrowest) narrowest = output_dims[i];
        outputs += output_dims[i];
    }
    const std::int64_t units = compute_units();
    const auto needed = [&](std::int64_t chunk) {
        std::int64_t largest = 0, floats = 0;
        std::int64_t here[kMaxProjections], required[kMaxProjections];
        for (int i = 0; i < count; ++i) {
            int same = 0;
            while (output_dims[same] != output_dims[i]) ++same;
            if (same == i) here[i] = most_partial_floats(chunk, output_dims[i], input_dim, units, &required[i]);
            largest = std::max(largest, required[same]);
            floats += here[same];
        }
        return std::max(largest, activation_bytes(chunk, input_dim) + 4 * floats + 256);
    };
    return largest_up_to(rows, narrowest, units, needed, [&](std::int64_t chunk) {
        return activation_bytes(chunk, input_dim) + 4 * kLowShares * chunk * outputs + 256;
    });
}

void launch_gemm_f16(const Descriptor* descriptors, int count, const float* input, float* const* outputs,
                     std::int64_t rows, void* workspace, std::int64_t workspace_bytes, hipStream_t stream) {
    const std::int64_t input_dim = descriptors[0].input_dim;
    convert_gemm_activations(input, rows, input_dim, workspace, stream);
    const std::uint8_t* activations = static_cast<const std::uint8_t*>(workspace);
    const float* inverse_scale = reinterpret_cast<const float*>(activations + padded_rows(rows) * input_dim * 2);
    float* partials = reinterpret_cast<float*>(static_cast<std::uint8_t*>(workspace) + activation_bytes(rows, input_dim));
    const std::int64_t room = (workspace_bytes - activation_bytes(rows, input_dim)) / 4;
    std::uint32_t encodings[kMaxProjections] = {};
    std::int64_t output_dims[kMaxProjections] = {};
    for (int i = 0; i < count; ++i) {
        encodings[i] = descriptors[i].encoding;
        output_dims[i] = descriptors[i].output_dim;
    }
    for_each_launch(encodings, output_dims, count, rows, input_dim, room,
                    [&](const int* members, int found, const int* shares) {
        GemmGroup group{};
        std::int64_t used = 0;
        for (int m = 0; m < found; ++m) {
            const int i = members[m];
            group.weights[m] = descriptors[i].data;
            group.row_stride = descriptors[i].row_stride_bytes;
            group.output[m] = outputs[i];
            group.partials[m] = partials + used;
            group.output_dim[m] = output_dims[i];
            group.shares[m] = shares[i];
            used += partial_floats(shares[i], rows, output_dims[i]);
        }
        switch (encodings[members[0]]) {
            case kEncQ4K: launch_group<kEncQ4K>(group, found, activations, inverse_scale, rows, input_dim, stream); break;
            case kEncQ5K: launch_group<kEncQ5K>(group, found, activations, inverse_scale, rows, input_dim, stream); break;
            case kEncQ6K: launch_group<kEncQ6K>(group, found, activations, inverse_scale, rows, input_dim, stream); break;
            default: launch_group<kEncQ8_0>(group, found, activations, inverse_scale, rows, input_dim, stream); break;
        }
    });
}

}  // namespace nfn
