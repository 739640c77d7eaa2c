// Verifier rows (4..16 tokens; two and three where that is faster) of K-quant projections on the int8 matrix cores, every row in
// the one-row kernel's arithmetic bit for bit.
//
// The contract (neuralfn/csrc/native_train/tile_ops.h:685-688; the reference's kernel:
// neuralfn/csrc/tile_cuda/glimmer_k_mmq.cu:1753-1925): row t of a batched call equals the
// one-row call on row t.  The one-row kernels (gemv_dot.hip, gemv_q6.hip, gemv_q8.hip) give
// lane L of a wave the units u = L, L + 64, ... of a weight row (a unit: 64 values), chain one
// fused multiply-add per unit,
//   Q4_K, Q5_K  acc = fmaf(scale, fmaf(-dmin, float(wmin), d * fmaf(float(whi), 256, float(wlo))), acc)
//   Q6_K        acc = fmaf(scale * d, ((sc0 * float(b0) + sc1 * float(b1)) + ...) in fused steps, acc)
//   Q8_0        acc = fmaf(scale, fmaf(d1, float(b1), d0 * float(b0)), acc)
// over them and sum the 64 lanes in a butterfly.  Everything up to the integers in these
// formulas is exact integer arithmetic, and float addition is commutative, so the result is
// fixed by
//   * which terms form a chain: the units 4b + p of the blocks b = c, c + 16, c + 32, ...
//     ("class" c = 0..15, p = 0..3; a block: 256 values), in that order,
//   * the balanced binary tree over the 64 chains in the order (c, p).
// Here a workgroup of 8 waves owns up to 32 consecutive weight rows.  A matrix instruction takes
// the values of a scale group (K: 32 values, 16 for Q6_K), 32 weight rows (operand B, lane l:
// row l % 32, half l / 32 of the group; the packed bytes are loaded coalesced and change lanes
// through a private LDS tile per wave) and the two int8 planes of up to 16 tokens (operand A,
// fetched in operand order from the image a quantizer launch left in the workspace beside the
// activation records: lanes that each pick their own 16 bytes out of sixteen records cost the
// memory pipeline four times the instructions' coalesced rate).  For Q4_K / Q5_K of more than eight tokens a second
// product against the sub-block minimums, spread over K, gives the sums the minimums
// multiply (fewer tokens: multiply-adds with the code sums of the records); Q6_K's offset of 32 is taken off the codes before the product.  A lane then holds,
// for its weight row and up to 8 tokens, the integers of a unit, and replays the float tail
// above.  Wave w takes the classes w and 15 - w (an even share of any row length), keeps the
// four chains of a class per token in registers, and leaves (c0 + c1) + (c2 + c3) per class,
// token and row in LDS; when all have, a thread per (token, row) adds the 16 classes in the
// tree's order (up to eight tokens a tile later, the waves waiting for each other's counts in LDS; more: after a
// barrier).  A workgroup walks the tiles blockIdx.x, blockIdx.x + gridDim.x, ... with the
// loads of the next tile's first block in flight under the last block of the one before.
// One pass over the weights for up to 16 tokens.
//
// What bounds it: more than eight tokens the vector ALU (the replayed tail).  Up to eight no unit is full:
// a wave issues an instruction every 5 to 8 cycles and two waves fit a SIMD.  Gate and up of seven tokens,
// Q4_K, share of the cycles: vector ALU 55 %, line look-ups 39, LDS 25, matrix cores 11, and waves wait
// 31 % of theirs; down, Q6_K, 46, 35, 43, 12 and 30; O, 208 tiles of sixteen blocks, vector ALU 33.  (Only the
// weights' loads take 23.4 us of gate and up's, with the operands' 28.5, everything 32 to 35.)  Up to
// eight tokens therefore: two or four scale groups to an operand fragment (half or a quarter of
// the operand bytes, registers for a second block of packed bytes in flight), the minimums'
// sums from the records instead of a second pair of products, products issued around the tail
// before.  Q4_K, 2 x 16,384 rows of 6,656 columns: 39.6 -> 31.2 us at four tokens, 41.9 -> 39.0 at
// seven, quantizer launch included; Q5_K 44.5 -> 35.8 and 48.2 -> 43.2, Q8_0 54.1 -> 48.2 and
// 57.0 -> 52.5, Q6_K 58.4 -> 53.3 and 63.1 -> 58.9.  With a barrier a tile its waves waited for the one with
// the most blocks (26 of a row are three for most waves, four for two): counts instead, at seven tokens,
// Q4_K 39.6 -> 38.3, Q6_K 58.9 -> 55.4 us, four projections of 8,704 rows 18.5 -> 17.3 and 26.0 -> 24.4;
// one tile a workgroup or even shares as before.  (More than eight tokens leave no memory for four tiles'
// sums; with two, and the counts to be cleared first, 3 to 7 % slower.)
#include "common.hpp"
#include "gemv_rows.hpp"
#include "wave_rows.hpp"

#include <algorithm>
#include <type_traits>

namespace nfn {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kRowsTile = 32;
constexpr int kRowsWaves = 8;
constexpr int kRowsThreads = kRowsWaves * kWave;
constexpr int kClasses = 16;
constexpr int kMaxRowsBlocks = 256;  // input_dim up to 65,536

constexpr int kImageFragments = kRowsImageFragments;
constexpr int kImageBlock = kRowsImageBlock;

// One wave per activation record: writes the (token, block) record of wave_rows.hpp and the
// token's share of the block's operand image.
// Workgroups past those of the records fill the outputs of `clear` with -0.0f, 1024 floats a
// workgroup: the split form of the kernel below adds the two halves of a row's butterfly
// onto them (-0 + x is x for every x, -0 included).
template <int P>
__global__ __launch_bounds__(256) void quantize_records_kernel(
    const float* __restrict__ first, const float* __restrict__ second,
    std::uint8_t* __restrict__ records, std::uint8_t* __restrict__ image, int blocks, int tokens,
    int record_groups, ProjectionSet clear) {
    if (static_cast<int>(blockIdx.x) >= record_groups) {
        std::int64_t chunk = static_cast<std::int64_t>(blockIdx.x) - record_groups;
#pragma unroll
        for (int index = 0; index < 4; ++index) {
            if (index >= clear.count) break;
            const std::int64_t floats = clear.op[index].output_dim * tokens;
            const std::int64_t chunks = (floats + 1023) >> 10;
            if (chunk < chunks) {
                float* output = clear.op[index].output;
                const std::int64_t begin = (chunk << 10) + threadIdx.x * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (begin + e < floats) output[begin + e] = -0.0f;
                }
                return;
            }
            chunk -= chunks;
        }
        return;
    }
    const int lane = threadIdx.x & 63;
    const int record = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6);
    if (record >= blocks * tokens) return;
    const float4 x = load_activations<P>(first, second,
                                         static_cast<std::int64_t>(record) * 256 + lane * 4);
    const ActivationCodes codes = activation_codes<P>(x);
    store_record(records + static_cast<std::int64_t>(record) * kActRecord, lane, codes);
    const int token = record / blocks;
    const int block = record - token * blocks;
    store_operand_image(image, block, token, tokens, lane, codes);
}

// How a block (256 values of one weight row) lies in memory and in a wave's LDS tile.
//   Q4_K / Q5_K: 144 / 176 bytes, 16-byte aligned; the tile is the same bytes row after row.
//   Q8_0: eight 34-byte blocks = 272 bytes; rows are as aligned as the tensor is.
//   Q6_K: 210 bytes, so every other block starts two bytes past a word.  A block is fetched as
//     fourteen 16-byte pieces from the word at or before its first byte (pieces 0..12 in a
//     row, piece 13 from byte 196, so that no load reaches past the word that holds the
//     block's last byte) and written to its 240-byte LDS slot two bytes down when it started
//     past a word: in LDS every block starts at byte 16 of its slot.
template <std::uint32_t ENC>
struct RowsFormat {
    static constexpr bool kQ6 = ENC == kEncQ6K;
    static constexpr bool kQ8 = ENC == kEncQ8_0;
    static constexpr int kBlockBytes = ENC == kEncQ4K ? 144 : ENC == kEncQ5K ? 176 : kQ6 ? 210 : 272;
    static constexpr int kChunks = kQ6 ? 14 : kBlockBytes / 16;  // 16-byte pieces of a block
    static constexpr int kTileChunks = kRowsTile * kChunks;      // of a block of 32 rows
    static constexpr int kLoads = (kTileChunks + kWave - 1) / kWave;
    static constexpr int kSlotBytes = kQ6 ? 240 : kBlockBytes;   // a row's place in the LDS tile
    static constexpr int kSlotOrigin = kQ6 ? 16 : 0;             // where the block starts in it
    static constexpr int kTileBytes = kRowsTile * kSlotBytes;
};

struct __attribute__((packed, aligned(2))) RowsPiece {
    std::uint32_t v[4];
};
struct __attribute__((packed, aligned(4))) RowsWords {
    std::uint32_t v[2];
};
struct __attribute__((packed, aligned(2))) RowsHalfPiece {
    std::uint32_t v[2];
};

typedef int v2i __attribute__((ext_vector_type(2)));

// The packed bytes of 32 rows x one block as a wave loads them, coalesced: one set of
// registers, up to eight tokens two (they go to the LDS tile as soon as they arrive, and the request of
// the next block, or the one after it, reuses them).
template <std::uint32_t ENC>
struct RowsPacked {
    v4u chunk[RowsFormat<ENC>::kLoads];
    std::uint32_t shifted;  // Q6_K: bit i = piece i of this lane starts two bytes past a word
};

// Operand A of the eight 32-value groups of a block: two sets, used by the matrix instructions
// where they arrive.
template <int S>
struct RowsOperands {
    static constexpr int kFragments = S;  // 8 / rows_groups(S)
    v4i a[kFragments];
    v2i extra;  // this lane's entry of the block's code sums and scales
};

__device__ __forceinline__ v16i mfma_i8(v4i a, v4i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// K = 16: operands of 8 bytes a lane (lane l: row l % 32, values 8 (l / 32)..+7)
__device__ __forceinline__ v16i mfma_i8_k16(v2i a, v2i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x16_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b),
                                                 c, 0, 0, 0);
}

__device__ __forceinline__ void rows_lds_fence() {
    // LDS traffic of one wave is in order; this only pins the compiler.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ std::uint32_t lds_address(const int* word) {
    return static_cast<std::uint32_t>(reinterpret_cast<std::uintptr_t>((const __attribute__((address_space(3))) int*)word));
}

// until each of the workgroup's waves has said `count` or more (the word of wave lane % 8 at `words`).  In
// assembly, so that the requests in flight stay counted as they are.
__device__ __forceinline__ void rows_wait_for_all(std::uint32_t words, int count) {
    std::uint32_t word;
    __asm__ volatile(
        ".Lwait%=:\n\t"
        "ds_read_b32 %0, %1\n\t"
        "s_waitcnt lgkmcnt(0)\n\t"
        "v_cmp_gt_i32 vcc, %2, %0\n\t"
        "s_cbranch_vccnz .Lwait%=\n"
        : "=&v"(word)
        : "v"(words), "s"(count)
        : "vcc", "memory");
}

// SPLIT: a workgroup computes one half of a row's butterfly, the classes 0..7 (the first
// left_groups workgroups) or 8..15 (the others), a wave one class, and adds (q0 + q1) or
// (q2 + q3) onto the output, which the quantizer launch has filled with -0: two terms commute,
// so the sum is the one-row kernel's whichever half arrives first.  Twice the work units of
// about half the length, shared out over the workgroups by what the halves cost (a row of 26
// blocks has 16 on the left and 10 on the right): for tile counts that leave much of the
// chip idle in the last pass over whole tiles (272 tiles on 256 units).
// rows_a_tile: kRowsTile; where whole tiles would not come out even, fewer (rows_of_tile).
template <std::uint32_t ENC, int S, bool SPLIT>
__global__ __launch_bounds__(kRowsThreads, 2) void gemv_rows_kernel(
    const std::uint8_t* __restrict__ image, const std::uint8_t* __restrict__ records, int tokens,
    int input_dim, std::uint32_t total_tiles, std::uint32_t left_groups, int rows_a_tile, ProjectionSet set) {
    constexpr bool kQ5 = ENC == kEncQ5K;
    using F = RowsFormat<ENC>;
    constexpr int kBlockBytes = F::kBlockBytes;
    constexpr int kQuants = kQ5 ? 48 : 16;
    constexpr int kTokens = 2 * S;
    constexpr int kGroups = rows_groups(S);
    constexpr bool kDeep = S <= 4;  // registers for two blocks of packed bytes in flight
    // class sums of so many tiles: two where the workgroup's waves meet at a barrier once per tile, four
    // where they wait for each other's counts (up to eight tokens)
    constexpr int kOwnClasses = SPLIT ? kClasses / 2 : kClasses;
    constexpr int kTilesHeld = kDeep ? 4 : 2;
    __shared__ float class_sums[kTilesHeld][kOwnClasses][kTokens][kRowsTile];
    // how many tiles a wave has left its sums of [0], and added its part of [1] (a word a lane: 64 writes
    // of one word would take turns)
    __shared__ int said[2][kDeep ? kRowsWaves : 1][kWave];
    __shared__ __attribute__((aligned(16))) std::uint8_t packed_tiles[kRowsWaves][F::kTileBytes];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 31;
    const int h = lane >> 5;
    const int blocks = input_dim >> 8;

    // A workgroup walks the tiles blockIdx.x, blockIdx.x + gridDim.x, ...; the loads of a
    // tile's first block go out under the arithmetic of the tile before.
    const bool right_half = SPLIT && blockIdx.x >= left_groups;
    const std::uint32_t first_tile = right_half ? blockIdx.x - left_groups : blockIdx.x;
    const std::uint32_t tile_stride =
        SPLIT ? (right_half ? gridDim.x - left_groups : left_groups) : gridDim.x;
    const int my_tiles = static_cast<int>((total_tiles - first_tile + tile_stride - 1) / tile_stride);
    if (kDeep && my_tiles > 1) {
        said[0][wave][lane] = 0;
        said[1][wave][lane] = 0;
        __syncthreads();
    }
    const auto wait_for_all = [&](int what, int count) {
        rows_wait_for_all(lds_address(&said[what][lane & (kRowsWaves - 1)][0]), count);
    };
    auto projection_of = [&](std::uint32_t tile) {
        int which = 0;
#pragma unroll
        for (int index = 1; index < 4; ++index) {
            if (index < set.count && tile >= set.op[index].first_tile) which = index;
        }
        return pick(set, which);
    };

    // What the loads of a tile need: its first row and, per lane, where the pieces it copies
    // per block lie: piece n = 64 i + lane of the 32 x kChunks, kChunks to a row (the lanes
    // past the last piece repeat it), and where in the LDS tile each goes.
    const std::uint8_t* tile_rows;
    std::uint32_t chunk_offset[F::kLoads];
    std::uint32_t row_parity = 0;  // Q6_K: bit i = the row of piece i starts two bytes past a word
    // (Q4_K, Q5_K, Q8_0: the LDS tile is the same bytes row after row, piece n at byte 16 n)
    std::uint32_t lds_offset[F::kQ6 ? F::kLoads : 1];
    if constexpr (F::kQ6) {
#pragma unroll
        for (int i = 0; i < F::kLoads; ++i) {
            const int chunk = i * kWave + lane;
            const int row = chunk / F::kChunks;
            const int col = chunk - row * F::kChunks;
            lds_offset[i] = row * F::kSlotBytes + F::kSlotOrigin + (col == 13 ? 196 : col * 16);
        }
    }
    const int last_slot = min((F::kLoads - 1) * kWave + lane, F::kTileChunks - 1) * 16;
    auto aim = [&](std::uint32_t tile) {
        const Projection op = projection_of(tile);
        const std::int64_t row0 = static_cast<std::int64_t>(tile - op.first_tile) * rows_a_tile;
        const int valid_rows =
            static_cast<int>(min(static_cast<std::int64_t>(rows_a_tile), op.output_dim - row0));
        tile_rows = op.data + row0 * op.row_stride;
        row_parity = 0;
#pragma unroll
        for (int i = 0; i < F::kLoads; ++i) {
            const int chunk = min(i * kWave + lane, F::kTileChunks - 1);
            const int row = chunk / F::kChunks;
            const int col = chunk - row * F::kChunks;
            const int within = F::kQ6 && col == 13 ? 196 : col * 16;
            const std::uint32_t row_offset = static_cast<std::uint32_t>(min(row, valid_rows - 1)) *
                    static_cast<std::uint32_t>(op.row_stride);
            chunk_offset[i] = row_offset + within;
            if constexpr (F::kQ6) {
                const std::uint32_t address_low = static_cast<std::uint32_t>(
                    reinterpret_cast<std::uintptr_t>(tile_rows)) + row_offset;
                row_parity |= ((address_low >> 1) & 1u) << i;
            }
        }
    };
    std::uint8_t* const my_tile = packed_tiles[wave];
    const std::uint8_t* const my_row = my_tile + j * F::kSlotBytes + F::kSlotOrigin;
    // What the float tails take from the activation records and the image.  Up to eight tokens it comes with a
    // block's operands, eight bytes a lane, and goes through LDS: for Q4_K and Q5_K the code sums
    // of two neighbouring 32-value groups of a token (entry [pair of groups][token]), then the
    // scale of every token.  More tokens leave no registers for that: the scales of all the wave's
    // blocks are brought to LDS when it starts.
    constexpr bool kSums = !F::kQ6 && !F::kQ8 && kDeep;
    constexpr int kScaleEntry = kSums ? 4 * kTokens : 0;
    constexpr int kEntries = kDeep ? kScaleEntry + kTokens : 1;
    constexpr int kMaxSteps = kDeep ? 1 : kMaxRowsBlocks / kRowsWaves;
    static_assert(kEntries <= kWave, "an entry a lane");
    __shared__ __attribute__((aligned(16))) v2i extras[kRowsWaves][kEntries];
    __shared__ __attribute__((aligned(16))) float step_scales[kRowsWaves][kMaxSteps][kDeep ? 1 : kTokens];
    v2i* const my_extras = extras[wave];
    const bool sums_lane = lane < kScaleEntry;
    const int extra_entry = sums_lane ? (lane & 3) * kTokens + (lane >> 2) : lane;
    const std::uint8_t* extra_base = nullptr;  // of block 0; from block to block `extra_stride` on
    std::uint32_t extra_stride = 0;
    if constexpr (kDeep) {
        const int token = sums_lane ? min(lane >> 2, tokens - 1) : min(lane - kScaleEntry, kTokens - 1);
        extra_base = sums_lane
            ? records + static_cast<std::uint32_t>(token * blocks) * kActRecord + kRecordSums + (lane & 3) * 8
            : image + kImageFragments + token * 4;
        extra_stride = sums_lane ? kActRecord : kImageBlock;
    }

    // A wave's steps of a tile: the blocks of class r, then those of class 15 - r (SPLIT: of the one
    // class r or 8 + r), r = wave for the first tile.  Rows whose blocks are no multiple of 16 give
    // some r a block more than others (26 blocks: r = 6 and 7 have four, the others three), so r
    // moves on by two with every tile and a wave has had every r of its parity after four tiles: even
    // shares where the extra blocks fall on both alike (26 blocks), a block more in four tiles for
    // one half of the waves where there is one (17 blocks: r = 0).  Rows of fewer than 16 blocks leave
    // some r nothing and stay.
    const int role_step = kDeep && blocks >= kClasses ? 2 : 0;
    struct Role {
        int class0, class1, count0, total;
    };
    const auto role_of = [&](int r) {
        Role role;
        role.class0 = (SPLIT && right_half ? 8 : 0) + r;
        role.class1 = kClasses - 1 - r;
        role.count0 = role.class0 < blocks ? (blocks - role.class0 + kClasses - 1) / kClasses : 0;
        int count1 = role.class1 < blocks ? (blocks - role.class1 + kClasses - 1) / kClasses : 0;
        if constexpr (SPLIT) {
            // (no second class; a value the optimizer cannot see through, so that the walk below
            // compiles as it does for two classes: with a known zero it is scheduled with far
            // more registers, and spills)
            count1 = 0;
            asm volatile("" : "+s"(count1));
        }
        role.total = role.count0 + count1;
        return role;
    };
    const auto block_of = [&](const Role& role, int step) {
        return step < role.count0 ? role.class0 + kClasses * step : role.class1 + kClasses * (step - role.count0);
    };
    int fetch_r = wave;
    Role fetch_role = role_of(fetch_r);
    Role role = fetch_role;  // of the tile being worked on
    std::uint32_t fetch_tile = first_tile;
    int fetch_step = 0;
    aim(fetch_tile);
    // the packed bytes of the next step of the walk; past its end the last block again
    auto fetch_packed = [&](RowsPacked<ENC>& stage) {
        const int block = min(block_of(fetch_role, min(fetch_step, max(fetch_role.total - 1, 0))), blocks - 1);
        const std::uint8_t* weights = tile_rows + static_cast<std::int64_t>(block) * kBlockBytes;
        // (a Q6_K block with an odd index lies two bytes further from a word than its row does)
        const std::uint32_t shifted = F::kQ6 ? row_parity ^ (0u - static_cast<std::uint32_t>(block & 1)) : 0u;
        if constexpr (F::kQ6) stage.shifted = shifted;
#pragma unroll
        for (int i = 0; i < F::kLoads; ++i) {
            if constexpr (F::kQ6 || F::kQ8) {
                // (Q8_0 rows are only as aligned as the tensor; Q6_K pieces start on a word, those of a tensor that does not
                // two bytes before it: the same aligned word, which is there, and what it brings is shifted out)
                const std::uint32_t back = F::kQ6 ? ((shifted >> i) & 1u) * 2u : 0u;
                const RowsPiece piece = *reinterpret_cast<const RowsPiece*>(weights + chunk_offset[i] - back);
                stage.chunk[i] = v4u{piece.v[0], piece.v[1], piece.v[2], piece.v[3]};
            } else {
                stage.chunk[i] = *reinterpret_cast<const v4u*>(weights + chunk_offset[i]);
            }
        }
        if (++fetch_step >= fetch_role.total && fetch_tile + tile_stride < total_tiles) {
            fetch_step = 0;
            fetch_tile += tile_stride;
            if constexpr (kDeep) {
                fetch_r = (fetch_r + role_step) & (kRowsWaves - 1);
                fetch_role = role_of(fetch_r);
            }
            aim(fetch_tile);
        }
    };
    // ... and the operands of a block
    auto fetch_operands = [&](RowsOperands<S>& operands, int wanted) {
        const int block = min(wanted, blocks - 1);
        if constexpr (kDeep) {
            // (the second word of a scale entry is the next token's: the image has 16)
            operands.extra = __builtin_bit_cast(
                v2i, *reinterpret_cast<const RowsWords*>(extra_base + static_cast<std::uint32_t>(block) * extra_stride));
        }
        const std::uint8_t* fragments = image + static_cast<std::int64_t>(block) * kImageBlock;
#pragma unroll
        for (int sub = 0; sub < RowsOperands<S>::kFragments; ++sub) {
            if constexpr (F::kQ6) {
                // the sixteen values 16 s..+15 of a 32-value group are what the image keeps for
                // lanes 32 s..+31: this lane takes bytes 8 h..+7 of row j's sixteen, for s = 0, 1
                const std::uint8_t* mine = fragments + sub * 1024 + j * 16 + h * 8;
                const v2i lower = *reinterpret_cast<const v2i*>(mine);
                const v2i upper = *reinterpret_cast<const v2i*>(mine + 512);
                operands.a[sub] = v4i{lower[0], lower[1], upper[0], upper[1]};
            } else {
                operands.a[sub] = *reinterpret_cast<const v4i*>(fragments + sub * 1024 + lane * 16);
            }
        }
    };

    float acc[4][S];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
        for (int slot = 0; slot < S; ++slot) acc[p][slot] = 0.0f;
    }

    // the packed bytes change lanes through the wave's LDS tile
    auto stage_to_lds = [&](const RowsPacked<ENC>& stage) {
        if constexpr (F::kQ6) {
#pragma unroll
            for (int i = 0; i < F::kLoads; ++i) {
                const std::uint32_t back = ((stage.shifted >> i) & 1u) * 2u;
                RowsPiece piece;
                piece.v[0] = stage.chunk[i][0];
                piece.v[1] = stage.chunk[i][1];
                piece.v[2] = stage.chunk[i][2];
                piece.v[3] = stage.chunk[i][3];
                *reinterpret_cast<RowsPiece*>(my_tile + lds_offset[i] - back) = piece;
            }
        } else {
#pragma unroll
            for (int i = 0; i + 1 < F::kLoads; ++i) {
                *reinterpret_cast<v4u*>(my_tile + lane * 16 + i * (kWave * 16)) = stage.chunk[i];
            }
            *reinterpret_cast<v4u*>(my_tile + last_slot) = stage.chunk[F::kLoads - 1];
        }
    };

    auto compute = [&](const RowsOperands<S>& stage, int step) {
        const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        float scale[S];
#pragma unroll
        for (int slot = 0; slot < S; ++slot) {
            scale[slot] = kDeep ? __int_as_float(my_extras[kScaleEntry + S * h + slot][0])
                                : step_scales[wave][step][S * h + slot];
        }
        if constexpr (F::kQ6) {
            // Q6_K (neuralfn/csrc/native_gpt2/resident_glimmer.cpp:591-616): per half of 128
            // values 64 bytes of low nibbles (quarters 0 / 2 in bytes 0..31, 1 / 3 in 32..63) and
            // 32 bytes of 2-bit tops; 16 int8 sub-scales (half, quarter, sixteen) and d.  This
            // lane decodes values 8 h..+7 of both sixteens of every quarter of row j.
            const RowsPiece sub_scales = *reinterpret_cast<const RowsPiece*>(my_row + 192);
            const float d = half_bits_to_float(*reinterpret_cast<const std::uint16_t*>(my_row + 208));
            float factor[S];
#pragma unroll
            for (int slot = 0; slot < S; ++slot) factor[slot] = scale[slot] * d;
            // The codes go into the product as 4 (q - 32), which is their six bits moved to the
            // top of a byte with the highest one flipped; the sub-scales as sc / 4, so that
            // every product sc * bracket keeps its value (both factors are exact) and every
            // rounding of the one-row kernel's chain happens on the same number.
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                float quarter_scale[8];
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const std::uint32_t biased = sub_scales.v[2 * half + w] ^ 0x80808080u;
#pragma unroll
                    for (int byte = 0; byte < 4; ++byte) {
                        quarter_scale[4 * w + byte] =
                            fmaf(static_cast<float>((biased >> (8 * byte)) & 0xffu), 0.25f, -32.0f);
                    }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const std::uint8_t* at = my_row + half * 64 + s * 16 + h * 8;
                    const RowsHalfPiece low_a = *reinterpret_cast<const RowsHalfPiece*>(at);
                    const RowsHalfPiece low_b = *reinterpret_cast<const RowsHalfPiece*>(at + 32);
                    const RowsHalfPiece top =
                        *reinterpret_cast<const RowsHalfPiece*>(my_row + 128 + half * 32 + s * 16 + h * 8);
                    v2i codes[4];
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        const std::uint32_t a = low_a.v[w], b = low_b.v[w];
                        const std::uint32_t t = top.v[w] ^ 0xaaaaaaaau;
                        codes[0][w] = static_cast<int>(((a << 2) & 0x3c3c3c3cu) | ((t << 6) & 0xc0c0c0c0u));
                        codes[1][w] = static_cast<int>(((b << 2) & 0x3c3c3c3cu) | ((t << 4) & 0xc0c0c0c0u));
                        codes[2][w] = static_cast<int>(((a >> 2) & 0x3c3c3c3cu) | ((t << 2) & 0xc0c0c0c0u));
                        codes[3][w] = static_cast<int>(((b >> 2) & 0x3c3c3c3cu) | (t & 0xc0c0c0c0u));
                    }
                    // quarter after quarter, so that one product's sixteen integers are live
                    float unit_value[S];
#pragma unroll
                    for (int slot = 0; slot < S; ++slot) unit_value[slot] = 0.0f;
                    const auto product = [&](int k) {
                        const v4i both = stage.a[(4 * half + k) / kGroups];
                        const v2i fragment = s == 0 ? v2i{both[0], both[1]} : v2i{both[2], both[3]};
                        return mfma_i8_k16(fragment, codes[k], zero);
                    };
                    const auto tail = [&](int k, const v16i& dots) {
#pragma unroll
                        for (int slot = 0; slot < S; ++slot) {
                            // |4 (256 hi + lo)| <= 4 * 16 * 32 * 32512 < 2^27: exact in int32
                            const int at = (4 * half + k) % kGroups * 2 * S + 2 * slot;
                            const int bracket = (dots[at] << 8) + dots[at + 1];
                            unit_value[slot] =
                                fmaf(quarter_scale[2 * k + s], static_cast<float>(bracket), unit_value[slot]);
                        }
                    };
                    if constexpr (kDeep) {
                        // (the next quarter's product under the tail of this one, as for Q4_K below)
                        v16i dots[2];
                        dots[0] = product(0);
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            if (k < 3) dots[(k + 1) & 1] = product(k + 1);
                            __builtin_amdgcn_sched_barrier(0);
                            tail(k, dots[k & 1]);
                            asm volatile("" : : "v"(dots[k & 1]));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k) tail(k, product(k));
                    }
#pragma unroll
                    for (int slot = 0; slot < S; ++slot) {
                        acc[2 * half + s][slot] = fmaf(factor[slot], unit_value[slot], acc[2 * half + s][slot]);
                    }
                }
            }
            rows_lds_fence();  // the next block's stores stay behind these reads
        } else if constexpr (F::kQ8) {
            // Q8_0: eight blocks of an fp16 scale and 32 int8 codes; the codes are operand B as
            // they lie, this lane's sixteen of each block from byte 34 b + 2 + 16 h
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const std::uint8_t* pair = my_row + 68 * p;
                const RowsPiece c0 = *reinterpret_cast<const RowsPiece*>(pair + 2 + 16 * h);
                const RowsPiece c1 = *reinterpret_cast<const RowsPiece*>(pair + 36 + 16 * h);
                const float d0 = half_bits_to_float(*reinterpret_cast<const std::uint16_t*>(pair));
                const float d1 = half_bits_to_float(*reinterpret_cast<const std::uint16_t*>(pair + 34));
                const v16i dots0 = mfma_i8(stage.a[2 * p / kGroups], v4i{static_cast<int>(c0.v[0]), static_cast<int>(c0.v[1]),
                                                                static_cast<int>(c0.v[2]), static_cast<int>(c0.v[3])}, zero);
                const v16i dots1 = mfma_i8(stage.a[(2 * p + 1) / kGroups], v4i{static_cast<int>(c1.v[0]), static_cast<int>(c1.v[1]),
                                                                    static_cast<int>(c1.v[2]), static_cast<int>(c1.v[3])}, zero);
#pragma unroll
                for (int slot = 0; slot < S; ++slot) {
                    // |256 hi + lo| <= 32 * 127 * 32512 < 2^28: exact in int32
                    const int at0 = 2 * p % kGroups * 2 * S + 2 * slot;
                    const int at1 = (2 * p + 1) % kGroups * 2 * S + 2 * slot;
                    const int bracket0 = (dots0[at0] << 8) + dots0[at0 + 1];
                    const int bracket1 = (dots1[at1] << 8) + dots1[at1 + 1];
                    const float value = fmaf(d1, static_cast<float>(bracket1), d0 * static_cast<float>(bracket0));
                    acc[p][slot] = fmaf(scale[slot], value, acc[p][slot]);
                }
            }
            rows_lds_fence();  // the next block's stores stay behind these reads
        } else {
            // Q4_K / Q5_K: a lane needs the header of row j and its half of the row's codes
            const uint4 head = *reinterpret_cast<const uint4*>(my_row);
            uint4 high = make_uint4(0, 0, 0, 0);
            if constexpr (kQ5) high = *reinterpret_cast<const uint4*>(my_row + 16 + h * 16);
            uint4 quants[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                quants[p] = *reinterpret_cast<const uint4*>(my_row + kQuants + p * 32 + h * 16);
            }
            rows_lds_fence();  // the next block's stores stay behind these reads
            // 6-bit scales and minimums of the eight sub-blocks, four per word
            const std::uint32_t sc_lo = head.y & 0x3f3f3f3fu;
            const std::uint32_t mn_lo = head.z & 0x3f3f3f3fu;
            const std::uint32_t sc_hi = (head.w & 0x0f0f0f0fu) | ((head.y >> 2) & 0x30303030u);
            const std::uint32_t mn_hi = ((head.w >> 4) & 0x0f0f0f0fu) | ((head.z >> 2) & 0x30303030u);
            const float d = half_bits_to_float(head.x & 0xffffu);
            const float dmin = half_bits_to_float(head.x >> 16);
            // the codes of pair p (sub-blocks 2p and 2p + 1), this lane's sixteen of each
            const auto unpack = [&](int p, v4i& low, v4i& upper) {
                const std::uint32_t packed[4] = {quants[p].x, quants[p].y, quants[p].z, quants[p].w};
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    std::uint32_t lo = packed[w] & 0x0f0f0f0fu;
                    std::uint32_t up = (packed[w] >> 4) & 0x0f0f0f0fu;
                    if constexpr (kQ5) {
                        const std::uint32_t bits[4] = {high.x, high.y, high.z, high.w};
                        const std::uint32_t shifted = bits[w] >> (2 * p);
                        lo |= (shifted & 0x01010101u) << 4;
                        up |= (shifted & 0x02020202u) << 3;
                    }
                    low[w] = static_cast<int>(lo);
                    upper[w] = static_cast<int>(up);
                }
            };
            // the float tail of pair p for the token slots first..last-1 (min_dots: the products with
            // the minimums, for more than eight tokens; fewer take the code sums of the records)
            const auto tail = [&](int p, const v16i& dots_a, const v16i& dots_b, const v16i& min_dots, int first,
                                  int last) {
                const std::uint32_t sc_word = p < 2 ? sc_lo : sc_hi;
                const std::uint32_t mn_word = p < 2 ? mn_lo : mn_hi;
                const int scale_a = static_cast<int>((sc_word >> (16 * (p & 1))) & 0xffu);
                const int scale_b = static_cast<int>((sc_word >> (16 * (p & 1) + 8)) & 0xffu);
                const int min_a = static_cast<int>((mn_word >> (16 * (p & 1))) & 0xffu);
                const int min_b = static_cast<int>((mn_word >> (16 * (p & 1) + 8)) & 0xffu);
                // the sub-block scales times 256, opaque to the optimizer: it would otherwise factor
                // scale * (256 * hi + lo) out and pay a full 32-bit multiplication for it
                int scale_a256, scale_b256;
                asm("v_lshlrev_b32 %0, 8, %1" : "=v"(scale_a256) : "v"(scale_a));
                asm("v_lshlrev_b32 %0, 8, %1" : "=v"(scale_b256) : "v"(scale_b));
#pragma unroll
                for (int slot = first; slot < last; slot += 2) {
                    // (sums of both sub-blocks for two tokens)
                    v4i sums = {0, 0, 0, 0};
                    if constexpr (kSums) sums = *reinterpret_cast<const v4i*>(my_extras + p * kTokens + S * h + slot);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const int at = slot + t;
                        const int in_a = 2 * p % kGroups * 2 * S + 2 * at;
                        const int in_b = (2 * p + 1) % kGroups * 2 * S + 2 * at;
                        float codes;
                        if constexpr (kQ5) {
                            const int weighted_hi =
                                __mul24(scale_a, dots_a[in_a]) + __mul24(scale_b, dots_b[in_b]);
                            const int weighted_lo =
                                __mul24(scale_a, dots_a[in_a + 1]) + __mul24(scale_b, dots_b[in_b + 1]);
                            codes = fmaf(static_cast<float>(weighted_hi), 256.0f, static_cast<float>(weighted_lo));
                        } else {
                            // 4-bit codes: 256 * weighted_hi + weighted_lo stays below 2^31
                            // (2 * 63 * 32 * 15 * (127 * 256 + 128)), and one conversion rounds the
                            // exact integer as the fused multiply-add of the two exact floats does
                            // (a chain of multiply-adds: the empty statements keep the optimizer from
                            // turning it into a tree with one more instruction)
                            int weighted = __mul24(scale_a256, dots_a[in_a]);
                            asm("" : "+v"(weighted));
                            weighted += __mul24(scale_b256, dots_b[in_b]);
                            asm("" : "+v"(weighted));
                            weighted += __mul24(scale_a, dots_a[in_a + 1]);
                            asm("" : "+v"(weighted));
                            weighted += __mul24(scale_b, dots_b[in_b + 1]);
                            codes = static_cast<float>(weighted);
                        }
                        int weighted_min;
                        if constexpr (kSums) {
                            // (a group's sum of codes stays below 32 * 32,512 < 2^23)
                            weighted_min = __mul24(min_a, sums[2 * t]);
                            asm("" : "+v"(weighted_min));
                            weighted_min += __mul24(min_b, sums[2 * t + 1]);
                        } else {
                            weighted_min = min_dots[2 * at] * 256 + min_dots[2 * at + 1];
                        }
                        const float value = fmaf(-dmin, static_cast<float>(weighted_min), d * codes);
                        acc[p][at] = fmaf(scale[at], value, acc[p][at]);
                    }
                }
            };
            if constexpr (!kSums) {
                // min_a * sum(codes of a) + min_b * sum(codes of b) per plane as products with the
                // minimums spread over K: more than eight tokens leave no registers for the code sums
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    v4i low, upper;
                    unpack(p, low, upper);
                    const std::uint32_t mn_word = p < 2 ? mn_lo : mn_hi;
                    const int min_a = static_cast<int>((mn_word >> (16 * (p & 1))) & 0xffu);
                    const int min_b = static_cast<int>((mn_word >> (16 * (p & 1) + 8)) & 0xffu);
                    const int spread_a = static_cast<int>(__umul24(min_a, 0x010101u)) | (min_a << 24);
                    const int spread_b = static_cast<int>(__umul24(min_b, 0x010101u)) | (min_b << 24);
                    const v4i mins_a = {spread_a, spread_a, spread_a, spread_a};
                    const v4i mins_b = {spread_b, spread_b, spread_b, spread_b};
                    const v16i dots_a = mfma_i8(stage.a[2 * p], low, zero);
                    const v16i dots_b = mfma_i8(stage.a[2 * p + 1], upper, zero);
                    const v16i min_dots = mfma_i8(stage.a[2 * p + 1], mins_b, mfma_i8(stage.a[2 * p], mins_a, zero));
                    tail(p, dots_a, dots_b, min_dots, 0, S);
                }
            } else {
                // The products of pair p + 1 are issued around the tail of pair p, into a second set of
                // result registers that stay whole until their tail has read them (the unused part of
                // a result handed to another value would make its writer wait for the product).
                constexpr int kHalf = S == 2 ? 2 : S / 2;
                v16i dots_a[2], dots_b[2];
                {
                    v4i low, upper;
                    unpack(0, low, upper);
                    dots_a[0] = mfma_i8(stage.a[0], low, zero);
                    dots_b[0] = mfma_i8(stage.a[1 / kGroups], upper, zero);
                }
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    v4i low, upper;
                    if (p < 3) {
                        unpack(p + 1, low, upper);
                        dots_a[(p + 1) & 1] = mfma_i8(stage.a[(2 * p + 2) / kGroups], low, zero);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    tail(p, dots_a[p & 1], dots_b[p & 1], zero, 0, kHalf);
                    __builtin_amdgcn_sched_barrier(0);
                    if (p < 3) dots_b[(p + 1) & 1] = mfma_i8(stage.a[(2 * p + 3) / kGroups], upper, zero);
                    __builtin_amdgcn_sched_barrier(0);
                    tail(p, dots_a[p & 1], dots_b[p & 1], zero, kHalf, S);
                    asm volatile("" : : "v"(dots_a[p & 1]), "v"(dots_b[p & 1]));
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            rows_lds_fence();  // the next block's entries stay behind these reads
        }
    };
    // a class is complete: (c0 + c1) + (c2 + c3) per token goes to LDS
    int work = 0;  // of the workgroup's tiles
    auto finish_class = [&](int cls) {
#pragma unroll
        for (int slot = 0; slot < S; ++slot) {
            class_sums[work % kTilesHeld][cls & (kOwnClasses - 1)][S * h + slot][j] =
                (acc[0][slot] + acc[1][slot]) + (acc[2][slot] + acc[3][slot]);
#pragma unroll
            for (int p = 0; p < 4; ++p) acc[p][slot] = 0.0f;
        }
    };
    // ... after all waves' have gone there, a thread per (token, row) adds the 16 classes of a tile in
    // the order of the one-row kernel's butterfly
    const int token = static_cast<int>(threadIdx.x) >> 5;
    auto add_classes = [&](int index) {
        const std::uint32_t tile = first_tile + static_cast<std::uint32_t>(index) * tile_stride;
        const Projection op = projection_of(tile);
        const std::int64_t row0 = static_cast<std::int64_t>(tile - op.first_tile) * rows_a_tile;
        const int valid_rows =
            static_cast<int>(min(static_cast<std::int64_t>(rows_a_tile), op.output_dim - row0));
        if (token < kTokens && token < tokens && j < valid_rows) {
            const auto& sums = class_sums[index % kTilesHeld];
            float pairs[kOwnClasses / 2];
#pragma unroll
            for (int m = 0; m < kOwnClasses / 2; ++m) pairs[m] = sums[2 * m][token][j] + sums[2 * m + 1][token][j];
            float* output = op.output + (static_cast<std::int64_t>(token) * op.output_dim + row0 + j);
            if constexpr (SPLIT) {
                // this half of the butterfly; the other workgroup's joins it in either order
                // (a compare-and-swap loop: the sum is a vector-ALU addition like every other)
                const float mine = (pairs[0] + pairs[1]) + (pairs[2] + pairs[3]);
                unsigned int* word = reinterpret_cast<unsigned int*>(output);
                unsigned int seen = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                while (true) {
                    const unsigned int wanted = __float_as_uint(__uint_as_float(seen) + mine);
                    if (__hip_atomic_compare_exchange_strong(word, &seen, wanted, __ATOMIC_RELAXED,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                        break;
                    }
                }
            } else {
                const float q0 = pairs[0] + pairs[1];
                const float q1 = pairs[2] + pairs[3];
                const float q2 = pairs[4] + pairs[5];
                const float q3 = pairs[6] + pairs[7];
                *output = (q0 + q1) + (q2 + q3);
            }
        }
    };
    // (behind what it announces: LDS takes a wave's operations in the order that the fences keep)
    const auto say = [&](int what, int count) {
        rows_lds_fence();
        __hip_atomic_store(&said[what][wave][lane], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        rows_lds_fence();
    };
    // A tile's waves do not meet: each says how many tiles it has left the sums of and how many it has
    // added its part of, adds a tile's when it has finished the next one, and waits only for what it
    // needs (a wave never waits for one that can wait for it: what is waited for lies a tile or more
    // behind).  The last tile's meet at a barrier.
    const auto finish_tile = [&]() {
        if constexpr (kDeep) {
            if (my_tiles > 1) say(0, work + 1);
            if (work > 0) {
                if (wave * 2 < tokens) {
                    wait_for_all(0, work);
                    add_classes(work - 1);
                }
                say(1, work);
            }
        }
        if (!kDeep || work + 1 == my_tiles) {
            __syncthreads();
            add_classes(work);
        }
        ++work;
    };
    // before the first class of a tile: its place was that of the tile kTilesHeld before
    const auto begin_sums = [&]() {
        if (kDeep && work >= kTilesHeld) wait_for_all(1, work - kTilesHeld + 1);
    };

    if (role.total == 0) {
        // (rows of fewer blocks than classes: this wave only takes part in the sums)
        for (int n = 0; n < my_tiles; ++n) {
            begin_sums();
            finish_class(role.class0);
            if constexpr (!SPLIT) finish_class(role.class1);
            finish_tile();
        }
        return;
    }
    // One set of registers for the packed bytes (up to eight tokens two), two for the operands, all
    // named (an array of them indexed in the loop ends up in scratch memory).  A block's loads are
    // requested when the block before it (two before it) has gone to LDS, so one block's
    // arithmetic (two blocks') covers them.  Past the end of the walk a request repeats the last
    // block, so that the number of loads in flight is the same on every path.
    RowsPacked<ENC> packed_even, packed_odd;
    RowsOperands<S> even, odd;
    fetch_packed(packed_even);
    fetch_operands(even, block_of(role, 0));
    if constexpr (kDeep) {
        fetch_packed(packed_odd);
    } else {
        // (requested behind the first block's loads, so that nothing waits for them alone)
        for (int index = lane; index < role.total * kTokens; index += kWave) {
            const int block = block_of(role, index / kTokens);
            step_scales[wave][index / kTokens][index % kTokens] = reinterpret_cast<const float*>(
                image + static_cast<std::int64_t>(block) * kImageBlock + kImageFragments)[index % kTokens];
        }
    }
    int work_step = 0;
    // (class0 = r has at least as many blocks as class1 = 15 - r; a class without blocks leaves
    // the zeros the sums start from)
    auto finish_step = [&]() {
        if (work_step == role.count0 - 1) {
            begin_sums();
            finish_class(role.class0);
        }
        if (work_step == role.total - 1) {
            if constexpr (!SPLIT) finish_class(role.class1);
            finish_tile();
            work_step = 0;
            if constexpr (kDeep) role = role_of((role.class0 + role_step) & (kRowsWaves - 1));
        } else {
            ++work_step;
        }
    };
    // the block after the one being worked on (past the end of the walk: any)
    auto next_block = [&]() {
        if (work_step < role.total - 1) return block_of(role, work_step + 1);
        if constexpr (!kDeep) return role.class0;
        return (SPLIT && right_half ? 8 : 0) + ((role.class0 + role_step) & (kRowsWaves - 1));
    };
    // one step of the walk: its packed bytes go to LDS, the operands of the next step and the packed
    // bytes of the one after that are requested (`last`: nothing is left to request), its products are
    // taken
    auto take_step = [&](RowsPacked<ENC>& packed, const RowsOperands<S>& here, RowsOperands<S>& next, auto last) {
        stage_to_lds(packed);
        if constexpr (kDeep) {
            if (lane < kEntries) my_extras[extra_entry] = here.extra;
        }
        rows_lds_fence();
        if constexpr (!last) {
            // (in the order in which they are waited for)
            if constexpr (!kDeep) fetch_packed(packed);
            fetch_operands(next, next_block());
            if constexpr (kDeep) fetch_packed(packed);
        }
        compute(here, work_step);
        finish_step();
    };
    // (a loop of whole pairs with one exit at its end, so that the number of loads in flight is the
    // same wherever a wait counts them)
    int steps = 0;
#pragma unroll
    for (int n = 0; n < 4; ++n) {  // (r comes round after four tiles)
        steps += role_of((wave + n * role_step) & (kRowsWaves - 1)).total * ((my_tiles - n + 3) >> 2);
    }
    if constexpr (kDeep) {
        if (steps >= 2) {
            do {
                take_step(packed_even, even, odd, std::false_type{});
                take_step(packed_odd, odd, even, std::false_type{});
                steps -= 2;
            } while (steps >= 2);
        }
        if (steps != 0) {
            // (a loop of one that the optimizer cannot see through, for the one form that would keep
            // registers in scratch without it: eight of Q6_K's split form, five to eight tokens)
            int once = 1;
            if constexpr (F::kQ6 && SPLIT && S == 4) asm volatile("" : "+s"(once));
            do {
                take_step(packed_even, even, odd, std::true_type{});
            } while (--once > 0);
        }
    } else {
        // (nothing is in flight behind the packed bytes that a step waits for; a third copy of
        // the step spills)
        while (true) {
            take_step(packed_even, even, odd, std::false_type{});
            if (--steps == 0) break;
            take_step(packed_even, odd, even, std::false_type{});
            if (--steps == 0) break;
        }
    }
}

std::uint32_t tiles_of(const ProjectionSet& set) {
    std::uint32_t tiles = 0;
    for (int index = 0; index < set.count; ++index) {
        tiles += static_cast<std::uint32_t>((set.op[index].output_dim + kRowsTile - 1) / kRowsTile);
    }
    return tiles;
}

// How a launch of `tiles` tiles of rows of `blocks` blocks is shared out.  Costs in half blocks that
// the slowest SIMD works through (two of a workgroup's eight waves to a SIMD, waves w and w + 4): of
// a whole tile wave w takes the classes w and 15 - w, of a half the class w (left) or 8 + w
// (right).  Up to eight tokens the shares move on by two waves with every tile (rows of 16 blocks and
// more), so a SIMD alternates between its share and that of the SIMD two further.  A block and a half
// per tile or half for its first loads and its stores, and more than eight tokens' barrier (measured:
// 1.1 us a block, 1.6 us a tile at 16 tokens).
struct RowsPlan {
    bool split;
    std::uint32_t left_groups;   // split: workgroups on the left halves
    std::uint32_t groups;        // workgroups of the launch
};

// fill_launch: the outputs are filled by a launch of its own (a prequantized call has no
// quantizer launch to do it), which the split form must win back as well (two blocks' time, up to
// eight tokens two and a half).
// Up to eight tokens the split form is taken wherever it costs no more (equal costs of one tile a
// workgroup are those of rows of up to eight blocks, whose right halves are empty: whole).  64 to 1,024 tiles of 2,048
// to 16,384 columns, the four formats, four and seven tokens, 800 calls of either form: the rule takes
// 0.2 % longer than the faster form on average, 7 % at most (prequantized 0.3 and 15; with fixed
// shares and a tenth asked for, as for more tokens, 1.5 and 16, prequantized 1.5 and 24).  264 tiles of
// 4,096 columns, Q6_K, seven tokens: whole 23.9 us, split 20.9; 256 of 6,656, Q8_0, four: 18.3 and 20.2.
RowsPlan plan_rows(std::uint32_t tiles, std::int64_t input_dim, std::int64_t tokens, bool may_split, bool fill_launch) {
    const std::uint32_t units = static_cast<std::uint32_t>(compute_units());
    const int blocks = static_cast<int>(input_dim >> 8);
    const bool few = tokens <= 8;
    const bool moves = few && blocks >= kClasses;
    const auto count = [blocks](int cls) { return cls < blocks ? (blocks - cls + kClasses - 1) / kClasses : 0; };
    int whole[4], left[4], right[4];
    for (int simd = 0; simd < 4; ++simd) {
        left[simd] = count(simd) + count(simd + 4);
        right[simd] = count(8 + simd) + count(12 + simd);
        whole[simd] = left[simd] + count(kClasses - 1 - simd) + count(kClasses - 1 - (simd + 4));
    }
    // a workgroup's walk over its share of the tiles, by the blocks of a SIMD
    const auto cost = [&](const int (&share)[4], std::uint32_t groups) {
        const std::uint64_t walk = (tiles + groups - 1) / groups, turned = moves ? walk / 2 : 0;
        std::uint64_t worst = 0;
        for (int simd = 0; simd < 4; ++simd) {
            const std::uint64_t here = (walk - turned) * share[simd] + turned * share[simd ^ 2];
            worst = here > worst ? here : worst;
        }
        return 2 * worst + 3 * walk;
    };
    RowsPlan plan{false, 0, tiles < units ? tiles : units};
    if (!may_split || units < 2) return plan;
    const std::uint64_t whole_cost = cost(whole, plan.groups);
    // The costlier side is least where the two sides cross (with more workgroups on the left the left
    // costs no more and the right no less); of equal ones the first.  By bisection: costing all 255
    // ways, twice a call, takes 2.5 us of the host each, this 0.14 (submitting a call of seven rows of
    // 6,656 columns 9.7 -> 7.3 us).
    const auto fewer = [tiles](std::uint32_t groups) { return groups < tiles ? groups : tiles; };
    const auto left_of = [&](std::uint32_t groups) { return cost(left, fewer(groups)); };
    const auto right_of = [&](std::uint32_t groups) { return cost(right, fewer(units - groups)); };
    const auto first_where = [units](const auto& holds) {  // 1..units - 1; units: nowhere
        std::uint32_t low = 1, high = units;
        while (low < high) {
            const std::uint32_t middle = (low + high) / 2;
            if (holds(middle)) {
                high = middle;
            } else {
                low = middle + 1;
            }
        }
        return low;
    };
    const std::uint32_t crossing = first_where([&](std::uint32_t groups) { return left_of(groups) <= right_of(groups); });
    std::uint64_t best = ~std::uint64_t(0);
    if (crossing < units) best = right_of(crossing);
    if (crossing > 1) best = std::min(best, left_of(crossing - 1));
    const std::uint32_t left_groups = first_where([&](std::uint32_t groups) { return left_of(groups) <= best; });
    const std::uint32_t best_left = fewer(left_groups), best_right = fewer(units - left_groups);
    if (fill_launch) best += few ? 5 : 4;
    // (more than eight tokens: the split form has to win by a tenth, the model is that coarse)
    if (few ? best < whole_cost || (best == whole_cost && tiles > units) : best * 10 <= whole_cost * 9) {
        plan.split = true;
        plan.left_groups = best_left;
        plan.groups = best_left + best_right;
    }
    return plan;
}

// Rows of a tile of the whole form: the fewest that send no workgroup round once more, so that 6,656 rows are 256 tiles of
// 26 and not 208 of 32.  us, seven tokens, 32 rows -> fewer: 16,384 -> 6,656 Q4_K 26.2 -> 24.2, Q5_K 28.0 -> 26.7, Q8_0 32.8 ->
// 31.0; 4,608 -> 4,608 Q4_K 11.6 -> 11.0.  1,700 calls of 5 to 16 tokens, geometric means: several tiles a workgroup 1.015 of
// all formats (the slowest 2 % longer), one of sixteen rows and more 1.02 of Q4_K and Q5_K, 1.03 of Q8_0; of fewer rows
// 1.00, and of Q6_K 0.99, down to 0.95: whole tiles.
int rows_of_tile(std::uint32_t encoding, const ProjectionSet& set) {
    const EvenTiles even = even_tiles(set, set.count, kRowsTile, 4);
    if (even.each > 6 || (even.each == 1 && (even.rows < 16 || encoding == kEncQ6K))) return kRowsTile;
    return even.rows;
}

template <std::uint32_t ENC, bool SPLIT>
void launch_form(const ProjectionSet& set, const std::uint8_t* image, const std::uint8_t* records,
                 int tokens, std::uint32_t tiles, int rows_a_tile, const RowsPlan& plan, hipStream_t stream) {
    const dim3 grid(plan.groups), block(kRowsThreads);
    const int input_dim = static_cast<int>(set.input_dim);
    if (tokens <= 4) {
        hipLaunchKernelGGL((gemv_rows_kernel<ENC, 2, SPLIT>), grid, block, 0, stream, image, records, tokens,
                           input_dim, tiles, plan.left_groups, rows_a_tile, set);
    } else if (tokens <= 8) {
        hipLaunchKernelGGL((gemv_rows_kernel<ENC, 4, SPLIT>), grid, block, 0, stream, image, records, tokens,
                           input_dim, tiles, plan.left_groups, rows_a_tile, set);
    } else {
        hipLaunchKernelGGL((gemv_rows_kernel<ENC, 8, SPLIT>), grid, block, 0, stream, image, records, tokens,
                           input_dim, tiles, plan.left_groups, rows_a_tile, set);
    }
}

template <std::uint32_t ENC>
void launch_encoding(ProjectionSet set, const std::uint8_t* image, const std::uint8_t* records,
                     int tokens, bool outputs_cleared, bool fill_launch, hipStream_t stream) {
    std::uint32_t tiles = 0;
    for (int index = 0; index < set.count; ++index) {
        set.op[index].first_tile = tiles;
        tiles += static_cast<std::uint32_t>((set.op[index].output_dim + kRowsTile - 1) / kRowsTile);
    }
    RowsPlan plan = plan_rows(tiles, set.input_dim, tokens, outputs_cleared, fill_launch);
    int rows = kRowsTile;
    if (!plan.split) {
        rows = rows_of_tile(ENC, set);
        tiles = 0;
        for (int index = 0; index < set.count; ++index) {
            set.op[index].first_tile = tiles;
            tiles += static_cast<std::uint32_t>((set.op[index].output_dim + rows - 1) / rows);
        }
        const std::uint32_t units = static_cast<std::uint32_t>(compute_units());
        plan.groups = tiles < units ? tiles : units;
    }
    if (plan.split) {
        launch_form<ENC, true>(set, image, records, tokens, tiles, rows, plan, stream);
    } else {
        launch_form<ENC, false>(set, image, records, tokens, tiles, rows, plan, stream);
    }
}

// the projections of one encoding, in the order of the set
ProjectionSet encoding_group(const ProjectionSet& set, std::uint32_t encoding) {
    ProjectionSet group{};
    group.input_dim = set.input_dim;
    for (int index = 0; index < set.count; ++index) {
        if (set.op[index].encoding == encoding) group.op[group.count++] = set.op[index];
    }
    return group;
}

constexpr std::uint32_t kRowsEncodings[4] = {kEncQ4K, kEncQ5K, kEncQ6K, kEncQ8_0};

}  // namespace

bool gemv_rows_supports(std::uint32_t encoding, std::int64_t input_dim) {
    return (encoding == kEncQ4K || encoding == kEncQ5K || encoding == kEncQ6K || encoding == kEncQ8_0) &&
        input_dim % 256 == 0 && input_dim <= kMaxRowsBlocks * 256;
}

std::int64_t gemv_rows_image_bytes(std::int64_t input_dim) {
    return (input_dim >> 8) * kImageBlock;
}

ProjectionSet gemv_rows_split_set(const ProjectionSet& set, std::int64_t rows, bool fill_launch) {
    ProjectionSet split{};
    split.input_dim = set.input_dim;
    for (const std::uint32_t encoding : kRowsEncodings) {
        const ProjectionSet group = encoding_group(set, encoding);
        if (group.count == 0 || !plan_rows(tiles_of(group), set.input_dim, rows, true, fill_launch).split) continue;
        for (int index = 0; index < group.count; ++index) split.op[split.count++] = group.op[index];
    }
    return split;
}

void launch_quantize_records(const float* first, const float* second, int prologue,
                             std::int64_t rows, std::int64_t input_dim, std::uint8_t* records,
                             std::uint8_t* image, const ProjectionSet& clear, hipStream_t stream) {
    const int blocks = static_cast<int>(input_dim >> 8);
    const int tokens = static_cast<int>(rows);
    const int record_groups = (blocks * tokens + 3) / 4;
    std::int64_t fill_groups = 0;
    for (int index = 0; index < clear.count; ++index) {
        fill_groups += (clear.op[index].output_dim * rows + 1023) >> 10;
    }
    const dim3 grid(static_cast<unsigned>(record_groups + fill_groups)), block(256);
    switch (prologue) {
        case kGated:
            hipLaunchKernelGGL((quantize_records_kernel<kGated>), grid, block, 0, stream, first,
                               second, records, image, blocks, tokens, record_groups, clear);
            break;
        case kSwiGlu:
            hipLaunchKernelGGL((quantize_records_kernel<kSwiGlu>), grid, block, 0, stream, first,
                               second, records, image, blocks, tokens, record_groups, clear);
            break;
        default:
            hipLaunchKernelGGL((quantize_records_kernel<kPlain>), grid, block, 0, stream, first,
                               second, records, image, blocks, tokens, record_groups, clear);
            break;
    }
}

void launch_fill_outputs(const ProjectionSet& clear, std::int64_t rows, hipStream_t stream) {
    std::int64_t fill_groups = 0;
    for (int index = 0; index < clear.count; ++index) {
        fill_groups += (clear.op[index].output_dim * rows + 1023) >> 10;
    }
    if (fill_groups == 0) return;
    // (the quantizer kernel with no records to write)
    hipLaunchKernelGGL((quantize_records_kernel<kPlain>), dim3(static_cast<unsigned>(fill_groups)),
                       dim3(256), 0, stream, static_cast<const float*>(nullptr),
                       static_cast<const float*>(nullptr), static_cast<std::uint8_t*>(nullptr),
                       static_cast<std::uint8_t*>(nullptr), 0, static_cast<int>(rows), 0, clear);
}

void launch_gemv_rows(const ProjectionSet& set, const std::uint8_t* image,
                      const std::uint8_t* records, std::int64_t rows,
                      bool outputs_cleared, bool fill_launch, hipStream_t stream) {
    for (const std::uint32_t encoding : kRowsEncodings) {
        const ProjectionSet group = encoding_group(set, encoding);
        if (group.count == 0) continue;
        const int tokens = static_cast<int>(rows);
        switch (encoding) {
            case kEncQ4K: launch_encoding<kEncQ4K>(group, image, records, tokens, outputs_cleared, fill_launch, stream); break;
            case kEncQ5K: launch_encoding<kEncQ5K>(group, image, records, tokens, outputs_cleared, fill_launch, stream); break;
            case kEncQ6K: launch_encoding<kEncQ6K>(group, image, records, tokens, outputs_cleared, fill_launch, stream); break;
            default: launch_encoding<kEncQ8_0>(group, image, records, tokens, outputs_cleared, fill_launch, stream); break;
        }
    }
}

}  // namespace nfn
