// One query row, or each row of a causal block, on the matrix cores (head_dim 128, four and more query
// heads per key/value head): the one-token attention of the decode loop, alone or with the per-head norms,
// the rotation and the cache commit before it, and the verifier's block attention where a row's share of
// the keys is short (semantics: neuralfn/csrc/native_train/tile_ops.h:308-339, 445-486, 905-943).
//
// One workgroup of eight waves per (query row, key/value head, group of up to 16 of its query heads, share
// of the keys).  All query heads of a group read a key/value row once.
//
// What bounds it is the number of instructions a wave issues one after the other (2 to 3 ns each for a
// wave that is alone on its SIMD) behind one round of requests, not memory: a 2,048-key window of two
// key/value heads is 2 MB.  So everything is dealt out over the waves, the 128 keys of a step twice:
//   query         wave w prepares the heads 2w and 2w + 1 and cuts them for the matrix cores,
//   scores        wave w takes keys 16w .. 16w + 15 against all 128 dimensions,
//   weighted sum  wave w takes dimensions 16w .. 16w + 15 of all 128 keys,
// with the query, the weights and the value rows changing waves through LDS in between.  The sums of a
// wave are then final: nothing is left to be added across waves at the end.  The requests for keys and
// values are out before the query arrives, and what they need (addresses, counts) comes in the kernel's
// first arguments, which are in registers at wave start.
//
// Lane = (j, i) = (lane / 16, lane % 16).  Both products run on v_mfma_f32_16x16x32_bf16 with float
// operands cut into three bf16 terms whose sum is the float, so that every product is exact (cache rows
// are bf16 already).
//
// Scores of 16 keys x 16 heads: operand A is the cached key as it lies in memory (lane (j, i): key i,
// dimensions 32s + 8j .. + 7), operand B the query of head i.  The result leaves lane (j, i) with keys
// 4j .. 4j + 3 of head i.
//
// Weighted sum over 32 keys at a time: operand A is the values (lane (j, i): dimension 16w + i of keys
// 8j .. 8j + 7, a column of the cache, which the transposing LDS read hands out four keys at a time),
// operand B the weights of head i for the same eight keys.  The result leaves lane (j, i) with dimensions
// 16w + 4j .. + 3 of head i, the head whose maximum and denominator the lane keeps: rescaling and the
// final division need no exchange.
//
// Before, waves walked 64-key tiles of their own, cut the whole query each, took the tile at the end of the ring and
// the last one a load behind the other (4.4 of 13 us), and met in LDS at the end (2.3 us); norms and rotation were a launch of
// 4.2 us.  Attention with its merge, us: 32 heads over 2, 2,048 keys 11.3 -> 8.3, 100 keys 8.4 -> 5.1, 32,768 18.3 -> 16.1; 48
// over 8, 772 keys 11.5 -> 8.3.  With the norms, rotation and commit: 15.1 -> 10.9, 12.0 -> 7.6, 21.7 -> 17.3 and, 607 keys of
// 48 over 4 without the rotation, 14.2 -> 9.0; a decode step of eight layers of 2,048 keys 722.6 -> 664.8.
#include "attention.hpp"

#include "common.hpp"
#include "kernels.hpp"
#include "wave_rows.hpp"

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace nfn {

namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int kRowWaves = 8;
constexpr int kWaveKeys = 16;  // keys a wave scores in a step
constexpr int kStepKeys = kRowWaves * kWaveKeys;
constexpr int kLoadsDone = 0x0f70;  // s_waitcnt: no load in flight
constexpr int kWaveHeads = kGroupHeads / kRowWaves;
constexpr std::int64_t kMostKeys = std::int64_t(1) << 30;  // of a ring or a call: sums of two fit 32 bits
static_assert(kGroupHeadDim == 16 * kRowWaves && kGroupHeadDim == 2 * kWave, "dimensions of a wave and a lane");

// Arguments that are needed once the first requests are out.
struct RowTail {
    const float* block_key;
    const float* block_value;
    std::int64_t block_stride;  // floats from a row of the block to the next
    float* output;
    float* partials;
    const std::int64_t* device_position;
    std::int64_t position;
    std::int64_t sliding_window;
    int whole_context;
    float* key_copy;  // where the prepared key goes (in place where no other workgroup reads it)
    RowPreparation preparation;
};

// What the lower two terms of a float contribute to its products with a bf16.  Where that is infinite and a lower term 0 the
// contribution is NaN and the upper term's product, an infinity, says it all; NaN for any other reason is in both.
__device__ __forceinline__ float finite_part(float lower) { return __builtin_amdgcn_fmed3f(lower, -FLT_MAX, FLT_MAX); }

// the four lanes (., i) of a wave meet
__device__ __forceinline__ float across_j_max(float value) {
    auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    value = fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    rows = __builtin_amdgcn_permlane32_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    return fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
}
__device__ __forceinline__ float across_j_sum(float value) {
    auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    value = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    rows = __builtin_amdgcn_permlane32_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
}

// The wave's sum as a halving tree (lane l and l + 32, then + 16, ...), in every lane: the bits of rms_tree_total's
// last six levels, since after a level both of its lanes hold the same number and addition is commutative.
__device__ __forceinline__ float tree_total(float value) {
    auto rows = __builtin_amdgcn_permlane32_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    value = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    value = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    value += dpp_move<0x128>(value);  // row_ror:8, 4, 2, 1: by now every lane stands for its class
    value += dpp_move<0x124>(value);
    value += dpp_move<0x122>(value);
    value += dpp_move<0x121>(value);
    return value;
}

// A head's columns `lane` and `lane + 64`.
struct HeadPair {
    float first, second;
};

// Columns c and c + 64 of the lanes to 2 c and 2 c + 1, or back, by way of the wave's own 128 floats of LDS.
__device__ __forceinline__ void turn_columns(float& first, float& second, int lane, bool back, float* exchange) {
    const auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    exchange[back ? 2 * lane : lane] = first;
    exchange[back ? 2 * lane + 1 : lane + kWave] = second;
    wave_sync();
    first = exchange[back ? lane : 2 * lane];
    second = exchange[back ? lane + kWave : 2 * lane + 1];
    wave_sync();
}

// The norm, scale and rotation of one head, operation for operation qk_norm_scale_rope_kernel's (rms.hip).
// `exchange`: 128 floats of LDS of this wave alone, used where a pair is two neighbouring columns.
__device__ __forceinline__ HeadPair prepare_head(HeadPair raw, const float (&scale)[2], bool scaled, float query_scale,
                                                 const RowPreparation& how, const RopeAngle& angle, int lane,
                                                 float* exchange) {
    const float squares = fmaf(raw.first, raw.first, 0.0f) + fmaf(raw.second, raw.second, 0.0f);
    const float inverse = 1.0f / sqrtf(tree_total(squares) / static_cast<float>(kGroupHeadDim) + how.eps);
    float a = __fmul_rn(__fmul_rn(raw.first, inverse), scale[0]);
    float b = __fmul_rn(__fmul_rn(raw.second, inverse), scale[1]);
    if (scaled) {
        a = __fmul_rn(a, query_scale);
        b = __fmul_rn(b, query_scale);
    }
    if (!how.apply_rope) return HeadPair{a, b};
    if (how.interleaved) turn_columns(a, b, lane, false, exchange);
    rope_apply(a, b, angle);
    if (how.interleaved) turn_columns(a, b, lane, true, exchange);
    return HeadPair{a, b};
}

// kBlock: several query rows, row r at context + r behind the cache's keys and the block's rows before it, which enter as
// the cache will hold them; `keys` is then the context and `first_slot` the most keys that a row sees before its own.
enum class RowMode { kPlain, kPrepare, kBlock };

// The leading arguments (14 dwords) arrive in registers.  `heads_splits`: query heads per key/value head, and from
// bit 16 on the shares; share_keys = 0: the position is in device memory.  first_slot: ring row of the first of `keys` cached keys.
template <RowMode MODE>
__global__ __launch_bounds__(kRowWaves * kWave) void attention_row_kernel(
    const float* query, const std::uint16_t* key_cache, const std::uint16_t* value_cache, std::uint32_t row_stride,
    std::uint32_t capacity, std::uint32_t first_slot, std::uint32_t keys, std::uint32_t share_keys,
    std::uint32_t heads_splits, std::uint32_t kv_heads, float scale, RowTail tail) {
    constexpr bool PREPARE = MODE == RowMode::kPrepare, BLOCK = MODE == RowMode::kBlock;
    __shared__ __attribute__((aligned(16))) std::uint8_t staged_values[kStepKeys * kStageRowBytes];
    // the weights' terms: [term][wave][head] x sixteen keys
    __shared__ __attribute__((aligned(16))) std::uint8_t staged_weights[3][kRowWaves][kGroupHeads][2 * kWaveKeys];
    __shared__ __attribute__((aligned(16))) float wave_maximum[kGroupHeads][kRowWaves];
    __shared__ __attribute__((aligned(16))) float wave_sum[kGroupHeads][kRowWaves];
    __shared__ float row_score[kGroupHeads];  // of the current key
    // before the first value rows: the query's terms, [term][head] rows of 128 dimensions and a pad
    std::uint8_t* const query_terms = staged_values;
    static_assert(3 * kGroupHeads * kStageRowBytes <= sizeof(staged_values), "the query's terms");
    static_assert(kRowWaves * kGroupHeadDim * sizeof(float) <= sizeof(staged_weights), "a head a wave");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane >> 4;
    const int i = lane & 15;
    const std::uint32_t heads = heads_splits & 0xffffu, splits = heads_splits >> 16;
    const std::uint32_t groups_per_kv = (heads + kGroupHeads - 1) / kGroupHeads;
    const std::uint32_t query_row = BLOCK ? blockIdx.x / (kv_heads * groups_per_kv) : 0;
    const std::uint32_t group = blockIdx.x - query_row * kv_heads * groups_per_kv;
    const std::uint32_t kv_head = groups_per_kv == 1 ? group : group / groups_per_kv;
    const std::uint32_t head_group = group - kv_head * groups_per_kv;
    const int heads_here = static_cast<int>(
        heads - head_group * kGroupHeads < kGroupHeads ? heads - head_group * kGroupHeads : kGroupHeads);
    const std::int64_t first_head = query_row * kv_heads * heads + kv_head * heads + head_group * kGroupHeads;
    const std::int64_t head_offset = static_cast<std::int64_t>(kv_head) * kGroupHeadDim;
    // the current key goes with the last share
    const bool has_row = blockIdx.y + 1 == splits;

    // this wave's query heads
    HeadPair mine[kWaveHeads];
#pragma unroll
    for (int h = 0; h < kWaveHeads; ++h) {
        const int head = kWaveHeads * wave + h;
        const float* row = query + (first_head + (head < heads_here ? head : 0)) * kGroupHeadDim;
        mine[h] = HeadPair{row[lane], row[lane + kWave]};
    }

    std::int64_t position = 0;
    if (share_keys == 0) {
        position = tail.device_position[0];
        std::int64_t first = tail.whole_context != 0 ? 0 : position - tail.sliding_window + 1;
        if (first < 0) first = 0;
        keys = static_cast<std::uint32_t>(position > first ? position - first : 0);
        first_slot = static_cast<std::uint32_t>(
            first < 2 * kMostKeys ? static_cast<std::uint32_t>(first) % capacity
                                  : static_cast<std::uint32_t>(first % static_cast<std::int64_t>(capacity)));
        share_keys = (keys + splits - 1) / splits;
        share_keys = (share_keys + kStepKeys - 1) / kStepKeys * kStepKeys;
        if (share_keys == 0) share_keys = kStepKeys;
    } else if constexpr (PREPARE) {
        position = tail.position;
    }
    [[maybe_unused]] int cached = 0;  // kBlock: keys of the share (later) that lie in the cache
    if constexpr (BLOCK) {
        const std::uint32_t end = keys + query_row;
        const std::uint32_t before = end < first_slot ? end : first_slot;
        cached = static_cast<int>(before) - static_cast<int>(query_row);  // (a window inside the block: negative)
        first_slot = cached > 0 ? (end - before) % capacity : 0;
        keys = before;
    }
    // the share's keys: `here` of them, the first at ring row `slot`
    const std::uint32_t share_begin = blockIdx.y * share_keys < keys ? blockIdx.y * share_keys : keys;
    const int here = static_cast<int>(keys - share_begin < share_keys ? keys - share_begin : share_keys);
    if constexpr (BLOCK) cached -= static_cast<int>(share_begin);
    const auto ring_row = [capacity](std::uint32_t slot) {  // slot < 2 * capacity
        return slot >= capacity ? slot - capacity : slot;
    };
    std::uint32_t slot = first_slot + share_begin;
    if (slot >= capacity) slot = slot < 2 * capacity ? slot - capacity : slot % capacity;
    // this wave's first row (the ring has at least 64 rows) and its way to the next step's
    slot = ring_row(ring_row(slot + wave * kWaveKeys));
    const std::uint32_t slot_step = capacity > kStepKeys ? kStepKeys : ring_row(ring_row(kStepKeys));

    // Requests of the wave's sixteen keys from `begin` of the share, at ring row `at`: key rows as operand A wants
    // them, value rows sixteen lanes to a row (row 4r + j).  Keys past the share repeat its last one and get weight 0;
    // a wave wholly past it requests nothing.
    uint4 key_raw[4], value_raw[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) key_raw[r] = value_raw[r] = make_uint4(0u, 0u, 0u, 0u);
    // (settle: requests of both kinds of row have landed where they end.  The lanes that keep the cache's row need not wait for
    // the block's, but the compiler then takes those loads for possibly in flight in every step and waits for the next
    // step's rows where their registers are used again: 7 rows of 48 heads over 8, 2,048 keys 16.8 -> 14.9 us, 12 of 16 over
    // 4, 4,000 20.4 -> 17.4.  A wave's first requests are waited for soon enough.)
    const auto keys_left = [&](int begin) {  // of the wave's sixteen, wave-uniform
        const int left = here - begin;
        return left < 0 ? 0 : left < kWaveKeys ? left : kWaveKeys;
    };
    const auto request_keys = [&](int begin, std::uint32_t at, [[maybe_unused]] auto settle) {
        const int count = keys_left(begin);
        if (count == 0) return;
        if constexpr (BLOCK) {
            if (begin + count > cached) {
                // every lane requests both kinds of row, so that nothing waits in between
                const int key = i < count ? i : count - 1, in_block = begin + key - cached;
                const bool from_block = in_block >= 0;
                const std::uint32_t row = from_block ? 0 : ring_row(at + key);
                const std::uint16_t* source = key_cache + static_cast<std::uint64_t>(row) * row_stride + head_offset + 8 * j;
                const float* floats = tail.block_key + (from_block ? in_block : 0) * tail.block_stride + head_offset + 8 * j;
                uint4 raw[4];
                float4 low[4], high[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    raw[s] = *reinterpret_cast<const uint4*>(source + 32 * s);
                    low[s] = *reinterpret_cast<const float4*>(floats + 32 * s);
                    high[s] = *reinterpret_cast<const float4*>(floats + 32 * s + 4);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) key_raw[s] = from_block ? pack_as_cached(low[s], high[s]) : raw[s];
                if constexpr (settle()) __builtin_amdgcn_s_waitcnt(kLoadsDone);
                return;
            }
        }
        const std::uint32_t row = ring_row(at + (i < count ? i : count - 1));
        const std::uint16_t* source = key_cache + static_cast<std::uint64_t>(row) * row_stride + head_offset + 8 * j;
#pragma unroll
        for (int s = 0; s < 4; ++s) key_raw[s] = *reinterpret_cast<const uint4*>(source + 32 * s);
    };
    const auto request_values = [&](int begin, std::uint32_t at, [[maybe_unused]] auto settle) {
        const int count = keys_left(begin);
        if (count == 0) return;
        if constexpr (BLOCK) {
            if (begin + count > cached) {
                uint4 raw[4];
                float4 low[4], high[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = 4 * r + j < count ? 4 * r + j : count - 1, in_block = begin + key - cached;
                    const std::uint32_t row = in_block >= 0 ? 0 : ring_row(at + key);
                    const float* floats = tail.block_value + (in_block >= 0 ? in_block : 0) * tail.block_stride + head_offset + 8 * i;
                    raw[r] = *reinterpret_cast<const uint4*>(
                        value_cache + static_cast<std::uint64_t>(row) * row_stride + head_offset + 8 * i);
                    low[r] = *reinterpret_cast<const float4*>(floats);
                    high[r] = *reinterpret_cast<const float4*>(floats + 4);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = 4 * r + j < count ? 4 * r + j : count - 1;
                    value_raw[r] = begin + key >= cached ? pack_as_cached(low[r], high[r]) : raw[r];
                }
                if constexpr (settle()) __builtin_amdgcn_s_waitcnt(kLoadsDone);
                return;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const std::uint32_t row = ring_row(at + (4 * r + j < count ? 4 * r + j : count - 1));
            value_raw[r] = *reinterpret_cast<const uint4*>(
                value_cache + static_cast<std::uint64_t>(row) * row_stride + head_offset + 8 * i);
        }
    };
    request_keys(wave * kWaveKeys, slot, std::false_type());
    request_values(wave * kWaveKeys, slot, std::false_type());

    // the current row's key and, of its value, the dimensions this lane adds up
    HeadPair row_key{0.0f, 0.0f}, row_value{0.0f, 0.0f};
    float4 row_sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (has_row) {
        const std::int64_t own = BLOCK ? query_row * tail.block_stride + head_offset : head_offset;
        const float* key = tail.block_key + own;
        const float* value = tail.block_value + own;
        row_key = HeadPair{key[lane], key[lane + kWave]};
        row_sum = *reinterpret_cast<const float4*>(value + 16 * wave + 4 * j);
        if constexpr (PREPARE) row_value = HeadPair{value[lane], value[lane + kWave]};
    }

    if constexpr (PREPARE) {
        const RowPreparation& how = tail.preparation;
        const int columns[2] = {lane, lane + kWave};
        float query_scales[2], key_scales[2] = {1.0f, 1.0f};
        norm_scales(how.query_weight, columns, query_scales);
        if (has_row) norm_scales(how.key_weight, columns, key_scales);
        // (the rotation's angle depends on the position alone: worked out while the requests are in flight; the
        // empty asm keeps the compiler from moving it behind the sums)
        RopeAngle angle{0.0, 1.0};
        if (how.apply_rope) {
            angle = rope_angle(position, lane, kGroupHeadDim, how.theta, false);
            asm volatile("" : "+v"(angle.sine), "+v"(angle.cosine));
        }
        float* exchange = reinterpret_cast<float*>(staged_weights) + wave * kGroupHeadDim;
#pragma unroll
        for (int h = 0; h < kWaveHeads; ++h) {
            mine[h] = prepare_head(mine[h], query_scales, true, how.query_scale, how, angle, lane, exchange);
        }
        if (has_row) row_key = prepare_head(row_key, key_scales, false, 1.0f, how, angle, lane, exchange);
        // the first share's workgroup hands the prepared query on: in place where it is alone, else by way of the
        // output rows (the other shares may still have to read the original), from where the merge moves it
        if (blockIdx.y == 0) {
            float* rows = (tail.partials != nullptr ? tail.output : how.query) +
                (first_head + kWaveHeads * wave) * kGroupHeadDim;
#pragma unroll
            for (int h = 0; h < kWaveHeads; ++h) {
                if (kWaveHeads * wave + h < heads_here) {
                    rows[h * kGroupHeadDim + lane] = mine[h].first;
                    rows[h * kGroupHeadDim + lane + kWave] = mine[h].second;
                }
            }
        }
    }
#pragma unroll
    for (int h = 0; h < kWaveHeads; ++h) {
        const int head = kWaveHeads * wave + h;
        if (head >= heads_here) mine[h] = HeadPair{0.0f, 0.0f};  // a head that the group lacks
        std::uint32_t first[3], second[3];
        split_term(mine[h].first, first);
        split_term(mine[h].second, second);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            std::uint8_t* row = query_terms + (t * kGroupHeads + head) * kStageRowBytes;
            *reinterpret_cast<std::uint16_t*>(row + 2 * lane) = static_cast<std::uint16_t>(first[t] >> 16);
            *reinterpret_cast<std::uint16_t*>(row + 2 * (lane + kWave)) = static_cast<std::uint16_t>(second[t] >> 16);
        }
        if (has_row) {
            const float dot = tree_total(fmaf(mine[h].second, row_key.second, mine[h].first * row_key.first));
            if (lane == 0) row_score[head] = dot * scale;
        }
    }
    __syncthreads();
    if constexpr (PREPARE) {  // every wave has read the key
        if (has_row && head_group == 0 && wave == 0) {
            const RowPreparation& how = tail.preparation;
            float* key = tail.key_copy + head_offset;
            key[lane] = row_key.first;
            key[lane + kWave] = row_key.second;
            // (the ring row that the new key takes is none that this call reads; a position below 0, which only device memory
            // can hold, has none)
            if (position >= 0) {
                const std::uint32_t ring = position < 2 * kMostKeys
                    ? static_cast<std::uint32_t>(position) % capacity
                    : static_cast<std::uint32_t>(position % static_cast<std::int64_t>(capacity));
                const std::uint64_t cache_row = static_cast<std::uint64_t>(ring) * row_stride + head_offset;
                how.key_cache[cache_row + lane] = to_bf16(row_key.first);
                how.key_cache[cache_row + lane + kWave] = to_bf16(row_key.second);
                how.value_cache[cache_row + lane] = to_bf16(row_value.first);
                how.value_cache[cache_row + lane + kWave] = to_bf16(row_value.second);
            }
        }
    }

    // operand B of the scores
    bf16x8 terms[3][4];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            terms[t][s] = *reinterpret_cast<const bf16x8*>(
                query_terms + (t * kGroupHeads + i) * kStageRowBytes + 2 * (32 * s + 8 * j));
        }
    }

    // The running maximum and denominator of head i (the same in every wave) and dimensions 16w + 4j + r of its sum
    // start with the current row, of weight 1; NaN for a score of +inf, and 0 for -inf, which leaves NaN only where no
    // other key has a finite score (0 / 0).
    float maximum = -INFINITY;
    float denominator = 0.0f;
    f32x4 accumulator = {0.0f, 0.0f, 0.0f, 0.0f};
    if (has_row) {
        maximum = row_score[i];
        denominator = maximum == -INFINITY ? 0.0f : expf(maximum - maximum);
        accumulator = f32x4{row_sum.x * denominator, row_sum.y * denominator, row_sum.z * denominator,
                            row_sum.w * denominator};
    }
    for (int begin = 0; begin < here; begin += kStepKeys) {
        const int wave_begin = begin + wave * kWaveKeys;
        const int count = keys_left(wave_begin);
        // A chain per term of the query.  Where they meet, the sum is as large as the score and rounds like it; the exponent
        // below takes them one by one on top of the maximum instead, where what is left of a key that matters is small.
        // Against float64, 100 to 2,047 keys: 1.53 to 1.86e-7, attention_grouped_kernel 1.59 to 1.98e-7 (the exponent from
        // the rounded score: 1.64 to 1.98e-7; one chain with the large term last: 1.50 to 1.86e-7, five steps 2 us longer).
        f32x4 chains[3] = {};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int t = 2; t >= 0; --t) {
                chains[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, key_raw[s]), terms[t][s], chains[t], 0, 0, 0);
            }
        }
        // the next step's keys are requested as soon as these have been used
        const std::uint32_t next_slot = ring_row(slot + slot_step);
        const bool more = begin + kStepKeys < here;
        if (more) request_keys(wave_begin + kStepKeys, next_slot, std::true_type());
        float lower[4];  // of the products, the lower terms' part
        float largest = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            lower[r] = finite_part(chains[2][r] + chains[1][r]);
            largest = fmaxf(largest, 4 * j + r < count ? (lower[r] + chains[0][r]) * scale : -INFINITY);
        }
        largest = across_j_max(largest);
        if (j == 0) wave_maximum[i][wave] = largest;
        __syncthreads();  // ... and the query's terms or the last step's weights and values have been read

        const float4 maxima[2] = {*reinterpret_cast<const float4*>(&wave_maximum[i][0]),
                                  *reinterpret_cast<const float4*>(&wave_maximum[i][4])};
        const float next_maximum = fmaxf(
            maximum, fmaxf(fmaxf(fmaxf(maxima[0].x, maxima[0].y), fmaxf(maxima[0].z, maxima[0].w)),
                           fmaxf(fmaxf(maxima[1].x, maxima[1].y), fmaxf(maxima[1].z, maxima[1].w))));
        // (without a finite score so far every weight is 0)
        const float reference = fmaxf(next_maximum, -FLT_MAX);
        const float keep = __expf(maximum - reference);
        maximum = next_maximum;
        float weight[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float exponent = fmaf(lower[r], scale, fmaf(chains[0][r], scale, -reference));
            weight[r] = 4 * j + r < count ? __expf(exponent) : 0.0f;
        }
        const float sum = across_j_sum((weight[0] + weight[1]) + (weight[2] + weight[3]));
        if (j == 0) wave_sum[i][wave] = sum;
        std::uint32_t words[3][2];
        split_terms(weight, words);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            *reinterpret_cast<uint2*>(&staged_weights[t][wave][i][8 * j]) = make_uint2(words[t][0], words[t][1]);
        }
        // the value rows; zeros for dead keys (their weight of 0 alone would let a NaN through)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint4 value = value_raw[r];
            if (4 * r + j >= count) value = make_uint4(0u, 0u, 0u, 0u);
            *reinterpret_cast<uint4*>(staged_values + (wave * kWaveKeys + 4 * r + j) * kStageRowBytes + 16 * i) = value;
        }
        if (more) request_values(wave_begin + kStepKeys, next_slot, std::true_type());
        slot = next_slot;
        __syncthreads();

        // weighted sum of the step's keys, 32 at a time
        f32x4 sums[3] = {};
#pragma unroll
        for (int t = 0; t < kStepKeys / 32; ++t) {
            if (begin + 32 * t >= here) break;  // workgroup-uniform
            typedef __attribute__((address_space(3))) i16x4* LdsColumns;
            const std::uint8_t* rows =
                staged_values + (32 * t + 8 * j + (i >> 2)) * kStageRowBytes + 32 * wave + 8 * (i & 3);
            const i16x4 first = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsColumns)rows);
            const i16x4 second = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsColumns)(rows + 4 * kStageRowBytes));
            const bf16x8 values =
                __builtin_bit_cast(bf16x8, __builtin_shufflevector(first, second, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int term = 2; term >= 0; --term) {
                const bf16x8 weights = *reinterpret_cast<const bf16x8*>(
                    &staged_weights[term][2 * t + (j >> 1)][i][16 * (j & 1)]);
                sums[term] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(values, weights, sums[term], 0, 0, 0);
            }
        }
        const float4 parts[2] = {*reinterpret_cast<const float4*>(&wave_sum[i][0]),
                                 *reinterpret_cast<const float4*>(&wave_sum[i][4])};
        denominator = denominator * keep +
            (((parts[0].x + parts[0].y) + (parts[0].z + parts[0].w)) +
             ((parts[1].x + parts[1].y) + (parts[1].z + parts[1].w)));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            accumulator[r] = accumulator[r] * keep + (finite_part(sums[2][r] + sums[1][r]) + sums[0][r]);
        }
    }

    // The split form leaves the sums unnormalised, relative to the share's maximum (an empty share says
    // (-inf, 0, 0)); otherwise the output row is written.
    if (i >= heads_here) return;
    if (tail.partials != nullptr) {
        // a partial row starts 8-byte aligned, and so does its third float
        float* partial =
            tail.partials + ((first_head + i) * splits + blockIdx.y) * partial_floats(kGroupHeadDim);
        if (wave == 0 && j == 0) *reinterpret_cast<float2*>(partial) = make_float2(maximum, denominator);
        float2* target = reinterpret_cast<float2*>(partial + 2 + 16 * wave + 4 * j);
        target[0] = make_float2(accumulator[0], accumulator[1]);
        target[1] = make_float2(accumulator[2], accumulator[3]);
    } else {
        *reinterpret_cast<float4*>(tail.output + (first_head + i) * kGroupHeadDim + 16 * wave + 4 * j) =
            make_float4(accumulator[0] / denominator, accumulator[1] / denominator,
                        accumulator[2] / denominator, accumulator[3] / denominator);
    }
}

// Keys that a workgroup walks alone although there is room for shares: a step of 128 keys more takes 1.5 us (32 heads over 2,
// 100 -> 200 keys 5.1 -> 6.6), shares with their merge from 300 keys on 7.7.
constexpr std::int64_t kAloneKeys = 256;

// The longest share of a block's row, in keys.  A step is 1.6 to 2 us for a workgroup that has a unit alone, since its waves
// meet twice a step; the waves of attention_grouped_kernel walk alone.  With merge, us, that kernel / this one: 128 keys a
// share (7 rows of 32 heads over 2, 2,048 keys) 12.8 / 10.9; 640 (7 of 48 over 8, 2,048) 16.0 / 14.7; 512 (10 of 32 over 8,
// 1,500) 16.8 / 16.3; 768 (16 of 32 over 8, 1,500) 19.6 / 19.5; 1,024 (16 of 32 over 8, 2,000) 23.4 / 22.2; 1,280 (16 of 32
// over 4, 4,802) 24.0 / 22.4, but (of 32 over 8, 2,500) 24.6 / 25.3; 2,176 (16 of 48 over 2, 8,192) 34.6 / 35.1; 4,224 (16
// of 32 over 8, 8,192) 57.4 / 58.4.  (Two workgroups a unit: 128 registers, of which 31 go to scratch memory, 64.7 and 117.)
// One row alone has no such limit: at 512 to 8,192 keys a share (16 heads over 1 to 256 over 64, up to 524,288 keys) it takes
// 0.80 to 0.95 of attention_grouped_kernel's time, with norms, rotation and commit 0.76 to 0.95; at 1,024 and 2,048 keys a
// share, which lie whole powers of two apart in the ring, 0.88 to 1.00 and 0.82 to 0.96.
constexpr std::int64_t kBlockKeys = 1024;

bool overlap(const void* a, std::int64_t a_bytes, const void* b, std::int64_t b_bytes) {
    const auto first = reinterpret_cast<std::uintptr_t>(a), second = reinterpret_cast<std::uintptr_t>(b);
    return first < second + static_cast<std::uintptr_t>(b_bytes) && second < first + static_cast<std::uintptr_t>(a_bytes);
}

}  // namespace

bool launch_attention_row(const RowAttention& call, float* partials, std::int64_t partial_bytes, hipStream_t stream) {
    const auto aligned = [](const void* pointer) { return reinterpret_cast<std::uintptr_t>(pointer) % 16 == 0; };
    const bool on_device = call.device_position != nullptr;
    // a position in device memory can be anything up to the ring's end, and a window is no longer than the ring
    // (several rows: the most that one sees before its own)
    const bool block = call.query_rows > 1;
    const std::int64_t keys = block ? std::min(call.position + call.query_rows, call.sliding_window) - 1
        : !on_device                ? call.position - call.first_key_position
        : call.whole_context        ? call.cache_capacity
                                    : call.sliding_window - 1;
    const std::int64_t heads_per_kv = call.query_heads / call.kv_heads;
    if (call.head_dim != kGroupHeadDim || heads_per_kv < kGroupMinHeads || call.query_heads > 65535 ||
        call.cache_row_stride % 8 != 0 || call.cache_row_stride >= (1 << 24) || call.cache_capacity < kWave ||
        call.cache_capacity > kMostKeys || keys > kMostKeys || !aligned(call.key_cache) || !aligned(call.value_cache) ||
        !aligned(call.current_value) || !aligned(call.output) ||
        (block && (call.position > kMostKeys || !aligned(call.current_key)))) {
        return false;
    }
    const std::int64_t groups_per_kv = (heads_per_kv + kGroupHeads - 1) / kGroupHeads;
    const std::int64_t groups = call.query_rows * call.kv_heads * groups_per_kv;
    const std::int64_t share_bytes = call.query_rows * call.query_heads * partial_floats(kGroupHeadDim) * 4;
    std::int64_t most = compute_units() / groups;
    if (most > kMaxSplits) most = kMaxSplits;
    if (partials == nullptr) most = 1;
    if (most > 1 && most > partial_bytes / share_bytes) most = partial_bytes / share_bytes;
    RowTail tail{};
    tail.block_key = call.current_key;
    tail.block_value = call.current_value;
    tail.block_stride = call.kv_heads * kGroupHeadDim;
    tail.output = call.output;
    tail.device_position = call.device_position;
    tail.position = call.position;
    tail.sliding_window = call.sliding_window;
    tail.whole_context = call.whole_context ? 1 : 0;
    float* key_copy = nullptr;
    if (call.preparation != nullptr) {
        const RowPreparation& how = *call.preparation;
        const std::int64_t query_bytes = call.query_heads * kGroupHeadDim * 4, key_bytes = call.kv_heads * kGroupHeadDim * 4;
        // the prepared query passes through the output rows, and nobody waits for the cache row that is written
        if (overlap(call.output, query_bytes, call.query, query_bytes) ||
            overlap(call.output, query_bytes, call.current_key, key_bytes) ||
            overlap(call.output, query_bytes, call.current_value, key_bytes) ||
            overlap(call.current_key, key_bytes, call.current_value, key_bytes) ||
            overlap(call.query, query_bytes, call.current_key, key_bytes) ||
            overlap(call.query, query_bytes, call.current_value, key_bytes) ||
            (on_device ? call.whole_context : keys >= call.cache_capacity)) {
            return false;
        }
        tail.preparation = how;
        tail.key_copy = how.key;
        // several workgroups read a key: it passes through the end of the workspace, and the merge copies it
        if (groups_per_kv > 1) {
            if (most > kMaxSplits - 1) most = kMaxSplits - 1;
            if (most < 2 || keys <= kAloneKeys || partial_bytes < kMaxSplits * share_bytes) return false;
            key_copy = partials + (kMaxSplits - 1) * share_bytes / 4;
            tail.key_copy = key_copy;
        }
    }
    if (most < 2 && keys > kAloneKeys) return false;
    std::int64_t share = 0, splits = 1;
    if (keys > kAloneKeys) {
        // whole steps of 128 keys a share
        share = ((keys + most - 1) / most + kStepKeys - 1) / kStepKeys * kStepKeys;
        splits = (keys + share - 1) / share;
    } else {
        share = kAloneKeys;
    }
    if (block && share > kBlockKeys) return false;
    if (splits > 1) tail.partials = partials;
    const std::uint32_t first_slot = static_cast<std::uint32_t>(
        block ? keys : on_device ? 0 : call.first_key_position % call.cache_capacity);
    const dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(splits)), threads(kRowWaves * kWave);
    const auto kernel = block               ? attention_row_kernel<RowMode::kBlock>
        : call.preparation != nullptr ? attention_row_kernel<RowMode::kPrepare>
                                      : attention_row_kernel<RowMode::kPlain>;
    hipLaunchKernelGGL(kernel, grid, threads, 0, stream, call.query, call.key_cache, call.value_cache,
                       static_cast<std::uint32_t>(call.cache_row_stride),
                       static_cast<std::uint32_t>(call.cache_capacity), first_slot,
                       static_cast<std::uint32_t>(block ? call.position : keys),
                       on_device ? 0u : static_cast<std::uint32_t>(share),
                       static_cast<std::uint32_t>(heads_per_kv | splits << 16),
                       static_cast<std::uint32_t>(call.kv_heads), call.scale, tail);
    if (splits > 1) {
        launch_attention_merge(partials, call.output, static_cast<int>(splits), call.query_rows * call.query_heads, kGroupHeadDim,
                               call.preparation != nullptr ? call.preparation->query : nullptr, key_copy,
                               call.preparation != nullptr ? call.preparation->key : nullptr,
                               call.kv_heads * kGroupHeadDim, stream);
    }
    return true;
}

}  // namespace nfn
