// Device code and launchers shared by the attention kernels: attention.hip (any row count, any
// head size) and attention_row.hip (one query row of 128-wide heads on the matrix cores).
#pragma once

#include "common.hpp"
#include "rms_device.hpp"

namespace nfn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxSplits = 128;      // most shares of one head's keys in the split form
constexpr int kGroupHeads = 16;      // query heads of one key/value head that a workgroup of the matrix-core kernels serves
constexpr int kGroupHeadDim = 128;   // ... and their size
constexpr int kGroupMinHeads = 4;    // fewer query heads per key/value head: the vector form
constexpr int kStageRowBytes = 2 * kGroupHeadDim + 16;  // a staged value row and its pad

// floats per (query row, query head, split) in the partial buffer: maximum, denominator, accumulator
__host__ __device__ constexpr std::int64_t partial_floats(std::int64_t head_dim) {
    return head_dim + 2;
}

// What the row kernel does besides when it also stands for the per-head norms, the query's scale, the rotation and
// the commit of the new cache row (the arithmetic of qk_norm_scale_rope_kernel, rms.hip).
struct RowPreparation {
    float* query;  // rewritten in place, as is the current key
    float* key;
    std::uint16_t* key_cache;
    std::uint16_t* value_cache;
    NormWeight query_weight, key_weight;
    float eps, query_scale;
    RopeBase theta;
    bool interleaved, apply_rope;
};

// One query row over a cache.  The keys are first_key_position .. position - 1 of the ring and the current one;
// with `device_position` the last `sliding_window` ones up to *device_position, or all when `whole_context`.
// With query_rows > 1 the rows of a causal block: row r at position + r, with the last `sliding_window` keys up to its
// own of the ring and of the block's rows (current_key, current_value).
struct RowAttention {
    const float* query;
    const float* current_key;
    const float* current_value;
    const std::uint16_t* key_cache;
    const std::uint16_t* value_cache;
    float* output;
    std::int64_t query_rows, query_heads, kv_heads, head_dim;
    std::int64_t position, first_key_position;
    std::int64_t cache_capacity, cache_row_stride;
    float scale;
    const std::int64_t* device_position;
    std::int64_t sliding_window;
    bool whole_context;
    const RowPreparation* preparation;  // null: query and key are final
};

// attention_row.hip: false (and nothing launched) where the kernel does not apply.  `partials`: room for
// partial_bytes of shares, or null.
bool launch_attention_row(const RowAttention& call, float* partials, std::int64_t partial_bytes, hipStream_t stream);

// attention.hip: merges the shares of `heads` rows of the output.  With `query` the output rows hold the prepared
// query, which moves there first; with key_copy its key_floats go to `key`.
void launch_attention_merge(const float* partials, float* output, int splits, std::int64_t heads, std::int64_t head_dim,
                            float* query, const float* key_copy, float* key, std::int64_t key_floats,
                            hipStream_t stream);

// eight floats as the bf16 row the cache would hold of them
__device__ __forceinline__ uint4 pack_as_cached(float4 low, float4 high) {
    const auto pair = [](float first, float second) {
        return static_cast<std::uint32_t>(to_bf16(first)) | (static_cast<std::uint32_t>(to_bf16(second)) << 16);
    };
    return make_uint4(pair(low.x, low.y), pair(low.z, low.w), pair(high.x, high.y), pair(high.z, high.w));
}

// x = high + middle + low exactly, every term a bf16 in the upper half of a word: each takes the next eight
// significant bits of what is left (truncation, so the remainders are exact; eight at most are left for the last,
// whose lower half holds none of them)
__device__ __forceinline__ void split_term(float x, std::uint32_t (&term)[3]) {
    float rest = x;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        term[t] = __float_as_uint(rest) & 0xffff0000u;
        rest -= __uint_as_float(term[t]);
    }
    term[2] = __float_as_uint(rest);
}

// ... of N values, two to a word, the first in its lower half
template <int N>
__device__ __forceinline__ void split_terms(const float (&x)[N], std::uint32_t (&words)[3][N / 2]) {
#pragma unroll
    for (int w = 0; w < N / 2; ++w) {
        std::uint32_t first[3], second[3];
        split_term(x[2 * w], first);
        split_term(x[2 * w + 1], second);
#pragma unroll
        for (int t = 0; t < 3; ++t) words[t][w] = __builtin_amdgcn_perm(second[t], first[t], 0x07060302u);
    }
}

}  // namespace nfn
