// lm_head GEMV with the argmax fused in.  Pass 1: every workgroup computes the
// logits of its vocabulary rows and keeps only the best (value, index) per
// input row in the workspace.  Pass 2: one workgroup per input row reduces the
// per-workgroup candidates.  The logits are never written to memory.
//
// The reference does this as two separate operations with an 808 KB logits
// buffer in between (neuralfn/csrc/native_gpt2/resident_glimmer_cuda.cpp:4087-4151:
// linear, then nfn_native_tile_argmax_rows_float32_v1).  Tie rule and NaN
// behaviour are those of neuralfn/csrc/tile_cuda/kernels.cu:1564-1602.
#include "common.hpp"
#include "exact_rows.hpp"
#include "gemv_f32_device.hpp"
#include "kernels.hpp"
#include "lm_head.hpp"

namespace nfn {

namespace {

constexpr int kWavesPerBlock = 4;

template <int R>
__global__ __launch_bounds__(kWavesPerBlock * kWave) void lm_head_partial_kernel(
    Projection op, std::int64_t input_dim, const float* __restrict__ input, std::int64_t rows,
    int columns_per_wave, LmHeadCandidate* __restrict__ candidates) {
    __shared__ float shared_values[kWavesPerBlock][R];
    __shared__ std::int64_t shared_indices[kWavesPerBlock][R];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const std::int64_t first_column =
        (static_cast<std::int64_t>(blockIdx.x) * kWavesPerBlock + wave) * columns_per_wave;
    float best_value[R];
    std::int64_t best_index[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        best_value[r] = -INFINITY;
        best_index[r] = 0;
    }
    const int active = static_cast<int>(rows);
    for (int step = 0; step < columns_per_wave; ++step) {
        const std::int64_t column = first_column + step;
        if (column >= op.output_dim) break;
        float sums[R];
        wave_row_partials<R, kPlain>(op.encoding, op.data + column * op.row_stride, input_dim,
                                     input, nullptr, 0, active, lane, sums);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float logit = wave_sum(sums[r]);
            better(logit, column, best_value[r], best_index[r]);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            shared_values[wave][r] = best_value[r];
            shared_indices[wave][r] = best_index[r];
        }
    }
    __syncthreads();
    if (threadIdx.x < R && threadIdx.x < rows) {
        float value = shared_values[0][threadIdx.x];
        std::int64_t index = shared_indices[0][threadIdx.x];
        for (int w = 1; w < kWavesPerBlock; ++w) {
            better(shared_values[w][threadIdx.x], shared_indices[w][threadIdx.x], value, index);
        }
        LmHeadCandidate candidate;
        candidate.index = index;
        candidate.value = value;
        candidate.pad = 0;
        candidates[static_cast<std::int64_t>(threadIdx.x) * gridDim.x + blockIdx.x] = candidate;
    }
}

// One input row of a packed format: the row in LDS, the vocabulary streamed by pairs of rows
// (exact_rows.hpp); a wave takes a contiguous run of pairs.  The kernel above loads two bytes a lane
// and waits for each block: 6,144 -> 15,734 rows of Q5_K took 454 us with it.
template <std::uint32_t ENC>
__global__ __launch_bounds__(kExactWaves * kWave) void lm_head_row_kernel(
    Projection op, std::int64_t input_dim, const float* __restrict__ input, LmHeadCandidate* __restrict__ candidates) {
    extern __shared__ __attribute__((aligned(16))) float staged[];
    __shared__ float wave_values[kExactWaves];
    __shared__ std::int64_t wave_indices[kExactWaves];
    exact_rows_stage<1>(input, input_dim, staged);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const std::int64_t pairs = (op.output_dim + kExactPair - 1) / kExactPair;
    const std::int64_t waves = static_cast<std::int64_t>(gridDim.x) * kExactWaves;
    const std::int64_t index = static_cast<std::int64_t>(blockIdx.x) * kExactWaves + wave;
    float best_value = -INFINITY;
    std::int64_t best_index = 0;
    exact_rows_walk<ENC, 1>(op.data, op.row_stride, op.output_dim, input_dim, staged, pairs * index / waves, 1,
                            pairs * (index + 1) / waves, [&](std::int64_t row, const float (&sums)[1]) {
                                better(sums[0], row, best_value, best_index);
                            });
    if ((threadIdx.x & 63) == 0) {
        wave_values[wave] = best_value;
        wave_indices[wave] = best_index;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kExactWaves; ++w) better(wave_values[w], wave_indices[w], best_value, best_index);
        LmHeadCandidate candidate;
        candidate.index = best_index;
        candidate.value = best_value;
        candidate.pad = 0;
        candidates[blockIdx.x] = candidate;
    }
}

template <std::uint32_t ENC>
void launch_row(const Projection& op, std::int64_t input_dim, const float* input, LmHeadCandidate* candidates,
                std::int64_t groups, hipStream_t stream) {
    allow_large_lds<lm_head_row_kernel<ENC>>(159 * 1024);
    hipLaunchKernelGGL((lm_head_row_kernel<ENC>), dim3(static_cast<unsigned>(groups)), dim3(kExactWaves * kWave),
                       static_cast<unsigned>(exact_rows_lds(1, input_dim)), stream, op, input_dim, input, candidates);
}

}  // namespace

constexpr int kFinalThreads = 1024;

__global__ __launch_bounds__(kFinalThreads) void lm_head_final_kernel(
    const LmHeadCandidate* __restrict__ candidates, std::int64_t candidate_count,
    std::int64_t* __restrict__ indices, float* __restrict__ maxima) {
    constexpr int kFinalWaves = kFinalThreads / kWave;
    __shared__ float wave_values[kFinalWaves];
    __shared__ std::int64_t wave_indices[kFinalWaves];
    const std::int64_t row = blockIdx.x;
    float best_value = -INFINITY;
    std::int64_t best_index = 0;
    for (std::int64_t i = threadIdx.x; i < candidate_count; i += kFinalThreads) {
        const LmHeadCandidate c = candidates[row * candidate_count + i];
        better(c.value, c.index, best_value, best_index);
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        const float other_value = __shfl_xor(best_value, offset, 64);
        const std::int64_t other_index = __shfl_xor(best_index, offset, 64);
        better(other_value, other_index, best_value, best_index);
    }
    if ((threadIdx.x & 63) == 0) {
        wave_values[threadIdx.x >> 6] = best_value;
        wave_indices[threadIdx.x >> 6] = best_index;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kFinalWaves; ++w) {
            better(wave_values[w], wave_indices[w], best_value, best_index);
        }
        indices[row] = best_index;
        maxima[row] = best_value;
    }
}

void launch_lm_head_final(const LmHeadCandidate* candidates, std::int64_t candidate_count,
                          std::int64_t* indices, float* maxima, std::int64_t rows,
                          hipStream_t stream) {
    hipLaunchKernelGGL(lm_head_final_kernel, dim3(static_cast<unsigned>(rows)),
                       dim3(kFinalThreads), 0, stream, candidates, candidate_count, indices,
                       maxima);
}

std::int64_t lm_head_f32_blocks(std::int64_t output_dim) {
    // 16 vocabulary rows per wave, 64 per workgroup.
    return (output_dim + 63) / 64;
}
// Workgroups of the one-row kernel, given room for their candidates (its sums and its choice do not hang on
// their number).  A vocabulary of up to two pairs of rows a wave at three workgroups a unit is spread over as
// many workgroups as that takes (64 rows each would leave most units idle, or waves with four pairs
// where others have none to hide behind): 4,608 -> 4,000 / 9,000 / 16,000 rows of Q4_K 24.4 / 24.4 / 25.2 ->
// 11.3 / 19.1 / 22.8 us; 30,000 would take 39.3 instead of 37.0.
std::int64_t row_pairs(std::int64_t output_dim) { return (output_dim + kExactPair - 1) / kExactPair; }
std::int64_t row_turns(std::int64_t output_dim) {  // of eight waves, three workgroups a unit
    const std::int64_t at_once = 24 * std::int64_t(compute_units());
    return (row_pairs(output_dim) + at_once - 1) / at_once;
}
std::int64_t lm_head_row_groups(std::int64_t output_dim) {
    const std::int64_t resident = 2 * std::int64_t(compute_units());
    const std::int64_t pairs = row_pairs(output_dim), turns = row_turns(output_dim);
    if (turns <= 2) return (pairs + kExactWaves * turns - 1) / (kExactWaves * turns);
    const std::int64_t blocks = lm_head_f32_blocks(output_dim);
    return blocks < resident ? blocks : resident;
}

void launch_lm_head_f32(const Descriptor& descriptor, const float* input, std::int64_t rows,
                        LmHeadCandidate* candidates, std::int64_t room, std::int64_t* indices, float* maxima,
                        hipStream_t stream) {
    Projection op{};
    op.data = descriptor.data;
    op.output = nullptr;
    op.output_dim = descriptor.output_dim;
    op.row_stride = descriptor.row_stride_bytes;
    op.encoding = descriptor.encoding;
    const std::int64_t blocks = lm_head_f32_blocks(descriptor.output_dim);
    // (two workgroups a compute unit; the row and the kernel's own few words have to fit LDS)
    if (rows == 1 && descriptor.input_dim % 64 == 0 &&
        exact_rows_lds(1, descriptor.input_dim) <= 159 * 1024) {
        std::int64_t groups = lm_head_row_groups(descriptor.output_dim);
        // (Q8_0, 12,289 to 16,384 rows: 64 each, one workgroup a unit.  In two turns some units would have two workgroups
        // and take as long as its four: 6,656 -> 13,001 and 7,936 -> 12,617 1.10 times, 2,560 to 5,120 columns as long;
        // more rows, where 64 each leave some units with two, take 0.85 to 0.89 times, like the other formats.)
        if (descriptor.encoding == kEncQ8_0 && row_turns(descriptor.output_dim) == 2 && blocks <= compute_units()) groups = blocks;
        if (groups > room) groups = room;
        bool launched = true;
        switch (descriptor.encoding) {
            case kEncQ4K: launch_row<kEncQ4K>(op, descriptor.input_dim, input, candidates, groups, stream); break;
            case kEncQ5K: launch_row<kEncQ5K>(op, descriptor.input_dim, input, candidates, groups, stream); break;
            case kEncQ6K: launch_row<kEncQ6K>(op, descriptor.input_dim, input, candidates, groups, stream); break;
            case kEncQ8_0: launch_row<kEncQ8_0>(op, descriptor.input_dim, input, candidates, groups, stream); break;
            default: launched = false; break;
        }
        if (launched) {
            launch_lm_head_final(candidates, groups, indices, maxima, rows, stream);
            return;
        }
    }
    const dim3 grid(static_cast<unsigned>(blocks));
    const dim3 block(kWavesPerBlock * kWave);
    if (rows == 1) {
        hipLaunchKernelGGL((lm_head_partial_kernel<1>), grid, block, 0, stream, op,
                           descriptor.input_dim, input, rows, 16, candidates);
    } else if (rows <= 4) {
        hipLaunchKernelGGL((lm_head_partial_kernel<4>), grid, block, 0, stream, op,
                           descriptor.input_dim, input, rows, 16, candidates);
    } else {
        hipLaunchKernelGGL((lm_head_partial_kernel<8>), grid, block, 0, stream, op,
                           descriptor.input_dim, input, rows, 16, candidates);
    }
    launch_lm_head_final(candidates, blocks, indices, maxima, rows, stream);
}

}  // namespace nfn
