// Prefill dequant-GEMM on the fp16 matrix cores (gemm_mfma.hip).
#pragma once

#include "common.hpp"

namespace nfn {

// Bytes of device workspace the fp16 path needs: a row-scaled fp16 copy of the
// activations in whole 256-row tiles, one inverse scale per row, and, where a
// small problem splits K over several workgroups per tile, one copy of the
// output per share.  required: of a call of so many rows; workspace: of any call of up to so many
// (fewer rows can take more K shares, and with them more memory).
std::int64_t gemm_f16_required_bytes(std::int64_t rows, std::int64_t input_dim, std::int64_t output_dim);
std::int64_t gemm_f16_workspace_bytes(std::int64_t rows, std::int64_t input_dim, std::int64_t output_dim);
bool gemm_f16_supports(std::uint32_t encoding, std::int64_t input_dim);
// The least that K is cut into by a launch of this geometry on the current device: the number of shares
// (1 = unsplit; more = one partial output per share, summed by a second launch; a call with room for more
// may take more), and the rows of the workgroup tile that they are cut for (256 or 128; 32 for up to 32 rows).
void gemm_f16_plan(std::uint32_t encoding, std::int64_t rows, std::int64_t input_dim,
                   std::int64_t output_dim, int* tile_rows, int* k_shares);
// What a call of `count` projections of one encoding with this workspace runs, for each of them: the rows of
// the workgroup tile (512, 256 or 128; 32 for up to 32 rows) in the launch that takes it, and its K shares.
void gemm_f16_launches(std::uint32_t encoding, std::int64_t rows, std::int64_t input_dim,
                       const std::int64_t* output_dims, int count, std::int64_t workspace_bytes, int* tile_rows,
                       int* k_shares);
// What 1..4 projections of one input, of up to so many rows, need to run in one launch an encoding;
// with the largest of the single sizes they still run, in as many launches as it takes.
std::int64_t gemm_f16_multi_workspace_bytes(std::int64_t rows, std::int64_t input_dim, const std::int64_t* output_dims,
                                            int count);
// outputs[i][rows, output_dim] = input[rows, input_dim] * W_i^T, float accumulation, for 1..4
// projections of one input width: the input is converted once.
void launch_gemm_f16(const Descriptor* descriptors, int count, const float* input, float* const* outputs,
                     std::int64_t rows, void* workspace, std::int64_t workspace_bytes, hipStream_t stream);

}  // namespace nfn
