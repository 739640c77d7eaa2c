// The exact tier at one to three input rows, and at more of them into few outputs: float activations
// from LDS, packed weights streamed once, a wave per pair of weight rows (exact_rows.hpp).  What bounds it
// is the weight stream for one row and the vector ALU (2.25 instructions to decode a weight, one per
// product) beyond.  More rows into many outputs are cheaper on the matrix cores (linear_exact.hip), where a
// product costs nothing on the vector ALU.  Into few outputs that kernel's tiles fill a fraction of the
// chip and walk K for as long as ever; here a workgroup takes two or three of the rows (blockIdx.y), and
// the call is done in what three rows take until there is a workgroup a unit (rows_pay below).
// 4,096 -> 6,656 of Q4_K at 1 / 3 rows: 30.4 / 40.3 -> 6.3 / 9.0 us
// against the wave-per-row kernel that loaded two bytes a lane.
#include "common.hpp"
#include "exact_rows.hpp"
#include "kernels.hpp"

namespace nfn {

namespace {

constexpr std::int64_t kMaxLds = 160 * 1024;
constexpr std::int64_t kMostRows = 3;  // of a workgroup

// The row count that the forms are chosen for: a row of a call of four to 32 rows has the same bits
// whichever other rows come with it, so that those calls take one form, which may not lose at 32.
std::int64_t rows_chosen_for(std::int64_t rows) { return rows > kMostRows && rows < 32 ? 32 : rows; }

constexpr std::int64_t kMaxDenseLds = 159 * 1024;  // beside the waves' meeting place

// GROUPS: of more than R rows, R (of the last group those that exist) a workgroup of blockIdx.y.
// Rows is empty or the row count's int: more than R rows.
// (A form of its own: the checks cost the call of up to three rows 3 %, and the argument alone as much, because
// it moves the grid's size, which a wave reads before its first pair, to a second line of arguments.)
template <std::uint32_t ENC, int R, typename... Rows>
__global__ __launch_bounds__(kExactWaves * kWave) void linear_rows_kernel(
    const std::uint8_t* __restrict__ data, std::int64_t row_stride, const float* __restrict__ input,
    const float* __restrict__ bias, float* __restrict__ output, std::int64_t input_dim, std::int64_t output_dim,
    Rows... rows) {
    constexpr bool GROUPS = sizeof...(Rows) > 0;
    extern __shared__ __attribute__((aligned(16))) float staged[];
    const int row0 = GROUPS ? static_cast<int>(blockIdx.y) * R : 0, there = min(R, (rows + ... + (GROUPS ? 0 : R)) - row0);
    input += row0 * input_dim;
    output += row0 * output_dim;
    exact_rows_stage<R, GROUPS>(input, input_dim, staged, there);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const std::int64_t pairs = (output_dim + kExactPair - 1) / kExactPair;
    exact_rows_walk<ENC, R>(data, row_stride, output_dim, input_dim, staged,
                            static_cast<std::int64_t>(blockIdx.x) * kExactWaves + wave,
                            static_cast<std::int64_t>(gridDim.x) * kExactWaves, pairs,
                            [&](std::int64_t row, const float (&sums)[R]) {
                                if ((threadIdx.x & 63) != 0) return;
                                const float offset = bias != nullptr ? bias[row] : 0.0f;
#pragma unroll
                                for (int r = 0; r < R; ++r) {
                                    if (r < there) output[r * output_dim + row] = sums[r] + offset;
                                }
                            });
}

template <std::uint32_t ENC, int R>
void launch_rows(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                 hipStream_t stream) {
    const std::int64_t pairs = (weight.output_dim + kExactPair - 1) / kExactPair;
    const std::int64_t lds = exact_rows_lds(R, weight.input_dim);
    // as many workgroups as the units hold at once, every wave with the same number of pairs
    const std::int64_t resident = std::int64_t(compute_units()) * (lds <= 40 * 1024 ? 4 : lds <= 80 * 1024 ? 2 : 1);
    const std::int64_t most = (pairs + kExactWaves - 1) / kExactWaves;
    const std::int64_t turns = (most + resident - 1) / resident;
    const std::int64_t groups = (most + turns - 1) / turns;
    const auto launch = [&](auto kernel, auto... count) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(groups), static_cast<unsigned>((rows + R - 1) / R)),
                           dim3(kExactWaves * kWave), static_cast<unsigned>(lds), stream, weight.data,
                           weight.row_stride_bytes, input, bias, output, weight.input_dim, weight.output_dim, count...);
    };
    if constexpr (R > 1) {
        if (rows > R) {
            allow_large_lds<linear_rows_kernel<ENC, R, int>>();
            return launch(linear_rows_kernel<ENC, R, int>, static_cast<int>(rows));
        }
    }
    allow_large_lds<linear_rows_kernel<ENC, R>>();
    launch(linear_rows_kernel<ENC, R>);
}

// Float and bf16 weights: a wave (SPLIT = 1) or the workgroup's eight waves together (SPLIT = 8, for
// few weight rows) take a pair of weight rows; a lane reads 16 neighbouring bytes of each, the
// next turn's requested before this one's are used.  Bound by the weight stream.
typedef std::uint32_t dense_u32x4 __attribute__((ext_vector_type(4), aligned(2)));

template <std::uint32_t ENC, int R, int SPLIT, typename... Rows>
__global__ __launch_bounds__(kExactWaves * kWave) void dense_rows_kernel(
    const std::uint8_t* __restrict__ data, std::int64_t row_stride, const float* __restrict__ input,
    const float* __restrict__ bias, float* __restrict__ output, std::int64_t input_dim, std::int64_t output_dim,
    Rows... rows) {
    constexpr bool GROUPS = sizeof...(Rows) > 0;
    constexpr int kValues = ENC == kEncF32 ? 4 : 8;  // of 16 bytes
    extern __shared__ __attribute__((aligned(16))) float staged[];
    __shared__ float meeting[kExactWaves][kExactPair * R];
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const int columns = static_cast<int>(input_dim);
    const int row0 = GROUPS ? static_cast<int>(blockIdx.y) * R : 0, there = min(R, (rows + ... + (GROUPS ? 0 : R)) - row0);
    input += row0 * input_dim;
    output += row0 * output_dim;
    for (int index = threadIdx.x * 4; index < R * columns; index += kExactWaves * kWave * 4) {
        // (rows past the end are whatever the first one has there; their sums are not stored)
        *reinterpret_cast<exact_f32x4*>(staged + index) =
            *reinterpret_cast<const f32x4_a4*>(input + (!GROUPS || index < there * columns ? index : index % columns));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pieces = columns / kValues;
    const int stride = SPLIT == 1 ? kWave : SPLIT * kWave;  // pieces from one turn to the next
    const int first = SPLIT == 1 ? lane : wave * kWave + lane;
    const std::int64_t pairs = (output_dim + kExactPair - 1) / kExactPair;
    const std::int64_t step = SPLIT == 1 ? static_cast<std::int64_t>(gridDim.x) * kExactWaves : gridDim.x;
    for (std::int64_t pair = SPLIT == 1 ? static_cast<std::int64_t>(blockIdx.x) * kExactWaves + wave : blockIdx.x;
         pair < pairs; pair += step) {
        const std::uint8_t* row[kExactPair];
#pragma unroll
        for (int k = 0; k < kExactPair; ++k) row[k] = data + min(pair * kExactPair + k, output_dim - 1) * row_stride;
        constexpr int kAhead = 4;
        dense_u32x4 held[kAhead][kExactPair];
        const auto load = [&](dense_u32x4 (&into)[kExactPair], int piece) {
#pragma unroll
            for (int k = 0; k < kExactPair; ++k) {
                into[k] = *reinterpret_cast<const dense_u32x4*>(row[k] + static_cast<std::int64_t>(min(piece, pieces - 1)) * 16);
            }
        };
#pragma unroll
        for (int turn = 0; turn < kAhead; ++turn) load(held[turn], first + turn * stride);
        float sums[kExactPair][R] = {}, odd_sums[kExactPair][R] = {};  // of the even and the odd columns
        for (int base = first; base < pieces; base += kAhead * stride) {
#pragma unroll
            for (int turn = 0; turn < kAhead; ++turn) {
                const int piece = base + turn * stride;
                float w[kExactPair][kValues];
#pragma unroll
                for (int k = 0; k < kExactPair; ++k) {
#pragma unroll
                    for (int j = 0; j < kValues; ++j) {
                        if constexpr (ENC == kEncF32) {
                            w[k][j] = __uint_as_float(held[turn][k][j]);
                        } else {
                            w[k][j] = __uint_as_float(j & 1 ? held[turn][k][j / 2] & 0xffff0000u
                                                            : held[turn][k][j / 2] << 16);
                        }
                    }
                }
                load(held[turn], piece + kAhead * stride);
                if (piece < pieces) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
#pragma unroll
                        for (int quad = 0; quad < kValues / 4; ++quad) {
                            const exact_f32x4 v =
                                *reinterpret_cast<const exact_f32x4*>(staged + r * columns + piece * kValues + 4 * quad);
#pragma unroll
                            for (int k = 0; k < kExactPair; ++k) {
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    float& sum = (j & 1) != 0 ? odd_sums[k][r] : sums[k][r];
                                    sum = fmaf(v[j], w[k][4 * quad + j], sum);
                                }
                            }
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < kExactPair; ++k) {
#pragma unroll
            for (int r = 0; r < R; ++r) sums[k][r] = wave_sum(sums[k][r] + odd_sums[k][r]);
        }
        if constexpr (SPLIT == 1) {
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < kExactPair; ++k) {
                    const std::int64_t at = pair * kExactPair + k;
                    if (at < output_dim) {
                        const float offset = bias != nullptr ? bias[at] : 0.0f;
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            if (r < there) output[r * output_dim + at] = sums[k][r] + offset;
                        }
                    }
                }
            }
        } else {
            __syncthreads();
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < kExactPair; ++k) {
#pragma unroll
                    for (int r = 0; r < R; ++r) meeting[wave][k * R + r] = sums[k][r];
                }
            }
            __syncthreads();
            if (threadIdx.x < kExactPair * R) {
                const int k = threadIdx.x / R, r = threadIdx.x % R;
                const std::int64_t at = pair * kExactPair + k;
                float total = meeting[0][threadIdx.x];
#pragma unroll
                for (int w = 1; w < kExactWaves; ++w) total += meeting[w][threadIdx.x];
                if (at < output_dim && r < there) output[r * output_dim + at] = total + (bias != nullptr ? bias[at] : 0.0f);
            }
        }
    }
}

template <std::uint32_t ENC, int R>
void launch_dense(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                  hipStream_t stream) {
    const std::int64_t pairs = (weight.output_dim + kExactPair - 1) / kExactPair;
    const std::int64_t lds = R * weight.input_dim * 4;
    const std::int64_t resident = std::int64_t(compute_units()) * (lds <= 40 * 1024 ? 4 : lds <= 78 * 1024 ? 2 : 1);
    // few pairs: a workgroup each, so that eight waves walk the row instead of one
    // (a form that a row's bits hang on)
    const std::int64_t row_groups_chosen_for = (rows_chosen_for(rows) + kMostRows - 1) / kMostRows;
    const bool split = pairs * row_groups_chosen_for <= 2 * std::int64_t(compute_units());
    const std::int64_t most = split ? pairs : (pairs + kExactWaves - 1) / kExactWaves;
    const unsigned groups = static_cast<unsigned>(most < resident ? most : resident);
    const unsigned row_groups = static_cast<unsigned>((rows + R - 1) / R);
    const auto launch = [&](auto kernel, auto... count) {
        hipLaunchKernelGGL(kernel, dim3(groups, row_groups), dim3(kExactWaves * kWave), static_cast<unsigned>(lds), stream,
                           weight.data, weight.row_stride_bytes, input, bias, output, weight.input_dim,
                           weight.output_dim, count...);
    };
    const auto form = [&](auto... count) {
        if (split) {
            allow_large_lds<dense_rows_kernel<ENC, R, kExactWaves, decltype(count)...>>(kMaxDenseLds);
            launch(dense_rows_kernel<ENC, R, kExactWaves, decltype(count)...>, count...);
        } else {
            allow_large_lds<dense_rows_kernel<ENC, R, 1, decltype(count)...>>(kMaxDenseLds);
            launch(dense_rows_kernel<ENC, R, 1, decltype(count)...>, count...);
        }
    };
    if constexpr (R > 1) {
        if (rows > R) return form(static_cast<int>(rows));
    }
    form();
}

template <std::uint32_t ENC>
void launch_for(const Descriptor& weight, const float* input, const float* bias, float* output, std::int64_t rows,
                hipStream_t stream) {
    const auto launch = [&](auto count) {
        constexpr int kRows = decltype(count)::value;
        if constexpr (kExactRowsFormat<ENC>) {
            launch_rows<ENC, kRows>(weight, input, bias, output, rows, stream);
        } else {
            launch_dense<ENC, kRows>(weight, input, bias, output, rows, stream);
        }
    };
    if (rows == 1) {
        launch(std::integral_constant<int, 1>{});
    } else if (rows == 2 || rows == 4) {
        launch(std::integral_constant<int, 2>{});
    } else {
        launch(std::integral_constant<int, 3>{});
    }
}

}  // namespace

namespace {

// Four rows and more: while the workgroups, of sixteen weight rows and three input rows each, are few enough.  A
// unit with two of them takes twice as long as one with one, so that the lines lie at whole workgroups a unit.
// Where it wins over linear_exact.hip, from 5,000 calls of 256 to 8,192 columns, 4 to 512 rows and up to four workgroups
// a unit; both in us, this one second, 32 rows if not named.  (Four to 32 rows, which take one form: where 32 lose up to
// a sixth, fewer gain up to half.)
//   None up to 1,024 columns, where that kernel needs a turn or two: 1,024 -> 439 of Q4_K 6.1 and 8.0, 512 -> 213 of Q8_0
//     5.3 and 5.9, -> 571 of Q5_K 6.0 and 10.1, -> 246 of Q6_K 5.7 and 10.6.
//   Q4_K, Q8_0   two: 2,048 -> 720 of Q4_K 9.8 and 8.8 (-> 915 9.8 and 11.7), 4,608 -> 592 19.1 and 14.9.  Three, up to 6,400
//     columns (three rows then leave a unit room for two) and from 2,049 (Q8_0: 2,048) on: 0.72 to 1.00 of the time up to
//     4,096, 0.85 to 1.07 from 5,121; between, 1.01 to 1.15, for up to 32 rows only: 4,608 -> 854 19.2 and 20.2, 8 rows of
//     4,608 -> 991 12.7 and 9.8, 19 of 6,144 -> 1,010 of Q8_0 28.3 and 15.4
//   Q5_K         two beyond 2,048 columns (4,608 -> 603 19.8 and 17.3; 0.67 to 0.92), and below for up to 32 rows (2,048 ->
//     447 10.4 and 10.9, -> 360 10.4 and 6.7)
//   Q6_K         two beyond 2,048 (0.58 to 1.06; 17 rows of 4,864 -> 467 31.7 and 13.2), around 4,608 for up to 32 rows only
//     (-> 408 24.8 and 29.0, -> 305 24.8 and 15.5); below one (2,048 -> 471 12.6 and 17.5, -> 350 12.6 and 9.8)
//   bf16         one (0.57 to 0.84; two 0.85 to 1.2): 8 rows of 6,400 into 300 18.5 and 8.9; 33 rows into 64 22.8 and 8.3
//   F32          one up to 256 columns, two beyond (0.36 to 0.89): 8 rows of 6,400 into 300 31.6 and 9.2
bool rows_pay(const Descriptor& weight, std::int64_t rows) {
    rows = rows_chosen_for(rows);
    const std::int64_t columns = weight.input_dim;
    const bool few = rows <= 32, q8 = weight.encoding == kEncQ8_0;
    const auto within = [columns](std::int64_t first, std::int64_t last) { return columns >= first && columns <= last; };
    std::int64_t most = 0;  // workgroups a unit
    switch (weight.encoding) {
        case kEncQ4K: case kEncQ8_0:
            most = within(q8 ? 2048 : 2049, few ? 6400 : 4096) || within(5121, 6400) ? 3 : 2;
            break;
        case kEncQ5K: most = columns > 2048 || few ? 2 : 1; break;
        case kEncQ6K: most = columns > 2048 && (few || !within(4353, 4863)) ? 2 : 1; break;
        case kEncBF16: most = 1; break;
        case kEncF32: most = columns <= 256 ? 1 : 2; break;
        default: return false;
    }
    if (columns <= 1024 && weight.encoding != kEncF32 && weight.encoding != kEncBF16) return false;
    const std::int64_t groups = (rows + kMostRows - 1) / kMostRows;
    constexpr std::int64_t kWorkgroupRows = kExactWaves * kExactPair;
    const std::int64_t workgroups = (weight.output_dim + kWorkgroupRows - 1) / kWorkgroupRows;
    return groups <= 65535 && workgroups <= most * compute_units() / groups;
}

}  // namespace

bool linear_rows_supports(const Descriptor& weight, std::int64_t rows) {
    if (rows < 1 || (rows > kMostRows && !rows_pay(weight, rows))) return false;
    if (rows > kMostRows) rows = kMostRows;
    switch (weight.encoding) {
        case kEncQ4K: case kEncQ5K: case kEncQ6K: case kEncQ8_0:
            return weight.input_dim % 64 == 0 && exact_rows_lds(rows, weight.input_dim) <= kMaxLds;
        case kEncF32: case kEncBF16:
            return weight.input_dim % 8 == 0 && rows * weight.input_dim * 4 <= kMaxDenseLds;
        default: return false;
    }
}

void launch_linear_rows(const Descriptor& weight, const float* input, const float* bias, float* output,
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
