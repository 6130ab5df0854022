// Cross-entropy of one chunk of logits, forward and backward, between the LM head's two matrix products.
//
// Two passes over the bf16 logits instead of the dozen of the same formulas written with tensor operations (fp32 copy,
// log-softmax, exponential, one-hot, mask, rounding and the packing of the result for the grad-input kernel):
//   loss_stats_kernel   reads a span of a row: its largest value and the sum of exponentials above it;
//   loss_grad_kernel    joins a row's spans, and writes (softmax - one_hot) / count, rounded to bf16, straight in the
//                       fragment order that the grad-input kernels read, so neither the softmax nor the row-major
//                       cotangent ever exists.
// Both are bound by memory: 256 rows of 248320 logits are 127 MB, read twice and written once; the two passes take
// 21 + 47 us for what took 465 us and another 43 us to pack.
//
// Exponentials and logarithms are the short forms (__expf, __logf; the full ones cost another 11 + 5 us a chunk).  With x <= 0 the
// product x * log2(e) is rounded once and the hardware's 2^t is good to 2^-23, so that e^x is off by at most
// (|x| + 2) * 2^-24 + |x| * 2^-26 of itself: 7e-6 at |x| = 88, where it underflows, against the 2^-9 that rounding the cotangent to bf16
// costs; in a row's sum the terms weigh |x| by e^x, which leaves (log(columns) + 2) * 2^-24 or less, 1e-6.  Measured against
// 64 bits on vocabularies of 1001 to 151936 and logits of rms 0.5 to 11: loss 4e-8 to 9e-8 of itself, the same figures with
// the full functions and with tensor operations; gradient 1e-5 to 5e-5 of its norm away from that of the exactly
// rounded cotangent, with any of the three.
#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

// ---- the number of counted rows -------------------------------------------------------------------------------
// count[0] = rows whose target is not ignored, at least 1, as a float: one workgroup, no atomics.
__global__ __launch_bounds__(1024) void count_targets_kernel(const int64_t * __restrict__ targets, int64_t rows,
                                                             int64_t ignore_index, float * __restrict__ count) {
    __shared__ int partial[16];
    int mine = 0;
    for (int64_t i = threadIdx.x; i < rows; i += 1024) {
        mine += targets[i] != ignore_index ? 1 : 0;
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        mine += __shfl_xor(mine, offset);
    }
    if ((threadIdx.x & 63) == 0) {
        partial[threadIdx.x >> 6] = mine;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
        for (int w = 0; w < 16; ++w) {
            total += partial[w];
        }
        count[0] = static_cast<float>(max(total, 1));
    }
}

// loss = (sum of the rows' losses) / count
__global__ __launch_bounds__(1024) void loss_total_kernel(const float * __restrict__ row_loss, int64_t rows,
                                                          const float * __restrict__ count, float * __restrict__ loss) {
    __shared__ float partial[16];
    float mine = 0.0f;
    for (int64_t i = threadIdx.x; i < rows; i += 1024) {
        mine += row_loss[i];
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        mine += __shfl_xor(mine, offset);
    }
    if ((threadIdx.x & 63) == 0) {
        partial[threadIdx.x >> 6] = mine;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.0f;
        for (int w = 0; w < 16; ++w) {
            total += partial[w];
        }
        loss[0] = total / count[0];
    }
}

// ---- statistics of a row's spans ------------------------------------------------------------------------------
// stats[row][span] = (m, sum of exp(x - m)) over LOSS_SPAN columns, m the largest value that is a number; where that is -inf,
// (-inf, sum of exp(x)): 0 of nothing but -inf, NaN with a NaN among them.  A NaN or +inf makes the sum NaN.  A thread holds four pieces of eight values, all
// requested before the first is used; enough workgroups for any row count (31 spans for a vocabulary of 248320).
__global__ __launch_bounds__(256) void loss_stats_kernel(const uint16_t * __restrict__ logits, int64_t pitch, int columns,
                                                         float2 * __restrict__ stats) {
    __shared__ float wave_value[2][4];
    const int tid = threadIdx.x;
    const int span = blockIdx.x, row = blockIdx.y;
    const uint16_t * const x = logits + row * pitch;
    const int first = span * LOSS_SPAN + tid * 8;
    float value[4][8];
    uint4 bits[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int column = first + p * 2048;
        // (the pitch is a multiple of eight and the buffer holds whole pieces: the piece that holds the last column may
        // be read as a whole)
        bits[p] = column < columns ? *reinterpret_cast<const uint4 *>(x + column) : uint4{0, 0, 0, 0};
    }
    float largest = -INFINITY;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        unpack_bf16x8(bits[p], value[p]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            value[p][e] = first + p * 2048 + e < columns ? value[p][e] : -INFINITY;
            largest = fmaxf(largest, value[p][e]);
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        largest = fmaxf(largest, __shfl_xor(largest, offset));
    }
    if ((tid & 63) == 0) {
        wave_value[0][tid >> 6] = largest;
    }
    __syncthreads();
    largest = fmaxf(fmaxf(wave_value[0][0], wave_value[0][1]), fmaxf(wave_value[0][2], wave_value[0][3]));
    const float above = largest == -INFINITY ? 0.0f : largest;   // (-inf - -inf would make a NaN of a span without one)
    float sum = 0.0f;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sum += __expf(value[p][e] - above);
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        sum += __shfl_xor(sum, offset);
    }
    if ((tid & 63) == 0) {
        wave_value[1][tid >> 6] = sum;
    }
    __syncthreads();
    if (tid == 0) {
        stats[static_cast<int64_t>(row) * gridDim.x + span] =
            make_float2(largest, (wave_value[1][0] + wave_value[1][1]) + (wave_value[1][2] + wave_value[1][3]));
    }
}

// ---- loss per row, and the cotangent of the logits --------------------------------------------------------------
// A workgroup holds 32 rows x LOSS_GRAD_COLUMNS columns.  Thread (rr, c) of the prologue joins every eighth span of row rr;
// in the loop it turns 16 neighbouring logits of row rr into 32 bytes of the packed cotangent (pack_cotangent_kernel's
// layout: [rows / 32][chunks of 16 columns][half][row][8 bf16], zeros behind the last row and column), which leave
// through LDS as one contiguous 8 KiB run.
// A target outside the vocabulary that is not the ignored one makes its row's loss and gradient NaN.
constexpr int LOSS_GRAD_COLUMNS = 1024;
__global__ __launch_bounds__(256) void loss_grad_kernel(const uint16_t * __restrict__ logits, int64_t pitch, int rows,
                                                        int columns, int n_chunks, const float2 * __restrict__ stats, int spans,
                                                        const int64_t * __restrict__ targets, int64_t ignore_index,
                                                        const float * __restrict__ count, float * __restrict__ row_loss,
                                                        uint8_t * __restrict__ cotangent) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[2][8 * 1024];
    const int tid = threadIdx.x;
    const int rr = tid >> 3;
    const int c = tid & 7;
    const int row = blockIdx.y * 32 + rr;
    const bool present = row < rows;
    const int row_read = min(row, rows - 1);
    const uint16_t * const x = logits + row_read * pitch;
    const int64_t target = targets[row_read];
    const bool counted = present && target != ignore_index;
    const bool known = target >= 0 && target < columns;
    // the row's largest value and its sum of exponentials: eight lanes of a row take every eighth span each
    float largest = -INFINITY, sum = 0.0f;
    const auto join = [&](float other_largest, float other_sum) {
        const float joined = fmaxf(largest, other_largest);
        // (a part without a finite maximum keeps its sum: 0, or NaN)
        sum = (largest == -INFINITY ? sum : sum * __expf(largest - joined)) +
              (other_largest == -INFINITY ? other_sum : other_sum * __expf(other_largest - joined));
        largest = joined;
    };
    for (int s = c; s < spans; s += 8) {
        const float2 part = stats[static_cast<int64_t>(row_read) * spans + s];
        join(part.x, part.y);
    }
#pragma unroll
    for (int offset = 1; offset < 8; offset <<= 1) {
        const float other_largest = __shfl_xor(largest, offset), other_sum = __shfl_xor(sum, offset);
        join(other_largest, other_sum);
    }
    const float log_sum = largest + __logf(sum);
    if (blockIdx.x == 0 && c == 0 && present) {
        row_loss[row] = !counted ? 0.0f : known ? log_sum - bf16_bits_to_float(x[target]) : NAN;
    }
    if (cotangent == nullptr) {
        return;
    }
    const float factor = !counted ? 0.0f : known ? 1.0f / count[0] : NAN;
    uint8_t * const out = cotangent + static_cast<int64_t>(blockIdx.y) * n_chunks * 1024;
    constexpr int PASSES = LOSS_GRAD_COLUMNS / 128;
    uint4 bits[2], next[2];
    auto request = [&](int chunk0, uint4 (&to)[2]) {
        const int n = (chunk0 + c) * 16;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            to[h] = n + 8 * h < columns ? *reinterpret_cast<const uint4 *>(x + n + 8 * h) : uint4{0, 0, 0, 0};
        }
    };
    const int first_chunk = blockIdx.x * (LOSS_GRAD_COLUMNS / 16);
    request(first_chunk, bits);
    for (int pass = 0; pass < PASSES; ++pass) {
        const int chunk0 = first_chunk + pass * 8;
        if (chunk0 >= n_chunks) {   // uniform
            return;
        }
        if (pass + 1 < PASSES) {
            request(chunk0 + 8, next);
        }
        const int n = (chunk0 + c) * 16;
        uint4 packed[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float value[8];
            unpack_bf16x8(bits[h], value);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int column = n + 8 * h + e;
                const float probability = __expf(value[e] - log_sum);
                // (rows that do not count get zeros whatever their logits are)
                value[e] = column < columns && factor != 0.0f ? (probability - (column == target ? 1.0f : 0.0f)) * factor : 0.0f;
            }
            packed[h] = make_uint4(pack_bf16x2(value[0], value[1]), pack_bf16x2(value[2], value[3]),
                                   pack_bf16x2(value[4], value[5]), pack_bf16x2(value[6], value[7]));
        }
        uint8_t * const slab = tile[pass & 1];
        *reinterpret_cast<uint4 *>(slab + c * 1024 + rr * 16) = packed[0];
        *reinterpret_cast<uint4 *>(slab + c * 1024 + (32 + rr) * 16) = packed[1];
        __syncthreads();   // (two slabs: the copy out of one needs no barrier before the next pass writes the other)
        const int pieces = min(8, n_chunks - chunk0) * 64;
        uint4 * const dst = reinterpret_cast<uint4 *>(out + static_cast<int64_t>(chunk0) * 1024);
        const uint4 * const src = reinterpret_cast<const uint4 *>(slab);
        if (tid < pieces) {
            dst[tid] = src[tid];
        }
        if (tid + 256 < pieces) {
            dst[tid + 256] = src[tid + 256];
        }
        bits[0] = next[0];
        bits[1] = next[1];
    }
}

hipError_t launch_count_targets(const int64_t * targets, int64_t rows, int64_t ignore_index, float * count, hipStream_t stream) {
    count_targets_kernel<<<1, 1024, 0, stream>>>(targets, rows, ignore_index, count);
    return hipGetLastError();
}

hipError_t launch_loss_total(const float * row_loss, int64_t rows, const float * count, float * loss, hipStream_t stream) {
    loss_total_kernel<<<1, 1024, 0, stream>>>(row_loss, rows, count, loss);
    return hipGetLastError();
}

hipError_t launch_cross_entropy(const uint16_t * logits, int64_t pitch, int rows, int columns, float2 * stats,
                                const int64_t * targets, int64_t ignore_index, const float * count, float * row_loss,
                                uint8_t * cotangent, hipStream_t stream) {
    if (pitch % 8 != 0) {
        return hipErrorInvalidValue;
    }
    const int spans = loss_spans(columns);
    const int row_tiles = (rows + 31) / 32;
    const int n_chunks = cotangent_chunks(columns);
    // (grid.y is at most 65535: callers keep a chunk below that many rows)
    loss_stats_kernel<<<dim3(static_cast<unsigned>(spans), static_cast<unsigned>(rows)), 256, 0, stream>>>(logits, pitch, columns, stats);
    const unsigned column_blocks = cotangent == nullptr ? 1 : static_cast<unsigned>((n_chunks * 16 + LOSS_GRAD_COLUMNS - 1) / LOSS_GRAD_COLUMNS);
    loss_grad_kernel<<<dim3(column_blocks, static_cast<unsigned>(row_tiles)), 256, 0, stream>>>(
        logits, pitch, rows, columns, n_chunks, stats, spans, targets, ignore_index, count, row_loss, cotangent);
    return hipGetLastError();
}

// out[i] = bf16(in[i] * factor[0]), `count` a multiple of 8
__global__ __launch_bounds__(256) void scale_bf16_kernel(const uint16_t * __restrict__ in, const float * __restrict__ factor,
                                                         uint16_t * __restrict__ out, int64_t pieces) {
    const float f = factor[0];
    for (int64_t piece = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; piece < pieces; piece += static_cast<int64_t>(gridDim.x) * 256) {
        float value[8];
        unpack_bf16x8(reinterpret_cast<const uint4 *>(in)[piece], value);
        reinterpret_cast<uint4 *>(out)[piece] =
            make_uint4(pack_bf16x2(value[0] * f, value[1] * f), pack_bf16x2(value[2] * f, value[3] * f),
                       pack_bf16x2(value[4] * f, value[5] * f), pack_bf16x2(value[6] * f, value[7] * f));
    }
}

hipError_t launch_scale_bf16(const uint16_t * in, const float * factor, uint16_t * out, int64_t count, hipStream_t stream) {
    const int64_t blocks = (count / 8 + 255) / 256;
    scale_bf16_kernel<<<static_cast<unsigned>(blocks < 1 ? 1 : blocks > 16384 ? 16384 : blocks), 256, 0, stream>>>(in, factor, out, count / 8);
    return hipGetLastError();
}

}  // namespace tgo
