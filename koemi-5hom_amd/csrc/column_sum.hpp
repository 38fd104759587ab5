// Column sums of fp32 partial rows, the last stage of reductions over rows that
// several workgroups share: out[c] = sum over b < blocks of partial[b * width + c].
#pragma once

#include "common.hpp"

namespace koemi {

// A workgroup takes 1024 / LANES or 256 / LANES columns (at least a 128-byte line of
// every partial row) and its row lanes stride the partial rows, eight loads in
// flight each; the row lanes' sums meet in LDS in a fixed tree: the same bits on
// every run. Bound by latency where the partials sit in L2. 1024 x 512: 4.8 us,
// against 240 us for a thread per column that walks the rows. Few rows take fewer
// lanes, so that none idle (2 x 262144: 12 -> 4 us).
template <typename T, int LANES>
__global__ __launch_bounds__(LANES == 32 ? 1024 : 256) void column_sum_kernel(
    const float* __restrict__ partial, T* __restrict__ out, int64_t blocks, int64_t width) {
    constexpr int kCols = (LANES == 32 ? 1024 : 256) / LANES;
    __shared__ float sums[LANES][kCols + 1];
    const int col = threadIdx.x % kCols, lane = threadIdx.x / kCols;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kCols + col;
    const float* p = partial + min(c, width - 1);
    float acc = 0.0f;
    for (int64_t b0 = lane; b0 < blocks; b0 += 8 * LANES) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = p[min(b0 + i * LANES, blocks - 1) * width];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc += b0 + i * LANES < blocks ? v[i] : 0.0f;
    }
    if constexpr (LANES > 1) {
        sums[lane][col] = acc;
        __syncthreads();
#pragma unroll
        for (int half = LANES / 2; half > 0; half >>= 1) {
            if (lane < half) sums[lane][col] += sums[lane + half][col];
            __syncthreads();
        }
        acc = sums[0][col];
    }
    if (lane == 0 && c < width) out[c] = from_f32<T>(acc);
}

template <typename T>
inline void launch_column_sum(const float* partial, T* out, int64_t blocks, int64_t width, hipStream_t stream) {
    if (blocks <= 8)
        hipLaunchKernelGGL((column_sum_kernel<T, 1>), dim3(grid_for(width, 256)), dim3(256), 0, stream, partial, out,
                           blocks, width);
    else if (blocks <= 64)
        hipLaunchKernelGGL((column_sum_kernel<T, 4>), dim3(grid_for(width, 64)), dim3(256), 0, stream, partial, out,
                           blocks, width);
    else
        hipLaunchKernelGGL((column_sum_kernel<T, 32>), dim3(grid_for(width, 32)), dim3(1024), 0, stream, partial, out,
                           blocks, width);
}

}  // namespace koemi
