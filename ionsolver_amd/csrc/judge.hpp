// Residual sums of the surrogate's judge, shared by the field kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ion {

// Judge partials of a block: the work-items' four sums (E error, E norm,
// B error, B norm) reduced in a fixed order (wavefront tree, then the
// wavefronts in order) into partial[blockIdx.x][4], in double.
__device__ __forceinline__ void judge_block_sums(const float v[4], double* partial) {
    __shared__ double jsh[16][4];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    double d[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        d[k] = (double)v[k];
        for (int o = 32; o >= 1; o >>= 1) d[k] += __shfl_down(d[k], o, 64);
    }
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 4; k++) jsh[wv][k] = d[k];
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (uint32_t w = 0; w < (blockDim.x + 63u) / 64u; w++) t += jsh[w][threadIdx.x];
        partial[(size_t)blockIdx.x * 4 + threadIdx.x] = t;
    }
}

}  // namespace ion
