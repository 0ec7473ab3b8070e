// What the field kernels write: a cell's fields, and the residual sums of the
// surrogate's judge.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"

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

// The cell's fields: raw sums, or E_dyn / B_dyn (compared with the surrogate's
// sums they replace, for the judge).
__device__ __forceinline__ void write_cell(const FieldArgs& f, uint64_t n, const float* v, float* jd) {
    const uint64_t N = f.N;
    if (f.raw != nullptr) {
#pragma unroll
        for (int c = 0; c < 6; c++) f.raw[(uint64_t)c * N + n] = v[c];
        return;
    }
#pragma unroll
    for (int c = 0; c < 6; c++) {
        float* const dyn = (c < 3 ? f.e_dyn : f.b_dyn) + (uint64_t)(c % 3) * N + n;
        const float* const stat = (c < 3 ? f.e_stat : f.b_stat) + (uint64_t)(c % 3) * N + n;
        if (f.judge != nullptr) {
            const float d = *dyn - v[c];
            jd[c < 3 ? 0 : 2] = __builtin_fmaf(d, d, jd[c < 3 ? 0 : 2]);
            jd[c < 3 ? 1 : 3] = __builtin_fmaf(v[c], v[c], jd[c < 3 ? 1 : 3]);
        }
        *dyn = *stat + (c < 3 ? f.ke : f.kmu) * v[c];
    }
}

}  // namespace ion
