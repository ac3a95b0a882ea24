// The fixed-order sums that end a backward pass: partial results of many workgroups into gradients of small parameters.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace bm2 {

// sum_i in[i * nj + j] for 16 columns j: 16 row slices per workgroup, added in a fixed order; store(j, sum) once per column
template <typename F> __device__ __forceinline__ void column_sums_body(const float *in, int ni, int nj, int block, F store) {
    __shared__ float red[16][17];
    const int jl = threadIdx.x & 15, sl = threadIdx.x >> 4, j = block * 16 + jl;
    float s = 0.f;
    if (j < nj) {
        // (bound by the rounds of loads that are waited for: sixteen go out at once)
        int i = sl;
        auto rounds = [&](auto R) __attribute__((always_inline)) {
            constexpr int n = decltype(R)::value;
            for (; i + (4 * n - 1) * 16 < ni; i += n * 64) {
                float v[4 * n];
#pragma unroll
                for (int q = 0; q < 4 * n; ++q) v[q] = in[(int64_t)(i + q * 16) * nj + j];
#pragma unroll
                for (int q = 0; q < 4 * n; q += 4) s += (v[q] + v[q + 1]) + (v[q + 2] + v[q + 3]);
            }
        };
        rounds(std::integral_constant<int, 4>());
        rounds(std::integral_constant<int, 1>());
        for (; i < ni; i += 16) s += in[(int64_t)i * nj + j];
    }
    red[sl][jl] = s;
    __syncthreads();
    if (sl == 0 && j < nj) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < 16; ++q) t += red[q][jl];
        store(j, t);
    }
}

// sum_i sum_k in[(i * nj + j) * nk + k] by one workgroup; store(sum) once
template <typename F> __device__ __forceinline__ void reduce_job_body(const ReduceJob &jb, int j, F store) {
    __shared__ float red[4];
    float s = 0.f;
    const int total = jb.ni * jb.nk;
    // eight loads go out before the first is added: a load that is waited for costs microseconds here
    for (int t0 = threadIdx.x; t0 < total; t0 += 8 * NTHREADS) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int t = min(t0 + u * NTHREADS, total - 1), i = t / jb.nk, kk = t - i * jb.nk;
            v[u] = jb.in[((int64_t)i * jb.nj + j) * jb.nk + kk];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (t0 + u * NTHREADS < total) s += v[u];
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) store(red[0] + red[1] + red[2] + red[3]);
}

}  // namespace bm2
