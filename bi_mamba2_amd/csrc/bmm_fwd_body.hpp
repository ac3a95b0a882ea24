// The work of one workgroup of the C.B^T kernel.
#pragma once
#include "common.hpp"

namespace bm2 {

// =========================================================================================================
// CB[t, s] = sum_n C[t, n] B[s, n]
// =========================================================================================================
template <typename T> constexpr int BMM_FWD_LDS = 2 * 64 * Mma<T>::LD * (int)sizeof(T);
// lds: BMM_FWD_LDS bytes; st, tt: tile of columns and of rows; bcg: (batch, chunk, group)
template <typename T>
__device__ __forceinline__ void bmm_chunk_fwd_body(const bimamba2_params &p, int nc, int st, int tt, int bcg, char *lds) {
    constexpr int LD = Mma<T>::LD;
    T *As = reinterpret_cast<T *>(lds), *Bs = As + 64 * LD;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = bcg % p.ngroups, bc = bcg / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, N = p.dstate;
    const int limit = min(Q, p.seqlen - c * Q);
    const T *Cp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + tt * 64) * p.C_sl + g * p.C_sg;
    const T *Bp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + st * 64) * p.B_sl + g * p.B_sg;
    f32x4 acc[4] = {};
    for (int k0 = 0; k0 < N; k0 += BK) {
        __syncthreads();
        tile_load_kcontig<T, T, 64>(As, Cp + k0, p.C_sl, limit - tt * 64, N - k0, Ident());
        tile_load_kcontig<T, T, 64>(Bs, Bp + k0, p.B_sl, limit - st * 64, N - k0, Ident());
        __syncthreads();
        mma_tile<T, 4>(acc, As + wave * 16 * LD, Bs, lane);
    }
    float *out = p.CB + (int64_t)bcg * Q * Q;
    float *outT = p.CBT ? p.CBT + (int64_t)bcg * Q * Q : nullptr;   // CBT[s, t] = CB[t, s], read by the dx kernel
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = tt * 64 + wave * 16 + (lane >> 4) * 4 + i, s = st * 64 + j * 16 + (lane & 15);
            if (t < Q && s < Q) {
                out[(int64_t)t * Q + s] = acc[j][i];
                if (outT && Q % 4) outT[(int64_t)s * Q + t] = acc[j][i];
            }
        }
    if (outT && Q % 4 == 0) {
        // a lane's four rows of the tile are four consecutive columns of the transposed one
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = tt * 64 + wave * 16 + (lane >> 4) * 4, s = st * 64 + j * 16 + (lane & 15);
            if (t < Q && s < Q) *reinterpret_cast<f32x4 *>(outT + (int64_t)s * Q + t) = acc[j];
        }
    }
}

}  // namespace bm2
