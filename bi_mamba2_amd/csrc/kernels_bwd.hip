// Backward kernels of the bidirectional SSD operator for gfx950 (the gradient of the chunk-entry states and dx
// reuse chunk_state_kernel / chunk_scan_kernel from kernels_fwd.hip).
//   bwd_dz             dz and dout*silu(z)
//   state_passing_bwd  both inter-chunk adjoint recurrences in one launch + the chunk-total decay gradients
//   bwd_dbdc           state part of dB (or dC) summed over the heads of a group + per-position decay terms
//   bwd_dcb            G = dy.x^T once per head -> dCB (summed over heads) and the within-chunk decay gradient
//   bmm_chunk_bwd      dB = dBs + dCB^T.C ; dC = dCs + dCB.B
//   chunk_cumsum_bwd   assembles d(dt*A) from its pieces with wavefront scans; ddt, dA, ddt_bias
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "sums_body.hpp"
#include "bmm_fwd_body.hpp"
#include "dbdc_body.hpp"
#include "dcb_body.hpp"
#include "dcb_heads_body.hpp"
#include "dbdc_heads_body.hpp"

namespace bm2 {

static inline int nchunks(const bimamba2_params *p) { return (p->seqlen + p->chunk_size - 1) / p->chunk_size; }
static inline hipStream_t stream_of(const bimamba2_params *p) { return reinterpret_cast<hipStream_t>(p->stream); }

// block index of a kernel body that may run as one of several roles of a launch

// =========================================================================================================
__global__ void fill_kernel(float *ptr, size_t n, float value) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) ptr[i] = value;
}
int launch_fill(float *ptr, size_t n, float value, hipStream_t stream) {
    if (n == 0) return BIMAMBA2_OK;
    const int blocks = (int)std::min<size_t>((n + 255) / 256, 2048);
    hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(256), 0, stream, ptr, n, value);
    return check_launch();
}

// out[j] = sum_i sum_k in[(i*nj + j)*nk + k]; one workgroup per j
__global__ __launch_bounds__(NTHREADS) void reduce_kernel(const float *in, float *out, int ni, int nj, int nk) {
    __shared__ float red[4];
    const int j = blockIdx.x;
    float s = 0.f;
    const int total = ni * nk;
    for (int t = threadIdx.x; t < total; t += NTHREADS) {
        const int i = t / nk, k = t - i * nk;
        s += in[((int64_t)i * nj + j) * nk + k];
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[j] = red[0] + red[1] + red[2] + red[3];
}
int launch_reduce(const float *in, float *out, int ni, int nj, int nk, hipStream_t stream) {
    hipLaunchKernelGGL(reduce_kernel, dim3(nj), dim3(NTHREADS), 0, stream, in, out, ni, nj, nk);
    return check_launch();
}

// several such reductions in one launch (the backward pass ends with three small ones)
__global__ __launch_bounds__(NTHREADS) void reduce_jobs_kernel(ReduceJobs jobs) {
    int j = blockIdx.x, k = 0;
    while (k + 1 < jobs.n && j >= jobs.job[k].nj) { j -= jobs.job[k].nj; ++k; }
    float *out = jobs.job[k].out;
    reduce_job_body(jobs.job[k], j, [&](float v) { out[j] = v; });
}
int launch_reduce_jobs(const ReduceJobs &jobs, hipStream_t stream) {
    int blocks = 0;
    for (int k = 0; k < jobs.n; ++k) blocks += jobs.job[k].nj;
    if (blocks == 0) return BIMAMBA2_OK;
    hipLaunchKernelGGL(reduce_jobs_kernel, dim3(blocks), dim3(NTHREADS), 0, stream, jobs);
    return check_launch();
}

// The sums of a layer's backward pass in one launch, each in its parameter's type: those of the norm's weight, of the convolution's
// filter and bias, of A, D and dt_bias, and what were a conversion of each afterwards.  Every one of them is a launch of 4 to 7 us
// of which the chip is busy for less than one.  16 x 1024 positions, d_model 768, bfloat16: 24 -> 11 us,
// the layer 938 -> 930 (two runs of one build differ by 1); 4 x 2000, 640: 554 -> 540; 16 x 4000, 256: 969 -> 950.
struct SumTarget { void *out; const float *mul; int dtype; };
struct SumArgs {
    ColumnSums cols[3];
    SumTarget to_cols[3], to_extra[3];
    ReduceJob jobs[4];
    SumTarget to_jobs[4];
    int ncols, njobs;
};
__device__ __forceinline__ void store_sum(const SumTarget &t, int i, float v) {
    if (t.mul) v *= t.mul[i];
    if (t.dtype == BIMAMBA2_F32) reinterpret_cast<float *>(t.out)[i] = v;
    else if (t.dtype == BIMAMBA2_BF16) reinterpret_cast<bf16_t *>(t.out)[i] = from_f<bf16_t>(v);
    else reinterpret_cast<f16_t *>(t.out)[i] = from_f<f16_t>(v);
}
__global__ __launch_bounds__(NTHREADS) void layer_sums_kernel(SumArgs a) {
    int j = blockIdx.x, k = 0;
    for (; k < a.ncols; ++k) {
        const int nb = (a.cols[k].nj + 15) / 16;
        if (j < nb) break;
        j -= nb;
    }
    if (k < a.ncols) {
        const int W = a.cols[k].width;
        column_sums_body(a.cols[k].in, a.cols[k].ni, a.cols[k].nj, j, [&](int at, float v) {
            if (W == 0) { store_sum(a.to_cols[k], at, v); return; }
            const int c = at / (W + 1), tap = at - c * (W + 1);
            if (tap < W) store_sum(a.to_cols[k], c * W + tap, v);
            else if (a.to_extra[k].out) store_sum(a.to_extra[k], c, v);
        });
        return;
    }
    for (k = 0; k + 1 < a.njobs && j >= a.jobs[k].nj; ++k) j -= a.jobs[k].nj;
    reduce_job_body(a.jobs[k], j, [&](float v) { store_sum(a.to_jobs[k], j, v); });
}
int launch_layer_sums(const LayerSums &sums, const bimamba2_cast_params *casts, hipStream_t stream) {
    SumArgs a{};
    int blocks = 0, used = 0;
    auto target = [&](float *place, int64_t n, SumTarget &t) {
        t = SumTarget{place, nullptr, BIMAMBA2_F32};
        for (int i = 0; place && i < casts->count; ++i) {
            const bimamba2_cast_item &it = casts->item[i];
            if (it.src != place) continue;
            if (it.n != n || it.src_dtype != BIMAMBA2_F32 || it.op == BIMAMBA2_CAST_NEG_EXP) continue;
            t = SumTarget{it.dst, it.op == BIMAMBA2_CAST_MUL ? it.aux : nullptr, it.dst_dtype};
            ++used;
            break;
        }
    };
    for (int k = 0; k < sums.ncols; ++k) {
        const ColumnSums &c = sums.cols[k];
        a.cols[a.ncols] = c;
        target(c.out, c.width ? (int64_t)c.nj / (c.width + 1) * c.width : c.nj, a.to_cols[a.ncols]);
        target(c.extra, c.width ? c.nj / (c.width + 1) : 0, a.to_extra[a.ncols]);
        ++a.ncols;
        blocks += (c.nj + 15) / 16;
    }
    for (int k = 0; k < sums.jobs.n; ++k) {
        const ReduceJob &r = sums.jobs.job[k];
        a.jobs[a.njobs] = r;
        target(r.out, r.nj, a.to_jobs[a.njobs]);
        ++a.njobs;
        blocks += r.nj;
    }
    if (used != casts->count) return BIMAMBA2_EINVAL;
    hipLaunchKernelGGL(layer_sums_kernel, dim3(blocks), dim3(NTHREADS), 0, stream, a);
    return check_launch();
}

// =========================================================================================================
// dz = dout * out_x * sigmoid(z) (1 + z (1 - sigmoid(z)));  dout_x = dout * z * sigmoid(z)
// (by their float32 values: the same bits as from the kernel that also forms the states' gradients)
// =========================================================================================================
template <typename T>
__device__ __forceinline__ void bwd_dz_body(const bimamba2_params &p, int id, int nblocks) {
    constexpr int VS = 16 / sizeof(T);
    const int P = p.headdim;
    const int pv = (P + VS - 1) / VS;
    const int64_t nrows = (int64_t)p.batch * p.seqlen * p.nheads;
    const T *zb = reinterpret_cast<const T *>(p.z);
    const T *db = reinterpret_cast<const T *>(p.dout);
    const T *ox = reinterpret_cast<const T *>(p.out_x);
    T *dz = reinterpret_cast<T *>(p.dz);
    T *dox = reinterpret_cast<T *>(p.dout_x);
    // z and dout laid out like out_x (rows of headdim one behind the other, headdim a multiple of the vector): a vector
    // unit's offset is the same in all of them and no index has to be taken apart (three 64-bit divisions per unit, most of
    // the kernel's instructions otherwise)
    const bool packed = P % VS == 0 && p.z_sh == P && p.z_sl == (int64_t)p.nheads * P && p.z_sb == (int64_t)p.seqlen * p.nheads * P &&
                        p.dout_sh == P && p.dout_sl == p.z_sl && p.dout_sb == p.z_sb;
    for (int64_t idx = id * (int64_t)NTHREADS + threadIdx.x; idx < nrows * pv; idx += (int64_t)nblocks * NTHREADS) {
        const T *zp, *dp;
        int64_t o;
        int c0;
        if (packed) {
            o = idx * VS;
            c0 = 0;                               // (only its distance from the row's end matters below: a whole vector fits)
            zp = zb + o;
            dp = db + o;
        } else {
            const int64_t row = idx / pv;
            c0 = (int)(idx - row * pv) * VS;
            const int h = (int)(row % p.nheads);
            const int64_t bl = row / p.nheads;
            const int l = (int)(bl % p.seqlen), b = (int)(bl / p.seqlen);
            zp = zb + b * p.z_sb + l * p.z_sl + h * p.z_sh + c0;
            dp = db + b * p.dout_sb + l * p.dout_sl + h * p.dout_sh + c0;
            o = row * P + c0;
        }
        const bool vec = (c0 + VS <= P) && aligned16(zp, 0) && aligned16(dp, 0) && aligned16(ox + o, 0);
        float zv[VS], dv[VS], ov[VS];
        if (vec) {
            // all three are read for the last time in this pass
            const Vec16<T> a = __builtin_bit_cast(Vec16<T>, __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(zp))),
                           d = __builtin_bit_cast(Vec16<T>, __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(dp))),
                           e = __builtin_bit_cast(Vec16<T>, __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(ox + o)));
#pragma unroll
            for (int i = 0; i < VS; ++i) { zv[i] = to_f(a.v[i]); dv[i] = to_f(d.v[i]); ov[i] = to_f(e.v[i]); }
        } else {
#pragma unroll
            for (int i = 0; i < VS; ++i) {
                const bool ok = c0 + i < P;
                zv[i] = ok ? to_f(zp[i]) : 0.f; dv[i] = ok ? to_f(dp[i]) : 0.f; ov[i] = ok ? to_f(ox[o + i]) : 0.f;
            }
        }
        Vec16<T> r1, r2;
#pragma unroll
        for (int i = 0; i < VS; ++i) {
            const float sg = sigmoid_f(zv[i]);
            r1.v[i] = from_f32<T>(dv[i] * ov[i] * sg * (1.f + zv[i] * (1.f - sg)));
            r2.v[i] = from_f32<T>(dv[i] * zv[i] * sg);
        }
        if (vec) {
            // dz is not read again inside the pass, dout_x by four kernels: the first goes past the caches
            __builtin_nontemporal_store(__builtin_bit_cast(f32x4, r1), reinterpret_cast<f32x4 *>(dz + o));
            *reinterpret_cast<Vec16<T> *>(dox + o) = r2;
        } else {
#pragma unroll
            for (int i = 0; i < VS; ++i)
                if (c0 + i < P) { dz[o + i] = r1.v[i]; dox[o + i] = r2.v[i]; }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void bwd_dz_kernel(const bimamba2_params p) {
    bwd_dz_body<T>(p, blockIdx.x, gridDim.x);
}

// dz and C.B^T (where the forward pass did not keep it) in one launch: the tiles first, they are chains, the rest streams.
// 4 x 2048, bfloat16, 16 heads of 16, dstate 16: 6 + 7 -> 9 us.
template <typename T>
__global__ __launch_bounds__(NTHREADS) void bwd_dz_bmm_kernel(const bimamba2_params p, int nc, int nqt, int nbmm) {
    __shared__ __attribute__((aligned(16))) char lds[BMM_FWD_LDS<T>];
    const int id = blockIdx.x;
    if (id < nbmm) bmm_chunk_fwd_body<T>(p, nc, id % nqt, id / nqt % nqt, id / (nqt * nqt), lds);
    else bwd_dz_body<T>(p, id - nbmm, gridDim.x - nbmm);
}

static int dz_blocks(const bimamba2_params *p) {
    const int64_t n = (int64_t)p->batch * p->seqlen * p->nheads * ((p->headdim + 3) / 4);
    return (int)std::min<int64_t>((n + NTHREADS - 1) / NTHREADS, 8192);
}

int launch_bwd_dz_bmm(const bimamba2_params *p) {
    const int nc = nchunks(p), nqt = (p->chunk_size + 63) / 64, nbmm = nqt * nqt * p->batch * nc * p->ngroups;
    const dim3 grid(nbmm + dz_blocks(p));
    switch (p->dtype) {
        case BIMAMBA2_F32: hipLaunchKernelGGL(bwd_dz_bmm_kernel<float>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nbmm); break;
        case BIMAMBA2_BF16: hipLaunchKernelGGL(bwd_dz_bmm_kernel<bf16_t>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nbmm); break;
        case BIMAMBA2_F16: hipLaunchKernelGGL(bwd_dz_bmm_kernel<f16_t>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nbmm); break;
        default: return BIMAMBA2_EUNSUPPORTED;
    }
    return check_launch();
}

int launch_bwd_dz(const bimamba2_params *p) {
    const int blocks = dz_blocks(p);
    switch (p->dtype) {
        case BIMAMBA2_F32: hipLaunchKernelGGL(bwd_dz_kernel<float>, dim3(blocks), dim3(NTHREADS), 0, stream_of(p), *p); break;
        case BIMAMBA2_BF16: hipLaunchKernelGGL(bwd_dz_kernel<bf16_t>, dim3(blocks), dim3(NTHREADS), 0, stream_of(p), *p); break;
        case BIMAMBA2_F16: hipLaunchKernelGGL(bwd_dz_kernel<f16_t>, dim3(blocks), dim3(NTHREADS), 0, stream_of(p), *p); break;
        default: return BIMAMBA2_EUNSUPPORTED;
    }
    return check_launch();
}

// =========================================================================================================
// adjoint of the inter-chunk recurrences.  On entry dstates_* hold the gradient w.r.t. the state entering
// each chunk (dprev); on exit they hold the gradient w.r.t. each chunk's own state S[c]:
//   forward dir : g = dfinal_f (or 0); for c = nc-1..0 : dS_f[c] = g; ddA_chunk_f[c] = e^{tot_c} <g, prev_f[c]>; g = dprev_f[c] + e^{tot_c} g
//   reverse dir : g = dfinal_b (or 0); for c = 0..nc-1 : dS_b[c] = g; ddA_chunk_b[c] = e^{tot_c} <g, prev_b[c]>; g = dprev_b[c] + e^{tot_c} g
// What g holds at the end is the gradient with respect to the initial state (written to dinitial_* when given).
// A workgroup owns SP_EPT*256 of the P*N elements of one (b, h); its partial inner products go to
// ddA_chunk_*[b, h, c, split].
// =========================================================================================================
constexpr int SP_EPT = 4;
__global__ __launch_bounds__(NTHREADS) void state_passing_bwd_kernel(const bimamba2_params p, int nc, int nsplit) {
    __shared__ float red[2][4];
    const int PN = p.headdim * p.dstate;
    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Q = p.chunk_size;
    const float *csf = p.cs_f + ((int64_t)b * p.nheads + h) * nc * Q;
    const float *csb = p.cs_b + ((int64_t)b * p.nheads + h) * nc * Q;
    const int64_t cstride = (int64_t)p.nheads * PN;
    const int64_t base = ((int64_t)b * nc * p.nheads + h) * PN;
    const int e0 = split * SP_EPT * NTHREADS + threadIdx.x;
    for (int dir = 0; dir < 2; ++dir) {
        const float *prev = (dir == 0 ? p.states_f : p.states_b) + base;
        float *ds = (dir == 0 ? p.dstates_f : p.dstates_b) + base;
        float *dda = (dir == 0 ? p.ddA_chunk_f : p.ddA_chunk_b) + ((int64_t)b * p.nheads + h) * nc * nsplit + split;
        const float *dfin = dir == 0 ? p.dfinal_f : p.dfinal_b;
        float *dini = dir == 0 ? p.dinitial_f : p.dinitial_b;
        const int64_t bh = ((int64_t)b * p.nheads + h) * PN;
        float g[SP_EPT];
#pragma unroll
        for (int i = 0; i < SP_EPT; ++i) {
            const int e = e0 + i * NTHREADS;
            g[i] = (dfin && e < PN) ? dfin[bh + e] : 0.f;
        }
        for (int step = 0; step < nc; ++step) {
            const int c = dir == 0 ? nc - 1 - step : step;
            const float dec = __expf(dir == 0 ? csf[(int64_t)c * Q + Q - 1] : csb[(int64_t)c * Q]);
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < SP_EPT; ++i) {
                const int e = e0 + i * NTHREADS;
                if (e < PN) {
                    const int64_t a = c * cstride + e;
                    const float dp = ds[a];
                    dot += g[i] * prev[a];
                    ds[a] = g[i];
                    g[i] = dp + dec * g[i];
                }
            }
            dot = wave_sum(dot);
            if (lane == 0) red[step & 1][wave] = dot;
            __syncthreads();
            if (threadIdx.x == 0) dda[(int64_t)c * nsplit] = dec * (red[step & 1][0] + red[step & 1][1] + red[step & 1][2] + red[step & 1][3]);
        }
        if (dini) {
#pragma unroll
            for (int i = 0; i < SP_EPT; ++i) {
                const int e = e0 + i * NTHREADS;
                if (e < PN) dini[bh + e] = g[i];
            }
        }
        __syncthreads();
    }
}

// The same with 16-byte accesses, one direction per workgroup (blockIdx.z = 2 b + dir) and the loads of SP_CH chunks in
// flight before the first of them is used: the recurrence is a chain over the chunks, and a global access that has to be
// waited for at every link costs microseconds.  Needs P*N % 4 == 0 and 16-byte aligned tensors.
// PREV16: the entering states are read from their 16-bit copies (states16_*); DS16: the gradients with respect to the
// entering states go to dstates16_* and the per-chunk gradients in dstates_* stay as they are.
// DP16 (with DS16): the per-chunk gradients lie in dstates16_* in the 16-bit type as well (no float32 tensors): every one is
// read once and replaced in place by the gradient with respect to the state entering its chunk.
constexpr int SP_CH = 8;
// AHEAD: the next SP_CH chunks are on their way while the present ones are worked on, and the inner products are handed out every
// SP_FLUSH chunks instead of every SP_CH (a barrier waits for the loads in flight): the launch of its own, whose workgroups have nothing
// else to cover a round trip with.  As a role beside dCB the kernel keeps to that one's registers and LDS.
constexpr int SP_FLUSH = 64;
// A workgroup takes one or several groups of SP_EPT * NTHREADS elements of a head.  Bound by the time of its one round trip to memory, so what
// counts is how much it asks for at once.  Short sequences: several groups, so that all its loads in flight are of use (with
// one group, and the loads behind the last chunk repeating it, a pass over one chunk asked eight times for everything).  As a role
// of the dCB launch, which has room for two of these a CU: two groups of long sequences too.  Both roles, heads of 64, bfloat16: 32 x 256, 24 heads,
// one chunk 60 -> 37 us; 16 x 512, 24 heads, 2 chunks 46 -> 36; 16 x 1024, 24 heads, 4 chunks 71 -> 64; 4 x 2048, 32 heads, 8 chunks 49 -> 43; 4 x 4096, 8
// groups, 16 chunks 129 -> 125; dstate 128, 2 x 3001, 24 heads 36 -> 34.
inline int sp_bwd_groups(int nc) { return nc <= 2 ? 4 : nc <= 4 ? 2 : 1; }
template <typename T16, bool PREV16, bool DS16, bool DP16, bool AHEAD, int NCH, int NG>
__device__ __forceinline__ void state_passing_bwd_groups(const bimamba2_params &p, int nc, int nsplit, int ndir, BlockId bid, float (*red)[4]) {
    struct alignas(8) V4 { T16 v[4]; };
    constexpr int NU = NCH * NG, FLUSH = AHEAD && NG == 1 ? SP_FLUSH : NU > SP_CH ? NU : SP_CH;
    static_assert(FLUSH <= SP_FLUSH, "rows of red");
    const int PN = p.headdim * p.dstate;
    const int split = bid.x * NG, h = bid.y, b = bid.z / ndir, dir = bid.z % ndir;   // ndir = 1: forward direction only
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Q = p.chunk_size;
    const float *cs = (dir == 0 ? p.cs_f : p.cs_b) + ((int64_t)b * p.nheads + h) * nc * Q + (dir == 0 ? Q - 1 : 0);
    const int64_t cstride = (int64_t)p.nheads * PN;
    const int64_t base = ((int64_t)b * nc * p.nheads + h) * PN;
    const float *prev = (dir == 0 ? p.states_f : p.states_b) + base;
    const T16 *prev16 = reinterpret_cast<const T16 *>(dir == 0 ? p.states16_f : p.states16_b) + base;
    float *ds = (dir == 0 ? p.dstates_f : p.dstates_b) + base;
    T16 *ds16 = reinterpret_cast<T16 *>(dir == 0 ? p.dstates16_f : p.dstates16_b) + base;
    float *dda = (dir == 0 ? p.ddA_chunk_f : p.ddA_chunk_b) + ((int64_t)b * p.nheads + h) * nc * nsplit + split;
    const float *dfin = dir == 0 ? p.dfinal_f : p.dfinal_b;
    float *dini = dir == 0 ? p.dinitial_f : p.dinitial_b;
    const int64_t bh = ((int64_t)b * p.nheads + h) * PN;
    bool live[NG];
    int e[NG];
    f32x4 g[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) {
        const int own = ((split + u) * NTHREADS + threadIdx.x) * SP_EPT;
        live[u] = own < PN;
        e[u] = live[u] ? own : PN - SP_EPT;                // loads are unconditional (so that they all go out together)
        g[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (dfin) g[u] = *reinterpret_cast<const f32x4 *>(dfin + bh + e[u]);
    }
    // the gradient of the recurrence's last chunk leads to the initial states only: without them its neighbour is read in its place
    const int last = dini || nc == 1 ? nc - 1 : nc - 2;
    // (as they lie in memory, converted where they are used: a conversion beside its load waits for it, and the loads went out one by one)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    struct Batch {
        typename std::conditional<DP16, f32x2, f32x4>::type dp[NU];
        typename std::conditional<PREV16, f32x2, f32x4>::type pv[NU];
        float dec[NCH];
    };
    auto wide = [](auto v) __attribute__((always_inline)) {
        if constexpr (sizeof(v) == 16) return v;
        else {
            const V4 t = __builtin_bit_cast(V4, v);
            return f32x4{to_f(t.v[0]), to_f(t.v[1]), to_f(t.v[2]), to_f(t.v[3])};
        }
    };
    auto load = [&](int s0, Batch &r) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int sj = min(s0 + j, nc - 1);            // past the last chunk: a valid chunk again, never used
            const int c = dir == 0 ? nc - 1 - sj : sj;
            r.dec[j] = cs[(int64_t)c * Q];
            const int sd = min(sj, last);
            const int64_t od = (dir == 0 ? nc - 1 - sd : sd) * cstride, op = c * cstride;
#pragma unroll
            for (int u = 0; u < NG; ++u) {
                const int k = j * NG + u;
                // (both are read for the last time in the pass: past the caches)
                if constexpr (DP16) r.dp[k] = *reinterpret_cast<const f32x2 *>(ds16 + e[u] + od);
                else r.dp[k] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(ds + e[u] + od));
                if constexpr (PREV16) r.pv[k] = __builtin_nontemporal_load(reinterpret_cast<const f32x2 *>(prev16 + e[u] + op));
                else r.pv[k] = *reinterpret_cast<const f32x4 *>(prev + e[u] + op);
            }
        }
    };
    // (the recurrence and its stores first, then all inner products' sums side by side: one after the other, each a chain of six
    // exchanges between the lanes, they were half of the kernel's time.  1 x 16384 in chunks of 128, 16 heads of 32, dstate 32: 61 -> 50 us
    // with the next chunks under way, -> 27 with the sums side by side; beside dCB, 1 x 16384, 8 heads of 64, the pass 186 -> 172)
    auto recur = [&](int s0, int nb, const Batch &r, float (&dot)[NU], auto WHOLE) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            if (decltype(WHOLE)::value || j < nb) {
                const int c = dir == 0 ? nc - 1 - (s0 + j) : s0 + j;
                const float d = __expf(r.dec[j]);
#pragma unroll
                for (int u = 0; u < NG; ++u) {
                    if (NG > 1 && !live[u]) continue;
                    const int k = j * NG + u;
                    f32x4 &gu = g[u];
                    const f32x4 pv = wide(r.pv[k]);
                    dot[k] = (gu[0] * pv[0] + gu[1] * pv[1] + gu[2] * pv[2] + gu[3] * pv[3]) * d;
                    if constexpr (DS16) {
                        V4 t;
                        // (by the float32 value: a row's gradients do not depend on how many rows there are, i.e. on NG)
#pragma unroll
                        for (int i = 0; i < 4; ++i) t.v[i] = from_f32<T16>(gu[i]);
                        *reinterpret_cast<V4 *>(ds16 + e[u] + c * cstride) = t;
                    } else {
                        *reinterpret_cast<f32x4 *>(ds + e[u] + c * cstride) = gu;
                    }
                    gu = wide(r.dp[k]) + d * gu;
                }
            }
        }
    };
    auto work = [&](int s0, const Batch &r) __attribute__((always_inline)) {
        const int nb = min(NCH, nc - s0);
        float dot[NU] = {};
        if (NG > 1 || live[0]) {
            if (nb == NCH) recur(s0, nb, r, dot, std::true_type());
            else recur(s0, nb, r, dot, std::false_type());
        }
#pragma unroll
        for (int j = 0; j < NU; ++j) dot[j] = row16_sum(dot[j]);
#pragma unroll
        for (int m = 16; m <= 32; m <<= 1)
#pragma unroll
            for (int j = 0; j < NU; ++j) dot[j] += __shfl_xor(dot[j], m, 64);
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < NU; ++j) red[s0 * NG % FLUSH + j][wave] = dot[j];      // (behind the last chunk: never read)
        }
        // chunks up to s0 + nb: hand the inner products out when their place is full, or at the end
        const int done = s0 + nb;
        if (done * NG % FLUSH == 0 || done == nc) {
            __syncthreads();
            const int from = (done - 1) / (FLUSH / NG) * (FLUSH / NG), i = threadIdx.x;
            if (i < (done - from) * NG && split + i % NG < nsplit) {
                const int c = dir == 0 ? nc - 1 - (from + i / NG) : from + i / NG;
                dda[(int64_t)c * nsplit + i % NG] = red[i][0] + red[i][1] + red[i][2] + red[i][3];
            }
            __syncthreads();
        }
    };
    if constexpr (AHEAD && NG == 1) {
        Batch one, two;
        load(0, one);
        for (int s0 = 0; s0 < nc; s0 += 2 * NCH) {
            if (s0 + NCH < nc) load(s0 + NCH, two);
            work(s0, one);
            if (s0 + NCH >= nc) break;
            if (s0 + 2 * NCH < nc) load(s0 + 2 * NCH, one);
            work(s0 + NCH, two);
        }
    } else {
        for (int s0 = 0; s0 < nc; s0 += NCH) {
            Batch one;
            load(s0, one);
            work(s0, one);
        }
    }
    if (dini)
#pragma unroll
        for (int u = 0; u < NG; ++u)
            if (live[u]) *reinterpret_cast<f32x4 *>(dini + bh + e[u]) = g[u];
}
// red: SP_FLUSH rows of LDS; ngr: groups a workgroup (2 also for long sequences, where TWO)
template <typename T16, bool PREV16, bool DS16, bool DP16 = false, bool AHEAD = false, bool TWO = false>
__device__ __forceinline__ void state_passing_bwd_vec_body(const bimamba2_params &p, int nc, int nsplit, int ndir, BlockId bid, float (*red)[4], int ngr = 1) {
    if (nc == 1) state_passing_bwd_groups<T16, PREV16, DS16, DP16, AHEAD, 1, 4>(p, nc, nsplit, ndir, bid, red);
    else if (nc == 2) state_passing_bwd_groups<T16, PREV16, DS16, DP16, AHEAD, 2, 4>(p, nc, nsplit, ndir, bid, red);
    else if (nc <= 4) state_passing_bwd_groups<T16, PREV16, DS16, DP16, AHEAD, 4, 2>(p, nc, nsplit, ndir, bid, red);
    else {
        if constexpr (TWO)
            if (ngr == 2) return state_passing_bwd_groups<T16, PREV16, DS16, DP16, AHEAD, SP_CH, 2>(p, nc, nsplit, ndir, bid, red);
        state_passing_bwd_groups<T16, PREV16, DS16, DP16, AHEAD, SP_CH, 1>(p, nc, nsplit, ndir, bid, red);
    }
}
template <typename T16, bool PREV16, bool DS16, bool DP16 = false>
__global__ __launch_bounds__(NTHREADS) void state_passing_bwd_vec_kernel(const bimamba2_params p, int nc, int nsplit, int ndir) {
    __shared__ float red[SP_FLUSH][4];
    state_passing_bwd_vec_body<T16, PREV16, DS16, DP16, true>(p, nc, nsplit, ndir, BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z}, red);
}

int launch_state_passing_bwd(const bimamba2_params *p) {
    const int nc = nchunks(p), PN = p->headdim * p->dstate;
    const int nsplit = (PN + SP_EPT * NTHREADS - 1) / (SP_EPT * NTHREADS);
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    const int ndir = p->causal ? 1 : 2;
    if (PN % 4 == 0 && al(p->states_f) && al(p->states_b) && al(p->dstates_f) && al(p->dstates_b) && al(p->dfinal_f) && al(p->dfinal_b) &&
        al(p->dinitial_f) && al(p->dinitial_b)) {
        const int ngr = sp_bwd_groups(nc);
        dim3 grid((nsplit + ngr - 1) / ngr, p->nheads, p->batch * ndir);
        const bool prev16 = p->states16_f != nullptr, ds16 = p->dstates16_f != nullptr;
        if (prev16 && (!(p->causal || p->states16_b) || !al(p->states16_f) || !al(p->states16_b))) return BIMAMBA2_EINVAL;
        if (ds16 && (!(p->causal || p->dstates16_b) || !al(p->dstates16_f) || !al(p->dstates16_b))) return BIMAMBA2_EINVAL;
        if ((prev16 || ds16) && p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
        if (!p->dstates_f) {
            // the per-chunk gradients lie in dstates16_* (16-bit): in place; known with the 16-bit copies on both sides only
            if (!(prev16 && ds16)) return BIMAMBA2_EINVAL;
            if (p->dtype == BIMAMBA2_F16) hipLaunchKernelGGL((state_passing_bwd_vec_kernel<f16_t, true, true, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsplit, ndir);
            else hipLaunchKernelGGL((state_passing_bwd_vec_kernel<bf16_t, true, true, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsplit, ndir);
            return check_launch();
        }
#define BM2_SPB(TT, A, B) hipLaunchKernelGGL((state_passing_bwd_vec_kernel<TT, A, B>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsplit, ndir)
        if (p->dtype == BIMAMBA2_F16) {
            if (prev16 && ds16) BM2_SPB(f16_t, true, true); else if (prev16) BM2_SPB(f16_t, true, false);
            else if (ds16) BM2_SPB(f16_t, false, true); else BM2_SPB(f16_t, false, false);
        } else {
            if (prev16 && ds16) BM2_SPB(bf16_t, true, true); else if (prev16) BM2_SPB(bf16_t, true, false);
            else if (ds16) BM2_SPB(bf16_t, false, true); else BM2_SPB(bf16_t, false, false);
        }
#undef BM2_SPB
        return check_launch();
    }
    if (p->states16_f || p->dstates16_f) return BIMAMBA2_EUNSUPPORTED;
    if (p->causal) return BIMAMBA2_EUNSUPPORTED;
    if (!p->dstates_f || !p->dstates_b) return BIMAMBA2_EINVAL;
    dim3 grid(nsplit, p->nheads, p->batch);
    hipLaunchKernelGGL(state_passing_bwd_kernel, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsplit);
    return check_launch();
}

// =========================================================================================================
// dB and dC, state part (the kernel for float32 state tensors: dbdc_body.hpp)
// =========================================================================================================
static bool dcb_aligned(const bimamba2_params *p);
static bool dcb_rows_in_32bit(const bimamba2_params *p);
static double dbdc_heads_cost(const bimamba2_params *p, int w, int hps);
static bool dx_db_dc_pays(const bimamba2_params *p);
// 16-byte aligned rows of B and C
static bool bmm_rows_aligned(const bimamba2_params *p) {
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    return al(p->Bm) && al(p->Cm) && p->B_sb % 8 == 0 && p->B_sl % 8 == 0 && p->B_sg % 8 == 0 && p->C_sb % 8 == 0 && p->C_sl % 8 == 0 && p->C_sg % 8 == 0;
}
static inline int dbdc_heads(const bimamba2_params *p) { return p->dbdc_heads > 0 ? p->dbdc_heads : DBDC_HEADS; }
static inline int dbdc_slices(const bimamba2_params *p) { return (p->nheads / p->ngroups + dbdc_heads(p) - 1) / dbdc_heads(p); }
// of them, those there are to add up: none where nothing wrote a state part (one_chunk())
static inline int state_slices(const bimamba2_params *p) { return p->dBs ? dbdc_slices(p) : 0; }

// Heads per slice where the caller leaves the choice (the partial sums are bimamba2_bwd's own).  A workgroup of the dB / dC
// kernels fills a CU, needs about three head steps to start (measured: 17 us for 8 heads, of which 5 before the first) and
// then one per head; each slice more is a partial sum of each of dB and dC that is written and read again.  With eight heads
// a slice, small problems leave most of the chip idle: 24 workgroups at batch 2 x 1500 with 8 heads of 128 channels, where the
// two kernels took 22 us each and take 12 with one head a slice.
static int dbdc_places(const bimamba2_params *p) { return p->dstate <= 32 ? 512 : 256; }      // workgroups on the chip at once (narrow states: two to a CU)
int choose_dbdc_heads(const bimamba2_params *p, bool by_heads, bool together) {
    const int hpg = p->nheads / p->ngroups, nc = nchunks(p);
    if (by_heads) {
        // the same for the kernel whose waves take whole heads, dB and dC in one launch (us; a partial sum of each at 5 TB/s)
        const double slice_cost = (double)p->batch * p->seqlen * p->ngroups * p->dstate * 8 * 2 / 5e6;
        int best = hpg;
        double best_cost = 0;
        for (int s = 1; s <= std::min(hpg, DBDC_SLICES_MAX); ++s) {
            const int hps = (hpg + s - 1) / s;
            if ((hpg + hps - 1) / hps != s) continue;
            double cost = dbdc_heads_cost(p, 4, hps);
            for (int w = 2; w >= 1; w /= 2) cost = std::min(cost, dbdc_heads_cost(p, w, hps));
            cost += s * slice_cost;
            if (s == 1 || cost < best_cost) { best = hps; best_cost = cost; }
        }
        return best;
    }
    const int64_t tiles = (int64_t)p->batch * nc * p->ngroups * ((p->chunk_size + 127) / 128);
    const double steps = ((p->headdim + 63) / 64) * ((p->dstate + 63) / 64);                             // per head
    const double slice_cost = (double)p->batch * p->seqlen * p->ngroups * p->dstate * 8 / 5e6 / 1.5;     // one partial sum at 5 TB/s, in steps of 1.5 us
    // Where both roles share a launch (db_dc_roles()) they share the chip, and half the slices are less to add up.  us a pass with one
    // launch, slices as for two launches and as here: float32, 2 x 1111, 16 heads of 64, dstate 64, 187 -> 177; 4 x 1024, 8 heads of 128
    // 222 -> 213.  With dx in front of them in it no round of theirs starts at once: they take the places that dx leaves one after the other, so
    // what counts is their work over all places, and the last workgroup, which ends alone.  us a pass, slices as for two launches / by half
    // the places / as here: bfloat16, heads of 32, dstate 16, two groups, 16 x 520, 16 heads 162 / 167 / 164; 20 x 500, heads of 16, dstate 32
    // 173 / 178 / 173; 4 x 2048, 16 heads of 16, dstate 16 137 / 132 / 133; float32, 1 x 6000, 16 heads of 32 179 / 182 / 180; 16 x 520
    // 265 / 247 / 247; 8 x 520 157 / 161 / 159.  (Wider states, whose workgroups have a CU each, keep to rounds: float32, 2 x 196, 8 groups of
    // 2 heads of 64, dstate 64 89 / 89, by the work 93; 2 x 300, 16 heads of 16 in two groups, dstate 96 103 / 101; bfloat16, 2 x 900, 16 heads of 16 in four, dstate 48
    // 91 / 86.)
    const int64_t places = dbdc_places(p) / (together ? 2 : 1);
    const bool behind_dx = together && p->dstate <= 32 && dx_db_dc_pays(p);
    int best = DBDC_HEADS;
    double best_cost = 0;
    for (int k = DBDC_HEADS; k >= 1; --k) {
        const int slices = (hpg + k - 1) / k;
        if (k < DBDC_HEADS && (slices > DBDC_SLICES_MAX || (hpg + slices - 1) / slices != k)) continue;  // (the fewest heads for this many slices)
        const double life = 3 + steps * std::min(k, hpg);
        const double cost = (behind_dx ? (double)(tiles * slices) / places + 1.5 : (double)((tiles * slices + places - 1) / places)) * life + slices * slice_cost;
        if (k == DBDC_HEADS || cost < best_cost) { best = k; best_cost = cost; }
    }
    return best;
}

// dB and dC by waves that take whole heads (dbdc_heads_body.hpp): headdim 64 or 128, dstate 64, the states and their gradients in 16-bit
// copies.  bwd_dbdc_dma_kernel below took 20.6 + 18.8 us for dC and dB at 4 x 2048 with 32 heads: its x and dout fragments come straight
// from memory, 16 bytes of 16 different rows to a request, so the address unit was busy four times as long as the bytes
// need, and a third of its life went by before the first product.  Here every request is of whole rows, a wave waits for nobody, and
// both roles share a launch: 28.7; 4 x 4096, 8 groups of 4 heads 108 -> 70; 16 x 1024, 24 heads 61.5 -> 37.8; heads
// of 128: 2 x 1500, 8 heads 18.6 -> 13.5; 4 x 2048, 16 heads 33.5 -> 28.5; 2 x 8192, 24 heads in 4 groups 97 -> 82.  What is left is the sums:
// 32 additions of a state's product into the lane's sums and 32 into the rows' per 16 matrix instructions of 8 cycles.
// (Counters, 4 x 2048, 32 heads: vector units busy 42 % of the time, matrix units 14 %, LDS 29 % without conflicts, and a third of the waves' time is spent
// waiting for an instruction: 219 registers leave two waves a SIMD, which do not cover each other.)
// (dC's workgroups in front, unless they form the product)
template <typename T, int W, bool PRODUCT>
__global__ __launch_bounds__(NTHREADS, 2) void bwd_dbdc_heads_kernel(const bimamba2_params p, int nc, int nqt, int hps, int gdx, int gdy, int gdz) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[DbdcHeadsMap<W>::LDS];
    const int per = gdx * gdy, half = per * gdz, lin = blockIdx.x;
    int id = lin % half;
    bool is_db = lin >= half;
    // With the product both roles read the (batch, chunk, group)'s dCB and its B and C rows: eight dC workgroups, one per XCD, then the eight of dB beside
    // them.  4 x 4096, 32 heads in 8 groups: 414 -> 363 MB read, 82 -> 81 us; 16 x 1024, 24 heads 44.6 -> 40.9; 16 heads 31.2 -> 29.5.
    if (PRODUCT && half % 8 == 0) {
        is_db = (lin >> 3) & 1;
        id = (lin >> 4) * 8 + (lin & 7);
    }
    BlockId bid = dcb_block_of(id % per, gdx, gdy, per, DCB_HEADS_RESIDENT);
    bid.z = id / per;
    if (is_db) bwd_dbdc_heads_body<T, true, W, PRODUCT>(p, nc, nqt, hps, bid, smem);
    else bwd_dbdc_heads_body<T, false, W, PRODUCT>(p, nc, nqt, hps, bid, smem);
}
// us: with the chip full (two workgroups on a CU) a wave's head takes 5.6, with one on a CU 3.8, start and end 6.  dC and dB
// in one launch: 4 x 2048, 32 heads, two slices: 28.7 with four waves to a tile (four heads each), one slice 34.5; with two waves
// 36.6, with one 58.4; 4 x 4096 with 8 groups of 4 heads: 96, 77, 70 with four, two and one.
static double dbdc_heads_cost(const bimamba2_params *p, int w, int hps) {
    const int hpg = p->nheads / p->ngroups, nqt = (p->chunk_size + 63) / 64, slices = (hpg + hps - 1) / hps;
    const double full = (double)p->batch * nchunks(p) * p->ngroups * nqt * w / 4 * slices * 2 / DCB_HEADS_RESIDENT;
    const double rounds = std::max(1.0, (full + std::ceil(full)) / 2);      // (a last round that is nearly empty costs more than its share)
    return rounds * (6 + (2 + 3.6 * std::min(std::max(full, 0.5), 1.0)) * ((std::min(hps, hpg) + w - 1) / w) * (p->headdim / 64));
}
static int dbdc_waves(const bimamba2_params *p, int hps) {
    int best = 4;
    for (int w = 2; w >= 1; w /= 2)
        if (dbdc_heads_cost(p, w, hps) < dbdc_heads_cost(p, best, hps)) best = w;
    return best;
}
// the states' copies aside, which a caller may bring
bool dbdc_by_heads(const bimamba2_params *p) {
    return p->dtype != BIMAMBA2_F32 && !p->causal && p->headdim % 64 == 0 && p->dstate == 64 && p->chunk_size % 64 == 0 && dcb_aligned(p) && dcb_rows_in_32bit(p) &&
           bmm_rows_aligned(p);
}
bool dbdc_both_by_heads(const bimamba2_params *p) {
    auto al = [](const void *q) { return q && (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    return dbdc_by_heads(p) && al(p->states16_f) && al(p->states16_b) && al(p->dstates16_f) && al(p->dstates16_b);
}
// Where one slice holds all heads of a group, the workgroup that has summed a tile's state parts forms the part inside the chunk too and writes dB and
// dC themselves: 16 MB of partial sums and 16 MB of dCB's transpose less per 64 (batch, chunk, group), and the last launch is left with the cumulative
// sums.  Not below 16 (batch, chunk, group), where the last launch ran beside them for nothing and the product is one more chain of
// waits.  us of the three launches (dCB, dB with dC, the last one), 16 bits, dstate 64, without -> with: 8 (b, c, g): 8 heads 29.1 -> 29.9, 4 heads 26.6 ->
// 27.7; 16: 3 heads 28.8 -> 29.1, 4 heads 30.7 -> 30.2, 4 heads of 128 33.5 -> 32.2; 32: 8 heads 37.1 -> 36.4; 64 of 8 heads in two groups 47.4 -> 44.4, of 16 in
// one 89.3 -> 90.1, of 24 130 -> 124; 128 of 4 heads 68 -> 58, of 8 heads 111 -> 98, of 4 heads of 128 104 -> 89; 512 of 4 heads 136 + 71 + 65 -> 131 + 81 + 15
// (4 x 4096, 32 heads in 8 groups), a training pass there 526 -> 485.
bool dbdc_with_product(const bimamba2_params *p) {
    auto in32 = [](int64_t stride) { return stride >= 0 && stride < (1 << 22); };      // (its rows of B and C are 32-bit offsets, as those of x)
    return dbdc_both_by_heads(p) && bwd_tail_merged(p) && dbdc_slices(p) == 1 && in32(p->B_sl) && in32(p->C_sl) &&
           (int64_t)p->batch * nchunks(p) * p->ngroups >= 16;
}
template <typename T, int W> static void launch_dbdc_both_w(const bimamba2_params *p, int nqt, int hps, bool product) {
    const int nc = nchunks(p), gdx = p->batch * nc * p->ngroups, gdy = (nqt * W + 3) / 4, gdz = dbdc_slices(p);
    const dim3 grid(2 * gdx * gdy * gdz);
    if (product) hipLaunchKernelGGL((bwd_dbdc_heads_kernel<T, W, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, hps, gdx, gdy, gdz);
    else hipLaunchKernelGGL((bwd_dbdc_heads_kernel<T, W, false>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, hps, gdx, gdy, gdz);
}
template <typename T> static int launch_dbdc_both_t(const bimamba2_params *p, bool product) {
    const int nqt = p->chunk_size / 64, hps = dbdc_heads(p), W = dbdc_waves(p, hps);
    if (W == 4) launch_dbdc_both_w<T, 4>(p, nqt, hps, product);
    else if (W == 2) launch_dbdc_both_w<T, 2>(p, nqt, hps, product);
    else launch_dbdc_both_w<T, 1>(p, nqt, hps, product);
    return check_launch();
}
int launch_dbdc_both(const bimamba2_params *p, bool product) {
    return p->dtype == BIMAMBA2_BF16 ? launch_dbdc_both_t<bf16_t>(p, product) : launch_dbdc_both_t<f16_t>(p, product);
}

// Two waves to a SIMD, said explicitly: with the bound left out the two-tile variant takes 140 us instead of 40 (float32, heads of 16,
// dstate 128, 4 x 2048, 16 heads; the same registers, another order of instructions).  With all four column tiles the registers do not allow more: held to
// four waves it spills 17 to 43 of them (33 -> 54 us).
template <typename T, int NT, int QT, bool IS_DB, bool FAST, bool UNI = false, int NJ = 4>
__global__ __launch_bounds__(DBDC_THREADS, NJ < 4 ? 4 : 2) void bwd_dbdc_kernel(const bimamba2_params p, int nc, int hps) {
    __shared__ __attribute__((aligned(16))) char lds[DbdcMap<T, QT>::LDS];
    bwd_dbdc_body<T, NT, QT, IS_DB, FAST, UNI, NJ>(p, nc, hps, BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z}, lds);
}

// ---------------------------------------------------------------------------------------------------------
// The same for 16-bit types with dstate 64 or 128 and headdim % 64 == 0, with every load of the head loop taken out of the
// compiler's hands.  The workgroup is alone on its CU (register-bound), so nothing hides a load it waits for; here the
// float32 state tiles of a step travel straight into a 3-slot LDS ring (no registers), two steps ahead of their use, and
// the x / dout fragments into registers, likewise two steps ahead, from inline assembly.  A step then reads its tiles
// from the ring, transposes them in registers into the 16-bit operand image as before, and multiplies.  All LDS traffic
// of the loop goes through the raw accessors (an access the compiler knows of would wait for every request in flight).
// Order of a wave's vector memory operations per step: NDIR * 2 ring requests, then QT * 2 fragment loads; "at most one
// step's worth outstanding" therefore means that the step in hand has landed.
// ---------------------------------------------------------------------------------------------------------
// S16: the state tiles come from their 16-bit copies (states16_* / dstates16_*).  They lie in the ring as they lie in
// memory ([p][n], 16-byte chunks swizzled as tile64_request does), and the operand fragments are LDS transpose reads
// straight from the ring slot: no operand image, one barrier per step, a third of the LDS.
// NT: 64-column tiles of the state dimension (1 or 2).  A step multiplies one of them: step = (head, n tile, headdim chunk).
template <typename T, int QT, bool IS_DB, bool UNI, bool S16, int NT = 1>
__global__ __launch_bounds__(DBDC_THREADS) void bwd_dbdc_dma_kernel(const bimamba2_params p, int nc, int hps) {
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    static_assert(sizeof(T) == 2, "16-bit operands");
    constexpr int KSTEP = 32, KC = 64, NKS = 2, VK = 8, LDX = KC + VK;
    constexpr int ROWS = DBDC_WAVES * 16 * QT;
    constexpr int NBLK = (KC / VK) * 16;                       // 8 x 4 blocks of a 64 x 64 tile
    constexpr int RING = 3, NDIR = UNI ? 1 : 2;
    constexpr int TILE_B = 64 * 64 * (S16 ? 2 : 4);            // bytes of a state tile
    constexpr int IMG_B = 64 * LDX * 2;                        // bytes of a 16-bit operand image
    constexpr int PER_STEP = NDIR * (S16 ? 1 : 2) + QT * NKS;  // vector memory operations of a wave per step
    static_assert(NDIR * NBLK <= DBDC_THREADS, "one block per thread");
    static_assert(NT == 1 || NT == 2, "state dimension 64 or 128");
    static_assert(DBDC_WAVES == 8, "a wave brings 8 (16-bit) resp. 2 x 4 (float32) rows of each tile");
    __shared__ __attribute__((aligned(16))) unsigned char ring[RING * NDIR * TILE_B];
    __shared__ __attribute__((aligned(16))) unsigned char img[S16 ? 16 : 2 * NDIR * IMG_B];
    __shared__ __attribute__((aligned(16))) float sfs[DBDC_HEADS][ROWS], sbs[DBDC_HEADS][ROWS];
    // the per-head decay gradients wait here for the end of the kernel: a global store inside the loop would sit in the
    // same counter as the requests and be waited for with them
    __shared__ __attribute__((aligned(16))) float uvs[DBDC_HEADS][NDIR][ROWS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int rt = blockIdx.y;
    const int g = blockIdx.x % p.ngroups, bc = blockIdx.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, N = p.dstate, P = p.headdim, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int r0 = rt * ROWS;
    const int hh0 = blockIdx.z * hps, hh_end = min(hpg, hh0 + hps);
    const int nkc = P / KC, per_head = nkc * NT, nsteps = (hh_end - hh0) * per_head;
    int arow[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) arow[q] = min(r0 + (wave * QT + q) * 16 + lr, limit - 1);

    // requests of a step: this wave's two 4-row units of each state tile, then its fragments
    auto issue_states = [&](int step) {
        const int hh = hh0 + step / per_head, kc = step % nkc, nt = NT == 1 ? 0 : (step / nkc) % NT, h = g * hpg + hh;
        const int64_t so = ((int64_t)(b * nc + c) * H + h) * P * N + (int64_t)kc * KC * N + nt * 64;
#pragma unroll
        for (int d = 0; d < NDIR; ++d) {
            if constexpr (S16) {
                // rows 8 wave .. 8 wave + 7, 16-byte chunk (lane % 8) ^ swizzle(row) at chunk position lane % 8
                const T *st = reinterpret_cast<const T *>(IS_DB ? (d ? p.dstates16_b : p.dstates16_f) : (d ? p.states16_b : p.states16_f)) + so;
                const int row = wave * 8 + (lane >> 3);
                load16_to_lds(st + row * (64 * NT) + (((lane & 7) ^ tile64_swz(row)) << 3), ring + ((step % RING) * NDIR + d) * TILE_B + wave * 1024);
            } else {
                const float *st = (IS_DB ? (d ? p.dstates_b : p.dstates_f) : (d ? p.states_b : p.states_f)) + so;
#pragma unroll
                for (int uu = 0; uu < 2; ++uu) {
                    const int u = wave * 2 + uu;
                    load16_to_lds(st + (4 * u + (lane >> 4)) * (64 * NT) + (lane & 15) * 4, ring + ((step % RING) * NDIR + d) * TILE_B + u * 1024);
                }
            }
        }
    };
    auto issue_frags = [&](int step, Frag (&af)[QT][NKS]) {
        const int hh = hh0 + step / per_head, kc = step % nkc, h = g * hpg + hh;
        const T *ap;
        int64_t as;
        if (IS_DB) { as = p.x_sl; ap = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * as + h * p.x_sh; }
        else if (p.has_z) { as = (int64_t)H * P; ap = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * as + (int64_t)h * P; }
        else { as = p.dout_sl; ap = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * as + h * p.dout_sh; }
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) af[q][ks] = raw_global_load_b128<Frag>(ap + (int64_t)arow[q] * as + kc * KC + ks * KSTEP + lg * 8);
    };
    Frag afA[QT][NKS], afB[QT][NKS];                           // fragments of the even / odd steps
    issue_states(0);
    issue_frags(0, afA);
    if (nsteps > 1) { issue_states(1); issue_frags(1, afB); }

    // ---- everything below up to the loop is ordinary code; its waits drain the requests above, which costs nothing here ----
    int tl[QT][4];
#pragma unroll
    for (int q = 0; q < QT; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) tl[q][i] = (wave * QT + q) * 16 + lg * 4 + i;
    // one round trip for everything the loop needs besides its requests: the decay vectors of the slice's heads and the
    // B / C values of this lane's output elements, all loaded unconditionally from clamped addresses before the first use
    constexpr int NTAB = DBDC_HEADS * ROWS / DBDC_THREADS;
    static_assert(NTAB * DBDC_THREADS == DBDC_HEADS * ROWS, "table entries per thread");
    float t_dt[NTAB], t_cf[NTAB], t_cb[NTAB], t_ef[NTAB], t_eb[NTAB];
#pragma unroll
    for (int it = 0; it < NTAB; ++it) {
        const int idx = threadIdx.x + it * DBDC_THREADS;
        const int hh = min(idx / ROWS, hh_end - hh0 - 1), r = min(r0 + idx % ROWS, limit - 1);
        const int64_t o = (((int64_t)b * H + g * hpg + hh0 + hh) * nc + c) * Q;
        t_cf[it] = p.cs_f[o + r];
        t_cb[it] = UNI ? 0.f : p.cs_b[o + r];
        t_dt[it] = IS_DB ? p.dt_out[o + r] : 0.f;
        t_ef[it] = IS_DB ? p.cs_f[o + Q - 1] : 0.f;
        t_eb[it] = (IS_DB && !UNI) ? p.cs_b[o] : 0.f;
    }
    const T *cbp;
    int64_t cbs;
    if (IS_DB) { cbs = p.B_sl; cbp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + r0) * cbs + g * p.B_sg; }
    else { cbs = p.C_sl; cbp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + r0) * cbs + g * p.C_sg; }
    float creg[NT][QT][4][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) creg[nt][q][j][i] = to_f(cbp[(int64_t)min(tl[q][i], limit - 1 - r0) * cbs + nt * 64 + j * 16 + lr]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (r0 + tl[q][i] >= limit) creg[nt][q][j][i] = 0.f;
#pragma unroll
    for (int it = 0; it < NTAB; ++it) {
        const int idx = threadIdx.x + it * DBDC_THREADS;
        const int hh = idx / ROWS, rl = idx % ROWS;
        if (hh < hh_end - hh0) {
            float f = 0.f, rv = 0.f;
            if (r0 + rl < limit) {
                if (IS_DB) {
                    f = t_dt[it] * __expf(t_ef[it] - t_cf[it]);
                    rv = UNI ? 0.f : t_dt[it] * __expf(t_eb[it] - t_cb[it]);
                } else {
                    f = __expf(t_cf[it]);
                    rv = UNI ? 0.f : __expf(t_cb[it]);
                }
            }
            sfs[hh][rl] = f;
            sbs[hh][rl] = rv;
        }
    }
    f32x4 tot[NT][QT][4] = {};
    __syncthreads();

    // ---- the head loop: raw LDS accesses and counted waits only ----
    const int sblk = threadIdx.x % NBLK, stile = threadIdx.x / NBLK;       // staging: tile stile, block (s_kb, s_rb)
    const int s_rb = sblk % 16, s_kb = sblk / 16;
    const unsigned ring_a = lds_addr(ring) + stile * TILE_B + (s_kb * VK) * 256 + s_rb * 16;
    const unsigned img_w = lds_addr(img) + stile * IMG_B;
    unsigned img_wo[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) img_wo[rr] = img_w + xt_index<T, LDX>(s_rb * 4 + rr, s_kb * VK) * 2;
    unsigned img_r[NKS][4];                                    // operand fragments of this lane (the swizzle depends on the row block)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int j = 0; j < 4; ++j) img_r[ks][j] = lds_addr(img) + xt_index<T, LDX>(j * 16 + lr, ks * KSTEP + lg * 8) * 2;
    const unsigned sfs_a = lds_addr(sfs) + ((wave * QT) * 16 + lg * 4) * 4, sbs_a = lds_addr(sbs) + ((wave * QT) * 16 + lg * 4) * 4;
    const unsigned uvs_a = lds_addr(uvs) + ((wave * QT) * 16 + lg * 4) * 4;
    // S16: lane parts of the transpose reads (see tile64_tr_frag): rows kk .. kk + 3 and kk + 4 .. kk + 7 of a K step,
    // 4 columns from 16 j + nn on; the K step adds 32 rows = 4096 bytes (the swizzle repeats every 16 rows)
    unsigned tr_lo[4], tr_hi[4];
    {
        const int kk = 8 * lg + (lr >> 2), nn = 4 * (lr & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            tr_lo[j] = lds_addr(ring) + tile64_tr_offset(kk, j * 16 + nn);
            tr_hi[j] = lds_addr(ring) + tile64_tr_offset(kk + 4, j * 16 + nn);
        }
    }
    f32x4 tf[QT][4], tb[QT][4];
    float uf[NT == 1 ? 1 : QT][4], ub[NT == 1 ? 1 : QT][4];     // (NT > 1: decay-gradient sums over the n tiles of a head)
    // SLOT = step % RING as a compile-time value: the slot's offset goes into the offset field of the LDS reads
    auto step_body = [&](int step, Frag (&af)[QT][NKS], auto SLOT) {
        constexpr int RB = decltype(SLOT)::value * NDIR * TILE_B;
        const int hh = hh0 + step / per_head, kc = step % nkc;
        // this wave's requests of the step have landed (those of the next step may be outstanding) ...
        if (step + 1 < nsteps) wait_vmcnt<PER_STEP>();
        else wait_vmcnt<0>();
        raw_lds_barrier();                                     // ... and everybody's; ring slot and image of step - 1 are free
        if (step + 2 < nsteps) issue_states(step + 2);
        const int buf = step & 1;
        if constexpr (!S16) {
        if (stile < NDIR) {
            // 8 rows (k = p) x 4 columns (n) of the tile from the ring, transposed into the image
            const unsigned ra = ring_a + ((step % RING) * NDIR) * TILE_B;
            f32x4 v[VK];
            v[0] = raw_lds_read_at<f32x4, 0>(ra); v[1] = raw_lds_read_at<f32x4, 256>(ra);
            v[2] = raw_lds_read_at<f32x4, 512>(ra); v[3] = raw_lds_read_at<f32x4, 768>(ra);
            v[4] = raw_lds_read_at<f32x4, 1024>(ra); v[5] = raw_lds_read_at<f32x4, 1280>(ra);
            v[6] = raw_lds_read_at<f32x4, 1536>(ra); v[7] = raw_lds_read_at<f32x4, 1792>(ra);
            raw_lds_wait();
#pragma unroll
            for (int kk = 0; kk < VK; ++kk) raw_lds_use(v[kk]);
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                Vec16<T> o;
#pragma unroll
                for (int kk = 0; kk < VK; ++kk) o.v[kk] = from_f<T>(v[kk][rr]);
                raw_lds_write128_at<0>(img_wo[rr] + buf * NDIR * IMG_B, __builtin_bit_cast(f32x4, o));
            }
        }
        raw_lds_wait();
        raw_lds_barrier();
        }
        // (the first products of a head start from a literal zero: no registers to clear between heads)
        const bool first = kc == 0;
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) raw_lds_use(af[q][ks]);
        const unsigned ib = buf * NDIR * IMG_B;
        if constexpr (S16) {
            // both K halves' fragments are asked for at once; the products of the first half run while the second half's
            // reads are still under way (LDS reads return in order: "at most NR outstanding" = the first half is there)
            static_assert(NKS == 2, "two K halves");
            constexpr int NR = UNI ? 8 : 16;                   // LDS reads per K half
            i16x4 flo[NKS][4], fhi[NKS][4], blo[NKS][4], bhi[NKS][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                flo[0][j] = raw_lds_tr16_read_at<RB>(tr_lo[j]); fhi[0][j] = raw_lds_tr16_read_at<RB>(tr_hi[j]);
                if (!UNI) { blo[0][j] = raw_lds_tr16_read_at<RB + TILE_B>(tr_lo[j]); bhi[0][j] = raw_lds_tr16_read_at<RB + TILE_B>(tr_hi[j]); }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                flo[1][j] = raw_lds_tr16_read_at<RB + 4096>(tr_lo[j]); fhi[1][j] = raw_lds_tr16_read_at<RB + 4096>(tr_hi[j]);
                if (!UNI) { blo[1][j] = raw_lds_tr16_read_at<RB + TILE_B + 4096>(tr_lo[j]); bhi[1][j] = raw_lds_tr16_read_at<RB + TILE_B + 4096>(tr_hi[j]); }
            }
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                // lgkmcnt(min(NR, 15)), vmcnt and expcnt left alone (the counter has four bits: 15 is its largest value)
                if (ks == 0) __builtin_amdgcn_s_waitcnt(0xC07F | ((NR < 15 ? NR : 15) << 8));
                else raw_lds_wait();
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    raw_lds_use(flo[ks][j]); raw_lds_use(fhi[ks][j]);
                    const Frag bff = __builtin_bit_cast(Frag, __builtin_shufflevector(flo[ks][j], fhi[ks][j], 0, 1, 2, 3, 4, 5, 6, 7));
                    Frag bfb = bff;
                    if (!UNI) {
                        raw_lds_use(blo[ks][j]); raw_lds_use(bhi[ks][j]);
                        bfb = __builtin_bit_cast(Frag, __builtin_shufflevector(blo[ks][j], bhi[ks][j], 0, 1, 2, 3, 4, 5, 6, 7));
                    }
#pragma unroll
                    for (int q = 0; q < QT; ++q) {
                        if (ks == 0 && first) {
                            tf[q][j] = M::mma(af[q][ks], bff, f32x4{0.f, 0.f, 0.f, 0.f});
                            if (!UNI) tb[q][j] = M::mma(af[q][ks], bfb, f32x4{0.f, 0.f, 0.f, 0.f});
                        } else {
                            tf[q][j] = M::mma(af[q][ks], bff, tf[q][j]);
                            if (!UNI) tb[q][j] = M::mma(af[q][ks], bfb, tb[q][j]);
                        }
                    }
                }
            }
        } else {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            Frag bff[4], bfb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                bff[j] = raw_lds_read_at<Frag, 0>(img_r[ks][j] + ib);
                if (!UNI) bfb[j] = raw_lds_read_at<Frag, IMG_B>(img_r[ks][j] + ib);
            }
            raw_lds_wait();
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                raw_lds_use(bff[j]);
                if (!UNI) raw_lds_use(bfb[j]);
#pragma unroll
                for (int q = 0; q < QT; ++q) {
                    if (ks == 0 && first) {
                        tf[q][j] = M::mma(af[q][ks], bff[j], f32x4{0.f, 0.f, 0.f, 0.f});
                        if (!UNI) tb[q][j] = M::mma(af[q][ks], bfb[j], f32x4{0.f, 0.f, 0.f, 0.f});
                    } else {
                        tf[q][j] = M::mma(af[q][ks], bff[j], tf[q][j]);
                        if (!UNI) tb[q][j] = M::mma(af[q][ks], bfb[j], tb[q][j]);
                    }
                }
            }
        }
        }
        // the fragments of step + 2 take the place of the ones just used
        if (step + 2 < nsteps) issue_frags(step + 2, af);
        if (kc == nkc - 1) {
            // ---- end of a head's n tile: its share of dB / dC and of the decay gradients.  (The tile's registers are picked by
            // a compile-time index: the caller's branch on the tile is uniform.)
            auto finish = [&](auto NTI) {
                constexpr int nt = decltype(NTI)::value;
#pragma unroll
                for (int q = 0; q < QT; ++q) {
                    f32x4 sf4 = raw_lds_read_at<f32x4, 0>(sfs_a + ((hh - hh0) * ROWS + q * 16) * 4);
                    f32x4 sb4 = raw_lds_read_at<f32x4, 0>(sbs_a + ((hh - hh0) * ROWS + q * 16) * 4);
                    raw_lds_wait();
                    raw_lds_use(sf4); raw_lds_use(sb4);
                    f32x4 av, bv;
                    constexpr int UQ = NT == 1 ? 0 : 1;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float fs = nt == 0 ? 0.f : uf[q * UQ][i], bs = nt == 0 ? 0.f : ub[q * UQ][i];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            fs += tf[q][j][i] * creg[nt][q][j][i];
                            if (!UNI) bs += tb[q][j][i] * creg[nt][q][j][i];
                            tot[nt][q][j][i] += UNI ? sf4[i] * tf[q][j][i] : sf4[i] * tf[q][j][i] + sb4[i] * tb[q][j][i];
                        }
                        if constexpr (nt < NT - 1) {
                            uf[q * UQ][i] = fs;
                            ub[q * UQ][i] = bs;
                        } else {
                            av[i] = row16_sum(fs) * sf4[i];
                            bv[i] = UNI ? 0.f : row16_sum(bs) * sb4[i];
                        }
                    }
                    if constexpr (nt == NT - 1) {
                        if (lr == 0) {
                            const unsigned ua = uvs_a + (((hh - hh0) * NDIR) * ROWS + q * 16) * 4;
                            raw_lds_write128_at<0>(ua, av);
                            if (!UNI) raw_lds_write128_at<ROWS * 4>(ua, bv);
                        }
                    }
                }
            };
            if constexpr (NT == 1) finish(std::integral_constant<int, 0>());
            else if ((step / nkc) % NT == 0) finish(std::integral_constant<int, 0>());
            else finish(std::integral_constant<int, 1>());
        }
    };
    static_assert(RING == 3, "six steps = one round of ring slots and of the two fragment sets");
    for (int step = 0; step < nsteps; step += 6) {
        step_body(step, afA, std::integral_constant<int, 0>());
        if (step + 1 < nsteps) step_body(step + 1, afB, std::integral_constant<int, 1>());
        if (step + 2 < nsteps) step_body(step + 2, afA, std::integral_constant<int, 2>());
        if (step + 3 < nsteps) step_body(step + 3, afB, std::integral_constant<int, 0>());
        if (step + 4 < nsteps) step_body(step + 4, afA, std::integral_constant<int, 1>());
        if (step + 5 < nsteps) step_body(step + 5, afB, std::integral_constant<int, 2>());
    }
    raw_lds_wait();
    __syncthreads();                                           // nothing is in flight any more: ordinary code again
    for (int idx = threadIdx.x; idx < (hh_end - hh0) * NDIR * ROWS; idx += DBDC_THREADS) {
        const int hh = idx / (NDIR * ROWS), d = (idx / ROWS) % NDIR, rl = idx % ROWS;
        if (r0 + rl < Q) {
            float *dst = IS_DB ? (d ? p.v_b : p.v_f) : (d ? p.u_b : p.u_f);
            dst[(((int64_t)b * H + g * hpg + hh0 + hh) * nc + c) * Q + r0 + rl] = uvs[hh][d][rl];
        }
    }
    float *out = (IS_DB ? p.dBs : p.dCs) + (int64_t)blockIdx.z * p.batch * p.seqlen * p.ngroups * N;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = nt * 64 + j * 16 + lr, r = r0 + tl[q][i];
                    if (r < limit) out[(((int64_t)b * p.seqlen + (int64_t)c * Q + r) * p.ngroups + g) * N + n] = tot[nt][q][j][i];
                }
}

template <typename T, bool IS_DB>
static int launch_dbdc_t(const bimamba2_params *p) {
    const int nc = nchunks(p);
    if (dbdc_heads(p) > DBDC_HEADS) return BIMAMBA2_EINVAL;
    const int nt = (p->dstate + 63) / 64;
    // 16-row tiles per wave: two (a 256-row chunk reads each state once) where that still gives every CU a workgroup
    int qt = (p->chunk_size > 128 && nt == 1 && (int64_t)p->batch * nc * p->ngroups * dbdc_slices(p) >= 256) ? 2 : 1;
    const int rows = DBDC_WAVES * 16 * qt;
    dim3 grid(p->batch * nc * p->ngroups, (p->chunk_size + rows - 1) / rows, dbdc_slices(p));
    constexpr int VS = 16 / (int)sizeof(T);
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    bool fast = p->headdim % 64 == 0 && p->dstate % 64 == 0;
    if (IS_DB) fast = fast && al(p->x) && p->x_sb % VS == 0 && p->x_sl % VS == 0 && p->x_sh % VS == 0;
    else fast = fast && (p->has_z ? al(p->dout_x) : (al(p->dout) && p->dout_sb % VS == 0 && p->dout_sl % VS == 0 && p->dout_sh % VS == 0));
#define BM2_DBDC(NTV, QTV)                                                                                                    \
    do {                                                                                                                  \
        if (fast) hipLaunchKernelGGL((bwd_dbdc_kernel<T, NTV, QTV, IS_DB, true>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p)); \
        else hipLaunchKernelGGL((bwd_dbdc_kernel<T, NTV, QTV, IS_DB, false>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));     \
    } while (0)
    if constexpr (sizeof(T) == 2) {
        // dstate 64 and 128: the variant with the ring of state tiles (16-byte aligned state tensors)
        const void *c16f = IS_DB ? p->dstates16_f : p->states16_f, *c16b = IS_DB ? p->dstates16_b : p->states16_b;
        const bool st_al = c16f ? al(c16f) && al(c16b) && (p->causal || c16b)
                                : (IS_DB ? al(p->dstates_f) && al(p->dstates_b) : al(p->states_f) && al(p->states_b));
        if (fast && p->dstate == 128 && st_al && !p->causal) {
            grid.y = (p->chunk_size + DBDC_WAVES * 16 - 1) / (DBDC_WAVES * 16);
            if (c16f) hipLaunchKernelGGL((bwd_dbdc_dma_kernel<T, 1, IS_DB, false, true, 2>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
            else hipLaunchKernelGGL((bwd_dbdc_dma_kernel<T, 1, IS_DB, false, false, 2>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
            return check_launch();
        }
        if (fast && p->dstate == 64 && st_al) {
            // 128-row tiles here: with eight heads per slice that is still one workgroup per CU at the usual sizes, and
            // the partial sums the slices leave behind (and bmm_chunk_bwd reads again) are half of what four heads give
            qt = 1;
            grid.y = (p->chunk_size + DBDC_WAVES * 16 - 1) / (DBDC_WAVES * 16);
#define BM2_DMA(QTV, UNIV)                                                                                                                  \
    do {                                                                                                                                    \
        if (c16f) hipLaunchKernelGGL((bwd_dbdc_dma_kernel<T, QTV, IS_DB, UNIV, true>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));   \
        else hipLaunchKernelGGL((bwd_dbdc_dma_kernel<T, QTV, IS_DB, UNIV, false>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));       \
    } while (0)
            if (p->causal) { BM2_DMA(1, true); }
            else { BM2_DMA(1, false); }
#undef BM2_DMA
            return check_launch();
        }
    }
    if (IS_DB ? p->dstates16_f : p->states16_f) return BIMAMBA2_EUNSUPPORTED;   // only the kernel above knows the 16-bit copies
    if (p->causal) {
        if constexpr (sizeof(T) == 2) {
            if (fast && nt == 1) {
                if (qt == 2) hipLaunchKernelGGL((bwd_dbdc_kernel<T, 1, 2, IS_DB, true, true>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
                else hipLaunchKernelGGL((bwd_dbdc_kernel<T, 1, 1, IS_DB, true, true>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
                return check_launch();
            }
        }
        return BIMAMBA2_EUNSUPPORTED;
    }
    if (nt == 1 && qt == 2) BM2_DBDC(1, 2);
    else if (p->dstate <= 16) hipLaunchKernelGGL((bwd_dbdc_kernel<T, 1, 1, IS_DB, false, false, 1>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
    else if (p->dstate <= 32) hipLaunchKernelGGL((bwd_dbdc_kernel<T, 1, 1, IS_DB, false, false, 2>), grid, dim3(DBDC_THREADS), 0, stream_of(p), *p, nc, dbdc_heads(p));
    else if (nt == 1) BM2_DBDC(1, 1);
    else if (nt == 2) BM2_DBDC(2, 1);
    else if (nt <= 4) BM2_DBDC(4, 1);
    else return BIMAMBA2_EUNSUPPORTED;
#undef BM2_DBDC
    return check_launch();
}

int launch_bwd_dbdc(const bimamba2_params *p, bool is_db) {
    switch (p->dtype) {
        case BIMAMBA2_F32: return is_db ? launch_dbdc_t<float, true>(p) : launch_dbdc_t<float, false>(p);
        case BIMAMBA2_BF16: return is_db ? launch_dbdc_t<bf16_t, true>(p) : launch_dbdc_t<bf16_t, false>(p);
        case BIMAMBA2_F16: return is_db ? launch_dbdc_t<f16_t, true>(p) : launch_dbdc_t<f16_t, false>(p);
        default: return BIMAMBA2_EUNSUPPORTED;
    }
}

// (what a workgroup does: dcb_body.hpp)
template <typename T, bool FAST>
__global__ __launch_bounds__(NTHREADS) void bwd_dcb_kernel(const bimamba2_params p, int nc, int nqt) {
    __shared__ __attribute__((aligned(16))) char lds[DcbMap::LDS];
    bwd_dcb_body<T, FAST>(p, nc, nqt, BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z}, gridDim.x, gridDim.z, lds);
}

// dst[i] += sum_{s=1..nslices-1} dst[s*n + i], for dst0 and dst1 (blockIdx.y)
__global__ __launch_bounds__(NTHREADS) void sum_slices_kernel(float *dst0, float *dst1, size_t n4, int nslices) {
    float4 *d = reinterpret_cast<float4 *>(blockIdx.y ? dst1 : dst0);
    for (size_t i = blockIdx.x * (size_t)NTHREADS + threadIdx.x; i < n4; i += (size_t)gridDim.x * NTHREADS) {
        float4 v = d[i];
        for (int s = 1; s < nslices; ++s) {
            const float4 u = d[s * n4 + i];
            v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
        }
        d[i] = v;
    }
}

// Head slices of the dCB kernel unless the caller says otherwise: one per 32 heads of a group (on grids that fill the chip more
// slices only cost traffic: 512 tiles of 24 heads 38 us in one slice, 42 in two; for small grids see choose_dcb_slices).
int dcb_slices(const bimamba2_params *p) {
    if (p->dcb_slices > 0) return p->dcb_slices;
    const int hpg = p->nheads / p->ngroups;
    return std::max(1, std::min(DCB_SLICES_MAX, hpg / DCB_SLICE_HEADS));
}

template <typename T, bool UNI = false, int KC = 64, bool WHOLE = true>
__global__ __launch_bounds__(NTHREADS) void bwd_dcb_ring_kernel(const bimamba2_params p, int nc, int nqt) {
    BlockId bid = dcb_block_of(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x, gridDim.y, gridDim.x * gridDim.y);
    bid.z = blockIdx.z;
    __shared__ __attribute__((aligned(16))) unsigned char smem[DcbRingMap<KC>::LDS];
    bwd_dcb_ring_body<T, UNI, KC, WHOLE>(p, nc, nqt, bid, gridDim.x, gridDim.z, smem);
}

template <typename T, bool UNI, int W>
__global__ __launch_bounds__(NTHREADS, 2) void bwd_dcb_heads_kernel(const bimamba2_params p, int nc, int nqt, int gdx, int gdy, int gdz) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[DcbHeadsMap<W>::LDS];
    const int id = blockIdx.x, per = gdx * gdy;
    BlockId bid = dcb_block_of(id % per, gdx, gdy, per, DCB_HEADS_RESIDENT);
    bid.z = id / per;
    bwd_dcb_heads_body<T, UNI, W>(p, nc, nqt, bid, gdx, gdz, smem, false);
}

// The dCB kernel and the backward state passing as roles of one launch: the first is bound by instruction issue and moves little data, the
// second streams 70 MB and needs few instructions, and the two depend on different kernels before them.  The first ndcb blocks are the
// dCB tiles, the rest are the state passing's, which take the places that the tiles leave one after the other: heads of 64, 45 us for both
// against 41 + 13 in two launches (4 x 2048, 32 heads), 121 against 109 + 23 (4 x 4096, 8 groups); with the state passing's blocks first
// 50 and 122, and 47 against 34 at dstate 128 (2 x 3001, 24 heads).
// W: the waves that share a tile in the kernel above (gdy: workgroups a (b, c, g)); 0: the ring, a tile a workgroup
template <typename T, bool UNI, int W>
__global__ __launch_bounds__(NTHREADS, W ? 2 : 1) void bwd_dcb_sp_kernel(const bimamba2_params p, int nc, int nqt, int gdx, int gdy, int gdz, int nsplit, int nspx, int ndir, bool out16) {
    const int id = blockIdx.x, per = gdx * gdy, ndcb = per * gdz;
    // (one place for both roles: with 1 KB more the ring's workgroups are three to a CU instead of four: 2 x 8192, 24 heads of 128 160 us instead of 148)
    __shared__ __attribute__((aligned(16))) unsigned char smem[W ? DcbHeadsMap<W ? W : 1>::LDS : DcbRingMap<64>::LDS];
    if (id < ndcb) {
        BlockId tile = dcb_block_of(id % per, gdx, gdy, per, W ? DCB_HEADS_RESIDENT : 1024);
        tile.z = id / per;
        if constexpr (W > 0) bwd_dcb_heads_body<T, UNI, W>(p, nc, nqt, tile, gdx, gdz, smem, out16);
        else bwd_dcb_ring_body<T, UNI, 64, true>(p, nc, nqt, tile, gdx, gdz, smem, out16);
    } else {
        const int k = id - ndcb;                  // grid (nspx, nheads, batch * ndir) of the state passing
        const BlockId sb{k % nspx, (k / nspx) % p.nheads, k / (nspx * p.nheads)};
        const int ngr = (nsplit + nspx - 1) / nspx;
        float (*red)[4] = reinterpret_cast<float (*)[4]>(smem);
        if (p.dstates_f == nullptr) state_passing_bwd_vec_body<T, true, true, true, false, W != 0>(p, nc, nsplit, ndir, sb, red, ngr);
        else if (p.dstates16_f == nullptr) state_passing_bwd_vec_body<T, false, false, false, false, W != 0>(p, nc, nsplit, ndir, sb, red, ngr);
        else state_passing_bwd_vec_body<T, true, true>(p, nc, nsplit, ndir, sb, red);
    }
}
// Waves that share a tile of the kernel above.  More of them split a tile's heads and finish sooner, fewer leave out the exchange at the end
// and the repeated C.B^T and keep their requests under way over more heads.  What is compared is rounds of the 512 workgroups that the
// chip holds times a workgroup's start and end (8 us) and heads (2.9 us each), and a tile to every wave pays for the unequal
// tiles (those on the diagonal take longer) while there are few rounds.  us with 4 / 2 / 1 waves (heads of 64, dstate 64):
//   512 tiles: 4 heads 12 / 14 / 19, 32 heads 34 / 51 / 90; 1024: 4 heads 20 / 16 / 20, 24 heads 47 / 45 / 70; 2048: 4 heads 37 / 27 / 27,
//   24 heads 93 / 78 / 102; 4096: 2 heads 62 / 41 / 34, 8 heads 90 / 80 / 72; 8192: 4 heads 130 / 98 / 81, 8 heads 181 / 149 / 137
static int dcb_waves(const bimamba2_params *p, int slices, double *us = nullptr) {
    const int nqt = (p->chunk_size + 63) / 64, heads = (p->nheads / p->ngroups + slices - 1) / slices;
    const double tiles = (double)p->batch * nchunks(p) * p->ngroups * nqt * nqt * slices;
    int best = 4;
    double best_cost = 0;
    for (int w = 4; w >= 1; w /= 2) {
        const double full = tiles * w / (4 * DCB_HEADS_RESIDENT), rounds = (full + std::ceil(full)) / 2;      // (a last round that is nearly empty costs more than its share)
        const double cost = (std::max(1.0, rounds) + (w == 1 ? 0.3 : 0.0)) * (8 + 2.9 * ((heads + w - 1) / w));
        if (w == 4 || cost < best_cost) { best = w; best_cost = cost; }
    }
    if (us) *us = best_cost;
    return best;
}
// Whether the state passing that shares dCB's launch is the longer part: float32 states (their gradients read and written, the states read:
// 12 bytes an element at 5 TB/s).  The ring's workgroups are four to a CU and stay so beside it, those of the kernel above fill the LDS by
// twos and it has to wait for them.  us ring / heads: 4 x 2048, 32 heads, dstate 96 (300 MB) 66 / 70, 12 heads in 4 groups, 2 x 8192, chunks of 128, dstate 96 (230 MB) 77 / 75
// to 91; but 8 groups of 4, dstate 32 (100 MB) 50 / 50, 1 x 4096, 24 heads, dstate 128 (75 MB) 40 / 30
static bool dcb_sp_streams(const bimamba2_params *p, int slices) {
    if (p->dstates16_f || !p->dstates_f) return false;
    double us;
    dcb_waves(p, slices, &us);
    return (double)p->batch * nchunks(p) * p->nheads * p->headdim * p->dstate * (p->causal ? 12 : 24) / 5e6 > us;
}
template <typename T, bool UNI> static void launch_dcb_heads(const bimamba2_params *p, int nc, int nqt, int slices) {
    const int W = dcb_waves(p, slices), gdx = p->batch * nc * p->ngroups, gdy = (nqt * nqt * W + 3) / 4;
    const dim3 g(gdx * gdy * slices);
    if (W == 4) hipLaunchKernelGGL((bwd_dcb_heads_kernel<T, UNI, 4>), g, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, gdx, gdy, slices);
    else if (W == 2) hipLaunchKernelGGL((bwd_dcb_heads_kernel<T, UNI, 2>), g, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, gdx, gdy, slices);
    else hipLaunchKernelGGL((bwd_dcb_heads_kernel<T, UNI, 1>), g, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, gdx, gdy, slices);
}
// Narrow heads (16-bit) take the ring as well: through registers a workgroup waits for its operands head by head.  4 x 2048 in chunks of
// 128, 16 heads of 16: 46 -> 21 us; 48 heads of 16: the whole pass 497 -> 389 us; in 8 groups (two heads a tile) 43 -> 28 us.
template <typename T> static void launch_dcb_ring(dim3 grid, const bimamba2_params *p, int nc, int nqt) {
    if constexpr (sizeof(T) == 2) {
        if (p->headdim == 64) {
            if (p->causal) launch_dcb_heads<T, true>(p, nc, nqt, grid.z);
            else launch_dcb_heads<T, false>(p, nc, nqt, grid.z);
        } else if (p->causal) hipLaunchKernelGGL((bwd_dcb_ring_kernel<T, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
        else if (p->headdim <= 32) hipLaunchKernelGGL((bwd_dcb_ring_kernel<T, false, 32, false>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
        else if (p->headdim % 64) hipLaunchKernelGGL((bwd_dcb_ring_kernel<T, false, 64, false>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
        else hipLaunchKernelGGL((bwd_dcb_ring_kernel<T>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
    }
}

// whether the dCB kernel can do without CB (it rebuilds its tile from the C and B rows): the 16-bit ring variant, dstate a
// multiple of 32, 16-byte aligned row matrices
// the ring variant addresses the rows of a chunk with 32-bit byte offsets from a per-head base
static bool dcb_rows_in_32bit(const bimamba2_params *p) {
    // (a query that comes before dout is known - no pointer, no strides yet - is answered for the contiguous tensor)
    const int64_t ys = (p->has_z || !p->dout) ? (int64_t)p->nheads * p->headdim : p->dout_sl;
    return p->x_sl > 0 && p->x_sl < (1 << 22) && ys > 0 && ys < (1 << 22);
}

bool dcb_recomputes_cb(const bimamba2_params *p) {
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    auto mult = [](int64_t a, int64_t b, int64_t c) { return a % 8 == 0 && b % 8 == 0 && c % 8 == 0; };
    if (p->dtype == BIMAMBA2_F32 || p->headdim % 64 || p->chunk_size % 64 || p->dstate % 32 || !dcb_rows_in_32bit(p)) return false;
    if (!(al(p->x) && mult(p->x_sb, p->x_sl, p->x_sh))) return false;
    if (!(p->has_z ? al(p->dout_x) : (al(p->dout) && mult(p->dout_sb, p->dout_sl, p->dout_sh)))) return false;
    return al(p->Bm) && mult(p->B_sb, p->B_sl, p->B_sg) && al(p->Cm) && mult(p->C_sb, p->C_sl, p->C_sg);
}

static bool dcb_aligned(const bimamba2_params *p) {
    const int vs = p->dtype == BIMAMBA2_F32 ? 4 : 8;
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    const bool x = al(p->x) && p->x_sb % vs == 0 && p->x_sl % vs == 0 && p->x_sh % vs == 0;
    return x && (p->has_z ? al(p->dout_x) : (al(p->dout) && p->dout_sb % vs == 0 && p->dout_sl % vs == 0 && p->dout_sh % vs == 0));
}
static bool dcb_ring_applies(const bimamba2_params *p) {
    return p->dtype != BIMAMBA2_F32 && dcb_aligned(p) && p->chunk_size % 64 == 0 && p->headdim % 8 == 0 && dcb_rows_in_32bit(p);
}

template <typename T>
static int launch_dcb_t(const bimamba2_params *p, bool add_up) {
    const int nc = nchunks(p), nqt = (p->chunk_size + 63) / 64;
    const int slices = dcb_slices(p);
    dim3 grid(p->batch * nc * p->ngroups, nqt * nqt, slices);
    const bool fast = dcb_aligned(p) && p->headdim % (sizeof(T) == 2 ? 64 : 16) == 0;
    if (!p->CB && !dcb_recomputes_cb(p)) return BIMAMBA2_EINVAL;
    const bool ring = dcb_ring_applies(p);
    if (p->causal && !(ring && fast)) return BIMAMBA2_EUNSUPPORTED;
    if (ring) launch_dcb_ring<T>(grid, p, nc, nqt);
    else if (fast) hipLaunchKernelGGL((bwd_dcb_kernel<T, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
    else hipLaunchKernelGGL((bwd_dcb_kernel<T, false>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt);
    if (slices > 1 && add_up) {
        // (Q*Q is a multiple of 4 only when Q is even; odd chunk sizes are rejected by the 16-byte requirement below)
        const size_t n = (size_t)p->batch * nc * p->ngroups * p->chunk_size * p->chunk_size;
        if (n % 4) return BIMAMBA2_EUNSUPPORTED;
        const int blocks = (int)std::min<size_t>((n / 4 + NTHREADS - 1) / NTHREADS, 4096);
        hipLaunchKernelGGL(sum_slices_kernel, dim3(blocks, 2), dim3(NTHREADS), 0, stream_of(p), p->dCB, p->dCBT, n / 4, slices);
    }
    return check_launch();
}

// Head slices where bimamba2_bwd owns dCB.
// The kernel rebuilds C.B^T (16 bits, wide heads): a slice starts with its own copy of the tile, and the last launch reads the slices in
// float32 instead of one in 16 bits; they pay while compute units are left without two workgroups.  us with 1 / 2 / 4 slices, chunks of 256:
//   heads of 128 (the ring), a training pass: dstate 64, 24 heads, 64 tiles 136 / 118 / 112, 128 tiles 157 / 138 / 136, 384 tiles 264 / 258 / 279; 16 heads, 512
//     tiles 214 / 222 / 244; dstate 128, 32 heads, 96 tiles 258 / 235 / 231
//   heads of 64 (waves that take whole heads split a tile's heads themselves), dCB with the state passing beside it + the last launch, dstate 64: 24 heads, 16
//     tiles 31 / 25 / 26, 32 tiles 33 / 27 / 28; 64 tiles: 12 heads 25 / 24 / 28, 24 34 / 28 / 28, 32 39 / 31 / 30, 48 50 / 36 / 33; 96 tiles: 16 heads 28 / 26 / 28,
//     24 34 / 29 / 33, 48 50 / 38 / 40; 128 tiles: 12 heads 26 / 25 / 29, 24 35 / 29 / 33, 48 51 / 38 / 38; 192 of 24 35 / 31 / 38; 256 of 24 36 / 34 / 41, of 32 43 / 40 / 46; 384
//     of 24 41 / 46 / 54, of 32 48 / 51 / 59; 512 of 16 36 / 47 / 54
// So four up to 95 tiles (fewer heads than 16 make fewer), then for heads of 64 two below 256 (at 256 from 32 heads on) and one beyond; for heads of
// 128 four up to 128, three up to 170, two up to 255, or 384 from 32 heads on.
// All of these are chunks of 256, where the last launch adds the slices up.  Where none does (dt of a type of its own in chunks of up to
// 128, chunks between, state dimensions other than 64 and 128 in chunks of 256) they take a launch for it and part the dCB launch from
// the state passing.  us a pass with one slice -> with the number chosen where a launch adds up (heads of 64, dstate 192): 8 heads, 64 tiles and up lose; 64
// tiles: 17 heads 218 -> 217, 24 228 -> 228, 32 255 -> 251, 48 310 -> 302; 128 tiles: 17 heads 241 -> 246, 24 260 -> 268, 48 401 -> 405; 224 tiles: 24 heads 340 ->
// 353, 48 573 -> 603; float16 dt beside bfloat16, dstate 64, chunks of 128: 32 tiles: 8 heads 81 -> 89, 32 112 -> 103, 48 135 -> 122; 96 tiles: 16 heads 114 -> 122,
// 24 134 -> 143, 32 150 -> 155, 48 194 -> 193.  So 16 heads or fewer are not cut, and up to 64 (of 64 channels) not from 96
// tiles on.
// The kernel reads C.B^T (float32, and 16-bit shapes whose state or headdim is no multiple of what the rebuilding kernel takes: the ring
// with a narrow state or narrow heads; through registers where rows are not aligned).
// A workgroup is one chain over its heads, 5 to 7 us a head through registers in float32, 3 to 5 in 16 bits and 1.5 in the ring,
// so slices pay on a small grid until there are three workgroups on every CU; against them stands a launch that adds them up
// (4 us, and 0.03 us per tile and slice), which few heads do not earn: in 16 bits a slice wants a head per 32 tiles of the grid,
// in float32 fewer than six heads are cut only where all slices are on the chip at once.  us with one slice -> with the number
// chosen here (-> with as many as three workgroups a CU would allow, where that is another number), the adding up included:
//   float32, headdim 64: 16 heads in 2 groups, 320 tiles 56 -> 42 + 6; 24 heads, 256 tiles 112 -> 82; 4 heads, 192 tiles 23 (-> 28)
//   16 bits through registers, headdim 32 or 16: 24 heads, 64 tiles 94 -> 30; 17 heads, 240 tiles 70 -> 51 (-> 62); 8 heads, 320 tiles 43 (-> 49);
//     6 heads, 384 tiles 33 (-> 46); the rule loses at 7 heads, 176 tiles (32 -> 29) and 15 heads, 256 tiles (62 -> 56)
//   ring, headdim 64, state 16: 48 heads, 64 tiles 62 -> 22; 24 heads, 256 tiles 36 -> 31; 16 heads, 160 tiles 26 -> 20 (-> 21);
//     8 heads, 320 tiles 17 (-> 22); 4 heads, 192 tiles 10 (-> 17); 8 heads, 128 tiles 15 -> 16 (-> 19)
int choose_dcb_slices(const bimamba2_params *p) {
    const int usual = dcb_slices(p), hpg = p->nheads / p->ngroups, nqt = (p->chunk_size + 63) / 64;
    const int64_t n = (int64_t)p->batch * nchunks(p) * p->ngroups * p->chunk_size * p->chunk_size;
    if (p->causal || n % 4) return usual;
    const int64_t wgs = (int64_t)p->batch * nchunks(p) * p->ngroups * nqt * nqt;
    int wanted = usual;
    if (dcb_recomputes_cb(p)) {
        const bool heads = p->headdim == 64;
        if (!bwd_tail_merged(p) && !bwd_tail_small(p)) {
            if (hpg <= 16) return usual;
            if (heads && wgs >= 96 && hpg <= 64) return 1;
        }
        if (wgs < 256 || (wgs <= (heads ? 256 : 384) && hpg >= DCB_SLICE_HEADS))
            wanted = (int)std::max<int64_t>(usual, std::min<int64_t>({hpg / 4, 4, heads && wgs >= 96 ? 2 : std::max<int64_t>(512 / wgs, 2)}));
    } else {
        const int most = p->dtype == BIMAMBA2_F32 ? (hpg < 6 ? 256 : 768) : std::min(768, 32 * hpg);      // workgroups
        wanted = (int)std::max<int64_t>(usual, std::min<int64_t>({hpg / 2, 8, most / wgs}));
    }
    const int heads = (hpg + wanted - 1) / wanted;               // (9 heads in 4 slices: three of 3, the fourth would be empty)
    return (hpg + heads - 1) / heads;
}

// whether bwd_dcb_sp_kernel exists for the problem (the ring variant of the dCB kernel, the vector
// variant of the state passing)
bool bwd_dcb_sp_merged(const bimamba2_params *p) {
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return false;
    if (!dcb_recomputes_cb(p)) return false;                             // (implies the conditions of the ring variant)
    // the entering states and their gradients both in 16 bits, or (state dimension 128) both in float32
    if (p->states16_f && p->dstates16_f ? !(p->causal || (p->states16_b && p->dstates16_b))
                                        : p->states16_f || p->dstates16_f || p->causal || !p->states_f || !p->states_b || !p->dstates_f || !p->dstates_b)
        return false;
    if (!al(p->states_f) || !al(p->states_b)) return false;
    if ((p->headdim * p->dstate) % 4) return false;
    return al(p->states16_f) && al(p->states16_b) && al(p->dstates16_f) && al(p->dstates16_b) && al(p->dstates_f) && al(p->dstates_b) &&
           al(p->dfinal_f) && al(p->dfinal_b) && al(p->dinitial_f) && al(p->dinitial_b);
}

// bimamba2_chunk_scan_bwd_dcb and bimamba2_state_passing_bwd in one launch (the caller checked bwd_dcb_sp_merged())
int launch_bwd_dcb_sp(const bimamba2_params *p, bool out16) {
    const int nc = nchunks(p), nqt = (p->chunk_size + 63) / 64, PN = p->headdim * p->dstate;
    const int nsplit = (PN + SP_EPT * NTHREADS - 1) / (SP_EPT * NTHREADS), ndir = p->causal ? 1 : 2;
    const int slices = dcb_slices(p), W = p->headdim == 64 && !dcb_sp_streams(p, slices) ? dcb_waves(p, slices) : 0;
    const int gdx = p->batch * nc * p->ngroups, gdy = W ? (nqt * nqt * W + 3) / 4 : nqt * nqt, nsp1 = nsplit * p->nheads * p->batch * ndir;
    // (two groups a workgroup of the state passing where that leaves as many workgroups as the chip holds beside the tiles, else fewer are
    // under way at once: 1 x 8192, 24 heads, 192 -> 96 workgroups 36.8 -> 37.5)
    const int ngr = nc > 4 && W && !(p->dstates_f && p->dstates16_f) && nsplit % 2 == 0 && nsp1 >= DCB_HEADS_RESIDENT ? 2 : sp_bwd_groups(nc);
    const int nspx = (nsplit + ngr - 1) / ngr, nsp = p->ddA_chunk_f ? nspx * p->nheads * p->batch * ndir : 0;      // (0: one_chunk())
    dim3 grid(gdx * gdy * slices + nsp);
#define BM2_D(TT, UNI, WV) hipLaunchKernelGGL((bwd_dcb_sp_kernel<TT, UNI, WV>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, gdx, gdy, slices, nsplit, nspx, ndir, out16)
#define BM2_DS(TT, UNI)                \
    do {                               \
        if (W == 4) BM2_D(TT, UNI, 4); \
        else if (W == 2) BM2_D(TT, UNI, 2); \
        else if (W == 1) BM2_D(TT, UNI, 1); \
        else BM2_D(TT, UNI, 0);        \
    } while (0)
    if (p->dtype == BIMAMBA2_BF16) { if (p->causal) BM2_DS(bf16_t, true); else BM2_DS(bf16_t, false); }
    else { if (p->causal) BM2_DS(f16_t, true); else BM2_DS(f16_t, false); }
#undef BM2_DS
#undef BM2_D
    return check_launch();
}

int launch_bwd_dcb(const bimamba2_params *p, bool add_up) {
    switch (p->dtype) {
        case BIMAMBA2_F32: return launch_dcb_t<float>(p, add_up);
        case BIMAMBA2_BF16: return launch_dcb_t<bf16_t>(p, add_up);
        case BIMAMBA2_F16: return launch_dcb_t<f16_t>(p, add_up);
        default: return BIMAMBA2_EUNSUPPORTED;
    }
}

// =========================================================================================================
// which = 0 : dB[s,n] = sum_slices dBs[s,n] + sum_t dCBT[s,t] C[t,n]     which = 1 : dC[t,n] = sum dCs + sum_s dCB[t,s] B[s,n]
// One workgroup: 64 rows x 64 dstate columns of one (b, c, g).  The K operand (C or B rows of the chunk) is staged
// transposed in LDS once; the A operand is read from the float32 dCB / dCBT rows straight into MFMA operand layout.
// =========================================================================================================
// FAST (16-bit types, chunk_size == QP, dstate a multiple of 64, aligned operands, at most 8 slices): every global load
// of a thread (its dCB row pieces, the slices it adds, the K operand) is requested before the first one is used.

// SLIM (with FAST): dCB / dCBT hold 16-bit elements (in16) and there are at most two slices to add: a quarter of the
// registers, and the staging tile of the result shares the LDS of the K operand, so that three workgroups fit a CU where
// the general variant fits two (with few heads per group the launch has thousands of workgroups: 83 -> 76 us at 8 groups
// of 4 heads, batch 4 x 4096, where the launch moves 250 MB).
template <typename T, int QP, bool FAST, bool SLIM = false>
__device__ __forceinline__ void bmm_chunk_bwd_body(const bimamba2_params &p, int nc, int nslices, BlockId bid, bool in16 = false, int ncb = 1) {
    // ncb: head slices of dCB / dCBT (float32) that are still to be added up
    typedef Mma<T> M;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP;
    constexpr int LDX = QP + 16 / (int)sizeof(T);
    constexpr int SLD = 64 + 4;
    constexpr int KT_BYTES = 64 * LDX * (int)sizeof(T), STG_BYTES = 64 * SLD * 4;
    __shared__ __attribute__((aligned(16))) unsigned char bmm_lds[SLIM ? (KT_BYTES > STG_BYTES ? KT_BYTES : STG_BYTES) : KT_BYTES + STG_BYTES];
    T *kT = reinterpret_cast<T *>(bmm_lds);
    float *stg = reinterpret_cast<float *>(bmm_lds + (SLIM ? 0 : KT_BYTES));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int nt = bid.x, rt = bid.y;
    const int which = bid.z & 1, bcg = bid.z >> 1;
    const int g = bcg % p.ngroups, bc = bcg / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, N = p.dstate;
    const int limit = min(Q, p.seqlen - c * Q);
    const int r0 = rt * 64;
    const T *op;
    int64_t os;
    if (which == 0) { os = p.C_sl; op = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + (int64_t)c * Q * os + g * p.C_sg + nt * 64; }
    else { os = p.B_sl; op = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * os + g * p.B_sg + nt * 64; }
    const float *arow = (which == 0 ? p.dCBT : p.dCB) + (int64_t)bcg * Q * Q + (int64_t)min(r0 + wave * 16 + lr, Q - 1) * Q;
    const int64_t cb_slice = (int64_t)p.batch * nc * p.ngroups * Q * Q;
    const float *res = which == 0 ? p.dBs : p.dCs;
    T *out = reinterpret_cast<T *>(which == 0 ? p.dB : p.dC);
    // (dB / dC may be slices of a wider buffer: their own position and batch strides; 0 = contiguous)
    const int64_t o_sl = (which == 0 ? p.dB_sl : p.dC_sl) ? (which == 0 ? p.dB_sl : p.dC_sl) : (int64_t)p.ngroups * p.dstate;
    const int64_t o_sb = (which == 0 ? p.dB_sl : p.dC_sl) ? (which == 0 ? p.dB_sb : p.dC_sb) : p.seqlen * o_sl;
    const int64_t slice = (int64_t)p.batch * p.seqlen * p.ngroups * N;
    constexpr int VS = 16 / (int)sizeof(T);
    if constexpr (FAST) {
        constexpr int NS = QP / KSTEP, NIT = 64 * (64 / VS) / NTHREADS, MAXSL = SLIM ? 2 : 8;
        // in16: dCB / dCBT hold elements of type T (written that way by the dCB kernel inside bimamba2_bwd): a row piece is
        // the MFMA operand as it lies in memory
        float4 raw[NS][SLIM ? 1 : 2];
        if (SLIM || in16) {
            const T *arow16 = reinterpret_cast<const T *>(which == 0 ? p.dCBT : p.dCB) + (int64_t)bcg * Q * Q + (int64_t)min(r0 + wave * 16 + lr, Q - 1) * Q;
#pragma unroll
            for (int s = 0; s < NS; ++s) raw[s][0] = *reinterpret_cast<const float4 *>(arow16 + s * KSTEP + lg * KPL);
        } else if constexpr (!SLIM) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                raw[s][0] = *reinterpret_cast<const float4 *>(arow + s * KSTEP + lg * KPL);
                raw[s][1] = *reinterpret_cast<const float4 *>(arow + s * KSTEP + lg * KPL + 4);
            }
            for (int sl = 1; sl < ncb; ++sl) {
                const float *more = arow + sl * cb_slice;
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const float4 u = *reinterpret_cast<const float4 *>(more + s * KSTEP + lg * KPL + 4 * half);
                        raw[s][half].x += u.x; raw[s][half].y += u.y; raw[s][half].z += u.z; raw[s][half].w += u.w;
                    }
            }
        }
        // slices: the first half is requested here, the second half after the products, into the registers of the row pieces
        // (keeps the kernel at two workgroups per CU)
        constexpr int HSL = MAXSL / 2;
        float4 sv[NIT][HSL][2];
        int64_t oa[NIT];
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int id = threadIdx.x + it * NTHREADS;
            const int rl = id / (64 / VS), cc = (id % (64 / VS)) * VS;
            const int r = min(r0 + rl, limit - 1);
            oa[it] = (((int64_t)b * p.seqlen + (int64_t)c * Q + r) * p.ngroups + g) * N + nt * 64 + cc;
#pragma unroll
            for (int sl = 0; sl < HSL; ++sl) {
                if (nslices == 0) continue;        // (uniform) no state part: a sequence of one chunk
                const float *q = res + oa[it] + (int64_t)min(sl, nslices - 1) * slice;
                sv[it][sl][0] = *reinterpret_cast<const float4 *>(q);
                sv[it][sl][1] = *reinterpret_cast<const float4 *>(q + 4);
            }
        }
        stage_transposed<T, QP, 64, LDX, true>(kT, op, os, limit, 64, [&](int k) { return k < limit ? 1.f : 0.f; });
        __syncthreads();
        f32x4 acc[4] = {};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s * KSTEP < limit) {
                // (chunks of 256 take dCB in 16 bits where it is bimamba2_bwd's own, and give the same bits where a caller brings it)
                constexpr bool SPLIT = QP < 256 && !SLIM;
                typename M::Frag af, rest{};
                if constexpr (SLIM) {
                    static_assert(!SLIM || sizeof(typename M::Frag) == 16, "16-bit operands");
                    af = __builtin_bit_cast(typename M::Frag, raw[s][0]);
                } else {
                    float v[KPL] = {raw[s][0].x, raw[s][0].y, raw[s][0].z, raw[s][0].w, raw[s][1].x, raw[s][1].y, raw[s][1].z, raw[s][1].w};
                    if constexpr (SPLIT) split_operand<T>(v, af, rest);
                    else if constexpr (sizeof(typename M::Frag) == 16) af = in16 ? __builtin_bit_cast(typename M::Frag, raw[s][0]) : M::pack(v);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const typename M::Frag bf = M::load(kT + xt_index<T, LDX>(j * 16 + lr, s * KSTEP + lg * KPL));
                    acc[j] = M::mma(af, bf, acc[j]);
                    if constexpr (SPLIT) acc[j] = M::mma(rest, bf, acc[j]);
                }
            }
        }
        float4 sw[NIT][HSL][2] = {};
        if (nslices > HSL) {                        // (with one half's worth of slices there is nothing more to wait for)
#pragma unroll
            for (int it = 0; it < NIT; ++it)
#pragma unroll
                for (int sl = 0; sl < HSL; ++sl) {
                    const float *q = res + oa[it] + (int64_t)min(HSL + sl, nslices - 1) * slice;
                    sw[it][sl][0] = *reinterpret_cast<const float4 *>(q);
                    sw[it][sl][1] = *reinterpret_cast<const float4 *>(q + 4);
                }
        }
        if constexpr (SLIM) __syncthreads();       // every wave is done with the K operand, whose LDS the staging tile shares
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) stg[(wave * 16 + lg * 4 + i) * SLD + j * 16 + lr] = acc[j][i];
        __syncthreads();
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int id = threadIdx.x + it * NTHREADS;
            const int rl = id / (64 / VS), cc = (id % (64 / VS)) * VS;
            float v[VS];
#pragma unroll
            for (int i = 0; i < VS; ++i) v[i] = stg[rl * SLD + cc + i];
#pragma unroll
            for (int sl = 0; sl < MAXSL; ++sl) {
                if (sl < nslices) {
                    const float4 a0 = sl < HSL ? sv[it][sl % HSL][0] : sw[it][sl % HSL][0], a1 = sl < HSL ? sv[it][sl % HSL][1] : sw[it][sl % HSL][1];
                    v[0] += a0.x; v[1] += a0.y; v[2] += a0.z; v[3] += a0.w;
                    v[4] += a1.x; v[5] += a1.y; v[6] += a1.z; v[7] += a1.w;
                }
            }
            if (r0 + rl < limit) {
                Vec16<T> ov;
#pragma unroll
                for (int i = 0; i < VS; ++i) ov.v[i] = from_f<T>(v[i]);
                *reinterpret_cast<Vec16<T> *>(out + (b * o_sb + ((int64_t)c * Q + r0 + rl) * o_sl + (int64_t)g * N + nt * 64 + cc)) = ov;
            }
        }
        return;
    }
    stage_transposed<T, QP, 64, LDX, false>(kT, op, os, limit, N - nt * 64, [&](int k) { return 1.f; });
    __syncthreads();
    const bool cvec = Q % 4 == 0;
    f32x4 acc[4] = {};
    for (int k0 = 0; k0 < limit; k0 += KSTEP) {
        const int kb = k0 + lg * KPL;
        float v[KPL];
        if (cvec && kb + KPL <= Q) {
            if (KPL >= 4) {
#pragma unroll
                for (int i = 0; i < KPL; i += 4) {
                    float4 t4 = *reinterpret_cast<const float4 *>(arow + kb + i);
                    for (int sl = 1; sl < ncb; ++sl) {
                        const float4 u = *reinterpret_cast<const float4 *>(arow + sl * cb_slice + kb + i);
                        t4.x += u.x; t4.y += u.y; t4.z += u.z; t4.w += u.w;
                    }
                    v[i] = t4.x; v[(i + 1) % KPL] = t4.y; v[(i + 2) % KPL] = t4.z; v[(i + 3) % KPL] = t4.w;
                }
            } else {
                v[0] = arow[kb];
            }
        } else {
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                v[i] = kb + i < Q ? arow[kb + i] : 0.f;
                for (int sl = 1; sl < ncb; ++sl)
                    if (kb + i < Q) v[i] += arow[sl * cb_slice + kb + i];
            }
        }
        typename M::Frag af, rest{};
        split_operand<T>(v, af, rest);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const typename M::Frag bf = M::load(kT + xt_index<T, LDX>(j * 16 + lr, kb));
            acc[j] = M::mma(af, bf, acc[j]);
            if constexpr (sizeof(T) == 2) acc[j] = M::mma(rest, bf, acc[j]);
        }
    }
    // pass the tile through LDS so that the slices are read and the result is written
    // as 16-byte vectors along dstate
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) stg[(wave * 16 + lg * 4 + i) * SLD + j * 16 + lr] = acc[j][i];
    __syncthreads();
    // (16-byte stores: the strides and the base of the destination slice must both allow them)
    const bool ovec = N % VS == 0 && o_sl % VS == 0 && o_sb % VS == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    for (int id = threadIdx.x; id < 64 * (64 / VS); id += NTHREADS) {
        const int rl = id / (64 / VS), cc = (id % (64 / VS)) * VS;
        const int r = r0 + rl, n = nt * 64 + cc;
        if (r >= limit || n >= N) continue;
        const int64_t a = (((int64_t)b * p.seqlen + (int64_t)c * Q + r) * p.ngroups + g) * N + n;
        const int64_t ao = b * o_sb + ((int64_t)c * Q + r) * o_sl + (int64_t)g * N + n;
        float v[VS];
#pragma unroll
        for (int i = 0; i < VS; ++i) v[i] = stg[rl * SLD + cc + i];
        if (ovec) {
            for (int sl = 0; sl < nslices; ++sl)
#pragma unroll
                for (int i = 0; i < VS; i += 4) {
                    const float4 t4 = *reinterpret_cast<const float4 *>(res + a + sl * slice + i);
                    v[i] += t4.x; v[i + 1] += t4.y; v[i + 2] += t4.z; v[i + 3] += t4.w;
                }
            Vec16<T> ov;
#pragma unroll
            for (int i = 0; i < VS; ++i) ov.v[i] = from_f<T>(v[i]);
            *reinterpret_cast<Vec16<T> *>(out + ao) = ov;
        } else {
#pragma unroll
            for (int i = 0; i < VS; ++i)
                if (n + i < N) {
                    float u = v[i];
                    for (int sl = 0; sl < nslices; ++sl) u += res[a + sl * slice + i];
                    out[ao + i] = from_f<T>(u);
                }
        }
    }
}

template <typename T, int QP, bool FAST>
__global__ __launch_bounds__(NTHREADS) void bmm_chunk_bwd_kernel(const bimamba2_params p, int nc, int nslices) {
    bmm_chunk_bwd_body<T, QP, FAST>(p, nc, nslices, BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z});
}

template <typename T>
static int launch_bmm_bwd_t(const bimamba2_params *p) {
    const int nc = nchunks(p), Q = p->chunk_size, nsl = state_slices(p);
    dim3 grid((p->dstate + 63) / 64, (Q + 63) / 64, p->batch * nc * p->ngroups * 2);
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    auto mult = [](int64_t a, int64_t b, int64_t c) { return a % 8 == 0 && b % 8 == 0 && c % 8 == 0; };
    const bool fast = sizeof(T) == 2 && (Q == 64 || Q == 128 || Q == 256) && p->dstate % 64 == 0 && nsl <= 8 && al(p->Bm) && al(p->Cm)
                      && mult(p->B_sb, p->B_sl, p->B_sg) && mult(p->C_sb, p->C_sl, p->C_sg) && al(p->dCB) && al(p->dCBT) && al(p->dBs)
                      && al(p->dCs) && al(p->dB) && al(p->dC) && mult(p->dB_sb, p->dB_sl, p->dC_sb) && p->dC_sl % 8 == 0;
#define BM2_BMMB(QPV)                                                                                                              \
    do {                                                                                                                       \
        if constexpr (sizeof(T) == 2) {                                                                                        \
            if (fast) { hipLaunchKernelGGL((bmm_chunk_bwd_kernel<T, QPV, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl); break; } \
        }                                                                                                                      \
        hipLaunchKernelGGL((bmm_chunk_bwd_kernel<T, QPV, false>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl);          \
    } while (0)
    if (Q <= 64) BM2_BMMB(64);
    else if (Q <= 128) BM2_BMMB(128);
    else BM2_BMMB(256);
#undef BM2_BMMB
    return check_launch();
}

int launch_bmm_chunk_bwd(const bimamba2_params *p) {
    switch (p->dtype) {
        case BIMAMBA2_F32: return launch_bmm_bwd_t<float>(p);
        case BIMAMBA2_BF16: return launch_bmm_bwd_t<bf16_t>(p);
        case BIMAMBA2_F16: return launch_bmm_bwd_t<f16_t>(p);
        default: return BIMAMBA2_EUNSUPPORTED;
    }
}

// =========================================================================================================
// one wave per (b, c, h); lane i owns positions 4i..4i+3.
//   da[q] = (within-chunk part from the tile vectors in da_intra) + sum_{s<q} v_f[s] + sum_{s>q} v_b[s] + sum_{t>=q} u_f[t] + sum_{t<=q} u_b[t]
//           + ddA_chunk_f + ddA_chunk_b
//   ddt' = da*A + ddt_direct ; through clamp and softplus -> ddt ; dA += sum da*dt' ; ddt_bias += sum ddt
// Partials per (b, c) go to red[(b*nc + c)*H + h] (dA) and red[B*nc*H + ...] (ddt_bias).
// =========================================================================================================
// k-th workgroup -> four heads of a (batch, chunk).  dt and ddt have the heads side by side, so the workgroups of a (batch, chunk) use the same
// lines and share an XCD: dealt to all eight, each L2 fetched the lines of dt and wrote its heads' bytes of those of ddt.  With a lane's four
// positions as one load: 4 x 4096, 32 heads 17.7 -> 14.6 us, 16 x 1024, 24 heads with dt and ddt in bfloat16 14.2 -> 12.1, 4 x 4096, 16 heads 10.2 -> 9.0.
__device__ __forceinline__ BlockId cumsum_block(int k, int gx, int nc, int batch) {
    int x, bc;
    xcd_order(k, gx, nc * batch, x, bc);
    return BlockId{x, bc % nc, bc / nc};
}
template <typename DT>
__device__ __forceinline__ void chunk_cumsum_bwd_body(const bimamba2_params &p, int nc, int nqt, int nsplit, BlockId bid) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = bid.x * 4 + wave, c = bid.y, b = bid.z;
    if (h >= p.nheads) return;
    const int Q = p.chunk_size, H = p.nheads;
    const int limit = min(Q, p.seqlen - c * Q);
    const int64_t o = (((int64_t)b * H + h) * nc + c) * Q;
    // Every load of the kernel goes out here, unconditionally and from clamped (valid) addresses, before anything is
    // used: a load that is waited for costs microseconds, and conditional loads get serialised by the compiler.
    float vf[4], vb[4], uf[4], ub[4], di[4], dtr[4], ddr[4];
    const int nplanes = ddt_direct_planes(p);
    const int64_t plane = (int64_t)p.batch * H * nc * Q;
    const DT *dt = reinterpret_cast<const DT *>(p.dt) + b * p.dt_sb + (int64_t)c * Q * p.dt_sl + h * p.dt_sh;
    const bool state_terms = p.u_f != nullptr;     // (else a sequence of one chunk: nothing crosses a boundary)
    // a lane's four positions as one load where they lie aligned (what stands behind the sequence's end is not used)
    const uintptr_t bits = reinterpret_cast<uintptr_t>(p.v_f) | reinterpret_cast<uintptr_t>(p.v_b) | reinterpret_cast<uintptr_t>(p.u_f) |
                           reinterpret_cast<uintptr_t>(p.u_b) | reinterpret_cast<uintptr_t>(p.ddt_direct);
    const bool wide = Q % 4 == 0 && bits % 16 == 0;
    auto load4 = [&](const float *from, float (&to)[4]) __attribute__((always_inline)) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(from + o + min(lane * 4, Q - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) to[e] = v[e];
    };
    if (state_terms && wide) {
        load4(p.v_f, vf);
        load4(p.v_b, vb);
        load4(p.u_f, uf);
        load4(p.u_b, ub);
    } else if (state_terms) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int qc = min(lane * 4 + e, limit - 1);
            vf[e] = p.v_f[o + qc];
            vb[e] = p.v_b[o + qc];
            uf[e] = p.u_f[o + qc];
            ub[e] = p.u_b[o + qc];
        }
    }
    // (ddt_direct: one plane per headdim tile of the dx kernel)
    if (wide) {
        load4(p.ddt_direct, ddr);
        for (int pl = 1; pl < nplanes; ++pl) {
            float more[4];
            load4(p.ddt_direct + pl * plane, more);
#pragma unroll
            for (int e = 0; e < 4; ++e) ddr[e] += more[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int qc = min(lane * 4 + e, limit - 1);
            ddr[e] = p.ddt_direct[o + qc];
            for (int pl = 1; pl < nplanes; ++pl) ddr[e] += p.ddt_direct[pl * plane + o + qc];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int qc = min(lane * 4 + e, limit - 1);
        dtr[e] = to_f(dt[(int64_t)qc * p.dt_sl]);
    }
    if (!state_terms) {
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[e] = vb[e] = uf[e] = ub[e] = 0.f;
    }
    if (p.causal) {                   // single-direction operator: nothing wrote the reverse direction's terms
#pragma unroll
        for (int e = 0; e < 4; ++e) vb[e] = ub[e] = 0.f;
    }
    const float A = p.A[h];
    const float bias = p.has_dt_bias ? p.dt_bias[h] : 0.f;
    float chunk_term = 0.f;
    for (int s = 0; state_terms && s < nsplit; ++s)
    {
        const float cf = p.ddA_chunk_f[(((int64_t)b * H + h) * nc + c) * nsplit + s], cr = p.ddA_chunk_b[(((int64_t)b * H + h) * nc + c) * nsplit + s];
        chunk_term += cf + (p.causal ? 0.f : cr);
    }
    // within-chunk part from the per-tile vectors of the dCB kernel; tile I = lane / 16 holds this lane's positions.
    // Four tiles per side at most (Q <= 256): tile indices past nqt are clamped for the loads and masked afterwards.
    const int I = lane >> 4, i0 = (lane & 15) * 4, Ic = min(I, nqt - 1);
    const float *tv = p.da_intra + (o / Q) * nqt * nqt * DCB_VEC;
    float4 colv[4], rowv[4], tot[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int ac = min(a, nqt - 1);
        colv[a] = *reinterpret_cast<const float4 *>(tv + (ac * nqt + Ic) * DCB_VEC + i0);          // [0] of tile (a, I)
        rowv[a] = *reinterpret_cast<const float4 *>(tv + (Ic * nqt + ac) * DCB_VEC + 64 + i0);     // [1] of tile (I, a)
#pragma unroll
        for (int bq = 0; bq < 4; ++bq) tot[a][bq] = *reinterpret_cast<const float4 *>(tv + (ac * nqt + min(bq, nqt - 1)) * DCB_VEC + i0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (lane * 4 + e >= limit) vf[e] = vb[e] = uf[e] = ub[e] = 0.f;
        di[e] = 0.f;
    }
    {
        if (I < nqt) {
            auto add = [](float (&r)[4], const float4 &v) { r[0] += v.x; r[1] += v.y; r[2] += v.z; r[3] += v.w; };
            // the diagonal tile's difference vectors join the exclusive scans: cwf gets cw_f - rw_f, cwb gets cw_b - rw_b
            float cwf[4] = {0.f, 0.f, 0.f, 0.f}, cwb[4] = {0.f, 0.f, 0.f, 0.f}, rwf[4] = {0.f, 0.f, 0.f, 0.f}, rwb[4] = {0.f, 0.f, 0.f, 0.f};
            float between = 0.f;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if (a < nqt) {
                    if (a == I) { add(cwf, colv[a]); add(cwb, rowv[a]); }
                    if (a > I) { add(cwf, colv[a]); add(rwb, rowv[a]); }
                    if (a < I) { add(rwf, rowv[a]); add(cwb, colv[a]); }
                    // tiles with this tile strictly between their row tile and column tile add their total
#pragma unroll
                    for (int bq = 0; bq < 4; ++bq)
                        if (bq < nqt && ((bq < I && I < a) || (a < I && I < bq))) between += tot[a][bq].x + tot[a][bq].y + tot[a][bq].z + tot[a][bq].w;
                }
            }
            between = row16_sum(between);
            // forward: exclusive prefix of cwf + inclusive suffix of rwf; reverse: inclusive prefix of rwb + exclusive suffix of cwb
            const float t_cwf = cwf[0] + cwf[1] + cwf[2] + cwf[3], t_rwb = rwb[0] + rwb[1] + rwb[2] + rwb[3];
            const float t_rwf = rwf[0] + rwf[1] + rwf[2] + rwf[3], t_cwb = cwb[0] + cwb[1] + cwb[2] + cwb[3];
            float ex = row16_incl_prefix(t_cwf) - t_cwf, in = row16_incl_prefix(t_rwb) - t_rwb;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                in += rwb[e];
                di[e] = between + ex + in;
                ex += cwf[e];
            }
            float exs = row16_incl_suffix(t_cwb) - t_cwb, ins = row16_incl_suffix(t_rwf) - t_rwf;
#pragma unroll
            for (int e = 3; e >= 0; --e) {
                ins += rwf[e];
                di[e] += exs + ins;
                exs += cwb[e];
            }
        }
    }
    // lane totals and cross-lane scans
    const float tvf = vf[0] + vf[1] + vf[2] + vf[3], tvb = vb[0] + vb[1] + vb[2] + vb[3];
    const float tuf = uf[0] + uf[1] + uf[2] + uf[3], tub = ub[0] + ub[1] + ub[2] + ub[3];
    const float vf_before = wave_incl_prefix(tvf, lane) - tvf;     // sum over lower lanes
    const float ub_before = wave_incl_prefix(tub, lane) - tub;
    const float vb_after = wave_incl_suffix(tvb, lane) - tvb;      // sum over higher lanes
    const float uf_after = wave_incl_suffix(tuf, lane) - tuf;
    float da[4];
    {
        float ex_vf = vf_before, in_ub = ub_before;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            in_ub += ub[e];
            da[e] = di[e] + ex_vf + in_ub + chunk_term;
            ex_vf += vf[e];
        }
        float ex_vb = vb_after, in_uf = uf_after;
#pragma unroll
        for (int e = 3; e >= 0; --e) {
            in_uf += uf[e];
            da[e] += ex_vb + in_uf;
            ex_vb += vb[e];
        }
    }
    const int64_t ddt_sl = p.ddt_sl ? p.ddt_sl : H, ddt_sb = p.ddt_sl ? p.ddt_sb : (int64_t)p.seqlen * H;
    DT *ddt = reinterpret_cast<DT *>(p.ddt) + b * ddt_sb + (int64_t)c * Q * ddt_sl + h;
    float sA = 0.f, sb = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int q = lane * 4 + e;
        if (q < limit) {
            const float pre = dtr[e] + bias;
            float d = pre;
            if (p.dt_softplus) d = d > 20.f ? d : log1pf(expf(d));
            const bool clamped = d < p.dt_min || d > p.dt_max;
            d = fminf(fmaxf(d, p.dt_min), p.dt_max);
            float g = da[e] * A + ddr[e];
            if (clamped) g = 0.f;
            if (p.dt_softplus && pre <= 20.f) g *= 1.f / (1.f + expf(-pre));
            ddt[q * ddt_sl] = from_f<DT>(g);
            sA += da[e] * d;
            sb += g;
        }
    }
    sA = wave_sum(sA);
    sb = wave_sum(sb);
    if (lane == 0) {
        p.red[(int64_t)(b * nc + c) * H + h] = sA;
        p.red[(int64_t)p.batch * nc * H + (int64_t)(b * nc + c) * H + h] = sb;
    }
}

template <typename DT>
__global__ __launch_bounds__(NTHREADS) void chunk_cumsum_bwd_kernel(const bimamba2_params p, int nc, int nqt, int nsplit) {
    chunk_cumsum_bwd_body<DT>(p, nc, nqt, nsplit, cumsum_block(blockIdx.x, (p.nheads + 3) / 4, nc, p.batch));
}

// The last two kernels of the backward pass in one launch: the first `nbmm` workgroups do the work of
// bmm_chunk_bwd_kernel (16-bit path, chunk_size 256), the others that of chunk_cumsum_bwd_kernel.  Neither depends on the
// other, both are short and latency-bound, and together they fit the machine in one wave of workgroups.
template <typename T, typename DT, bool SLIM = false>
__global__ __launch_bounds__(NTHREADS) void bwd_tail_kernel(const bimamba2_params p, int nc, int nslices, int nqt, int nsplit, int nbmm,
                                                            int bmm_gy, int cs_gx, bool in16, int ncb) {
    const int id = blockIdx.x;
    if (id < nbmm) {
        // bmm grid (n tiles, bmm_gy, z), bmm_gy here counting both.  The bmm_gy tiles of one z = (which, b, c, g) stage the same
        // K operand (the chunk's C or B rows, or the 64 columns of them that the n tile takes): consecutive ids are dealt round-robin to the 8 XCDs, so eight z at a time, one per XCD, go through their
        // row tiles (with the row tile fastest every XCD fetched every K operand: +100 MB of reads at 8 groups)
        const int nz = nbmm / bmm_gy, k = id >> 3;
        const int t = nz % 8 == 0 ? k % bmm_gy : id % bmm_gy, ntiles = p.dstate >> 6;
        const BlockId bb{t % ntiles, t / ntiles, nz % 8 == 0 ? (k / bmm_gy) * 8 + (id & 7) : id / bmm_gy};
        bmm_chunk_bwd_body<T, 256, true, SLIM>(p, nc, nslices, bb, in16, ncb);
    } else {
        chunk_cumsum_bwd_body<DT>(p, nc, nqt, nsplit, cumsum_block(id - nbmm, cs_gx, nc, p.batch));
    }
}

// The same for chunks of up to 128 positions and any type and shape, with the head slices of dCB added up by their reader (instead of
// a launch of their own): what ends a pass whose kernels for wide 16-bit heads and states do not apply.  4 x 2048, bfloat16, 16 heads
// of 16, dstate 16: 10 + 8 + 5 -> 14 us; float32, 16 heads of 64, dstate 64: 14 + 9 + 6 -> 18.
template <typename T, int QP, bool FAST, typename DT>
__global__ __launch_bounds__(NTHREADS) void bwd_tail_small_kernel(const bimamba2_params p, int nc, int nslices, int nqt, int nsplit, int nbmm,
                                                                  int nnt, int cs_gx, int ncb) {
    const int id = blockIdx.x;
    if (id < nbmm) bmm_chunk_bwd_body<T, QP, FAST>(p, nc, nslices, BlockId{id % nnt, id / nnt % nqt, id / (nnt * nqt)}, false, ncb);
    else {
        const int k = id - nbmm;                  // cumsum grid (cs_gx, nc, batch): few workgroups, which XCD makes no difference
        chunk_cumsum_bwd_body<DT>(p, nc, nqt, nsplit, BlockId{k % cs_gx, (k / cs_gx) % nc, k / (cs_gx * nc)});
    }
}

static bool bmm_bwd_fast(const bimamba2_params *p) {
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    auto mult = [](int64_t a, int64_t b, int64_t c) { return a % 8 == 0 && b % 8 == 0 && c % 8 == 0; };
    const int Q = p->chunk_size;
    return p->dtype != BIMAMBA2_F32 && (Q == 64 || Q == 128 || Q == 256) && p->dstate % 64 == 0 && dbdc_slices(p) <= 8 && al(p->Bm) &&
           al(p->Cm) && mult(p->B_sb, p->B_sl, p->B_sg) && mult(p->C_sb, p->C_sl, p->C_sg) && al(p->dCB) && al(p->dCBT) && al(p->dBs) &&
           al(p->dCs) && al(p->dB) && al(p->dC) && mult(p->dB_sb, p->dB_sl, p->dC_sb) && p->dC_sl % 8 == 0;
}

// whether launch_bwd_tail() exists for this problem
bool bwd_tail_merged(const bimamba2_params *p) { return bmm_bwd_fast(p) && p->chunk_size == 256 && (p->dstate == 64 || p->dstate == 128); }

template <typename T>
static int launch_bwd_tail_t(const bimamba2_params *p, int nc, int nqt, int nsplit, bool in16, int ncb) {
    const int bmm_gy = (p->chunk_size + 63) / 64 * (p->dstate / 64), nbmm = bmm_gy * p->batch * nc * p->ngroups * 2;
    const int cs_gx = (p->nheads + 3) / 4, ncs = cs_gx * nc * p->batch;
    dim3 grid(nbmm + ncs);
    const int nsl = state_slices(p);
    if (in16 && nsl <= 2) {
        switch (p->dt_dtype) {
            case BIMAMBA2_F32: hipLaunchKernelGGL((bwd_tail_kernel<T, float, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
            case BIMAMBA2_BF16: hipLaunchKernelGGL((bwd_tail_kernel<T, bf16_t, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
            case BIMAMBA2_F16: hipLaunchKernelGGL((bwd_tail_kernel<T, f16_t, true>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
            default: return BIMAMBA2_EUNSUPPORTED;
        }
        return check_launch();
    }
    switch (p->dt_dtype) {
        case BIMAMBA2_F32: hipLaunchKernelGGL((bwd_tail_kernel<T, float>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
        case BIMAMBA2_BF16: hipLaunchKernelGGL((bwd_tail_kernel<T, bf16_t>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
        case BIMAMBA2_F16: hipLaunchKernelGGL((bwd_tail_kernel<T, f16_t>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nsl, nqt, nsplit, nbmm, bmm_gy, cs_gx, in16, ncb); break;
        default: return BIMAMBA2_EUNSUPPORTED;
    }
    return check_launch();
}

// dt in float32 or in the type of x (two instantiations of each)
bool bwd_tail_small(const bimamba2_params *p) {
    return !p->causal && p->chunk_size <= 128 && (p->dt_dtype == BIMAMBA2_F32 || p->dt_dtype == p->dtype);
}

template <typename T, int QP, bool FAST>
static void launch_bwd_tail_small_t(const bimamba2_params *p, int nc, int nsplit, int ncb) {
    const int nqt = (p->chunk_size + 63) / 64, nnt = (p->dstate + 63) / 64, nbmm = nnt * nqt * p->batch * nc * p->ngroups * 2;
    const int cs_gx = (p->nheads + 3) / 4;
    const dim3 grid(nbmm + cs_gx * nc * p->batch);
    if (p->dt_dtype == BIMAMBA2_F32) hipLaunchKernelGGL((bwd_tail_small_kernel<T, QP, FAST, float>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, state_slices(p), nqt, nsplit, nbmm, nnt, cs_gx, ncb);
    else hipLaunchKernelGGL((bwd_tail_small_kernel<T, QP, FAST, T>), grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, state_slices(p), nqt, nsplit, nbmm, nnt, cs_gx, ncb);
}

// ncb: head slices of dCB that nobody has added up yet
int launch_bwd_tail_small(const bimamba2_params *p, ReduceJobs *defer, int ncb) {
    const int nc = nchunks(p), nsplit = (p->headdim * p->dstate + SP_EPT * NTHREADS - 1) / (SP_EPT * NTHREADS);
    const bool fast = bmm_bwd_fast(p), half = p->chunk_size <= 64;
    switch (p->dtype) {
        case BIMAMBA2_F32: if (half) launch_bwd_tail_small_t<float, 64, false>(p, nc, nsplit, ncb); else launch_bwd_tail_small_t<float, 128, false>(p, nc, nsplit, ncb); break;
#define BM2_TAIL(TT)                                                                                                                   \
    if (fast && half) launch_bwd_tail_small_t<TT, 64, true>(p, nc, nsplit, ncb); else if (fast) launch_bwd_tail_small_t<TT, 128, true>(p, nc, nsplit, ncb); \
    else if (half) launch_bwd_tail_small_t<TT, 64, false>(p, nc, nsplit, ncb); else launch_bwd_tail_small_t<TT, 128, false>(p, nc, nsplit, ncb)
        case BIMAMBA2_BF16: BM2_TAIL(bf16_t); break;
        case BIMAMBA2_F16: BM2_TAIL(f16_t); break;
#undef BM2_TAIL
        default: return BIMAMBA2_EUNSUPPORTED;
    }
    const int rc = check_launch();
    if (rc) return rc;
    const int ni = p->batch * nc;
    defer->job[defer->n++] = ReduceJob{p->red, p->dA, ni, p->nheads, 1};
    if (p->has_dt_bias && p->ddt_bias) defer->job[defer->n++] = ReduceJob{p->red + (int64_t)ni * p->nheads, p->ddt_bias, ni, p->nheads, 1};
    return BIMAMBA2_OK;
}

// bmm_chunk_bwd + chunk_cumsum_bwd in one launch (the caller checked bwd_tail_merged()); reductions as in
// launch_chunk_cumsum_bwd
int launch_bwd_tail(const bimamba2_params *p, ReduceJobs *defer, bool in16, int ncb) {
    const int nc = nchunks(p), nqt = (p->chunk_size + 63) / 64;
    const int PN = p->headdim * p->dstate;
    const int nsplit = (PN + SP_EPT * NTHREADS - 1) / (SP_EPT * NTHREADS);
    int rc = p->dtype == BIMAMBA2_BF16 ? launch_bwd_tail_t<bf16_t>(p, nc, nqt, nsplit, in16, ncb) : launch_bwd_tail_t<f16_t>(p, nc, nqt, nsplit, in16, ncb);
    if (rc) return rc;
    const int ni = p->batch * nc;
    defer->job[defer->n++] = ReduceJob{p->red, p->dA, ni, p->nheads, 1};
    if (p->has_dt_bias && p->ddt_bias) defer->job[defer->n++] = ReduceJob{p->red + (int64_t)ni * p->nheads, p->ddt_bias, ni, p->nheads, 1};
    return BIMAMBA2_OK;
}

int launch_chunk_cumsum_bwd(const bimamba2_params *p, ReduceJobs *defer) {
    const int nc = nchunks(p), nqt = (p->chunk_size + 63) / 64;
    const int PN = p->headdim * p->dstate;
    const int nsplit = (PN + SP_EPT * NTHREADS - 1) / (SP_EPT * NTHREADS);
    dim3 grid((p->nheads + 3) / 4 * nc * p->batch);
    switch (p->dt_dtype) {
        case BIMAMBA2_F32: hipLaunchKernelGGL(chunk_cumsum_bwd_kernel<float>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nsplit); break;
        case BIMAMBA2_BF16: hipLaunchKernelGGL(chunk_cumsum_bwd_kernel<bf16_t>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nsplit); break;
        case BIMAMBA2_F16: hipLaunchKernelGGL(chunk_cumsum_bwd_kernel<f16_t>, grid, dim3(NTHREADS), 0, stream_of(p), *p, nc, nqt, nsplit); break;
        default: return BIMAMBA2_EUNSUPPORTED;
    }
    int rc = check_launch();
    if (rc) return rc;
    const int ni = p->batch * nc;
    if (defer) {
        // the caller runs these together with its other reductions
        defer->job[defer->n++] = ReduceJob{p->red, p->dA, ni, p->nheads, 1};
        if (p->has_dt_bias && p->ddt_bias) defer->job[defer->n++] = ReduceJob{p->red + (int64_t)ni * p->nheads, p->ddt_bias, ni, p->nheads, 1};
        return BIMAMBA2_OK;
    }
    rc = launch_reduce(p->red, p->dA, ni, p->nheads, 1, stream_of(p));
    if (rc) return rc;
    if (p->has_dt_bias && p->ddt_bias) rc = launch_reduce(p->red + (int64_t)ni * p->nheads, p->ddt_bias, ni, p->nheads, 1, stream_of(p));
    return rc;
}

// ---------------------------------------------------------------------------------------------------------
// launches of several roles (roles.hpp)
// ---------------------------------------------------------------------------------------------------------
static bool dbdc_wide16(const bimamba2_params *p) {      // the dB / dC kernels with the ring of state tiles
    return p->dtype != BIMAMBA2_F32 && p->headdim % 64 == 0 && (p->dstate == 64 || p->dstate == 128);
}
static RolesShape roles_shape(const bimamba2_params *p) {
    const int vs = p->dtype == BIMAMBA2_F32 ? 4 : 8;
    RolesShape r;
    r.nchunks = nchunks(p);
    r.dcb_slices = dcb_slices(p);
    r.dbdc_slices = dbdc_slices(p);
    r.dbdc_heads = dbdc_heads(p);
    r.dcb_ring = dcb_ring_applies(p);
    r.dcb_fast = dcb_aligned(p) && p->headdim % 16 == 0;
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    r.dstates_fast = dcb_aligned(p) && p->headdim % 64 == 0 && p->dstate % 64 == 0 && al(p->Cm) && p->C_sb % vs == 0 && p->C_sl % vs == 0 && p->C_sg % vs == 0;
    r.dstates_narrow = chunk_state_narrow(p, true);
    r.dx = true;
    r.dbdc_fast = dcb_aligned(p) && p->headdim % 64 == 0 && p->dstate % 64 == 0;
    return r;
}

// (faster at every size measured, 1 x 300 to 8 x 2048 with 8 to 32 heads of 16 to 128 and dstate 16 to 128: 4 x 2048, 16 heads of 16, dstate 16,
// bfloat16 158 -> 150 us a pass, float32 174 -> 171; 8 x 2048, 32 heads of 64, dstate 64, float32 1544 -> 1513)
bool dcb_dstates_merged(const bimamba2_params *p) {
    if (p->causal || p->chunk_size > 128 || !p->CB || !p->dstates_f || !p->dstates_b || p->dstates16_f) return false;
    // 16 bits: the ring variant of dCB, and the generic kernel of the states' gradients
    return p->dtype == BIMAMBA2_F32 || (dcb_ring_applies(p) && !(p->headdim % 64 == 0 && p->dstate % 64 == 0));
}
int launch_dcb_dstates(const bimamba2_params *p) {
    const RolesShape r = roles_shape(p);
    return p->dtype == BIMAMBA2_F32 ? launch_dcb_dstates_f32(p, r) : p->dtype == BIMAMBA2_BF16 ? launch_dcb_dstates_bf16(p, r) : launch_dcb_dstates_f16(p, r);
}

// One launch holds the registers of the dB / dC role (128 for states of up to 32 columns, 165 for 64, 245 for 128) for the dx role too,
// which then has one workgroup a CU above 128: it pays while most of the dx workgroups are on the chip at once anyway.
// us a pass over 16 heads, three launches -> one: 16 bits, heads of 16, dstate 16: 4 x 1024 (512 dx workgroups) 122 -> 101, 4 x 2048 (1024) 153 ->
// 149, 32 heads 8 x 2048 (4096) 398 -> 395, but heads of 64, dstate 32 573 -> 580; heads of 128, dstate 32: 4 x 2048 (2048) 306 -> 302.  dstate 64,
// heads of 32: 4 x 1024 (512) 123 -> 121, but 4 x 2048 186 -> 192.  dstate 128: 163 -> 170 (512).  float32, heads of 64, dstate 32: 4 x 1024 (1024)
// 204 -> 198, 4 x 2048 (2048) 323 -> 324; dstate 64: 4 x 1024 (1024) 238 -> 246.
static bool dx_db_dc_pays(const bimamba2_params *p) {
    const int pw = scan_col_tile_of(p->headdim, p->dtype);
    const int64_t dx = (int64_t)p->batch * nchunks(p) * p->nheads * ((p->headdim + pw - 1) / pw);
    return dx <= (p->dstate <= 32 ? 2048 : p->dstate <= 64 ? 512 : 256);
}

// dB and dC in one launch, without dx where that does not pay (us a pass, two launches -> one: float32, 2 x 1111, 16 heads of 64, dstate
// 64 190 -> 181; 4 x 1024, 8 heads of 128 235 -> 225; 4 x 2048, 16 heads of 64, dstate 128 598 -> 586; bfloat16, 8 x 1000, 16 heads
// of 32, dstate 64 176 -> 169): neither role fills the chip for long, and each alone ends with a wait for its slowest workgroup.
// 16-bit types lose by it where a role is many rounds of workgroups by itself, counted in heads of a place (8 x 2048: 32 heads of 64,
// dstate 32, eight of them, 554 -> 567; 16 heads of 40, dstate 48, eight, 345 -> 349; the case above four); float32 does
// not (8 x 2048, 32 heads of 64, dstate 64, sixteen, 1356 -> 1358; 2 x 3000, 8 groups of 8 heads of 32, twelve, 762 -> 716).
bool db_dc_roles(const bimamba2_params *p, bool states16) {
    const int64_t heads = (int64_t)p->batch * nchunks(p) * p->nheads * ((p->headdim + 63) / 64) * ((p->dstate + 63) / 64);
    return !p->causal && p->chunk_size <= 128 && !states16 && !dbdc_wide16(p) && p->dstate <= 128 && (p->dtype == BIMAMBA2_F32 || heads <= 4 * dbdc_places(p));
}
bool db_dc_merged(const bimamba2_params *p) { return db_dc_roles(p, p->states16_f || p->dstates16_f) && dbdc_heads(p) <= DBDC_HEADS; }
bool dx_db_dc_merged(const bimamba2_params *p) {
    return db_dc_merged(p) && p->CBT && dx_db_dc_pays(p) && scan_is_fast(p, true);
}
int launch_db_dc(const bimamba2_params *p) {
    RolesShape r = roles_shape(p);
    r.dx = false;
    return p->dtype == BIMAMBA2_F32 ? launch_dx_db_dc_f32(p, r) : p->dtype == BIMAMBA2_BF16 ? launch_dx_db_dc_bf16(p, r) : launch_dx_db_dc_f16(p, r);
}
int launch_dx_db_dc(const bimamba2_params *p) {
    const RolesShape r = roles_shape(p);
    return p->dtype == BIMAMBA2_F32 ? launch_dx_db_dc_f32(p, r) : p->dtype == BIMAMBA2_BF16 ? launch_dx_db_dc_bf16(p, r) : launch_dx_db_dc_f16(p, r);
}

}  // namespace bm2
