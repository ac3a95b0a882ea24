// One wave's work of the chunk cumsum, and the work of one workgroup of the generic chunk-state kernel.
#pragma once
#include <type_traits>

#include "common.hpp"

namespace bm2 {

// =========================================================================================================
// chunk cumsum: one wave per (b, c, h); lane i owns positions 4i..4i+3 of the chunk (Q <= 256)
// =========================================================================================================
// One wave's work for (b, c, h): dt' (v) and the two cumulative sums (cf, cb) at this lane's four positions.
// ACC: the type of the sums.  float32 problems take them in 64 bits and round once: a result there is off by little else than the
// resolution of these sums (their differences are exponents), and with every addition rounded it was off by 1.7 times as much.
// 16-bit results are not, and 64 bits would cost them 2 of 13 us over 2 x 16384 positions of 48 heads.
// The sums of a lane's four positions with the products dt * A unrounded, as the chunk-state kernel with direct loads takes them.  (Written
// out: with the cuts' conditions between product and sum the compiler does not fuse the two by itself.)  cut_*: of packed sequences, in
// front of a position in the forward sums and behind it in the reverse ones.
__device__ __forceinline__ void chunk_sums_unrounded(const float (&dt)[4], float A, const float (&cut_f)[4], const float (&cut_b)[4], int lane, float (&cf)[4], float (&cb)[4]) {
    float pf[4], sb[4];
    pf[0] = fmaf(dt[0], A, cut_f[0]);
    sb[3] = fmaf(dt[3], A, cut_b[3]);
#pragma unroll
    for (int e = 1; e < 4; ++e) {
        pf[e] = fmaf(dt[e], A, pf[e - 1] + cut_f[e]);
        sb[3 - e] = fmaf(dt[3 - e], A, sb[4 - e] + cut_b[3 - e]);
    }
    const float tot = pf[3], tot_r = sb[0];
    const float before = wave_incl_prefix(tot, lane) - tot, after = wave_incl_suffix(tot_r, lane) - tot_r;
    cf[0] = fmaf(dt[0], A, before + cut_f[0]);
    cb[3] = fmaf(dt[3], A, after + cut_b[3]);
#pragma unroll
    for (int e = 1; e < 4; ++e) {
        cf[e] = before + pf[e];
        cb[3 - e] = after + sb[3 - e];
    }
}
// UNROUNDED: the sums as above
template <typename DT, typename ACC, bool UNROUNDED = false>
__device__ __forceinline__ void chunk_cumsum_wave(const bimamba2_params &p, int b, int c, int h, int lane, float (&v)[4], float (&cf)[4], float (&cb)[4]) {
    const int Q = p.chunk_size;
    const int limit = min(Q, p.seqlen - c * Q);
    const DT *dt = reinterpret_cast<const DT *>(p.dt) + b * p.dt_sb + (int64_t)c * Q * p.dt_sl + h * p.dt_sh;
    const float A = p.A[h];
    const float bias = p.has_dt_bias ? p.dt_bias[h] : 0.f;
    ACC a[4], ar[4];                                  // ar: exponents of the reverse direction (differ with seq_idx only)
    float cut_f[4] = {}, cut_b[4] = {};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int q = lane * 4 + e;
        float d = 0.f;
        if (q < limit) {
            d = to_f(dt[(int64_t)q * p.dt_sl]) + bias;
            if (p.dt_softplus) d = d > 20.f ? d : log1pf(expf(d));
            d = fminf(fmaxf(d, p.dt_min), p.dt_max);
        }
        v[e] = d;
        a[e] = ar[e] = (ACC)d * A;
        if (p.seq_idx && q < limit) {
            // packed sequences: cut the forward recurrence in front of a sequence's first position, the reverse one
            // behind its last
            const int l = c * Q + q;
            const int32_t *si = p.seq_idx + (int64_t)b * p.seqlen + l;
            const int32_t cur = si[0];
            if (l > 0 && si[-1] != cur) { a[e] += BIMAMBA2_SEQ_CUT; cut_f[e] = BIMAMBA2_SEQ_CUT; }
            if (l + 1 < p.seqlen && si[1] != cur) { ar[e] += BIMAMBA2_SEQ_CUT; cut_b[e] = BIMAMBA2_SEQ_CUT; }
        }
    }
    if constexpr (UNROUNDED) return chunk_sums_unrounded(v, A, cut_f, cut_b, lane, cf, cb);
    // forward inclusive scan, reverse inclusive scan
    ACC pf[4], sb[4];
    pf[0] = a[0]; pf[1] = pf[0] + a[1]; pf[2] = pf[1] + a[2]; pf[3] = pf[2] + a[3];
    sb[3] = ar[3]; sb[2] = sb[3] + ar[2]; sb[1] = sb[2] + ar[1]; sb[0] = sb[1] + ar[0];
    const ACC tot = pf[3], tot_r = sb[0];
    const ACC before = wave_incl_prefix(tot, lane) - tot, after = wave_incl_suffix(tot_r, lane) - tot_r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        cf[e] = (float)(before + pf[e]);
        cb[e] = (float)(after + sb[e]);
    }
}
// ... and their way to dt_out, cs_f, cs_b (o: offset of the (b, c, h) there)
__device__ __forceinline__ void chunk_cumsum_store(const bimamba2_params &p, int64_t o, int lane, const float (&v)[4], const float (&cf)[4], const float (&cb)[4]) {
    const int Q = p.chunk_size;
    if (Q % 4 == 0) {
        // a lane's four positions are contiguous: 16-byte stores (the three tensors are contiguous and Q * 4 bytes per row)
        if (lane * 4 < Q) {
            *reinterpret_cast<f32x4 *>(p.dt_out + o + lane * 4) = f32x4{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<f32x4 *>(p.cs_f + o + lane * 4) = f32x4{cf[0], cf[1], cf[2], cf[3]};
            *reinterpret_cast<f32x4 *>(p.cs_b + o + lane * 4) = f32x4{cb[0], cb[1], cb[2], cb[3]};
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int q = lane * 4 + e;
        if (q < Q) {
            p.dt_out[o + q] = v[e];
            p.cs_f[o + q] = cf[e];
            p.cs_b[o + q] = cb[e];
        }
    }
}

// =========================================================================================================
// chunk state (DSTATES = false):  S_f[p,n] = sum_k x[k,p] B[k,n] e^{cs_f[Q-1]-cs_f[k]} dt[k],  S_b with
//                                 e^{cs_b[0]-cs_b[k]}
// gradient of the chunk-entry states (DSTATES = true):  dprev_f[p,n] = sum_k dy[k,p] C[k,n] e^{cs_f[k]},
//                                 dprev_b with e^{cs_b[k]}
// =========================================================================================================
// Both operands have K = chunk position as their slow dimension, so both are staged transposed (8x8 in-register
// transposes) into LDS, KH positions at a time; the decay weights are applied to the B-side image while staging.
template <typename T> struct ChunkStateMap {
    static constexpr int KH = 128 / (int)sizeof(T);                                   // chunk positions staged per round
    static constexpr int LDX = KH + 16 / (int)sizeof(T), IMAGE = 64 * LDX * (int)sizeof(T);
    static constexpr int BLOCKS = (KH / (16 / (int)sizeof(T))) * (64 / (16 / (int)sizeof(T)));   // of x, staged by as many threads; B is the next ones' work
    static constexpr int WF = 3 * IMAGE, WB = WF + 4 * BIMAMBA2_MAX_CHUNK, LDS = WB + 4 * BIMAMBA2_MAX_CHUNK;
};
// lds: ChunkStateMap<T>::LDS bytes; bch: (batch, chunk, head)
// CUMSUM (states only): the workgroup's first wave does the work of chunk_cumsum_fwd_kernel for its (b, c, h) on the way, and the
// first tile's workgroup writes dt_out, cs_f, cs_b for the later kernels.
template <typename T, bool DSTATES, bool FAST, bool CUMSUM = false>
__device__ __forceinline__ void chunk_state_body(const bimamba2_params &p, int nc, int nt, int pt, int bch, char *lds) {
    typedef Mma<T> M;
    typedef ChunkStateMap<T> Map;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP, KH = Map::KH, LDX = Map::LDX;
    T *xT = reinterpret_cast<T *>(lds), *Bf = reinterpret_cast<T *>(lds + Map::IMAGE), *Bb = reinterpret_cast<T *>(lds + 2 * Map::IMAGE);
    float *wf = reinterpret_cast<float *>(lds + Map::WF), *wb = reinterpret_cast<float *>(lds + Map::WB);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int h = bch % p.nheads, bc = bch / p.nheads, c = bc % nc, b = bc / nc;
    const int g = h / (p.nheads / p.ngroups);
    const int Q = p.chunk_size, N = p.dstate, P = p.headdim;
    const int limit = min(Q, p.seqlen - c * Q);
    const int64_t o = (((int64_t)b * p.nheads + h) * nc + c) * Q;
    if constexpr (CUMSUM && !DSTATES) {
        if (wave == 0) {
            typedef std::conditional_t<sizeof(T) == 4, double, float> ACC;
            float v[4], cf[4], cb[4];
            if (p.dt_dtype == BIMAMBA2_F32) chunk_cumsum_wave<float, ACC>(p, b, c, h, lane, v, cf, cb);
            else if (p.dt_dtype == BIMAMBA2_BF16) chunk_cumsum_wave<bf16_t, ACC>(p, b, c, h, lane, v, cf, cb);
            else chunk_cumsum_wave<f16_t, ACC>(p, b, c, h, lane, v, cf, cb);
            if (nt == 0 && pt == 0) chunk_cumsum_store(p, o, lane, v, cf, cb);
            // cs_f at the chunk's last position (past the sequence's end: what it was there), cs_b at its first
            const float ef = __shfl(cf[(Q - 1) & 3], (Q - 1) >> 2, 64), eb = __shfl(cb[0], 0, 64);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wf[lane * 4 + e] = __expf(ef - cf[e]) * v[e];              // (v is 0 past the end)
                wb[lane * 4 + e] = __expf(eb - cb[e]) * v[e];
            }
        }
    } else
    for (int q = threadIdx.x; q < Q; q += NTHREADS) {
        float f = 0.f, r = 0.f;
        if (q < limit) {
            if (DSTATES) {
                f = __expf(p.cs_f[o + q]);
                r = __expf(p.cs_b[o + q]);
            } else {
                const float d = p.dt_out[o + q];
                f = __expf(p.cs_f[o + Q - 1] - p.cs_f[o + q]) * d;
                r = __expf(p.cs_b[o] - p.cs_b[o + q]) * d;
            }
        }
        wf[q] = f;
        wb[q] = r;
    }
    const T *xp;
    int64_t xs;
    if (DSTATES) {
        const T *src = reinterpret_cast<const T *>(p.has_z ? p.dout_x : p.dout);
        if (p.has_z) { xs = (int64_t)p.nheads * P; xp = src + ((int64_t)b * p.seqlen + (int64_t)c * Q) * xs + (int64_t)h * P; }
        else { xs = p.dout_sl; xp = src + b * p.dout_sb + (int64_t)c * Q * xs + h * p.dout_sh; }
    } else {
        xs = p.x_sl;
        xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * xs + h * p.x_sh;
    }
    xp += pt * 64;
    const T *bp;
    int64_t bs;
    if (DSTATES) { bs = p.C_sl; bp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + (int64_t)c * Q * bs + g * p.C_sg; }
    else { bs = p.B_sl; bp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * bs + g * p.B_sg; }
    bp += nt * 64;
    f32x4 accf[4] = {}, accb[4] = {};
    for (int k0 = 0; k0 < limit; k0 += KH) {
        __syncthreads();       // weights written / previous round consumed
        const int kv = limit - k0;
        stage_transposed<T, KH, 64, LDX, FAST>(xT, xp + (int64_t)k0 * xs, xs, kv, P - pt * 64,
                                               [&](int k) { return k < kv ? 1.f : 0.f; });
        stage_transposed2<T, KH, 64, LDX, FAST, Map::BLOCKS % NTHREADS>(Bf, Bb, bp + (int64_t)k0 * bs, bs, kv, N - nt * 64,
                                                [&](int k) { return k < kv ? wf[k0 + k] : 0.f; },
                                                [&](int k) { return k < kv ? wb[k0 + k] : 0.f; });
        __syncthreads();
        const int kend = min(KH, (kv + KSTEP - 1) / KSTEP * KSTEP);
        for (int ks = 0; ks < kend; ks += KSTEP) {
            const int kq = ks + lg * KPL;
            const typename M::Frag a = M::load(xT + xt_index<T, LDX>(wave * 16 + lr, kq));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!FAST && nt * 64 + j * 16 >= N) continue;      // (uniform) narrow states: nothing in this column tile
                accf[j] = M::mma(a, M::load(Bf + xt_index<T, LDX>(j * 16 + lr, kq)), accf[j]);
                accb[j] = M::mma(a, M::load(Bb + xt_index<T, LDX>(j * 16 + lr, kq)), accb[j]);
            }
        }
    }
    float *of = (DSTATES ? p.dstates_f : p.states_f) + (int64_t)bch * P * N;
    float *ob = (DSTATES ? p.dstates_b : p.states_b) + (int64_t)bch * P * N;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int pp = pt * 64 + wave * 16 + lg * 4 + i, n = nt * 64 + j * 16 + lr;
            if (pp < P && n < N) {
                of[(int64_t)pp * N + n] = accf[j][i];
                ob[(int64_t)pp * N + n] = accb[j][i];
            }
        }
}

// ---------------------------------------------------------------------------------------------------------
// The same for 16-bit types in chunks of up to 128 positions, headdim and dstate multiples of 8, aligned rows: the whole x tile and
// the whole B tile of the chunk come by direct loads, all requested at once, and the operands are LDS transpose reads (no registers
// to stage in, 143 of them above: four workgroups fit a CU instead of three, and each waits for memory once).  A row's units past
// headdim or dstate are not requested: what lies there gives outputs that nobody stores.
// The weighted operand enters in two 16-bit parts: the kernel waits for memory, and states that were off by its rounding made dA up to
// 32 % less exact in chunks of 128 than in the ones of 256 that a caller asked for.  Time with two parts and one: 39.5 and 38.3 us a
// forward pass over 4 x 2048, 16 heads of 16, dstate 16, two boxes; 134 and 133.5 in training.
// 4 x 2048 in chunks of 128, bfloat16, 16 heads, headdim 16, dstate 16: the forward launch 24 -> 15 us, beside dCB 27 -> 22; headdim 128, dstate 32: 35 -> 27 and 26 -> 18.
// ---------------------------------------------------------------------------------------------------------
struct ChunkStateNarrowMap {
    static constexpr int ROWS = 128, TILE = ROWS * 128;                                  // rows of 64 elements, tile64 swizzle
    static constexpr int WF = 2 * TILE, WB = WF + 4 * BIMAMBA2_MAX_CHUNK, LDS = WB + 4 * BIMAMBA2_MAX_CHUNK;
};
template <typename T, bool DSTATES, bool CUMSUM = false>
__device__ __forceinline__ void chunk_state_narrow_body(const bimamba2_params &p, int nc, int nt, int pt, int bch, char *lds) {
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    typedef ChunkStateNarrowMap Map;
    static_assert(sizeof(T) == 2, "16-bit operands");
    T *xt = reinterpret_cast<T *>(lds), *bt = reinterpret_cast<T *>(lds + Map::TILE);
    float *wf = reinterpret_cast<float *>(lds + Map::WF), *wb = reinterpret_cast<float *>(lds + Map::WB);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int h = bch % p.nheads, bc = bch / p.nheads, c = bc % nc, b = bc / nc;
    const int g = h / (p.nheads / p.ngroups);
    const int Q = p.chunk_size, N = p.dstate, P = p.headdim;
    const int limit = min(Q, p.seqlen - c * Q), rows = (limit + 31) & ~31;
    const int64_t o = (((int64_t)b * p.nheads + h) * nc + c) * Q;
    const T *xp, *bp;
    int64_t xs, bs;
    if (DSTATES) {
        if (p.has_z) { xs = (int64_t)p.nheads * P; xp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * xs + (int64_t)h * P; }
        else { xs = p.dout_sl; xp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * xs + h * p.dout_sh; }
        bs = p.C_sl;
        bp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + (int64_t)c * Q * bs + g * p.C_sg;
    } else {
        xs = p.x_sl;
        xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * xs + h * p.x_sh;
        bs = p.B_sl;
        bp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * bs + g * p.B_sg;
    }
    // unit of 8 rows: lane l brings 16 bytes of row l / 8 (rows behind the sequence's end read its last row: weight 0)
    for (int u = wave; u < rows / 8; u += NTHREADS / 64) {
        const int row = u * 8 + (lane >> 3), col = ((lane & 7) ^ tile64_swz(row)) << 3;
        const int64_t r = min(row, limit - 1);
        if (pt * 64 + col < P) load16_to_lds(xp + r * xs + pt * 64 + col, xt + u * 512);
        if (nt * 64 + col < N) load16_to_lds(bp + r * bs + nt * 64 + col, bt + u * 512);
    }
    if constexpr (CUMSUM && !DSTATES) {
        if (wave == 0) {
            float v[4], cf[4], cb[4];
            if (p.dt_dtype == BIMAMBA2_F32) chunk_cumsum_wave<float, float>(p, b, c, h, lane, v, cf, cb);
            else if (p.dt_dtype == BIMAMBA2_BF16) chunk_cumsum_wave<bf16_t, float>(p, b, c, h, lane, v, cf, cb);
            else chunk_cumsum_wave<f16_t, float>(p, b, c, h, lane, v, cf, cb);
            if (nt == 0 && pt == 0) chunk_cumsum_store(p, o, lane, v, cf, cb);
            const float ef = __shfl(cf[(Q - 1) & 3], (Q - 1) >> 2, 64), eb = __shfl(cb[0], 0, 64);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wf[lane * 4 + e] = __expf(ef - cf[e]) * v[e];              // (v is 0 past the end)
                wb[lane * 4 + e] = __expf(eb - cb[e]) * v[e];
            }
        }
    } else {
        for (int q = threadIdx.x; q < rows; q += NTHREADS) {
            const int qc = min(q, limit - 1);
            const float cf = p.cs_f[o + qc], cb = p.cs_b[o + qc];
            float f, r;
            if (DSTATES) { f = __expf(cf); r = __expf(cb); }
            else {
                const float d = p.dt_out[o + qc];
                f = __expf(p.cs_f[o + Q - 1] - cf) * d;
                r = __expf(p.cs_b[o] - cb) * d;
            }
            wf[q] = q < limit ? f : 0.f;
            wb[q] = q < limit ? r : 0.f;
        }
    }
    wait_vmcnt<0>();
    __syncthreads();
    if (pt * 64 + wave * 16 >= P) return;
    f32x4 accf[4] = {}, accb[4] = {};
    for (int ks = 0; ks < rows; ks += 32) {
        const Frag a = tile64_tr_frag<Frag>(xt, ks, wave * 16, lr, lg);
        float vf[8], vb[8];
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            const f32x4 f4 = *reinterpret_cast<const f32x4 *>(wf + ks + lg * 8 + i), b4 = *reinterpret_cast<const f32x4 *>(wb + ks + lg * 8 + i);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const T x = a[i + k];
                vf[i + k] = to_f(x) * f4[k];
                vb[i + k] = to_f(x) * b4[k];
            }
        }
        Frag af, ab, af_rest, ab_rest;
        split_operand<T>(vf, af, af_rest);
        split_operand<T>(vb, ab, ab_rest);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (nt * 64 + j * 16 >= N) continue;               // (uniform)
            const Frag bf = tile64_tr_frag<Frag>(bt, ks, j * 16, lr, lg);
            accf[j] = M::mma(af_rest, bf, M::mma(af, bf, accf[j]));
            accb[j] = M::mma(ab_rest, bf, M::mma(ab, bf, accb[j]));
        }
    }
    float *of = (DSTATES ? p.dstates_f : p.states_f) + (int64_t)bch * P * N, *ob = (DSTATES ? p.dstates_b : p.states_b) + (int64_t)bch * P * N;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int pp = pt * 64 + wave * 16 + lg * 4 + i, n = nt * 64 + j * 16 + lr;
            if (pp < P && n < N) {
                of[(int64_t)pp * N + n] = accf[j][i];
                ob[(int64_t)pp * N + n] = accb[j][i];
            }
        }
}

}  // namespace bm2
