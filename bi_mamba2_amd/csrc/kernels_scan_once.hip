// A forward pass over a short sequence in one launch: without states going in or out and without anything kept for a backward pass, a sequence
// of at most 256 positions is the sum over its pairs of positions,
//
//   acc[t,p] = sum_s (C_t . B_s) m(t,s) dt[s] x[s,p],    m = e^{cs_f[t]-cs_f[s]} (s<t), e^{cs_b[t]-cs_b[s]} (s>t), 2 (s=t)
//   out = (acc + D x[t,p]) silu(z)
//
// A workgroup (8 waves) owns 64 positions (float32: 32) of one (batch, head) and a tile of headdim columns.  It brings the sequence's x and B rows into
// LDS, forms the head's decays itself, and its waves take 16 rows and every second (fourth) step of columns each.  Everything else such a pass is made of - the
// chunk cumsum, C.B^T, the states and their passing - would be a launch of 3 to 8 us of its own, of which the work is a fraction.
// Bound by the chain load - decays - barrier - steps - barrier - store, 5.5 us at 197 positions, 12 heads of 64 (bfloat16, dstate 64): 2.5 until
// the decays stand, 1.9 for the steps, 1.1 for the rest.  What made it short: loads without conditions and without the LDS copies that a
// struct in a select became (13 -> 5.5 us to the barrier), decays by four waves with row shifts instead of LDS permutes, two steps at a
// time.  us a call: 2 x 256, 4 heads of 32, dstate 16, float32 18.0 -> 7.2; 1 x 197, 12 heads of 64, dstate 64, bfloat16 17.0 -> 7.9; 4 x 256, 8 heads of 128,
// dstate 128 24.0 -> 9.7.  Error against 64 bits: float32 0.60 to 0.78 of the chunked pass's, float16 0.81 to 0.86, bfloat16 0.98 to 1.003.
// The decays are exact to the last rounding of an exponent: the sums are kept in 64 bits and only differences within a block of 16
// positions, or between a row and a block's edge, are rounded to 32 (the chunked pass rounds the sums of a chunk).
#include <type_traits>

#include "chunk_state_body.hpp"
#include "common.hpp"
#include "launch.hpp"

namespace bm2 {
namespace {

constexpr int ONCE_L = 256, ONCE_THREADS = 512;

template <typename T, int NS> struct OnceMap {
    // positions of a workgroup (float32, whose products are 16 times as long: 32), waves that share a row tile's columns
    static constexpr int ROWS = sizeof(T) == 4 ? 32 : 64, SHARE = 8 / (ROWS / 16);
    static constexpr int NJ = sizeof(T) == 4 ? 2 : 4, PW = 16 * NJ, N = NS * Mma<T>::KSTEP;      // headdim columns of a workgroup, dstate
    static constexpr int XP = sizeof(T) == 4 ? PW + 4 : PW, BP = N + 16 / (int)sizeof(T), RP = PW + 4;  // row pitches of x, B and of the two halves of the result, elements
};

// inclusive prefix sums over the 64 lanes without a trip through LDS per step (row shifts, then the last lanes of the rows of 16 and of 32)
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_shifted(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true), hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_incl_prefix_dpp(double v) {
    v += dpp_shifted<0x111, 0xf>(v);
    v += dpp_shifted<0x112, 0xf>(v);
    v += dpp_shifted<0x114, 0xf>(v);
    v += dpp_shifted<0x118, 0xf>(v);
    v += dpp_shifted<0x142, 0xa>(v);
    v += dpp_shifted<0x143, 0xc>(v);
    return v;
}

}  // namespace

template <typename T, int NS>
__global__ __launch_bounds__(ONCE_THREADS) void scan_once_kernel(const bimamba2_params p, int nrt, int npt) {
    typedef OnceMap<T, NS> Map;
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP, VS = 16 / (int)sizeof(T), NJ = Map::NJ, PW = Map::PW, N = Map::N;
    constexpr int XP = Map::XP, BP = Map::BP, RP = Map::RP, HALVES = KPL / 4, ROWS = Map::ROWS, SHARE = Map::SHARE;
    constexpr int BS_B = ONCE_L * BP * (int)sizeof(T), RED_B = SHARE * ROWS * RP * 4;
    __shared__ __attribute__((aligned(16))) T xs[ONCE_L * XP];
    __shared__ __attribute__((aligned(16))) char bs_red[BS_B > RED_B ? BS_B : RED_B];     // the B rows, then the waves' shares of the result
    T *bs = reinterpret_cast<T *>(bs_red);
    float *red = reinterpret_cast<float *>(bs_red);
    __shared__ __attribute__((aligned(16))) float gf[ONCE_L], gb[ONCE_L], lf[ONCE_L], lb[ONCE_L], dts[ONCE_L];    // column factors e^{-l} dt, sums relative to the edge of the block of 16, dt
    __shared__ double sf[ONCE_L], sb[ONCE_L], totals[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4, rtile = wave % (ROWS / 16), share = wave / (ROWS / 16);
    const int L = p.seqlen, P = p.headdim, H = p.nheads;
    const int rt = blockIdx.x % nrt, hp = blockIdx.x / nrt, pt = hp % npt, bh = hp / npt, h = bh % H, b = bh / H, g = h / (H / p.ngroups);
    const int p0 = pt * PW, r0 = rt * ROWS + rtile * 16;

    // ---- everything from memory at once ----
    const T *xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + h * p.x_sh + p0;
    const T *bp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + g * p.B_sg;
    const T *cp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + g * p.C_sg;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 zero = {0, 0, 0, 0};
    // (a thread's result: 16 bytes of one row)
    const int orow = rt * ROWS + (threadIdx.x >> 3), ocol = (threadIdx.x & 7) * VS;
    const bool mine = threadIdx.x < ROWS * 8 && orow < L && p0 + ocol < P;
    // (No load stands under a condition: the compiler would wait for each before the next.  What lies outside reads a valid neighbour.)
    const float A = p.A[h], bias = p.has_dt_bias ? p.dt_bias[h] : 0.f;
    const int q = min((int)threadIdx.x, ONCE_L - 1);          // the first four waves form the decays, one position a lane
    unsigned raw = 0;
    if (wave < 4) {
        const int64_t at = b * p.dt_sb + (int64_t)min(q, L - 1) * p.dt_sl + h * p.dt_sh;
        if (p.dt_dtype == BIMAMBA2_F32) raw = reinterpret_cast<const unsigned *>(p.dt)[at];
        else raw = reinterpret_cast<const unsigned short *>(p.dt)[at];
    }
    constexpr int XC = PW / VS, BC = N / VS;                  // 16-byte chunks of a row
    constexpr int XI = ONCE_L * XC / ONCE_THREADS, BI = ONCE_L * BC / ONCE_THREADS;
    u32x4 xr[XI], br[BI];
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        const int id = threadIdx.x + i * ONCE_THREADS, r = id / BC, c = id % BC;
        br[i] = *reinterpret_cast<const u32x4 *>(bp + (int64_t)min(r, L - 1) * p.B_sl + c * VS);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int id = threadIdx.x + i * ONCE_THREADS, r = id / XC, c = id % XC;
        xr[i] = *reinterpret_cast<const u32x4 *>(xp + (int64_t)min(r, L - 1) * p.x_sl + min(c * VS, P - p0 - VS));
    }
    Frag own[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) own[s] = M::load(cp + (int64_t)min(r0 + lr, L - 1) * p.C_sl + s * KSTEP + lg * KPL);
    u32x4 zraw = zero;
    if (p.has_z) zraw = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const T *>(p.z) + b * p.z_sb + (int64_t)min(orow, L - 1) * p.z_sl + h * p.z_sh + p0 + min(ocol, P - p0 - VS));
    float dv[VS] = {};
    if (p.has_D) {
        const float *dp = p.D_has_hdim ? p.D + h * P + p0 + min(ocol, P - p0 - VS) : p.D + h;
        const int step = p.D_has_hdim ? 1 : 0;
#pragma unroll
        for (int i = 0; i < VS; ++i) dv[i] = dp[i * step];
    }
    float v = 0.f;
    double step = 0., incl = 0.;
    if (wave < 4) {
        const unsigned short u = (unsigned short)raw;
        float d = p.dt_dtype == BIMAMBA2_F32 ? __uint_as_float(raw) : p.dt_dtype == BIMAMBA2_BF16 ? __uint_as_float(raw << 16) : (float)__builtin_bit_cast(f16_t, u);
        d += bias;
        if (p.dt_softplus) d = d > 20.f ? d : log1pf(expf(d));
        d = fminf(fmaxf(d, p.dt_min), p.dt_max);
        v = q < L ? d : 0.f;
        step = (double)v * A;
        incl = wave_incl_prefix_dpp(step);
        if (lane == 63) totals[wave] = incl;
    }
    raw_lds_wait();
    raw_lds_barrier();                                        // (not __syncthreads(), which would wait for the loads)
    asm volatile("" ::: "memory");
    if (wave < 4) {
        const double t0 = totals[0], t1 = totals[1], t2 = totals[2], t3 = totals[3];
        const double cf = incl + (wave == 0 ? 0. : wave == 1 ? t0 : wave == 2 ? t0 + t1 : t0 + t1 + t2), cb = (t0 + t1 + t2 + t3) - cf + step;
        // ... and the sums relative to those at the last position of the block of 16 (forward) and at its first (reverse)
        const float f = (float)(cf - __shfl(cf, lane | 15, 64)), r = (float)(cb - __shfl(cb, lane & ~15, 64));
        sf[q] = cf; sb[q] = cb;
        lf[q] = f; lb[q] = r;
        gf[q] = __expf(-f) * v; gb[q] = __expf(-r) * v;
        dts[q] = v;
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        const int id = threadIdx.x + i * ONCE_THREADS, r = id / BC, c = id % BC;
        *reinterpret_cast<u32x4 *>(bs + r * BP + c * VS) = r < L ? br[i] : zero;      // (zeros behind the end: the factors are, but what lies there may be no number)
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int id = threadIdx.x + i * ONCE_THREADS, r = id / XC, c = id % XC;
        *reinterpret_cast<u32x4 *>(xs + r * XP + (sizeof(T) == 2 ? c ^ tile64_swz(r) : c) * VS) = r < L && p0 + c * VS < P ? xr[i] : zero;
    }
    __syncthreads();

    // ---- this wave's 16 rows and its share of the columns ----
    f32x4 acc[NJ] = {};
    const int row = min(r0 + lr, L - 1);
    const double rf = sf[row], rb = sb[row];
    const float lrf = lf[row], lrb = lb[row];
    // two steps at a time, whose chains of reads, products and exponentials cover each other (a second one behind the end is zeros)
    for (int k0 = share * KSTEP; k0 < L; k0 += 2 * SHARE * KSTEP) {
        float c[2][KPL];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int hh = 0; hh < HALVES; ++hh) {
                // D[m][n] = B row k + KPL (m / 4) + 4 hh + m % 4 times C row n: a lane has four consecutive columns of its row
                f32x4 d = {};
                const T *brow = bs + (k0 + u * SHARE * KSTEP + KPL * (lr >> 2) + 4 * hh + (lr & 3)) * BP + lg * KPL;
#pragma unroll
                for (int s = 0; s < NS; ++s) d = M::mma(M::load(brow + s * KSTEP), own[s], d);
#pragma unroll
                for (int i = 0; i < 4; ++i) c[u][4 * hh + i] = d[i];
            }
        Frag a[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int ku = k0 + u * SHARE * KSTEP, k = ku + KPL * lg, kb = k & ~15;       // this lane's columns lie in one block of 16
            float w[KPL];
            const bool below = kb < r0;
            const double edge = *(below ? sf + (kb | 15) : sb + kb);
            const float ef = __expf((float)((below ? rf : rb) - edge));
            const float *gt = below ? gf : gb;
#pragma unroll
            for (int i = 0; i < KPL; i += 4) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(gt + k + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) w[i + j] = c[u][i + j] * ef * t[j];
            }
            if (ku <= r0 + 15 && ku + KSTEP > r0 && kb == r0) {       // across the diagonal
#pragma unroll
                for (int i = 0; i < KPL; ++i) {
                    const int s = k + i, r = r0 + lr;
                    const float e = s < r ? lrf - lf[s] : lrb - lb[s];
                    w[i] = c[u][i] * (s == r ? 2.f : __expf(e)) * dts[s];
                }
            }
            a[u] = M::pack(w);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                Frag xf;
                if constexpr (sizeof(T) == 2) xf = tile64_tr_frag<Frag>(xs, k0 + u * SHARE * KSTEP, j * 16, lr, lg);
                else {
#pragma unroll
                    for (int i = 0; i < KPL; ++i) xf[i] = xs[(k0 + u * SHARE * KSTEP + KPL * lg + i) * XP + j * 16 + lr];
                }
                acc[j] = M::mma(a[u], xf, acc[j]);
            }
    }
    __syncthreads();                                          // (the B rows lie where the result goes)
    float *mineh = red + (share * ROWS + rtile * 16) * RP;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) mineh[(4 * lg + i) * RP + j * 16 + lr] = acc[j][i];
    __syncthreads();

    // ---- the shares together, D, the gate ----
    if (!mine) return;
    const float *part = red + (threadIdx.x >> 3) * RP + ocol;
    Vec16<T> o;
    const Vec16<T> zv = __builtin_bit_cast(Vec16<T>, zraw);
    const Vec16<T> xv = *reinterpret_cast<const Vec16<T> *>(xs + orow * XP + (sizeof(T) == 2 ? (threadIdx.x & 7) ^ tile64_swz(orow) : (int)(threadIdx.x & 7)) * VS);
#pragma unroll
    for (int i = 0; i < VS; ++i) {
        float y = part[i];
#pragma unroll
        for (int t = 1; t < SHARE; ++t) y += part[t * ROWS * RP + i];
        if (p.has_D) y = __builtin_fmaf(dv[i], to_f(xv.v[i]), y);
        if (p.has_z) y *= silu_f(to_f(zv.v[i]));
        o.v[i] = from_f<T>(y);
    }
    *reinterpret_cast<Vec16<T> *>(reinterpret_cast<T *>(p.out) + (((int64_t)b * L + orow) * H + h) * P + p0 + ocol) = o;
}

static int once_row_tiles(const bimamba2_params *p) {
    const int rows = p->dtype == BIMAMBA2_F32 ? OnceMap<float, 1>::ROWS : OnceMap<bf16_t, 1>::ROWS;
    return (p->seqlen + rows - 1) / rows;
}
static int once_tiles(const bimamba2_params *p) {             // workgroups of a head
    const int columns = p->dtype == BIMAMBA2_F32 ? OnceMap<float, 1>::PW : OnceMap<bf16_t, 1>::PW;
    return once_row_tiles(p) * ((p->headdim + columns - 1) / columns);
}

// Where it runs: no intermediates are asked for (final states are: bimamba2_fwd forms them besides), no states go in, no packed sequences, at most 256 positions, and vector loads throughout.
bool scan_once_applies(const bimamba2_params *p) {
    if (p->seqlen > ONCE_L || p->causal || p->fwd_saved || p->seq_idx || p->out_x || p->dt_out || p->cs_f || p->cs_b || p->CB || p->CBT) return false;
    if (p->states_f || p->states_b || p->states16_f || p->states16_b || p->initial_f || p->initial_b) return false;
    const int N = p->dstate, e = p->dtype == BIMAMBA2_F32 ? 4 : 2, kstep = e == 4 ? 16 : 32, ns = N / kstep;
    if (N % kstep || (ns != 1 && ns != 2 && ns != 4) || p->headdim % (e == 4 ? 16 : 64)) return false;
    auto rows = [&](const void *t, int64_t s0, int64_t s1, int64_t s2) { return (reinterpret_cast<uintptr_t>(t) & 15) == 0 && ((s0 | s1 | s2) * e & 15) == 0; };
    if (!rows(p->x, p->x_sb, p->x_sl, p->x_sh) || !rows(p->Bm, p->B_sb, p->B_sl, p->B_sg) || !rows(p->Cm, p->C_sb, p->C_sl, p->C_sg) || !rows(p->out, 0, 0, 0) ||
        (p->has_z && !rows(p->z, p->z_sb, p->z_sl, p->z_sh)))
        return false;
    // Up to so many workgroups of one row.  The lines do not follow the number of rows, so that a row's result is the same alone and in any
    // batch; they lie where sixteen rows are as fast either way.  Time of the launches it replaces over its own, one row and sixteen:
    //   bfloat16, heads of 64, dstate 64: 16 workgroups (256 positions, 4 heads) 2.3 and 2.1; 48 (256, 12 heads) 2.2 and 1.08; 64 2.3 and 0.89
    //   dstate 128: 32 (256, 8 heads) 2.7 and 1.32; 36 (130, 12 heads) 2.0 and 0.84
    //   float32, heads of 64, dstate 64, whose chunk of 64 is one launch less up to there: 16 (64, 4 heads) 1.5 and 1.34; 32 1.45 and 0.80; behind: 40 (130, 4
    //     heads) 2.3 and 1.30; 64 (256, 4 heads) 2.1 and 0.88.  Heads of 32, dstate 16: 48 (64, 24 heads) 1.8 and 1.10; 64 0.93; 128 (256, 16 heads)
    //     2.5 and 0.99
    const int per_row = p->nheads * once_tiles(p);
    if (e == 2) return per_row <= (ns == 4 ? 32 : 48);
    return p->seqlen <= 64 ? per_row <= (ns == 4 ? 24 : ns == 2 ? 32 : 48) : per_row <= (ns == 4 ? 48 : ns == 2 ? 80 : 128);
}

int launch_scan_once(const bimamba2_params *p) {
    const int nrt = once_row_tiles(p), npt = once_tiles(p) / nrt;
    const int64_t grid = (int64_t)p->batch * p->nheads * nrt * npt;
    if (grid > 0x7fffffff) return BIMAMBA2_EUNSUPPORTED;
#define BM2_ONCE(T, NS) hipLaunchKernelGGL((scan_once_kernel<T, NS>), dim3((unsigned)grid), dim3(ONCE_THREADS), 0, reinterpret_cast<hipStream_t>(p->stream), *p, nrt, npt)
#define BM2_ONCE_T(T)                                   \
    switch (p->dstate / Mma<T>::KSTEP) {                \
        case 1: BM2_ONCE(T, 1); break;                  \
        case 2: BM2_ONCE(T, 2); break;                  \
        case 4: BM2_ONCE(T, 4); break;                  \
        default: return BIMAMBA2_EUNSUPPORTED;          \
    }
    if (p->dtype == BIMAMBA2_F32) { BM2_ONCE_T(float) }
    else if (p->dtype == BIMAMBA2_BF16) { BM2_ONCE_T(bf16_t) }
    else { BM2_ONCE_T(f16_t) }
#undef BM2_ONCE_T
#undef BM2_ONCE
    return check_launch();
}

}  // namespace bm2
