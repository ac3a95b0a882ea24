// A forward pass over a short sequence in one launch: without states going in or out and without anything kept for a backward pass, a sequence
// of at most 256 positions is the sum over its pairs of positions,
//
//   acc[t,p] = sum_s (C_t . B_s) m(t,s) dt[s] x[s,p],    m = e^{cs_f[t]-cs_f[s]} (s<t), e^{cs_b[t]-cs_b[s]} (s>t), 2 (s=t)
//   out = (acc + D x[t,p]) silu(z)
//
// scan_once_kernel, for few rows of more than 128 positions: a workgroup (8 waves) owns 64 positions (float32: 32) of one (batch, head) and a tile of headdim columns.  It brings the sequence's x and B rows into
// LDS, forms the head's decays itself, and its waves take 16 rows and every second (fourth) step of columns each.  Everything else such a pass is made of - the
// chunk cumsum, C.B^T, the states and their passing - would be a launch of 3 to 8 us of its own, of which the work is a fraction.
// Bound by the chain load - decays - barrier - steps - barrier - store, a few hundred workgroups at most: 8.2 us in the trace of a layer at 197 positions,
// 12 heads of 64 (bfloat16, dstate 64, 48 workgroups).  What made it short: loads without conditions and without the LDS copies that a
// struct in a select became, decays by four waves with row shifts instead of LDS permutes, two steps at a time.  us a call, from the chunked launches: 2 x 256, 4 heads of 32, dstate 16, float32 18.0 -> 7.2; 1 x 197, 12 heads of 64, dstate 64, bfloat16 17.0 -> 7.9; 4 x 256, 8 heads of 128,
// dstate 128 24.0 -> 9.7.  Error against 64 bits: float32 0.60 to 1.0 of the chunked pass's, float16 0.81 to 0.86, bfloat16 0.98 to 1.000.
// The decays are exact to the last rounding of an exponent: the sums are kept in 64 bits and only differences within a block of 16
// positions, or between a row and a block's edge, are rounded to 32 (the chunked pass rounds the sums of a chunk).
#include <algorithm>
#include <type_traits>

#include "chunk_state_body.hpp"
#include "common.hpp"
#include "launch.hpp"

namespace bm2 {
namespace {

constexpr int ONCE_L = 256, ONCE_THREADS = 512, WALK_GRID = 2097152;

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

// a position's dt as it lies in memory, and its step
__device__ __forceinline__ unsigned once_dt_raw(const bimamba2_params &p, int b, int h, int q) {
    const int64_t at = b * p.dt_sb + (int64_t)min(q, p.seqlen - 1) * p.dt_sl + h * p.dt_sh;
    return p.dt_dtype == BIMAMBA2_F32 ? reinterpret_cast<const unsigned *>(p.dt)[at] : reinterpret_cast<const unsigned short *>(p.dt)[at];
}
__device__ __forceinline__ float once_dt(const bimamba2_params &p, unsigned raw, float bias) {
    const unsigned short u = (unsigned short)raw;
    float d = p.dt_dtype == BIMAMBA2_F32 ? __uint_as_float(raw) : p.dt_dtype == BIMAMBA2_BF16 ? __uint_as_float(raw << 16) : (float)__builtin_bit_cast(f16_t, u);
    d += bias;
    if (p.dt_softplus) d = d > 20.f ? d : log1pf(expf(d));
    return fminf(fmaxf(d, p.dt_min), p.dt_max);
}
// a position's entries of the tables; incl: its sum within the block of 64 positions whose wave this is, totals: those of the four blocks
__device__ __forceinline__ void once_decays(double step, double incl, const double *totals, int wave, int lane, int q, float v, float *gf, float *gb, float *lf, float *lb,
                                            float *dts, double *sf, double *sb) {
    const double t0 = totals[0], t1 = totals[1], t2 = totals[2], t3 = totals[3];
    const double cf = incl + (wave == 0 ? 0. : wave == 1 ? t0 : wave == 2 ? t0 + t1 : t0 + t1 + t2), cb = (t0 + t1 + t2 + t3) - cf + step;
    // ... and the sums relative to those at the last position of the block of 16 (forward) and at its first (reverse)
    const float f = (float)(cf - __shfl(cf, lane | 15, 64)), r = (float)(cb - __shfl(cb, lane & ~15, 64));
    sf[q] = cf; sb[q] = cb;
    lf[q] = f; lb[q] = r;
    gf[q] = __expf(-f) * v; gb[q] = __expf(-r) * v;
    dts[q] = v;
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
    if (wave < 4) raw = once_dt_raw(p, b, h, q);
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
        const float d = once_dt(p, raw, bias);
        v = q < L ? d : 0.f;
        step = (double)v * A;
        incl = wave_incl_prefix_dpp(step);
        if (lane == 63) totals[wave] = incl;
    }
    ordered_lds_barrier();
    if (wave < 4) once_decays(step, incl, totals, wave, lane, q, v, gf, gb, lf, lb, dts, sf, sb);
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

// The same sums where there is work for the whole chip, and for up to 128 positions: a workgroup owns a whole sequence of up to LP positions and walks through
// heads of one group, where scan_once_kernel fetches x and B for every 64 positions and forms C.B^T for every head again.  A wave takes one row tile (of more
// than 128 positions two, one after the other) and all columns: C.B^T is formed once and stays in registers, nothing is exchanged between waves, and a head's x and
// decays are brought while the head before is worked on.  Steps, and which of them add up to which sum, are those of scan_once_kernel, so that the results
// are the same bits and the number of rows may choose between the two (launch_scan_once).
// Bound by vector instructions: at 256 x 256 positions, 12 heads of 64 (bfloat16, dstate 64, two waves a SIMD) they are issued 62 % of the time, two products and
// half a conversion per pair of positions most of them; a head takes 6.3 us with the chip half empty and 8 with 256 workgroups on it.  What made it so:
// whole columns a wave instead of shares that meet in LDS (four barriers a head less, 159 -> 127 us), results as 16-byte stores from the sums of transposed products,
// z and x never waited for behind stores (118 -> 101), addresses by immediates.  us a call, scan_once_kernel for every 64 positions -> this one (before: the chunked launches):
// 64 x 256, 12 heads, z, dstate 64 53 -> 31 (33); 256 x 256, 8 heads, dstate 128 245 -> 66 (65); 256 x 256, 16 heads of 32, dstate 16, float32 419 -> 213 (355);
// 64 x 64, 48 heads 43 -> 22 (44).
template <typename T, int NS, int LP> struct WalkMap {
    typedef OnceMap<T, NS> Once;
    static constexpr int WAVES = LP == 64 ? 4 : 8, THREADS = 64 * WAVES, NRT = LP / (16 * WAVES), NSTEP = LP / Mma<T>::KSTEP;     // row tiles and steps of a wave
    static constexpr int XS_B = LP * Once::XP * (int)sizeof(T), BS_B = LP * Once::BP * (int)sizeof(T);
    static constexpr int BODY_B = XS_B + (BS_B > XS_B ? BS_B : XS_B);                   // x of the head in hand; the B rows, then x of the next
    static_assert(Once::SHARE * Mma<T>::KSTEP == 64 && BODY_B + 2 * LP * 36 + 8 * Once::PW + 64 <= 160 * 1024, "LDS");
};

template <typename T, int NS, int LP, bool Z>
__global__ __launch_bounds__((WalkMap<T, NS, LP>::THREADS), LP == 256 ? 2 : 4) void scan_once_walk_kernel(const bimamba2_params p, int npt, int hpw, int first_row) {
    typedef WalkMap<T, NS, LP> W;
    typedef OnceMap<T, NS> Map;
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP, VS = 16 / (int)sizeof(T), NJ = Map::NJ, PW = Map::PW, N = Map::N, THREADS = W::THREADS;
    constexpr int XP = Map::XP, BP = Map::BP, HALVES = KPL / 4, SHARE = Map::SHARE, NRT = W::NRT, NSTEP = W::NSTEP, DW = LP / 64;
    __shared__ __attribute__((aligned(16))) char body[W::BODY_B];
    __shared__ __attribute__((aligned(16))) float tables[2][5][LP];       // gf, gb, lf, lb, dts of scan_once_kernel
    __shared__ __attribute__((aligned(16))) float ds[2][PW];
    __shared__ double sums[2][2][LP], totals[4];
    T *bs = reinterpret_cast<T *>(body + W::XS_B);
    // (what follows from the lane is worked out anew for each head: kept, it would take the registers that C.B^T lies in)
    int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int L = p.seqlen, P = p.headdim, H = p.nheads, hpg = H / p.ngroups, nsl = (hpg + hpw - 1) / hpw;
    const int pt = blockIdx.x % npt, unit = blockIdx.x / npt, sl = unit % nsl, bg = unit / nsl, g = bg % p.ngroups, b = first_row + bg / p.ngroups;
    const int p0 = pt * PW, h0 = g * hpg + sl * hpw, nh = min(hpw, hpg - sl * hpw);
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 zero = {0, 0, 0, 0};
    const bool has_D = p.has_D, d_cols = p.has_D && p.D_has_hdim;

    // ---- a head's x and dt, requested ahead ----
    constexpr int XC = PW / VS, BC = N / VS, XI = LP * XC / THREADS, BI = (LP * BC + THREADS - 1) / THREADS, XROWS = THREADS / XC;
    static_assert(XROWS % 16 == 0, "the image's swizzle repeats");
    u32x4 xr[XI];
    unsigned raw = 0;
    float A = 0.f, bias = 0.f, D = 0.f;
    auto request = [&](int h) __attribute__((always_inline)) {
        // (loads without conditions and without arithmetic behind them: a wait for one of these would be for x as well)
        A = p.A[h];
        bias = (p.has_dt_bias ? p.dt_bias : p.A)[h];
        D = (has_D ? p.D : p.A)[d_cols ? h * P + min(p0 + tid, P - 1) : h];
        if (wave < DW) raw = once_dt_raw(p, b, h, tid);
        // (this thread's column unit of rows xrow, xrow + XROWS ...)
        const int xrow = (unsigned)tid / XC;
        const T *xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + h * p.x_sh + p0 + min((int)((unsigned)tid % XC) * VS, P - p0 - VS);
#pragma unroll
        for (int i = 0; i < XI; ++i) xr[i] = *reinterpret_cast<const u32x4 *>(xp + (int64_t)min(xrow + i * XROWS, L - 1) * p.x_sl);
    };
    // (between the two a position's step and sum wait where its entries will lie)
    auto form_sums = [&](int k) __attribute__((always_inline)) {
        if (tid < PW) ds[k][tid] = D;
        if (wave >= DW) return;
        const float d = once_dt(p, raw, p.has_dt_bias ? bias : 0.f), v = tid < L ? d : 0.f;
        const double step = (double)v * A, incl = wave_incl_prefix_dpp(step);
        if ((tid & 63) == 63) totals[wave] = incl;
        tables[k][4][tid] = v;
        sums[k][0][tid] = incl;
        sums[k][1][tid] = step;
    };
    auto form_tables = [&](int k) __attribute__((always_inline)) {
        if (wave < DW)
            once_decays(sums[k][1][tid], sums[k][0][tid], totals, wave, tid & 63, tid, tables[k][4][tid], tables[k][0], tables[k][1], tables[k][2], tables[k][3], tables[k][4], sums[k][0],
                        sums[k][1]);
    };
    auto store_x = [&](int k) __attribute__((always_inline)) {
        const unsigned xrow = (unsigned)tid / XC, c = (unsigned)tid % XC;
        T *xs = reinterpret_cast<T *>(body + k * W::XS_B) + xrow * XP + (sizeof(T) == 2 ? c ^ tile64_swz(xrow) : c) * VS;
        const bool in = sizeof(T) == 2 || p0 + (int)c * VS < P;      // (16 bits: whole tiles of columns)
#pragma unroll
        for (int i = 0; i < XI; ++i) *reinterpret_cast<u32x4 *>(xs + i * XROWS * XP) = (int)xrow + i * XROWS < L && in ? xr[i] : zero;
    };
    // The products are formed transposed (rows of the matrix instruction are columns of x), and which column of x such a row stands for is chosen so that
    // a lane holds 2 x 16 bytes of one row of the result: column(k) on, k = 0, 1.
    auto column = [&](int k) __attribute__((always_inline)) { return (sizeof(T) == 2 ? 32 : 16) * k + VS * ((tid >> 4) & 3); };

    u32x4 zraw[2] = {zero, zero};
    auto request_z = [&](int h, int row) __attribute__((always_inline)) {
        const T *zp = reinterpret_cast<const T *>(p.z) + b * p.z_sb + h * p.z_sh + row * p.z_sl + p0;
#pragma unroll
        for (int k = 0; k < 2; ++k) zraw[k] = *reinterpret_cast<const u32x4 *>(zp + min(column(k), P - p0 - VS));
    };

    // ---- C.B^T of the wave's rows ----
    const T *bp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + g * p.B_sg;
    const T *cp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + g * p.C_sg;
    u32x4 br[BI];
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        const int id = min(tid + i * THREADS, LP * BC - 1), r = id / BC, c = id % BC;
        br[i] = *reinterpret_cast<const u32x4 *>(bp + (int64_t)min(r, L - 1) * p.B_sl + c * VS);
    }
    request(h0);
    float cb[NRT][NSTEP][KPL];
    {
        const int lr = tid & 15, lg = (tid >> 4) & 3;
        Frag own[NRT][NS];
#pragma unroll
        for (int t = 0; t < NRT; ++t)
#pragma unroll
            for (int s = 0; s < NS; ++s) own[t][s] = M::load(cp + (int64_t)min((t * W::WAVES + wave) * 16 + lr, L - 1) * p.C_sl + s * KSTEP + lg * KPL);
        if (tid >= DW && tid < 4) totals[tid] = 0.;
        form_sums(0);
#pragma unroll
        for (int i = 0; i < BI; ++i) {
            const int id = tid + i * THREADS, r = id / BC, c = id % BC;
            if (id < LP * BC) *reinterpret_cast<u32x4 *>(bs + r * BP + c * VS) = r < L ? br[i] : zero;
        }
        store_x(0);
        ordered_lds_barrier();
        form_tables(0);
        if (nh > 1) request(h0 + 1);
#pragma unroll
        for (int n = 0; n < NSTEP; ++n)
#pragma unroll
            for (int hh = 0; hh < HALVES; ++hh) {
                const T *brow = bs + (n * KSTEP + KPL * (lr >> 2) + 4 * hh + (lr & 3)) * BP + lg * KPL;
                Frag bf[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) bf[s] = M::load(brow + s * KSTEP);
#pragma unroll
                for (int t = 0; t < NRT; ++t) {
                    f32x4 d = {};
#pragma unroll
                    for (int s = 0; s < NS; ++s) d = M::mma(bf[s], own[t][s], d);
#pragma unroll
                    for (int j = 0; j < 4; ++j) cb[t][n][4 * hh + j] = d[j];
                }
            }
        ordered_lds_barrier();                                       // (x of the next head lies where the B rows did)
    }

    // ---- the heads ----
#pragma unroll 1
    for (int hi = 0; hi < nh; ++hi) {
        const int h = h0 + hi, cur = hi & 1;
        const bool more = hi + 1 < nh;
        const T *xs = reinterpret_cast<const T *>(body + cur * W::XS_B);
        asm volatile("" : "+v"(tid));
        const int lr = tid & 15, lg = (tid >> 4) & 3;
        // what this lane reads of step 0 (KSTEP columns on for the next one): the columns' entries, the sums at the edges of their block
        // of 16, and the image of x
        const int kl = KPL * lg, kb = kl & ~15;
        const float *tf = &tables[cur][0][kl], *tb = &tables[cur][1][kl];
        const double *edge_f = &sums[cur][0][kb + 15], *edge_b = &sums[cur][1][kb];
        const char *xl[2] = {};
        if constexpr (sizeof(T) == 2) {
            // (rows kl + lr / 4 of the image, columns 32 (j / 2) + 4 (j % 2) + 8 (lr % 4) for tile j; the four rows below and the other half of the
            // columns flip bit 2 of the 16-byte unit, see tile64_swz())
            xl[0] = reinterpret_cast<const char *>(xs) + (kl + (lr >> 2)) * 128 + ((((lr & 3) ^ (lr >> 2)) + ((lg & 1) << 2)) << 4);
            xl[1] = reinterpret_cast<const char *>(xs) + (kl + (lr >> 2)) * 128 + ((((lr & 3) ^ (lr >> 2)) + ((~lg & 1) << 2)) << 4);
        }
        if (more) form_sums(cur ^ 1);
        static_for<0, NRT>([&](auto RT) __attribute__((always_inline)) {
            constexpr int rt = decltype(RT)::value;
            const int r0 = (rt * W::WAVES + wave) * 16, orow = r0 + lr;
            Vec16<T> o[2] = {};
            if (r0 < L) {
                const int row = min(r0 + lr, L - 1);
                if constexpr (Z) request_z(h, row);           // (used behind the products, which cover it)
                const double rf = sums[cur][0][row], rb = sums[cur][1][row];
                f32x4 acc[SHARE][NJ] = {};                    // (the sums of scan_once_kernel's waves that share a row tile)
                // 64 columns, from 64 q on: all in front of the rows of this round, all behind them, or in front of some and behind others
                auto columns = [&](auto GROUP, auto STEPS) __attribute__((always_inline)) {
                    constexpr int q = decltype(GROUP)::value, k0 = 64 * q, NU = decltype(STEPS)::value;
                    constexpr bool FRONT = k0 + 64 <= rt * 16 * W::WAVES, BEHIND = k0 >= (rt + 1) * 16 * W::WAVES;
                    Frag a[NU];
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        const int ku = k0 + u * KSTEP;
                        const bool below = FRONT || (!BEHIND && kb < r0 - ku);
                        const float ef = __expf((float)((below ? rf : rb) - (below ? edge_f : edge_b)[ku]));
                        const float *gt = (below ? tf : tb) + ku;
                        float w[KPL];
#pragma unroll
                        for (int e = 0; e < KPL; e += 4) {
                            const f32x4 t = *reinterpret_cast<const f32x4 *>(gt + e);
#pragma unroll
                            for (int j = 0; j < 4; ++j) w[e + j] = cb[rt][q * SHARE + u][e + j] * ef * t[j];
                        }
                        a[u] = M::pack(w);
                    }
                    if constexpr (!FRONT && !BEHIND) {
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const int at = r0 - (k0 + u * KSTEP);        // the diagonal's first column within the step
                            if (at >= 0 && at < KSTEP) {
                                const float lrf = tables[cur][2][row], lrb = tables[cur][3][row];
                                if (kb == at) {
                                    const float *ll = tf + 2 * LP + k0 + u * KSTEP;
                                    const int diag = lr + at - kl;       // ... and this row's within the lane's
                                    float w[KPL];
#pragma unroll
                                    for (int e = 0; e < KPL; e += 4) {
                                        const f32x4 lf = *reinterpret_cast<const f32x4 *>(ll + e), lb = *reinterpret_cast<const f32x4 *>(ll + LP + e);
                                        const f32x4 dts = *reinterpret_cast<const f32x4 *>(ll + 2 * LP + e);
#pragma unroll
                                        for (int j = 0; j < 4; ++j) {
                                            const float x = e + j < diag ? lrf - lf[j] : lrb - lb[j];
                                            w[e + j] = cb[rt][q * SHARE + u][e + j] * (e + j == diag ? 2.f : __expf(x)) * dts[j];
                                        }
                                    }
                                    a[u] = M::pack(w);
                                }
                            }
                        }
                    }
#pragma unroll
                    for (int u = 0; u < NU; ++u)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const int ku = k0 + u * KSTEP;
                            Frag xf;
                            if constexpr (sizeof(T) == 2) {
                                typedef __attribute__((address_space(3))) i16x4 *lds_i16x4_ptr;
                                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(xl[j >> 1] + ku * 128 + 8 * (j & 1)));
                                const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(xl[~j >> 1 & 1] + ku * 128 + 512 + 8 * (j & 1)));
                                xf = __builtin_bit_cast(Frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                            } else {
#pragma unroll
                                for (int e = 0; e < KPL; ++e) xf[e] = xs[(kl + ku + e) * XP + j * 16 + lr];
                            }
                            acc[u][j] = M::mma(xf, a[u], acc[u][j]);
                        }
                };
                // (there are more than LP / 2 positions: of four groups the last may be behind the end, or half of it)
                static_for<0, LP == 256 ? 3 : LP / 64>([&](auto GROUP) __attribute__((always_inline)) { columns(GROUP, std::integral_constant<int, SHARE>()); });
                if constexpr (LP == 256) {
                    if (L > 224) columns(std::integral_constant<int, 3>(), std::integral_constant<int, SHARE>());
                    else if (L > 192) columns(std::integral_constant<int, 3>(), std::integral_constant<int, SHARE / 2>());
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int col = column(k);
                    float y[VS];
#pragma unroll
                    for (int e = 0; e < VS; ++e) {
                        const int j = sizeof(T) == 2 ? 2 * k + (e >> 2) : k;
                        y[e] = acc[0][j][e & 3];
#pragma unroll
                        for (int u = 1; u < SHARE; ++u) y[e] += acc[u][j][e & 3];
                    }
                    if (has_D) {
                        const Vec16<T> xv = *reinterpret_cast<const Vec16<T> *>(xs + orow * XP + (sizeof(T) == 2 ? ((col >> 3) ^ tile64_swz(orow)) << 3 : col));
#pragma unroll
                        for (int e = 0; e < VS; ++e) y[e] = __builtin_fmaf(ds[cur][col + e], to_f(xv.v[e]), y[e]);
                    }
                    if constexpr (Z) {
                        const Vec16<T> zv = __builtin_bit_cast(Vec16<T>, zraw[k]);
#pragma unroll
                        for (int e = 0; e < VS; ++e) y[e] *= silu_f(to_f(zv.v[e]));
                    }
#pragma unroll
                    for (int e = 0; e < VS; ++e) {
                        asm("" : "+v"(y[e]));                 // (rounded to 32 bits first: not one instruction with the conversion)
                        o[k].v[e] = from_f<T>(y[e]);
                    }
                }
            }
            // (in front of the stores: a wait for x behind them would be for them as well)
            if (rt == 0 && more) store_x(cur ^ 1);
            T *out = reinterpret_cast<T *>(p.out) + ((int64_t)b * L * H + h) * P + p0 + (unsigned)(orow * (H * P));
#pragma unroll
            for (int k = 0; k < 2; ++k)
                if (orow < L && p0 + column(k) < P) *reinterpret_cast<Vec16<T> *>(out + column(k)) = o[k];
            if (more) {
                if (rt == 0) {
                    ordered_lds_barrier();
                    form_tables(cur ^ 1);
                    if (hi + 2 < nh) request(h + 2);
                }
                if (rt == NRT - 1) ordered_lds_barrier();
            }
        });
    }
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
    // Up to so many workgroups (of scan_once_kernel) of one row.  The lines do not follow the number of rows, so that a row's result is the same alone and
    // in any batch.  Time of the launches replaced over that of the one launch, at 1, 16, 64 and 256 rows (heads of 64 without remark):
    //   bfloat16, dstate 64: 16 workgroups (256 positions, 4 heads, z) 2.3, 1.84, 1.22, 1.05; 48 (256, 12 heads, z) 2.3, 1.39, 1.08, 0.95; 48 (197, 12 heads, no z) 2.2, 1.47,
    //     1.06, 0.88; 18 (160, 6 heads, z) 2.1, 1.52, 1.19, 0.88; 48 (64, 48 heads, z) 2.6, 2.3, 2.0, 2.0; 48 (128, 24 heads, z) 2.1, 1.74, 1.31, 1.19
    //   dstate 128: 32 (256, 8 heads) 2.7, 1.53, 1.19, 0.97; 32 (16, 32 heads) 3.0, 2.8, 2.9, 3.6.  dstate 32: 48 (256, 12 heads) 2.8, 2.6, 2.5, 2.9
    //   float32, dstate 64: 48 (192, 4 heads, z) 2.2, 1.13, 1.51, 1.87; 24 (64, 6 heads, z) 1.77, 1.67, 1.40, 1.37.  Heads of 32, dstate 32: 80 (256, 10 heads, z) 2.5, 1.35,
    //     1.48, 2.1; dstate 16: 128 (256, 16 heads) 2.6, 1.54, 1.60, 1.74; 48 (64, 24 heads) 2.0, 1.88, 1.64, 1.66
    // Below 1 are 16 bits over more than 128 positions at dstate 64 from some 200 rows on, where the chunked launches move two entries an instruction: the price of
    // the same bits in any batch.  Final states besides (the launches that form them stay, and the one launch takes the place of their scan only): bfloat16, 197
    // positions, 12 heads 1.36, 1.12, 1.00, 0.97; float32 in one chunk, 64 positions, 6 heads 1.15, 1.16, 1.20, 1.38, in several chunks, where the
    // chunked scan takes a quarter of the pairs, 256 positions, 4 heads of 32, dstate 16 1.07, 0.86, 0.92, 0.95, and 192 positions, 4 heads, dstate 64 0.99, 0.75, 0.89, 1.04: the
    // price of a result that is the same in bits whether or not they are asked for.
    const int per_row = p->nheads * once_tiles(p);
    if (e == 2) return per_row <= (ns == 4 ? 32 : 48);
    return p->seqlen <= 64 ? per_row <= (ns == 4 ? 24 : ns == 2 ? 32 : 48) : per_row <= (ns == 4 ? 48 : ns == 2 ? 80 : 128);
}

// Which of the two kernels: the walk wherever its chain of waits is not the longer one, by all rows' workgroups of the other.  us, scan_once_kernel / walk:
//   up to 128 positions always the walk: one row of 64 positions, 48 heads, bfloat16 6.7 / 5.1, 16 rows 14.4 / 8.8; 128 positions, 24 heads 6.7 / 6.5, 14.6 / 10.7;
//     float32, 64 positions, 24 heads of 32 5.5 / 5.1, 11.1 / 6.8
//   16 bits (256 positions, 12 heads, dstate 64): 192 workgroups 8.7 / 11.7, 384 12.4 / 12.6, 576 16.4 / 13.2; 6 heads over 160 positions: 216 8.4 / 9.7, 288 11.3 / 9.9;
//     dstate 128, 8 heads: 256 10.2 / 13.3, 384 17.1 / 14.0
//   float32, 256 positions: dstate 16, 16 heads: 1024 18.3 / 19.7, 1536 24.2 / 20.7; dstate 32, 10 heads: 640 22.1 / 23.6, 960 28.6 / 24.4; dstate 64, 3 heads: 768 26 / 32, 1152 40 / 32
static bool once_walks(const bimamba2_params *p) {
    if (p->seqlen <= 128) return true;
    const int line = p->dtype != BIMAMBA2_F32 ? 256 : p->dstate <= 16 ? 1024 : 768;
    return (int64_t)p->batch * p->nheads * once_tiles(p) > line;
}
// Heads that a workgroup walks through: rounds of workgroups (in half a round or less those that share a CU do not wait for each other) times their heads
// and the start, C.B^T and the first head's operands, in heads' worth.  256 positions, 12 heads, dstate 64, 64 rows: 1, 2, 3, 6 heads 41, 41, 31, 47 us; 256 rows 146,
// 125, 115, 107, all twelve 101.
static int walk_heads(const bimamba2_params *p, int npt) {
    const int hpg = p->nheads / p->ngroups, places = p->seqlen > 128 ? 256 : p->seqlen > 64 ? 512 : 1280;
    int best = 1;
    double best_cost = 1e30;
    for (int hpw = 1; hpw <= hpg; ++hpw) {
        const int64_t wgs = (int64_t)p->batch * p->ngroups * ((hpg + hpw - 1) / hpw) * npt, rest = wgs % places;
        const double rounds = (double)(wgs / places) + (!rest ? 0. : places > 256 && 2 * rest <= places ? 0.7 : 1.);
        const double cost = rounds * ((places > 256 ? 0.3 : 0.5) + hpw);
        if (cost < best_cost) { best_cost = cost; best = hpw; }
    }
    return best;
}

template <typename T, int NS, int LP> static void launch_walk(const bimamba2_params *p, int grid, int npt, int hpw, int first_row) {
    const dim3 block(WalkMap<T, NS, LP>::THREADS);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
    if (p->has_z) hipLaunchKernelGGL((scan_once_walk_kernel<T, NS, LP, true>), dim3(grid), block, 0, s, *p, npt, hpw, first_row);
    else hipLaunchKernelGGL((scan_once_walk_kernel<T, NS, LP, false>), dim3(grid), block, 0, s, *p, npt, hpw, first_row);
}
template <typename T, int NS> static int launch_once_t(const bimamba2_params *p) {
    const int nrt = once_row_tiles(p), npt = once_tiles(p) / nrt;
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
    if (!once_walks(p)) {
        hipLaunchKernelGGL((scan_once_kernel<T, NS>), dim3(p->batch * p->nheads * nrt * npt), dim3(ONCE_THREADS), 0, s, *p, nrt, npt);
        return check_launch();
    }
    const int hpw = walk_heads(p, npt), hpg = p->nheads / p->ngroups, per_row = p->ngroups * ((hpg + hpw - 1) / hpw) * npt;
    const int rows = WALK_GRID / per_row;                      // (the threads of a launch are counted in 32 bits)
    for (int b = 0; b < p->batch; b += rows) {
        const int grid = std::min(rows, p->batch - b) * per_row;
        if (p->seqlen <= 64) launch_walk<T, NS, 64>(p, grid, npt, hpw, b);
        else if (p->seqlen <= 128) launch_walk<T, NS, 128>(p, grid, npt, hpw, b);
        else launch_walk<T, NS, 256>(p, grid, npt, hpw, b);
        if (int rc = check_launch()) return rc;
    }
    return BIMAMBA2_OK;
}

template <typename T> static int launch_once_n(const bimamba2_params *p) {
    switch (p->dstate / Mma<T>::KSTEP) {
        case 1: return launch_once_t<T, 1>(p);
        case 2: return launch_once_t<T, 2>(p);
        case 4: return launch_once_t<T, 4>(p);
        default: return BIMAMBA2_EUNSUPPORTED;
    }
}

bool scan_once_walks(const bimamba2_params *p) { return once_walks(p); }

int launch_scan_once(const bimamba2_params *p) {
    return p->dtype == BIMAMBA2_F32 ? launch_once_n<float>(p) : p->dtype == BIMAMBA2_BF16 ? launch_once_n<bf16_t>(p) : launch_once_n<f16_t>(p);
}

}  // namespace bm2
