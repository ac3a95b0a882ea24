// The work of one workgroup of the dB / dC kernels for float32 state tensors, any shape.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace bm2 {

// =========================================================================================================
// state part of dC (IS_DB = false), rows r = positions t of a 64-row tile, summed over the heads of a group:
//   tmp_f = dy_h[r,:] . prev_f[h]  (K = headdim),  dCs[r,n] += e^{cs_f[r]} tmp_f + e^{cs_b[r]} tmp_b
//   u_f[h,r] = e^{cs_f[r]} sum_n tmp_f[r,n] C[r,n]      (same for b)
// state part of dB (IS_DB = true), rows r = positions s:
//   tmp_f = x_h[r,:] . dS_f[h],  dBs[r,n] += dt[r] (e^{cs_f[Q-1]-cs_f[r]} tmp_f + e^{cs_b[0]-cs_b[r]} tmp_b)
//   v_f[h,r] = dt[r] e^{cs_f[Q-1]-cs_f[r]} sum_n tmp_f[r,n] B[r,n]
// =========================================================================================================
constexpr int DBDC_HEADS = 8;         // heads per slice at most (measured against 4 with 256-row tiles: dB / dC / tail 0.323 -> 0.316 ms per step)
constexpr int DBDC_SLICES_MAX = 8;    // what bmm_chunk_bwd adds up in its fast variant
constexpr int DBDC_WAVES = 8, DBDC_THREADS = 64 * DBDC_WAVES;

// The A operand (x or dout rows, K = headdim contiguous) is read from global memory straight into MFMA operand
// registers; the states, stored [p][n], are staged transposed ([n][p], 64 x 64 at a time) in LDS, double-buffered for
// 16-bit types so that one barrier per step suffices.
// 8 waves; wave w owns QT 16-row tiles: the workgroup covers 128*QT rows, so that with QT = 2 a 256-row chunk reads
// each state once.  Global memory latency is hidden by software pipelining over "steps" (head, dstate tile, headdim
// chunk): the state blocks and A fragments of step s+1 are requested into registers before step s is multiplied, and
// only then written to the LDS image.
// UNI: the forward direction's state only (single-direction comparator).
template <typename T, int QT> struct DbdcMap {
    static constexpr int KC = 64, VK = 16 / (int)sizeof(T), LDX = KC + VK, NBUF = sizeof(T) == 2 ? 2 : 1, ROWS = DBDC_WAVES * 16 * QT;
    static constexpr int IMAGE = 64 * LDX * (int)sizeof(T);
    static constexpr int SB = NBUF * IMAGE, SFS = 2 * NBUF * IMAGE, SBS = SFS + 4 * DBDC_HEADS * ROWS, LDS = SBS + 4 * DBDC_HEADS * ROWS;
};
// lds: DbdcMap::LDS bytes, 16-byte aligned; bid: (batch, chunk, group), row tile, head slice
// NT: 64-column tiles of the state dimension, NJ: 16-column tiles in use of each (below 4 with NT = 1 only): a narrow state does not
// hold registers for 64 columns, and two workgroups fit a CU, which cover each other's waits (one step of one head is a chain of
// 2 to 3 us: requests, LDS image, barrier, products, sums).  4 x 2048, bfloat16, 16 heads of 16, dstate 16: 17 -> 11 us each.
template <typename T, int NT, int QT, bool IS_DB, bool FAST, bool UNI = false, int NJ = 4>
__device__ __forceinline__ void bwd_dbdc_body(const bimamba2_params &p, int nc, int hps, BlockId bid, char *lds) {
    typedef Mma<T> M;
    typedef DbdcMap<T, QT> Map;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP, KC = Map::KC, NKS = KC / KSTEP;
    constexpr int VK = Map::VK;                                            // image rows (k) per staged block; 4 columns (n)
    constexpr int LDX = Map::LDX, NBUF = Map::NBUF, ROWS = Map::ROWS;
    constexpr int NBLK = (KC / VK) * (64 / 4);                             // staged blocks per 64 x 64 state tile
    static_assert(2 * NBLK <= DBDC_THREADS, "one staged block per thread");
    T (*sF)[64 * LDX] = reinterpret_cast<T (*)[64 * LDX]>(lds), (*sB)[64 * LDX] = reinterpret_cast<T (*)[64 * LDX]>(lds + Map::SB);
    float (*sfs)[ROWS] = reinterpret_cast<float (*)[ROWS]>(lds + Map::SFS), (*sbs)[ROWS] = reinterpret_cast<float (*)[ROWS]>(lds + Map::SBS);   // row scales of the heads of this slice
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    // bid.x = (b, c, g) varies fastest: consecutive workgroups are dealt round-robin to the 8 XCDs, so the row
    // tiles of one (b, c, g), which read the same states, land on the same XCD and share its L2
    const int rt = bid.y;
    const int g = bid.x % p.ngroups, bc = bid.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, N = p.dstate, P = p.headdim, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int r0 = rt * ROWS;
    // bid.z selects a slice of hps (at most DBDC_HEADS) heads of the group; its partial sum goes to slice bid.z of
    // the output, and bmm_chunk_bwd adds the slices up
    const int hh0 = bid.z * hps, hh_end = min(hpg, hh0 + hps);
    const int nkc = (P + KC - 1) / KC, nnt = (N + 63) / 64;
    const int per_head = nnt * nkc, nsteps = (hh_end - hh0) * per_head;

    // ---- software pipeline, stage 1: requests for a step (state blocks of two tiles, A fragments) ----
    Vec16<float> sreg[VK];                                                 // one VK x 4 block of a state tile
    typename M::Frag af[QT][NKS];
    int arow[QT];                                                          // this lane's A-operand rows
#pragma unroll
    for (int q = 0; q < QT; ++q) arow[q] = min(r0 + (wave * QT + q) * 16 + lr, limit - 1);
    const int sblk = threadIdx.x % NBLK, stile = threadIdx.x / NBLK;       // stile 0: forward state, 1: reverse state
    const int s_rb = sblk % 16, s_kb = sblk / 16;
    // without FAST: whole vectors of the states (columns) and of the x / dout rows, or element by element
    const bool whole_s = !FAST && N % 4 == 0 && aligned16(IS_DB ? p.dstates_f : p.states_f, 0) && aligned16(IS_DB ? p.dstates_b : p.states_b, 0);
    const bool whole_a = !FAST && P % KPL == 0 &&
                         (IS_DB ? aligned16(reinterpret_cast<const T *>(p.x), p.x_sb | p.x_sl | p.x_sh)
                                : p.has_z ? aligned16(reinterpret_cast<const T *>(p.dout_x), P) : aligned16(reinterpret_cast<const T *>(p.dout), p.dout_sb | p.dout_sl | p.dout_sh));
    int s_kc = 0, s_nt = 0;                                                // the step whose state block sreg holds
    auto request = [&](int step) __attribute__((always_inline)) {
        const int hh = hh0 + step / per_head, rem = step % per_head, nt = rem / nkc, kc = rem % nkc;
        s_kc = kc;
        s_nt = nt;
        const int h = g * hpg + hh;
        if (stile < (UNI ? 1 : 2)) {
            const int64_t so = ((int64_t)(b * nc + c) * H + h) * P * N;
            const float *st = (IS_DB ? (stile ? p.dstates_b : p.dstates_f) : (stile ? p.states_b : p.states_f)) + so;
#pragma unroll
            for (int kk = 0; kk < VK; ++kk) {
                const int pp = kc * KC + s_kb * VK + kk, n = nt * 64 + s_rb * 4;
                if (FAST) sreg[kk] = *reinterpret_cast<const Vec16<float> *>(st + (int64_t)pp * N + n);
                else if (whole_s) {                        // unconditional, from clamped addresses; zeroed in commit()
                    sreg[kk] = *reinterpret_cast<const Vec16<float> *>(st + (int64_t)min(pp, P - 1) * N + min(n, N - 4));
                } else
#pragma unroll
                    for (int i = 0; i < 4; ++i) sreg[kk].v[i] = (pp < P && n + i < N) ? st[(int64_t)pp * N + n + i] : 0.f;
            }
        }
        const T *ap;
        int64_t as;
        if (IS_DB) { as = p.x_sl; ap = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * as + h * p.x_sh; }
        else if (p.has_z) { as = (int64_t)H * P; ap = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * as + (int64_t)h * P; }
        else { as = p.dout_sl; ap = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * as + h * p.dout_sh; }
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int kb = kc * KC + ks * KSTEP + lg * KPL;
                const T *row = ap + (int64_t)arow[q] * as;
                if (FAST) af[q][ks] = M::load(row + kb);
                else if (whole_a) {
                    af[q][ks] = M::load(row + min(kb, P - KPL));
                    if (kb >= P) af[q][ks] = typename M::Frag{};
                } else {
                    float v[KPL];
#pragma unroll
                    for (int i = 0; i < KPL; ++i) v[i] = kb + i < P ? to_f(row[kb + i]) : 0.f;
                    af[q][ks] = M::pack(v);
                }
            }
    };
    // stage 2: the requested state block goes, transposed, into the LDS image (r = n, k = p)
    auto commit = [&](int buf) __attribute__((always_inline)) {
        if (stile < (UNI ? 1 : 2)) {
            T *dst = stile ? sB[buf] : sF[buf];
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                Vec16<T> o;
#pragma unroll
                for (int kk = 0; kk < VK; ++kk) {
                    const bool in = FAST || (s_kc * KC + s_kb * VK + kk < P && s_nt * 64 + s_rb * 4 + rr < N);
                    o.v[kk] = from_f<T>(in ? sreg[kk].v[rr] : 0.f);
                }
                *reinterpret_cast<Vec16<T> *>(dst + xt_index<T, LDX>(s_rb * 4 + rr, s_kb * VK)) = o;
            }
        }
    };
    request(0);

    int tl[QT][4];                                                         // rows of this lane's accumulator elements
#pragma unroll
    for (int q = 0; q < QT; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) tl[q][i] = (wave * QT + q) * 16 + lg * 4 + i;
    // row scales of every head of the slice
    for (int idx = threadIdx.x; idx < (hh_end - hh0) * ROWS; idx += DBDC_THREADS) {
        const int hh = idx / ROWS, rl = idx % ROWS, r = r0 + rl;
        const int64_t o = (((int64_t)b * H + g * hpg + hh0 + hh) * nc + c) * Q;
        float f = 0.f, rv = 0.f;
        if (r < limit) {
            if (IS_DB) {
                const float d = p.dt_out[o + r];
                f = d * __expf(p.cs_f[o + Q - 1] - p.cs_f[o + r]);
                rv = UNI ? 0.f : d * __expf(p.cs_b[o] - p.cs_b[o + r]);
            } else {
                f = __expf(p.cs_f[o + r]);
                rv = UNI ? 0.f : __expf(p.cs_b[o + r]);
            }
        }
        sfs[hh][rl] = f;
        sbs[hh][rl] = rv;
    }
    // B or C values of this lane's output elements
    const T *cbp;
    int64_t cbs;
    if (IS_DB) { cbs = p.B_sl; cbp = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + r0) * cbs + g * p.B_sg; }
    else { cbs = p.C_sl; cbp = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + r0) * cbs + g * p.C_sg; }
    float creg[NT][QT][NJ][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // unconditional loads from clamped addresses (conditional ones are waited for one by one), masked after
                    const int n = nt * 64 + j * 16 + lr;
                    const float v = to_f(cbp[(int64_t)min(tl[q][i], limit - 1 - r0) * cbs + min(n, N - 1)]);
                    creg[nt][q][j][i] = (r0 + tl[q][i] < limit && n < N) ? v : 0.f;
                }
    f32x4 tot[NT][QT][NJ] = {};

    int step = 0;
    for (int hh = hh0; hh < hh_end; ++hh) {
        const int h = g * hpg + hh;
        const int64_t o = (((int64_t)b * H + h) * nc + c) * Q;
        float uf[QT][4], ub[QT][4];
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) { uf[q][i] = 0.f; ub[q][i] = 0.f; }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if (nt >= nnt) break;
            f32x4 tf[QT][NJ] = {}, tb[QT][NJ] = {};
            for (int kc = 0; kc < nkc; ++kc, ++step) {
                const int buf = NBUF == 2 ? (step & 1) : 0;
                if (NBUF == 1) __syncthreads();            // the single image is still being read by slower waves
                commit(buf);
                typename M::Frag afc[QT][NKS];
#pragma unroll
                for (int q = 0; q < QT; ++q)
#pragma unroll
                    for (int ks = 0; ks < NKS; ++ks) afc[q][ks] = af[q][ks];
                __syncthreads();
                if (step + 1 < nsteps) request(step + 1);  // in flight while this step is multiplied
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    if (!FAST && kc * KC + ks * KSTEP >= P) continue;      // (uniform) nothing there: narrow heads and states
                    const int kq = ks * KSTEP + lg * KPL;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        if (!FAST && nt * 64 + j * 16 >= N) continue;
                        const typename M::Frag bff = M::load(sF[buf] + xt_index<T, LDX>(j * 16 + lr, kq));
                        const typename M::Frag bfb = UNI ? bff : M::load(sB[buf] + xt_index<T, LDX>(j * 16 + lr, kq));
#pragma unroll
                        for (int q = 0; q < QT; ++q) {
                            tf[q][j] = M::mma(afc[q][ks], bff, tf[q][j]);
                            if (!UNI) tb[q][j] = M::mma(afc[q][ks], bfb, tb[q][j]);
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float sf = sfs[hh - hh0][tl[q][i]], sb = sbs[hh - hh0][tl[q][i]];
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        uf[q][i] += tf[q][j][i] * creg[nt][q][j][i];
                        ub[q][i] += tb[q][j][i] * creg[nt][q][j][i];
                        tot[nt][q][j][i] += sf * tf[q][j][i] + sb * tb[q][j][i];
                    }
                }
        }
        float *of = IS_DB ? p.v_f : p.u_f, *ob = IS_DB ? p.v_b : p.u_b;
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = row16_sum(uf[q][i]) * sfs[hh - hh0][tl[q][i]], bb = row16_sum(ub[q][i]) * sbs[hh - hh0][tl[q][i]];
                if (lr == 0 && r0 + tl[q][i] < Q) {
                    of[o + r0 + tl[q][i]] = a;
                    if (!UNI) ob[o + r0 + tl[q][i]] = bb;
                }
            }
    }
    float *out = (IS_DB ? p.dBs : p.dCs) + (int64_t)bid.z * p.batch * p.seqlen * p.ngroups * N;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = nt * 64 + j * 16 + lr, r = r0 + tl[q][i];
                    if (r < limit && n < N)
                        out[(((int64_t)b * p.seqlen + (int64_t)c * Q + r) * p.ngroups + g) * N + n] = tot[nt][q][j][i];
                }
}

}  // namespace bm2
