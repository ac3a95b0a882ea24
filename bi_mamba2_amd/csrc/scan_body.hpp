// The work of one workgroup of the chunk-scan kernel (forward output) and its mirror (dx in the backward pass) for gfx950.
//
// One workgroup (8 waves) owns one (batch, chunk, head) and a tile of up to 64 headdim columns; wave w owns the
// rows [w*16*QT, (w+1)*16*QT) of the chunk.  The K operand of the big product (x * dt, resp. dy) is staged ONCE,
// transposed, into LDS; the A operand (CB times the decay factors) is built directly in registers in the MFMA
// operand layout from float32 CB rows, so the main loop has no barrier and no LDS round trip for A.
//
//   forward (BWD = false), rows r = output positions t, k = source positions s:
//     acc[r,p] = e^{cs_f[r]} C_r.prev_f[p,:] + e^{cs_b[r]} C_r.prev_b[p,:]
//              + sum_k CB[r,k] m(r,k) dt[k] x[k,p],    m = e^{cs_f[r]-cs_f[k]} (k<r), e^{cs_b[r]-cs_b[k]} (k>r), 2 (k=r)
//     out_x = acc + D x[r,p];  out = out_x * silu(z)
//   mirror (BWD = true), rows r = input positions s, k = output positions t, CBT[r,k] = CB[k,r]:
//     acc[r,p] = e^{cs_f[Q-1]-cs_f[r]} B_r.dS_f[p,:] + e^{cs_b[0]-cs_b[r]} B_r.dS_b[p,:]
//              + sum_k CBT[r,k] m'(r,k) dy[k,p],       m' = e^{cs_f[k]-cs_f[r]} (k>r), e^{cs_b[k]-cs_b[r]} (k<r), 2 (k=r)
//     dx = acc dt[r] + D dy[r,p];  ddt_direct[r] = sum_p acc x[r,p];  dD partial = sum_r dy x
#pragma once
#include <type_traits>

#include "common.hpp"

namespace bm2 {

constexpr int SCAN_WAVES = 8, SCAN_THREADS = 64 * SCAN_WAVES;

// FAST = true is chosen by the launcher when chunk_size % 32 == 0, headdim is a multiple of the column tile,
// dstate a multiple of the elements in 16 bytes and every operand is 16-byte aligned with strides that keep rows aligned: all guarded scalar
// fallbacks compile away and loads become unconditional (rows past the end of the sequence are read from a valid
// row and never stored).
//
// NF > 0 (16-bit types, FAST, dstate = 32 * NF): CB is not read at all.  The 16 x 32 piece of CB (resp. CB^T) a wave needs
// for a K step is recomputed with MFMAs from the C and B rows, arranged so that the product comes out in the A operand
// layout: D[m][n] = sum_d Krow[k(m)][d] * Ownrow[n][d] with k(m) = k0 + 8*(m/4) + m%4 (+4 for the second product) leaves
// lane (l%16 = row, l/16 = g) with columns k0 + 8g + 0..3 (resp. +4..7) of its row.  All waves of a workgroup read the
// same 32 K rows per step, so they come from L1, where the CB rows were 256 KB of L2 traffic per workgroup.  The state
// products use the raw rows as well and scale the accumulator instead of the operand.
// UNI (with NF > 0 only): the single-direction (causal) operator - the reverse direction's state product, the K steps on
// the far side of the diagonal and the far half of the diagonal step are left out.
template <typename T, int QT, int NJ, bool BWD, int NF> struct ScanMap {
    static constexpr int QP = SCAN_WAVES * 16 * QT, PW = 16 * NJ, LDX = QP + 16 / (int)sizeof(T), LDS_ = Mma<T>::LD - BK + 64;
    static constexpr int XT_BYTES = PW * LDX * (int)sizeof(T), ST_BYTES = 2 * PW * LDS_ * (int)sizeof(T), STG_BYTES = SCAN_WAVES * 16 * (PW + 4) * 4;
    // the operand images (xT and the two state tiles) and the per-wave epilogue staging patches are never live together
    static constexpr int LO = XT_BYTES + ST_BYTES > STG_BYTES ? XT_BYTES + ST_BYTES : STG_BYTES, UP = LO + 4 * QP, GLO = UP + 4 * QP, GUP = GLO + 4 * QP;
    static constexpr int DTL = GUP + 4 * QP, RED = DTL + 4 * (BWD ? 4 : QP), KRL = RED + (BWD ? 4 * SCAN_WAVES * PW : 0);
    static constexpr int KRING = 4;                // slots of the K-row image (NF > 0): requests run KRING - 1 steps ahead
    static constexpr int LDS = KRL + (NF > 0 ? KRING * 32 * 64 * (int)sizeof(T) : 0);
};
// (the pieces of LDS are arguments that do not alias: through one pointer the compiler ordered the reads of one behind the writes
// of another, 70 -> 76 us for the float32 kernel over 4 x 2048, 16 heads of 64, dstate 64)
// STATES = false: a sequence of one chunk without states of its own: the states entering it are zero and have no tensors.  (A kernel of its own: asked at
// run time the question keeps the state tiles' loads behind it, 28.0 -> 28.4 us over 8 x 339, 36 heads of 64, dstate 16, in bfloat16.)
template <typename T, int QT, int NJ, bool BWD, bool FAST, int NF, bool UNI, bool STATES>
__device__ __forceinline__ void chunk_scan_work(const bimamba2_params &p, int nc, int npt, unsigned id, char *__restrict__ shared_u,
                                                float *__restrict__ lo, float *__restrict__ up,      // decay exponents, see below
                                                float *__restrict__ glo, float *__restrict__ gup,    // their column factors relative to the edge of the 16-block
                                                float *__restrict__ dtl,                             // forward: dt of the columns, for the step across the diagonal
                                                float (*__restrict__ red)[16 * NJ], T *__restrict__ krl) {
    typedef ScanMap<T, QT, NJ, BWD, NF> Map;
    typedef Mma<T> M;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP;
    constexpr int VS = 16 / (int)sizeof(T);
    constexpr int QP = SCAN_WAVES * 16 * QT;      // rows the workgroup covers (>= chunk_size); QT row tiles per wave
    constexpr int PW = 16 * NJ;                   // headdim columns the workgroup covers
    constexpr int LDX = QP + VS;
    constexpr int NW = 64;                        // dstate columns of the state tiles held in LDS at a time
    constexpr int LDS_ = M::LD - BK + NW;         // their leading dimension
    constexpr int SLD = PW + 4;                   // float32 row of the epilogue staging patches
    constexpr int XT_BYTES = Map::XT_BYTES;
    T *xT = reinterpret_cast<T *>(shared_u);
    T *sF = reinterpret_cast<T *>(shared_u + XT_BYTES), *sB = sF + PW * LDS_;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    // linear block id -> (pt, h, bc) with bc fastest: all heads of one (batch, chunk) share CB and C, and
    // consecutive ids are dealt round-robin to the 8 XCDs, so equal bc % 8 keeps them on one XCD's L2
    const int nbc = p.batch * nc;
    const int bc = id % nbc, hp = id / nbc, pt = hp % npt, h = hp / npt;
    const int c = bc % nc, b = bc / nc;
    const int g = h / (p.nheads / p.ngroups);
    const int Q = p.chunk_size, N = p.dstate, P = p.headdim, H = p.nheads;
    const int limit = min(Q, p.seqlen - c * Q);
    const int p0 = pt * PW;
    const int64_t o = (((int64_t)b * H + h) * nc + c) * Q;
    const float *csf = p.cs_f + o, *csb = p.cs_b + o, *dto = p.dt_out + o;
    const float d_head = (p.has_D && !p.D_has_hdim) ? p.D[h] : 0.f;   // read here: in the epilogue its latency would be exposed
    // NF > 0: the K rows of part 2 (forward: B rows, mirror: C rows) travel straight into a ring of LDS slots, KRING - 1
    // K steps (of 32 rows) ahead of their use: a global access takes microseconds when the memory system is busy.  Wave w brings rows 4w..4w+3 of the step: unit u = 32*w + lane (lane < 32) is row
    // u/8, chunk position u%8, which holds the row's 16-byte chunk (u%8) ^ (row % 8).
    constexpr int KRING = Map::KRING;
    const char *krbase = nullptr;                  // uniform: row 0 of the chunk in the K-row matrix
    unsigned krs_bytes = 0;                        // its row stride (the launcher checks that 256 rows fit 32 bits)
    if constexpr (NF > 0) {
        if (BWD) { krs_bytes = (unsigned)p.C_sl * sizeof(T); krbase = reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + (int64_t)c * Q * p.C_sl + g * p.C_sg); }
        else { krs_bytes = (unsigned)p.B_sl * sizeof(T); krbase = reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * p.B_sl + g * p.B_sg); }
    }
    if constexpr (NF > 0) {
        // keep the base in scalar registers (it is uniform, but that is not visible through the 64-bit arithmetic)
        const uint64_t kb64 = reinterpret_cast<uint64_t>(krbase);
        const uint32_t klo = __builtin_amdgcn_readfirstlane((uint32_t)kb64), khi = __builtin_amdgcn_readfirstlane((uint32_t)(kb64 >> 32));
        krbase = reinterpret_cast<const char *>(((uint64_t)khi << 32) | klo);
    }
    auto kr_issue = [&](int step) {
        if (lane < 32) {
            int ln = lane;
            asm volatile("" : "+v"(ln));           // recompute the few lane terms per call rather than keep them in registers
            const int rowl = wave * 4 + (ln >> 3);
            const unsigned off = (unsigned)min(step * 32 + rowl, limit - 1) * krs_bytes + (((ln & 7) ^ (rowl & 7)) * 16);
            load16_to_lds(krbase + off, krl + (step % KRING) * (32 * 64) + wave * 256);
        }
    };
    if constexpr (NF > 0) {
#pragma unroll
        for (int st = 0; st < KRING - 1; ++st)
            if (st * 32 < limit) kr_issue(st);
    }
    int rowi[QT];                                  // this lane's A-operand row in each row tile
#pragma unroll
    for (int rt = 0; rt < QT; ++rt) rowi[rt] = (wave * QT + rt) * 16 + lr;

    // A operand of part 1: C rows (forward) or B rows (mirror), straight from global memory in operand layout
    const T *ap;
    int64_t as;
    if (BWD) { as = p.B_sl; ap = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * as + g * p.B_sg; }
    else { as = p.C_sl; ap = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + (int64_t)c * Q * as + g * p.C_sg; }
    const bool avec = aligned16(ap, as) && (N % VS == 0);
    // rows of NW dstate columns, as they are (the row factors go onto the accumulators: a factor on a 16-bit operand would be
    // one more rounding of it), the first ones requested up front
    typename M::Frag own[QT][NW / KSTEP];
    auto load_arows = [&](int n0) {
#pragma unroll
        for (int rt = 0; rt < QT; ++rt)
#pragma unroll
            for (int s = 0; s < NW / KSTEP; ++s) {
                const int r = rowi[rt], kb = n0 + s * KSTEP + lg * KPL;
                if (NF > 0) own[rt][s] = M::load(ap + (int64_t)min(r, limit - 1) * as + kb);
                else if (FAST) {
                    // (zeros behind the state dimension by masking the 16 bytes: a select per element cost the kernel 20 of 55 us)
                    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
                    const u32x4 bits = *reinterpret_cast<const u32x4 *>(ap + (int64_t)min(r, limit - 1) * as + min(kb, N - KPL));
                    own[rt][s] = __builtin_bit_cast(typename M::Frag, bits & (kb < N ? ~0u : 0u));
                } else if (r < limit && avec && kb + KPL <= N) {
                    own[rt][s] = M::load(ap + (int64_t)r * as + kb);
                } else {
                    float v[KPL];
#pragma unroll
                    for (int i = 0; i < KPL; ++i) v[i] = (r < limit && kb + i < N) ? to_f(ap[(int64_t)r * as + kb + i]) : 0.f;
                    own[rt][s] = M::pack(v);
                }
            }
    };

    // forward: k<r uses lo[r]-lo[k] with lo = cs_f, k>r uses up[r]-up[k] with up = cs_b
    // mirror : k<r uses e^{cs_b[k]-cs_b[r]} -> lo = -cs_b;  k>r uses e^{cs_f[k]-cs_f[r]} -> up = -cs_f
    // Away from the diagonal the factor separates: with m = lo at the last position of k's block of 16 (which lies
    // between k and r), e^{lo[r]-lo[k]} = e^{lo[r]-m} * glo[k], glo[k] = e^{m-lo[k]}, both factors <= 1 for A <= 0;
    // likewise gup[k] = e^{up[first of k's block] - up[k]}.  One exponential per lane and K step instead of one per element.
    // (The sums stay as they are here and only their differences are scaled to base 2: scaled first, each would be rounded
    // once more at the size of the sum, which is most of what a float32 result is off by.)
    for (int q = threadIdx.x; q < QP; q += SCAN_THREADS) {
        const int qq = min(q, Q - 1), qe = min(q | 15, Q - 1), qs = min(q & ~15, Q - 1);
        const float f = csf[qq], r = csb[qq];
        const float l = BWD ? -r : f, u = BWD ? -f : r;
        lo[q] = l;
        up[q] = u;
        // forward: dt[k] of the source position rides on the column factors (and on the diagonal step through dtl), so
        // that the operand image holds x as it is and the D term can take x from there
        const float dtq = BWD ? 1.f : dto[qq];
        glo[q] = __expf((BWD ? -csb[qe] : csf[qe]) - l) * dtq;
        gup[q] = __expf((BWD ? -csf[qs] : csb[qs]) - u) * dtq;
        if (!BWD) dtl[q] = dtq;
    }
    // K operand of part 2, transposed into LDS
    const T *kp;
    int64_t ks;
    if (!BWD) { ks = p.x_sl; kp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * ks + h * p.x_sh; }
    else if (p.has_z) { ks = (int64_t)H * P; kp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * ks + (int64_t)h * P; }
    else { ks = p.dout_sl; kp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * ks + h * p.dout_sh; }
    stage_transposed<T, QP, PW, LDX, FAST>(xT, kp + p0, ks, limit, P - p0, [&](int k) { return k < limit ? 1.f : 0.f; });

    // (two row tiles of four column tiles have no registers to hold them over the loads of the state tiles)
    constexpr bool ROWS_FIRST = NF > 0 || QT * NJ <= 4;
    if (ROWS_FIRST) load_arows(0);
    f32x4 acc[QT][NJ] = {};

    // ---- part 1: states.  A = (C or B rows) * row scale, K = dstate; B operand = state tiles [p][n] in LDS ----
    if constexpr (!STATES) __syncthreads();
    else {
        const int64_t so = ((int64_t)(b * nc + c) * H + h) * P * N + (int64_t)p0 * N;
        const float *stf = (BWD ? p.dstates_f : p.states_f) + so, *stb = (BWD ? p.dstates_b : p.states_b) + so;
        // one direction's product of the rows with the state tile in LDS, scaled row by row (rows 4*(l/16)+i of each tile) on
        // its way to acc; one direction after the other, and without CB fragments to spare registers for also one row tile
        // after the other, to keep one small set of temporaries (both row tiles at once: 32 registers spilled)
        constexpr int RT = NF == 0 && QT * NJ > 4 ? 1 : QT;
        auto state_product = [&](int dir, int nleft) __attribute__((always_inline)) {
            const T *st = dir ? sB : sF;
            // forward: e^{cs_f[r]}, e^{cs_b[r]}; mirror: e^{cs_f[Q-1] - cs_f[r]}, e^{cs_b[0] - cs_b[r]} (lo, up: see above)
            const float ref = BWD ? (dir ? lo[0] : up[Q - 1]) : 0.f;
            const float *tab = BWD ? (dir ? lo : up) : (dir ? up : lo);
#pragma unroll
            for (int r0 = 0; r0 < QT; r0 += RT) {
                if (RT < QT) __builtin_amdgcn_sched_barrier(0);
                f32x4 tmp[RT][NJ] = {};
#pragma unroll
                for (int s = 0; s < NW / KSTEP; ++s) {
                    if (NF == 0 && s * KSTEP >= nleft) break;
                    typename M::Frag bfs[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; ++j) bfs[j] = M::load(st + (j * 16 + lr) * LDS_ + s * KSTEP + lg * KPL);
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) tmp[rt][j] = M::mma(own[r0 + rt][s], bfs[j], tmp[rt][j]);
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const f32x4 cs4 = *reinterpret_cast<const f32x4 *>(tab + (wave * QT + r0 + rt) * 16 + lg * 4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = __expf(cs4[i] - ref);
#pragma unroll
                        for (int j = 0; j < NJ; ++j) acc[r0 + rt][j][i] = __builtin_fmaf(tmp[rt][j][i], e, acc[r0 + rt][j][i]);
                    }
                }
            }
        };
        if constexpr (NF > 0) {
            static_assert(NF == 0 || NF * KSTEP == NW, "one round of state tiles");
            // full 64 x 64 float tiles (the launcher checked it): every 16-byte load of both tiles goes out
            // before the first one is converted
            const T *s16f = reinterpret_cast<const T *>(BWD ? p.dstates16_f : p.states16_f);
            if (s16f) {
                // the 16-bit copies of the entering states: 64 x 64 elements per direction, 16 bytes per thread
                static_assert(PW * NW * (int)sizeof(T) == SCAN_THREADS * 16, "one 16-byte unit per thread and direction");
                const T *s16b = reinterpret_cast<const T *>(BWD ? p.dstates16_b : p.states16_b);
                const f32x4 rf = *reinterpret_cast<const f32x4 *>(s16f + so + threadIdx.x * VS);
                const f32x4 rb = UNI ? rf : *reinterpret_cast<const f32x4 *>(s16b + so + threadIdx.x * VS);
                const int r = threadIdx.x / (NW / VS), k0 = (threadIdx.x % (NW / VS)) * VS;
                *reinterpret_cast<f32x4 *>(sF + r * LDS_ + k0) = rf;
                *reinterpret_cast<f32x4 *>(sB + r * LDS_ + k0) = rb;
            } else {
                constexpr int PER = PW * NW / 4 / SCAN_THREADS;
                float4 rawf[PER], rawb[PER];
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    const int idx = threadIdx.x + i * SCAN_THREADS;
                    rawf[i] = *reinterpret_cast<const float4 *>(stf + idx * 4);
                    rawb[i] = UNI ? rawf[i] : *reinterpret_cast<const float4 *>(stb + idx * 4);
                }
                struct alignas(sizeof(T) * 4) Out { T v[4]; };
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    const int idx = threadIdx.x + i * SCAN_THREADS, r = idx / (NW / 4), k0 = (idx % (NW / 4)) * 4;
                    Out of, ob;
                    of.v[0] = from_f<T>(rawf[i].x); of.v[1] = from_f<T>(rawf[i].y); of.v[2] = from_f<T>(rawf[i].z); of.v[3] = from_f<T>(rawf[i].w);
                    ob.v[0] = from_f<T>(rawb[i].x); ob.v[1] = from_f<T>(rawb[i].y); ob.v[2] = from_f<T>(rawb[i].z); ob.v[3] = from_f<T>(rawb[i].w);
                    *reinterpret_cast<Out *>(sF + r * LDS_ + k0) = of;
                    *reinterpret_cast<Out *>(sB + r * LDS_ + k0) = ob;
                }
            }
            __syncthreads();
            state_product(0, NW);
            if (!UNI) state_product(1, NW);
        } else
        for (int n0 = 0; n0 < N; n0 += NW) {
            if (n0) {
                __syncthreads();
                if (ROWS_FIRST) load_arows(n0);
            }
            if (sizeof(T) == 2 && !BWD && p.states16_f) {
                // the 16-bit copies of the entering states (a forward pass whose caller keeps no states: half the bytes)
                tile_load_kcontig<T, T, PW, NW>(sF, reinterpret_cast<const T *>(p.states16_f) + so + n0, N, P - p0, N - n0, Ident());
                tile_load_kcontig<T, T, PW, NW>(sB, reinterpret_cast<const T *>(p.states16_b) + so + n0, N, P - p0, N - n0, Ident());
            } else {
                tile_load_kcontig<T, float, PW, NW>(sF, stf + n0, N, P - p0, N - n0, Ident());
                tile_load_kcontig<T, float, PW, NW>(sB, stb + n0, N, P - p0, N - n0, Ident());
            }
            if (!ROWS_FIRST) load_arows(n0);
            __syncthreads();
            state_product(0, N - n0);
            state_product(1, N - n0);
        }
    }

    // ---- epilogue operands (x and z, resp. x and dy) are requested one row tile ahead of their use ----
    constexpr int CPR = PW / VS;                   // 16-byte chunks per row
    constexpr int NPASS = (16 * CPR + 63) / 64;    // chunks per lane and row tile
    const T *xrow = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * p.x_sl + h * p.x_sh;
    const T *zrow = (!BWD && p.has_z) ? reinterpret_cast<const T *>(p.z) + b * p.z_sb + (int64_t)c * Q * p.z_sl + h * p.z_sh : nullptr;
    const bool need2 = BWD ? (bool)p.has_D : (bool)p.has_z;      // second operand: dy (for D) resp. z
    const T *row2 = BWD ? kp : zrow;
    const int64_t s2 = BWD ? ks : p.z_sl;
    const bool xvec = aligned16(xrow + p0, p.x_sl) && (P % VS == 0);
    const bool vec2 = need2 && aligned16(row2 + p0, s2) && (P % VS == 0);
    const bool ovec = (P % VS == 0);
    Vec16<T> ex[QT][NPASS], e2[QT][NPASS];         // kept as loaded; converted where they are used
    auto load_vec = [&](const T *ptr, bool vec, int ncol, Vec16<T> &v) {
        if (FAST || (vec && ncol >= VS)) {
            v = *reinterpret_cast<const Vec16<T> *>(ptr);
        } else {
#pragma unroll
            for (int i = 0; i < VS; ++i) v.v[i] = i < ncol ? ptr[i] : from_f<T>(0.f);
        }
    };
    // past_caches: a result that no kernel of the pass reads again (out, dx) leaves the caches to what is read again
    auto store_vec = [&](T *ptr, bool vec, int ncol, const float (&v)[VS], bool past_caches = false) {
        if (FAST || (vec && ncol >= VS)) {
            Vec16<T> ov;
#pragma unroll
            for (int i = 0; i < VS; ++i) ov.v[i] = from_f<T>(v[i]);
            if (past_caches) __builtin_nontemporal_store(__builtin_bit_cast(f32x4, ov), reinterpret_cast<f32x4 *>(ptr));
            else *reinterpret_cast<Vec16<T> *>(ptr) = ov;
        } else {
#pragma unroll
            for (int i = 0; i < VS; ++i)
                if (i < ncol) ptr[i] = from_f<T>(v[i]);
        }
    };
    auto epi_issue = [&](int rt) {
        const int B_ = rt;
        const int r0 = (wave * QT + rt) * 16;
#pragma unroll
        for (int ps = 0; ps < NPASS; ++ps) {
            const int id = lane + ps * 64;
            const int r = r0 + id / CPR, col = p0 + (id % CPR) * VS;
            const int ncol = (id < 16 * CPR && r < limit) ? P - col : 0;
            if (FAST && id >= 16 * CPR) continue;
            const int rc = min(r, limit - 1);
            if (BWD) load_vec(xrow + (int64_t)rc * p.x_sl + col, xvec, ncol, ex[B_][ps]);
            if (need2 && !BWD) load_vec(row2 + (int64_t)rc * s2 + col, vec2, ncol, e2[B_][ps]);
        }
    };
    typedef std::integral_constant<int, 0> B0;
    typedef std::integral_constant<int, 1> B1;
    // ---- part 2: inside the chunk.  A built in registers from CB (forward) or CB^T (mirror) ----
    {
        const float *cb = (BWD ? p.CBT : p.CB) + ((int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
        const bool cvec = (Q % 4 == 0);
        float lor[QT], upr[QT];
        const float *rowp[QT];
#pragma unroll
        for (int rt = 0; rt < QT; ++rt) {
            lor[rt] = lo[rowi[rt]];
            upr[rt] = up[rowi[rt]];
            rowp[rt] = cb + (int64_t)min(rowi[rt], Q - 1) * Q;
        }
        // two register buffers where there is room for them: the CB rows of the next K step are on their way while the current
        // step is consumed (with 2 x 4 tiles of accumulators the kernel is at its 128 registers)
        constexpr bool AHEAD = QT * NJ <= 4;
        float cbv[AHEAD ? 2 : 1][QT][KPL];
        auto issue = [&](auto BUF, int k0) {
            constexpr int B_ = decltype(BUF)::value;
            const int kb = k0 + lg * KPL;
#pragma unroll
            for (int rt = 0; rt < QT; ++rt) {
                if (FAST || (cvec && kb + KPL <= Q)) {
                    if (KPL >= 4) {
#pragma unroll
                        for (int i = 0; i < KPL; i += 4) {
                            const float4 t4 = *reinterpret_cast<const float4 *>(rowp[rt] + kb + i);
                            cbv[B_][rt][i] = t4.x; cbv[B_][rt][(i + 1) % KPL] = t4.y;
                            cbv[B_][rt][(i + 2) % KPL] = t4.z; cbv[B_][rt][(i + 3) % KPL] = t4.w;
                        }
                    } else {
                        cbv[B_][rt][0] = rowp[rt][kb];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < KPL; ++i) cbv[B_][rt][i] = (kb + i < Q) ? rowp[rt][kb + i] : 0.f;
                }
            }
        };
        auto process = [&](auto BUF, int k0) {
            constexpr int B_ = decltype(BUF)::value;
            const int kb = k0 + lg * KPL;
            typename M::Frag bf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) bf[j] = M::load(xT + xt_index<T, LDX>(j * 16 + lr, kb));
            // this lane's KPL columns lie in one block of 16
#pragma unroll
            for (int rt = 0; rt < QT; ++rt) {
                const int r = rowi[rt], r0 = (wave * QT + rt) * 16;
                float v[KPL];
                if (k0 + KSTEP - 1 < r0) {            // every k of this step is below every row of the tile
                    const float rf = __expf(lor[rt] - lo[kb | 15]);
#pragma unroll
                    for (int i = 0; i < KPL; ++i) v[i] = cbv[B_][rt][i] * rf * glo[kb + i];
                } else if (k0 > r0 + 15) {            // every k above every row
                    const float rf = __expf(upr[rt] - up[kb & ~15]);
#pragma unroll
                    for (int i = 0; i < KPL; ++i) v[i] = cbv[B_][rt][i] * rf * gup[kb + i];
                } else {
#pragma unroll
                    for (int i = 0; i < KPL; ++i) {
                        const int k = kb + i;
                        const float e = k < r ? lor[rt] - lo[k] : upr[rt] - up[k];
                        v[i] = cbv[B_][rt][i] * ((k == r) ? 2.f : __expf(e));
                        if (!BWD) v[i] *= dtl[min(k, QP - 1)];
                    }
                }
                const typename M::Frag af = M::pack(v);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[rt][j] = M::mma(af, bf[j], acc[rt][j]);
            }
        };
        if constexpr (NF > 0) {
            static_assert(NF == 0 || (NF == 2 && KPL == 8 && KSTEP == 32), "K-row image: 32 rows of 64 elements per step");
            // fragment (hh, f): K row krow + 4*hh of the step, 16-byte chunk lg + 4*f, stored at chunk ^ (row % 8); with
            // krow % 8 = lr % 4 that is element kfb + 256*hh + 32*(f ^ hh) of the slot
            const int kfb = (8 * (lr >> 2) + (lr & 3)) * 64 + (lg ^ (lr & 3)) * 8;
            // x^T fragment j of step s (xt_index(16j + lr, 32s + 8lg)): lane part by the parity of j, the rest is uniform
            static_assert(NF == 0 || NJ == 4, "fragment addresses below are written out for four column tiles");
            const int xl0 = lr * LDX + 8 * (lg ^ (lr >> 3)), xl1 = lr * LDX + 8 * (lg ^ ((lr >> 3) + 2));
            // While requests are in flight every LDS access goes through the raw accessors (the compiler would make an
            // access it knows of wait for all of them), and the barrier is the bare instruction.
            const unsigned krl_a = lds_addr(krl) + kfb * 2, xt_a = lds_addr(xT);
            const unsigned lg32 = lg * 32;             // this lane's 8 columns inside a step of the float tables
            const int nsteps = (limit + KSTEP - 1) / KSTEP;
            typedef typename M::Frag Frag;
            for (int step = 0; step < nsteps; ++step) {
                const int k0 = step * KSTEP;
                // this wave's request for the step has landed: one request per step, up to KRING - 2 newer ones
                const int newer = min(KRING - 2, nsteps - 1 - step);
                if (newer >= 2) wait_vmcnt<2>();
                else if (newer == 1) wait_vmcnt<1>();
                else wait_vmcnt<0>();
                raw_lds_barrier();                     // ... and everybody else's; the slot of step - 1 is free again
                if (step + KRING - 1 < nsteps) kr_issue(step + KRING - 1);
                if (UNI && (BWD ? k0 + KSTEP - 1 < wave * QT * 16 : k0 > wave * QT * 16 + QT * 16 - 1)) continue;   // far side of the diagonal
                const unsigned slot = krl_a + (step % KRING) * (32 * 64 * 2);
                // the CB tiles of both row tiles first; the K fragments are dead after that
                f32x4 cb1[QT], cb2[QT];
                {
                    Frag kf00 = raw_lds_read_at<Frag, 0>(slot), kf01 = raw_lds_read_at<Frag, 64>(slot);
                    Frag kf10 = raw_lds_read_at<Frag, 512 + 64>(slot), kf11 = raw_lds_read_at<Frag, 512>(slot);
                    raw_lds_wait();
                    raw_lds_use(kf00); raw_lds_use(kf01); raw_lds_use(kf10); raw_lds_use(kf11);
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) {
                        cb1[rt] = M::mma(kf00, own[rt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                        cb2[rt] = M::mma(kf10, own[rt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                        cb1[rt] = M::mma(kf01, own[rt][1], cb1[rt]);
                        cb2[rt] = M::mma(kf11, own[rt][1], cb2[rt]);
                    }
                }
                // the wave's rows [wr0, wr0 + 16*QT) meet the step's columns [k0, k0 + 32) in one step only
                const int wr0 = wave * QT * 16;
                const int cls = (k0 + KSTEP - 1 < wr0) ? 0 : (k0 > wr0 + QT * 16 - 1) ? 1 : 2;   // below, above, across the diagonal
                const int kb = k0 + lg * KPL;
                // ---- A operands of both row tiles: CB times the decay factors
                Frag af[QT];
                if (cls != 2) {
                    const unsigned ta = lds_addr(cls == 0 ? glo : gup) + k0 * 4 + lg32;
                    f32x4 ga0 = raw_lds_read_at<f32x4, 0>(ta), ga1 = raw_lds_read_at<f32x4, 16>(ta);
                    float mref = raw_lds_read_at<float, 0>(cls == 0 ? lds_addr(lo) + (kb | 15) * 4 : lds_addr(up) + (kb & ~15) * 4);
                    raw_lds_wait();
                    raw_lds_use(ga0); raw_lds_use(ga1); raw_lds_use(mref);
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) {
                        const float rf = __expf((cls == 0 ? lor[rt] : upr[rt]) - mref);
                        float v[KPL];
#pragma unroll
                        for (int i = 0; i < 4; ++i) { v[i] = cb1[rt][i] * rf * ga0[i]; v[i + 4] = cb2[rt][i] * rf * ga1[i]; }
                        af[rt] = M::pack(v);
                    }
                } else {
                    // the one step across the diagonal: element by element
                    const unsigned la = lds_addr(lo) + k0 * 4 + lg32, ua = lds_addr(up) + k0 * 4 + lg32;
                    f32x4 l0 = raw_lds_read_at<f32x4, 0>(la), l1 = raw_lds_read_at<f32x4, 16>(la);
                    f32x4 u0 = raw_lds_read_at<f32x4, 0>(ua), u1 = raw_lds_read_at<f32x4, 16>(ua);
                    f32x4 d0 = {1.f, 1.f, 1.f, 1.f}, d1 = d0;
                    if (!BWD) {
                        const unsigned da = lds_addr(dtl) + k0 * 4 + lg32;
                        d0 = raw_lds_read_at<f32x4, 0>(da);
                        d1 = raw_lds_read_at<f32x4, 16>(da);
                    }
                    raw_lds_wait();
                    raw_lds_use(l0); raw_lds_use(l1); raw_lds_use(u0); raw_lds_use(u1);
                    if (!BWD) { raw_lds_use(d0); raw_lds_use(d1); }
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) {
                        const int r = (wave * QT + rt) * 16 + lr;
                        float v[KPL];
#pragma unroll
                        for (int i = 0; i < KPL; ++i) {
                            const int k = kb + i;
                            const float lk = i < 4 ? l0[i & 3] : l1[i & 3], uk = i < 4 ? u0[i & 3] : u1[i & 3];
                            const float e = k < r ? lor[rt] - lk : upr[rt] - uk;
                            float w = (k == r) ? (UNI ? 1.f : 2.f) : __expf(e);
                            if (UNI && (BWD ? k < r : k > r)) w = 0.f;
                            if (!BWD) w *= i < 4 ? d0[i & 3] : d1[i & 3];
                            v[i] = (i < 4 ? cb1[rt][i & 3] : cb2[rt][i & 3]) * w;
                        }
                        af[rt] = M::pack(v);
                    }
                }
                // ---- the x product, two column tiles at a time
                const unsigned xa = xt_a + 64 * step, xb = xt_a + 64 * (step ^ 1);
                {
                    Frag b0 = raw_lds_read_at<Frag, 0>(xa + 2 * xl0), b1 = raw_lds_read_at<Frag, 32 * LDX>(xa + 2 * xl1);
                    raw_lds_wait();
                    raw_lds_use(b0); raw_lds_use(b1);
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) {
                        acc[rt][0] = M::mma(af[rt], b0, acc[rt][0]);
                        acc[rt][1] = M::mma(af[rt], b1, acc[rt][1]);
                    }
                }
                {
                    Frag b2 = raw_lds_read_at<Frag, 64 * LDX>(xb + 2 * xl0), b3 = raw_lds_read_at<Frag, 96 * LDX>(xb + 2 * xl1);
                    raw_lds_wait();
                    raw_lds_use(b2); raw_lds_use(b3);
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) {
                        acc[rt][2] = M::mma(af[rt], b2, acc[rt][2]);
                        acc[rt][3] = M::mma(af[rt], b3, acc[rt][3]);
                    }
                }
            }
            wait_vmcnt<0>();
            __syncthreads();
        } else {
            if constexpr (AHEAD) {
                issue(B0(), 0);
                for (int k0 = 0; k0 < limit; k0 += 2 * KSTEP) {
                    if (k0 + KSTEP < limit) issue(B1(), k0 + KSTEP);
                    process(B0(), k0);
                    if (k0 + KSTEP < limit) {
                        if (k0 + 2 * KSTEP < limit) issue(B0(), k0 + 2 * KSTEP);
                        process(B1(), k0 + KSTEP);
                    }
                }
            } else {
                for (int k0 = 0; k0 < limit; k0 += KSTEP) {
                    issue(B0(), k0);
                    process(B0(), k0);
                }
            }
        }
    }

    // ---- epilogue.  Each wave passes its 16-row accumulator tiles through a private LDS patch so that out, out_x,
    // dx are written (and x, z, dy were read) as 16-byte vectors along headdim ----
    // the rows that the D term needs (forward: x, mirror: dy) lie in the operand image (transposed, unscaled; zero past the
    // end of the sequence and of headdim): they are read from there, elements a row of the image apart, before the image
    // becomes the staging area - and before the global requests below, which an LDS access known to the compiler would
    // wait for
    if (BWD ? need2 : (bool)p.has_D) {
#pragma unroll
        for (int rt = 0; rt < QT; ++rt) {
            if ((wave * QT + rt) * 16 < limit) {
#pragma unroll
                for (int ps = 0; ps < NPASS; ++ps) {
                    const int id = lane + ps * 64;
                    if (FAST && id >= 16 * CPR) continue;
                    const int r = (wave * QT + rt) * 16 + min(id / CPR, 15), cc = (id % CPR) * VS;
#pragma unroll
                    for (int i = 0; i < VS; ++i) (BWD ? e2 : ex)[rt][ps].v[i] = xT[xt_index<T, LDX>(cc + i, r)];
                }
            }
        }
    }
    // the epilogue operands of all row tiles are requested before the barrier
#pragma unroll
    for (int rt = 0; rt < QT; ++rt) {
        if ((wave * QT + rt) * 16 < limit) epi_issue(rt);
    }
    __syncthreads();   // every wave is done with xT: the operand images become the staging area
    float *stg = reinterpret_cast<float *>(shared_u) + wave * 16 * SLD;
    float dsum[VS];
#pragma unroll
    for (int i = 0; i < VS; ++i) dsum[i] = 0.f;
    auto epi_consume = [&](int rt) {
        const int B_ = rt;
        const int r0 = (wave * QT + rt) * 16;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) stg[(lg * 4 + i) * SLD + j * 16 + lr] = acc[rt][j][i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int ps = 0; ps < NPASS; ++ps) {
            const int id = lane + ps * 64;
            const int rl = id / CPR, cc = (id % CPR) * VS;
            const int r = r0 + rl, col = p0 + cc;
            const int ncol = P - col;              // valid columns from col on
            const bool ok = id < 16 * CPR && r < limit && ncol > 0;
            float a[VS];
#pragma unroll
            for (int i = 0; i < VS; i += 4) {
                const float4 t4 = *reinterpret_cast<const float4 *>(stg + (rl & 15) * SLD + cc + i);
                a[i] = t4.x; a[i + 1] = t4.y; a[i + 2] = t4.z; a[i + 3] = t4.w;
            }
            const int64_t orow = (((int64_t)b * p.seqlen + (int64_t)c * Q + r) * H + h) * P + col;
            float rsum = 0.f;
            if (ok) {
                if (!BWD) {
                    if (p.has_D) {
#pragma unroll
                        for (int i = 0; i < VS; ++i)
                            a[i] += (p.D_has_hdim ? (i < ncol ? p.D[h * P + col + i] : 0.f) : d_head) * to_f(ex[B_][ps].v[i]);
                    }
                    if (p.has_z) {
                        if (p.out_x) store_vec(reinterpret_cast<T *>(p.out_x) + orow, ovec, ncol, a);
#pragma unroll
                        for (int i = 0; i < VS; ++i) a[i] *= silu_f(to_f(e2[B_][ps].v[i]));
                    }
                    store_vec(reinterpret_cast<T *>(p.out) + orow, ovec, ncol, a, true);
                } else {
                    const float dtr = dto[r];
                    float dxv[VS];
#pragma unroll
                    for (int i = 0; i < VS; ++i) { rsum += a[i] * to_f(ex[B_][ps].v[i]); dxv[i] = a[i] * dtr; }
                    if (p.has_D) {
#pragma unroll
                        for (int i = 0; i < VS; ++i) {
                            dxv[i] += (p.D_has_hdim ? (i < ncol ? p.D[h * P + col + i] : 0.f) : d_head) * to_f(e2[B_][ps].v[i]);
                            dsum[i] += to_f(e2[B_][ps].v[i]) * to_f(ex[B_][ps].v[i]);
                        }
                    }
                    // (dx may be a slice of a wider buffer: its own position and batch strides)
                    const int64_t dxo = p.dx_sl ? b * p.dx_sb + ((int64_t)c * Q + r) * p.dx_sl + (int64_t)h * P + col : orow;
                    store_vec(reinterpret_cast<T *>(p.dx) + dxo, ovec && (p.dx_sl % VS == 0) && (p.dx_sb % VS == 0), ncol, dxv, true);
                }
            }
            if (BWD) {
                // the CPR lanes of a row sit next to each other: butterfly over them
#pragma unroll
                for (int d = 1; d < CPR; d <<= 1) rsum += __shfl_xor(rsum, d, 64);
                if (id < 16 * CPR && r < limit && (id % CPR) == 0) {
                    // (several headdim tiles share a row: each writes the plane of its tile, the reader adds them)
                    p.ddt_direct[(int64_t)pt * ((int64_t)p.batch * H * nc * Q) + o + r] = rsum;
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int rt = 0; rt < QT; ++rt) {
        if ((wave * QT + rt) * 16 < limit) epi_consume(rt);
    }
    if (BWD && p.has_D) {
        // dsum[i]: this lane's share of column (lane % CPR)*VS + i; add the lanes that hold other rows
#pragma unroll
        for (int i = 0; i < VS; ++i) {
            float v = dsum[i];
#pragma unroll
            for (int d = CPR; d < 64; d <<= 1) v += __shfl_xor(v, d, 64);
            dsum[i] = v;
        }
        if (lane < CPR) {
#pragma unroll
            for (int i = 0; i < VS; ++i) red[wave][lane * VS + i] = dsum[i];
        }
        __syncthreads();
        if (threadIdx.x < PW && p0 + (int)threadIdx.x < P) {
            float v = 0.f;
#pragma unroll
            for (int wv = 0; wv < SCAN_WAVES; ++wv) v += red[wv][threadIdx.x];
            p.red[((int64_t)(b * nc + c) * H + h) * P + p0 + threadIdx.x] = v;   // partials [(b, c)][h][P]
        }
    }
}

// lds: ScanMap::LDS bytes, 16-byte aligned; id: the workgroup's place in the launch
template <typename T, int QT, int NJ, bool BWD, bool FAST, int NF, bool UNI = false, bool STATES = true>
__device__ __forceinline__ void chunk_scan_body(const bimamba2_params &p, int nc, int npt, unsigned id, char *lds) {
    typedef ScanMap<T, QT, NJ, BWD, NF> Map;
    auto at = [&](int offset) { return reinterpret_cast<float *>(lds + offset); };
    chunk_scan_work<T, QT, NJ, BWD, FAST, NF, UNI, STATES>(p, nc, npt, id, lds, at(Map::LO), at(Map::UP), at(Map::GLO), at(Map::GUP), at(Map::DTL),
                                                           reinterpret_cast<float (*)[16 * NJ]>(lds + Map::RED), reinterpret_cast<T *>(lds + Map::KRL));
}

}  // namespace bm2
