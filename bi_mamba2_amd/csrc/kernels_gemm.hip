// Matrix products of the BiMamba2 layer's two projections (forward, input gradient, weight gradient) for 16-bit operands.
//
//   C[m, n] = sum_k A(m, k) B(n, k)  (+ bias[n]),   float32 accumulation, C in the operands' type
//
// Either operand may have k contiguous in memory (x and W of a forward product) or its rows contiguous (W in an input
// gradient, both operands of a weight gradient).  What it replaces at these places is a library product whose call costs the
// host 18 to 22 us - more than the product at small sizes - and whose weight gradients (few output tiles, a long sum) ran at 330 to
// 460 TFLOP/s.
//
// A workgroup owns a BM x BN tile and goes through k in steps of 32.  The operand tiles of a step travel straight into a ring
// of four LDS slots (direct loads, requested three steps ahead), a step's fragments are read into registers while the products
// of the step before run, and there is one barrier per step.  (Steps of 64 with two slots: the registers of a 256 x 256 tile no
// longer suffice, weight gradients 93 -> 120 us.)  Tiles with k contiguous lie in LDS as rows of 64 bytes whose 16-byte chunks
// are XOR-swizzled, the others as [k][64] blocks that are read with LDS transpose reads (tile64_swz).  The
// products are computed transposed (rows of the matrix instruction are n) and the n of a row is chosen so that a lane holds
// eight consecutive columns of one output row: the result leaves as 16-byte stores straight from the accumulators.
// Products with few output tiles are cut along k (blockIdx): the float32 partial tiles are added up by a second kernel in a
// fixed order.
#include <atomic>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace bm2 {
namespace {

constexpr int GK = 32, GRING = 4;                 // k of a step, slots of the ring

template <int BM, int BN, int WR, int WC> struct GemmTile {
    static constexpr int WAVES = WR * WC, THREADS = 64 * WAVES;
    static constexpr int MT = BM / WR / 16, NT = BN / WC / 16;        // 16-row / 16-column tiles of a wave
    static constexpr int A_B = BM * GK * 2, B_B = BN * GK * 2, SLOT = A_B + B_B;
    static constexpr int LOADS = (BM + BN) / 16 / WAVES;              // requests of a wave per step (1 KB each)
    static_assert((BM + BN) / 16 % WAVES == 0 && BM / 16 % WAVES == 0, "a wave's requests lie in one operand each");
    static_assert(NT % 2 == 0 && MT >= 1, "pairs of column tiles");
};

__device__ __forceinline__ unsigned mask_from(int k, int K) { return k + 1 < K ? ~0u : k < K ? 0xFFFFu : 0u; }

}  // namespace

// AKC / BKC: k contiguous in A / B.  F32: the tile goes to the float32 partial sums of its k slice.
template <typename T, int BM, int BN, int WR, int WC, bool AKC, bool BKC, bool F32>
__global__ __launch_bounds__(64 * WR * WC) void gemm_kernel(const bimamba2_gemm_params p, int mtiles, int ntiles, int kper) {
    typedef GemmTile<BM, BN, WR, WC> G;
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    constexpr int MT = G::MT, NT = G::NT, L = G::LOADS;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[GRING * G::SLOT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4, wm = wave / WC, wn = wave % WC;
    // Workgroups are dealt to the 8 XCDs one after the other: each XCD gets a contiguous run of tiles, which goes through bands
    // of 4 row tiles column by column, so that its L2 serves the operand rows several times.
    int mt_, nt_, split;
    {
        const int total = gridDim.x, id = blockIdx.x, xcd = id & 7, per = total >> 3, rem = total & 7;
        const int lin = xcd * per + min(xcd, rem) + (id >> 3), tiles = mtiles * ntiles;
        split = lin / tiles;
        const int t = lin - split * tiles, band = t / (4 * ntiles), in = t - band * 4 * ntiles, rows = min(4, mtiles - band * 4);
        mt_ = band * 4 + in % rows;
        nt_ = in / rows;
    }
    const int m0 = mt_ * BM, n0 = nt_ * BN, kbeg = split * kper, K = min(p.k - kbeg, kper), nk = (K + GK - 1) / GK;
    const unsigned lda = (unsigned)(p.lda * 2), ldb = (unsigned)(p.ldb * 2);
    const char *abase = uniform_ptr(reinterpret_cast<const T *>(p.a) + (AKC ? (int64_t)m0 * p.lda + kbeg : (int64_t)kbeg * p.lda + m0));
    const char *bbase = uniform_ptr(reinterpret_cast<const T *>(p.b) + (BKC ? (int64_t)n0 * p.ldb + kbeg : (int64_t)kbeg * p.ldb + n0));
    const int mvalid = p.m - m0, nvalid = p.n - n0;

    // one request: unit u (1 KB) of an operand tile, step it.  k contiguous: 16 rows x 64 bytes; else 8 k x 128 bytes of a
    // 64-column block.  Rows, columns and k outside the matrix read a valid neighbour (k is masked later, in the fragments).
    auto request = [&](auto KC, const char *base, unsigned ld, int valid, int u, int it, unsigned char *dst) __attribute__((always_inline)) {
        if constexpr (decltype(KC)::value) {
            const int row = u * 16 + (lane >> 2), chunk = (lane & 3) ^ ((row >> 2) & 3);
            const int kk = min(it * GK + chunk * 8, (K - 1) & ~7);
            load16_to_lds(base + (__umul24(min(row, valid - 1), ld) + (unsigned)kk * 2), dst + u * 1024);
        } else {
            const int row = (u & 3) * 8 + (lane >> 3), col = (u >> 2) * 64 + (((lane & 7) ^ tile64_swz(row)) << 3);
            load16_to_lds(base + (__umul24(min(it * GK + row, K - 1), ld) + (unsigned)min(col, (valid - 1) & ~7) * 2), dst + u * 1024);
        }
    };
    auto issue = [&](int it) __attribute__((always_inline)) {
        unsigned char *slot = smem + (it & (GRING - 1)) * G::SLOT;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int u = wave + i * G::WAVES;
            if (i < BM / 16 / G::WAVES) request(std::integral_constant<bool, AKC>(), abase, lda, mvalid, u, it, slot);
            else request(std::integral_constant<bool, BKC>(), bbase, ldb, nvalid, u - BM / 16, it, slot + G::A_B);
        }
    };

    // this lane's fragment addresses inside a slot
    const unsigned sb = lds_addr(smem);
    unsigned a_l[4], b_l[2];
    if constexpr (AKC) {
        a_l[0] = sb + (wm * MT * 16 + lr) * 64 + ((lg ^ (lr >> 2)) << 4);
    } else {
        // tile mt: 64-column block (wm MT + mt) / 4, columns 16 ((wm MT + mt) % 4): the chunk position's bits 1, 2 flip with it
#pragma unroll
        for (int j = 0; j < 4; ++j) a_l[j] = sb + (tile64_tr_offset(8 * lg + (lr >> 2), 4 * (lr & 3)) ^ (j << 5));
    }
    if constexpr (BKC) {
        b_l[0] = sb + G::A_B + (wn * NT * 16 + 8 * (lr >> 2) + (lr & 3)) * 64 + ((lg ^ ((2 * (lr >> 2)) & 3)) << 4);
        b_l[1] = (b_l[0] ^ 16u) + 256u;
    } else {
        b_l[0] = sb + G::A_B + tile64_tr_offset(8 * lg + (lr >> 2), 8 * (lr & 3));
        b_l[1] = b_l[0] ^ 64u;
    }
    struct Frags {
        Frag a[AKC ? MT : 1], b[BKC ? NT : 1];
        i16x4 al[AKC ? 1 : MT], ah[AKC ? 1 : MT], bl[BKC ? 1 : NT], bh[BKC ? 1 : NT];
    };
    auto read = [&](Frags &f, int it) __attribute__((always_inline)) {
        const unsigned so = (unsigned)(it & (GRING - 1)) * G::SLOT;
        if constexpr (BKC) {
            const unsigned b0 = b_l[0] + so, b1 = b_l[1] + so;
#define BM2_RB(J) if constexpr (J < NT) f.b[J] = raw_lds_read_at<Frag, (J >> 1) * 2048>((J & 1) ? b1 : b0)
            BM2_RB(0); BM2_RB(1); BM2_RB(2); BM2_RB(3);
#undef BM2_RB
        } else {
            // column pair t of the wave: block (wn NT + 2 t) / 4, half ((wn NT / 2) + t) % 2
            constexpr int HALVES = NT / 2;
            const unsigned blk = so + (unsigned)((wn * HALVES) >> 1) * 4096u;
            const bool odd = (wn * HALVES) & 1;                // (HALVES is 2, or 1 where a wave owns half a block)
            const unsigned h0 = (odd ? b_l[1] : b_l[0]) + blk, h1 = (odd ? b_l[0] : b_l[1]) + blk;
#define BM2_RB(J)                                                                                     \
    if constexpr (J < NT) {                                                                           \
        constexpr int O = (J & 1) * 8;                                                                \
        f.bl[J] = raw_lds_tr16_read_at<O>((J >> 1) ? h1 : h0);                                        \
        f.bh[J] = raw_lds_tr16_read_at<O + 512>((J >> 1) ? h0 : h1);                                  \
    }
            BM2_RB(0) BM2_RB(1) BM2_RB(2) BM2_RB(3)
#undef BM2_RB
        }
        if constexpr (AKC) {
            const unsigned a0 = a_l[0] + so;
#define BM2_RA(J) if constexpr (J < MT) f.a[J] = raw_lds_read_at<Frag, J * 1024>(a0)
            BM2_RA(0); BM2_RA(1); BM2_RA(2); BM2_RA(3); BM2_RA(4); BM2_RA(5); BM2_RA(6); BM2_RA(7);
#undef BM2_RA
        } else {
            constexpr bool WHOLE = MT % 4 == 0;                // a wave owns whole 64-column blocks (else half of one)
            const unsigned blk = so + (unsigned)(wm * MT / 4) * 4096u;
            unsigned ta[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) ta[j] = (WHOLE ? a_l[j] : a_l[(j + 2 * (wm & 1)) & 3]) + blk;
#define BM2_RA(J)                                                                  \
    if constexpr (J < MT) {                                                        \
        f.al[J] = raw_lds_tr16_read_at<(J >> 2) * 4096>(ta[J & 3]);                \
        f.ah[J] = raw_lds_tr16_read_at<(J >> 2) * 4096 + 512>(ta[(J & 3) ^ 2]);    \
    }
            BM2_RA(0) BM2_RA(1) BM2_RA(2) BM2_RA(3) BM2_RA(4) BM2_RA(5) BM2_RA(6) BM2_RA(7)
#undef BM2_RA
        }
    };
    auto use = [&](Frags &f) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < (AKC ? MT : 0); ++j) raw_lds_use(f.a[j]);
#pragma unroll
        for (int j = 0; j < (AKC ? 0 : MT); ++j) { raw_lds_use(f.al[j]); raw_lds_use(f.ah[j]); }
#pragma unroll
        for (int j = 0; j < (BKC ? NT : 0); ++j) raw_lds_use(f.b[j]);
#pragma unroll
        for (int j = 0; j < (BKC ? 0 : NT); ++j) { raw_lds_use(f.bl[j]); raw_lds_use(f.bh[j]); }
    };
    f32x4 acc[MT][NT] = {};
    // the last step of a k that is no multiple of 32: the elements behind the end become zero on both sides (what the loads
    // found there may be an infinity, or no number at all)
    auto mask_tail = [&](Frags &f) __attribute__((always_inline)) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        const int k = (nk - 1) * GK + 8 * lg;
        const u32x4 msk = {mask_from(k, K), mask_from(k + 2, K), mask_from(k + 4, K), mask_from(k + 6, K)};
#pragma unroll
        for (int j = 0; j < (AKC ? MT : 0); ++j) f.a[j] = __builtin_bit_cast(Frag, __builtin_bit_cast(u32x4, f.a[j]) & msk);
#pragma unroll
        for (int j = 0; j < (AKC ? 0 : MT); ++j) {
            f.al[j] = __builtin_bit_cast(i16x4, __builtin_bit_cast(u32x2, f.al[j]) & u32x2{msk[0], msk[1]});
            f.ah[j] = __builtin_bit_cast(i16x4, __builtin_bit_cast(u32x2, f.ah[j]) & u32x2{msk[2], msk[3]});
        }
#pragma unroll
        for (int j = 0; j < (BKC ? NT : 0); ++j) f.b[j] = __builtin_bit_cast(Frag, __builtin_bit_cast(u32x4, f.b[j]) & msk);
#pragma unroll
        for (int j = 0; j < (BKC ? 0 : NT); ++j) {
            f.bl[j] = __builtin_bit_cast(i16x4, __builtin_bit_cast(u32x2, f.bl[j]) & u32x2{msk[0], msk[1]});
            f.bh[j] = __builtin_bit_cast(i16x4, __builtin_bit_cast(u32x2, f.bh[j]) & u32x2{msk[2], msk[3]});
        }
    };
    auto multiply = [&](Frags &f) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            Frag a;
            if constexpr (AKC) a = f.a[mt];
            else a = __builtin_bit_cast(Frag, __builtin_shufflevector(f.al[mt], f.ah[mt], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                Frag b;
                if constexpr (BKC) b = f.b[nt];
                else b = __builtin_bit_cast(Frag, __builtin_shufflevector(f.bl[nt], f.bh[nt], 0, 1, 2, 3, 4, 5, 6, 7));
                acc[mt][nt] = M::mma(b, a, acc[mt][nt]);
            }
        }
    };
    const bool ragged = K % GK != 0;

    issue(0);
    if (nk > 1) issue(1);
    if (nk > 2) issue(2);
    if (nk > 2) wait_vmcnt<2 * L>();
    else if (nk > 1) wait_vmcnt<L>();
    else wait_vmcnt<0>();
    raw_lds_barrier();
    Frags fa, fb;
    read(fa, 0);
    // one step: the fragments in `cur` are multiplied while those of the next step are read into `nxt`
    auto step = [&](int it, Frags &cur, Frags &nxt) __attribute__((always_inline)) {
        raw_lds_wait();
        use(cur);
        if (it + 1 < nk) {
            if (it + 2 < nk) wait_vmcnt<L>();              // step it + 1 has landed, it + 2 may be outstanding
            else wait_vmcnt<0>();
            raw_lds_barrier();                             // ... everybody's share of it; the slot of step it - 1 is free
            if (it + 3 < nk) issue(it + 3);
            read(nxt, it + 1);
        }
        if (ragged && it == nk - 1) mask_tail(cur);
        multiply(cur);
    };
    for (int it = 0; it < nk; it += 2) {
        step(it, fa, fb);
        if (it + 1 < nk) step(it + 1, fb, fa);
    }

    // a lane holds, per row tile and column pair t, the columns 32 t + 8 lg .. + 7 of row lr
#pragma unroll
    for (int t = 0; t < NT / 2; ++t) {
        const int n = n0 + (wn * NT + 2 * t) * 16 + 8 * lg;
        const int nn = min(8, p.n - n);
        float bias[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (!F32 && p.bias) {
#pragma unroll
            for (int i = 0; i < 8; ++i) bias[i] = i < nn ? to_f(reinterpret_cast<const T *>(p.bias)[n + i]) : 0.f;
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = m0 + (wm * MT + mt) * 16 + lr;
            if (m >= p.m || nn <= 0) continue;
            const f32x4 lo = acc[mt][2 * t], hi = acc[mt][2 * t + 1];
            if constexpr (F32) {
                const int np = (p.n + 7) & ~7;
                float *o = p.partial + ((int64_t)split * p.m + m) * np + n;
                *reinterpret_cast<f32x4 *>(o) = lo;
                *reinterpret_cast<f32x4 *>(o + 4) = hi;
            } else {
                Vec16<T> v;
#pragma unroll
                for (int i = 0; i < 4; ++i) { v.v[i] = from_f<T>(lo[i] + bias[i]); v.v[4 + i] = from_f<T>(hi[i] + bias[4 + i]); }
                T *o = reinterpret_cast<T *>(p.c) + (int64_t)m * p.ldc + n;
                if (nn == 8 && p.ldc % 8 == 0) *reinterpret_cast<Vec16<T> *>(o) = v;
                else
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (i < nn) o[i] = v.v[i];
            }
        }
    }
}

// C = sum of the k slices' float32 tiles (+ bias), eight columns per thread
template <typename T>
__global__ __launch_bounds__(NTHREADS) void gemm_reduce_kernel(const bimamba2_gemm_params p, int nsplit) {
    const int nv = (p.n + 7) / 8, np = nv * 8;
    const int64_t id = (int64_t)blockIdx.x * NTHREADS + threadIdx.x;
    if (id >= (int64_t)p.m * nv) return;
    const int64_t m = id / nv;
    const int n = (int)(id % nv) * 8, nn = min(8, p.n - n);
    const float *src = p.partial + m * np + n;
    const int64_t slice = (int64_t)p.m * np;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    int s = 0;
    for (; s + 4 <= nsplit; s += 4) {
        f32x4 a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = *reinterpret_cast<const f32x4 *>(src + (s + q) * slice);
            b[q] = *reinterpret_cast<const f32x4 *>(src + (s + q) * slice + 4);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) { lo += a[q]; hi += b[q]; }
    }
    for (; s < nsplit; ++s) {
        lo += *reinterpret_cast<const f32x4 *>(src + s * slice);
        hi += *reinterpret_cast<const f32x4 *>(src + s * slice + 4);
    }
    T *o = reinterpret_cast<T *>(p.c) + m * p.ldc + n;
    Vec16<T> v;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float bias = p.bias && i < nn ? to_f(reinterpret_cast<const T *>(p.bias)[n + i]) : 0.f;
        v.v[i] = from_f<T>((i < 4 ? lo[i & 3] : hi[i & 3]) + bias);
    }
    if (nn == 8 && p.ldc % 8 == 0) *reinterpret_cast<Vec16<T> *>(o) = v;
    else
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < nn) o[i] = v.v[i];
}

namespace {

struct GemmPlan {
    int tile;        // 0: 256 x 256, 1: 128 x 128, 2: 64 x 64
    int nsplit, kper;
};

struct GemmTileCost {
    int bm, bn, per_cu;
    double fixed_us, each_us;     // 32 k of one tile: fixed + each * (tiles that share the CU)
};
// measured on weight gradients (both operands with k outermost); products with k contiguous take about 1.4 times as long
constexpr GemmTileCost GEMM_TILES[3] = {{256, 256, 1, 0.66, 0.12}, {128, 128, 2, 0.22, 0.12}, {64, 64, 4, 0.12, 0.10}};

// Tile and number of k slices by the estimated time: per round of workgroups a start and an end (3 us) and its steps at the
// round's occupancy; for k slices the partial tiles that are written and read again (5 TB/s) and the launch that adds them.
// Against a sweep of tiles and slices: 3224 x 768 over 16384 rows takes 93 us with three slices of 128 x 128 tiles (chosen), 120
// with four of 256 x 256; 768 x 1536: 52 with six (chosen), 402 uncut; 648 x 128 over 17927 rows: 18 with sixteen slices of 64 x 64.
GemmPlan gemm_plan(const bimamba2_gemm_params *p) {
    const int64_t m = p->m, n = p->n, steps = (p->k + 31) / 32;
    const double slow = p->a_kcontig ? 1.4 : 1.0;
    GemmPlan best{2, 1, (int)steps * 32};
    double best_cost = 1e30;
    for (int t = 0; t < 3; ++t) {
        const GemmTileCost &c = GEMM_TILES[t];
        const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn), slots = 256 * c.per_cu;
        for (int s = 1; s <= 16; ++s) {
            const int64_t per = (steps + s - 1) / s;
            if (s > 1 && (per < 8 || (steps + per - 1) / per != s)) continue;
            const int64_t full = tiles * s / slots, rest = tiles * s % slots;
            auto round = [&](int64_t wgs) { return 3.0 + per * slow * (c.fixed_us + c.each_us * ((wgs + 255) / 256)); };
            double cost = full * round(slots) + (rest ? round(rest) : 0.0);
            if (s > 1) cost += 4.0 + (double)m * n * 8 * s / 5e6;
            if (cost < best_cost) { best_cost = cost; best = GemmPlan{t, s, (int)(per * 32)}; }
        }
    }
    return best;
}

template <typename T, int BM, int BN, int WR, int WC>
int launch_gemm_tile(const bimamba2_gemm_params *p, const GemmPlan &g) {
    const int mt = (p->m + BM - 1) / BM, nt = (p->n + BN - 1) / BN;
    const dim3 grid((unsigned)(mt * nt * g.nsplit)), block(64 * WR * WC);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
#define BM2_GEMM(AKC, BKC)                                                                                                                      \
    do {                                                                                                                                        \
        if (g.nsplit > 1) hipLaunchKernelGGL((gemm_kernel<T, BM, BN, WR, WC, AKC, BKC, true>), grid, block, 0, s, *p, mt, nt, g.kper);          \
        else hipLaunchKernelGGL((gemm_kernel<T, BM, BN, WR, WC, AKC, BKC, false>), grid, block, 0, s, *p, mt, nt, g.kper);                      \
    } while (0)
    if (p->a_kcontig && p->b_kcontig) BM2_GEMM(true, true);
    else if (p->a_kcontig) BM2_GEMM(true, false);
    else if (!p->b_kcontig) BM2_GEMM(false, false);
    else return BIMAMBA2_EUNSUPPORTED;
#undef BM2_GEMM
    return check_launch();
}

template <typename T> int launch_gemm_t(const bimamba2_gemm_params *p) {
    const GemmPlan g = gemm_plan(p);
    if (g.nsplit > 1 && !p->partial) return BIMAMBA2_EWORKSPACE;
    int rc = g.tile == 0 ? launch_gemm_tile<T, 256, 256, 2, 4>(p, g) : g.tile == 1 ? launch_gemm_tile<T, 128, 128, 2, 2>(p, g)
                                                                                  : launch_gemm_tile<T, 64, 64, 2, 2>(p, g);
    if (rc || g.nsplit == 1) return rc;
    const int64_t threads = (int64_t)p->m * ((p->n + 7) / 8);
    hipLaunchKernelGGL(gemm_reduce_kernel<T>, dim3((unsigned)((threads + NTHREADS - 1) / NTHREADS)), dim3(NTHREADS), 0,
                       reinterpret_cast<hipStream_t>(p->stream), *p, g.nsplit);
    return check_launch();
}

}  // namespace

size_t gemm_workspace_bytes(const bimamba2_gemm_params *p) {
    const GemmPlan g = gemm_plan(p);
    return g.nsplit > 1 ? (size_t)g.nsplit * p->m * ((p->n + 7) / 8 * 8) * sizeof(float) : 0;
}

int launch_gemm(const bimamba2_gemm_params *p) {
    if (p->dtype == BIMAMBA2_BF16) return launch_gemm_t<bf16_t>(p);
    if (p->dtype == BIMAMBA2_F16) return launch_gemm_t<f16_t>(p);
    return BIMAMBA2_EUNSUPPORTED;
}

}  // namespace bm2
