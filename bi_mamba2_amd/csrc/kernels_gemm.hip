// Matrix products of the BiMamba2 layer's two projections (forward, input gradient, weight gradient) for 16-bit operands.
//
//   C[m, n] = sum_k A(m, k) B(n, k)  (+ bias[n]),   float32 accumulation, C in the operands' type
//
// Either operand may have k contiguous in memory (x and W of a forward product) or its rows contiguous (W in an input
// gradient, both operands of a weight gradient).  What it replaces at these places is a library product whose call costs the
// host 18 to 22 us - more than the product at small sizes - and whose weight gradients (few output tiles, a long sum) ran at 330 to
// 460 TFLOP/s.
//
// Two kernels, both with the operand tiles of a step of 32 k travelling straight into a ring of LDS slots (direct loads, requested
// several steps ahead) and a step's fragments read into registers while the products of the step before run, one barrier per step:
//   gemm_big_kernel  256 x 256 or 256 x 192 tiles, four waves, each alone on its SIMD with 128 x 128 (128 x 96) sums in the accumulation
//                    registers: the work of long products
//   gemm_kernel      128 x 128 and 64 x 64 tiles, two and more workgroups a CU: small products and short sums
// Tiles with k contiguous lie in LDS as rows of 64 bytes whose 16-byte chunks are XOR-swizzled, the others as [k][64] blocks that are
// read with LDS transpose reads (tile64_swz).  The products are computed transposed (rows of the matrix instruction are n) and the n
// of a row is chosen so that a lane holds eight consecutive columns of one output row.
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
    static_assert(NT % 2 == 0 && NT <= 4 && MT <= 4, "pairs of column tiles; what the fragment reads below are written out for");
};

// the large kernel's tiles: MT x NT tiles of 16 a wave, 2 x 2 waves; BRING slots in its ring
constexpr int BRING = 5;
template <int NT> struct BigTile {
    static constexpr int MT = 8, BM = 256, BN = 32 * NT;
    static constexpr int A_B = BM * GK * 2, B_B = BN * GK * 2, SLOT = A_B + B_B;
    static constexpr int AL = BM / 64, BL = BN / 64;                  // requests of a wave per step (1 KB each), A and B
};

__device__ __forceinline__ unsigned mask_from(int k, int K) { return k + 1 < K ? ~0u : k < K ? 0xFFFFu : 0u; }

// A wave's tile of 16 MT rows x 16 NT columns at (m0, n0) goes to memory: a lane holds, per row tile and column pair t, the columns 32 t + 8 lg .. + 7 of
// row lr.  Straight from there a store would hold 64 bytes of each of 16 rows; the tile goes through LDS instead and leaves as whole
// rows (16384 x 3072 from 64 columns, 256 x 256 tiles: 74 -> 42 us; 768 x 1536 over 16384 rows in ten slices 49 -> 41).  A wave of two column tiles stores them as they are: there the extra
// step costs more than it gives (128 x 256 over 1609 rows, seven slices 8.5 against 8.8 us).
// AGPR: the sums lie in accumulation registers.  LDS_B: bytes of smem, which nothing is on its way to.
template <typename T, int MT, int NT, bool F32, bool AGPR, int WAVES, int LDS_B>
__device__ __forceinline__ void store_tile(const bimamba2_gemm_params &p, f32x4 (&acc)[MT][NT], unsigned char *smem, int wave, int lane, int m0, int n0, int split) {
    constexpr int E = F32 ? 4 : 2, RCH = NT * E;              // bytes of a result, 16-byte chunks of a row
    const int lr = lane & 15, lg = lane >> 4;
    const int np = F32 ? (p.n + 7) & ~7 : p.n;
    float bias[NT / 2][8] = {};
    if (!F32 && p.bias) {
#pragma unroll
        for (int t = 0; t < NT / 2; ++t)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int n = n0 + t * 32 + 8 * lg + i;
                if (n < p.n) bias[t][i] = to_f(reinterpret_cast<const T *>(p.bias)[n]);
            }
    }
    auto rounded = [&](const f32x4 &lo, const f32x4 &hi, int t) __attribute__((always_inline)) {
        Vec16<T> v;
#pragma unroll
        for (int i = 0; i < 4; ++i) { v.v[i] = from_f<T>(lo[i] + bias[t][i]); v.v[4 + i] = from_f<T>(hi[i] + bias[t][4 + i]); }
        return v;
    };
    auto store = [&](int m, int n, const Vec16<T> &v) __attribute__((always_inline)) {
        if (m >= p.m || n >= np) return;
        if constexpr (F32) *reinterpret_cast<Vec16<T> *>(p.partial + ((int64_t)split * p.m + m) * np + n) = v;
        else {
            T *o = reinterpret_cast<T *>(p.c) + (int64_t)m * p.ldc + n;
            if (n + 8 <= p.n && p.ldc % 8 == 0) *reinterpret_cast<Vec16<T> *>(o) = v;
            else
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (n + j < p.n) o[j] = v.v[j];
        }
    };
    if constexpr (NT == 2) {
        const int n = n0 + 8 * lg, nn = min(8, p.n - n);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = m0 + mt * 16 + lr;
            if (m >= p.m || nn <= 0) continue;
            if constexpr (F32) {
                float *o = p.partial + ((int64_t)split * p.m + m) * np + n;
                *reinterpret_cast<f32x4 *>(o) = acc[mt][0];
                *reinterpret_cast<f32x4 *>(o + 4) = acc[mt][1];
            } else store(m, n, rounded(acc[mt][0], acc[mt][1], 0));
        }
    } else {
        constexpr int PITCH = RCH * 16 + 16;                  // (an odd number of chunks: 16 rows' chunks lie in different banks)
        constexpr int MG = WAVES * MT * 16 * PITCH <= LDS_B ? MT : MT / 2;      // row tiles at a time
        static_assert(WAVES * MG * 16 * PITCH <= LDS_B && MG * 16 * RCH % 64 == 0, "staging of the result");
        unsigned char *mine = smem + wave * (MG * 16 * PITCH);
        ordered_lds_barrier();                                // (the fragments that others read lie there)
        static_for<0, MT / MG>([&](auto GI) __attribute__((always_inline)) {
            constexpr int g = decltype(GI)::value;
#pragma unroll
            for (int q = 0; q < MG; ++q) {
                unsigned char *row = mine + (q * 16 + lr) * PITCH + lg * (8 * E);
#pragma unroll
                for (int t = 0; t < NT / 2; ++t) {
                    f32x4 &lo = acc[g * MG + q][2 * t], &hi = acc[g * MG + q][2 * t + 1];
                    if constexpr (AGPR) asm volatile("" : "+a"(lo), "+a"(hi));       // (they leave the accumulation registers here, not all at once)
                    if constexpr (F32) {
                        *reinterpret_cast<f32x4 *>(row + t * 128) = lo;
                        *reinterpret_cast<f32x4 *>(row + t * 128 + 16) = hi;
                    } else *reinterpret_cast<Vec16<T> *>(row + t * 64) = rounded(lo, hi, t);
                }
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll 8
            for (int i = 0; i < MG * 16 * RCH / 64; ++i) {
                const int id = i * 64 + lane, row = id / RCH, ch = id % RCH;
                store(m0 + g * MG * 16 + row, n0 + ch * (16 / E), *reinterpret_cast<const Vec16<T> *>(mine + row * PITCH + ch * 16));
            }
            __builtin_amdgcn_wave_barrier();
        });
    }
}

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
            BM2_RA(0); BM2_RA(1); BM2_RA(2); BM2_RA(3);
#undef BM2_RA
        } else {
            constexpr bool WHOLE = MT % 4 == 0;                // a wave owns whole 64-column blocks (else half of one)
            const unsigned blk = so + (unsigned)(wm * MT / 4) * 4096u;
            unsigned ta[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) ta[j] = (WHOLE ? a_l[j] : a_l[(j + 2 * (wm & 1)) & 3]) + blk;
#define BM2_RA(J)                                          \
    if constexpr (J < MT) {                                \
        f.al[J] = raw_lds_tr16_read_at<0>(ta[J]);          \
        f.ah[J] = raw_lds_tr16_read_at<512>(ta[J ^ 2]);    \
    }
            BM2_RA(0) BM2_RA(1) BM2_RA(2) BM2_RA(3)
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

    store_tile<T, MT, NT, F32, false, G::WAVES, GRING * G::SLOT>(p, acc, smem, wave, lane, m0 + wm * MT * 16, n0 + wn * NT * 16, split);
}

// acc += B A with the sums in accumulation registers
template <typename T, typename Frag> __device__ __forceinline__ void big_mma(Frag b, Frag a, f32x4 &acc) {
    if constexpr (std::is_same<T, bf16_t>::value) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}
// Wait states between these products and other instructions that touch their sums (the compiler does not know what the assembly holds)
template <int N, int MT, int NT> __device__ __forceinline__ void big_settle(f32x4 (&acc)[MT][NT]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("s_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j]));
    __builtin_amdgcn_sched_barrier(0);
}

// 256 x (32 NT) tiles.  What bounds it: the products of a step take 1024 (NT = 8) cycles of a SIMD's matrix unit and the step 1480 (8192 cubed: 765 us, 1437 TFLOP/s;
// the unit is busy 73 % of the time there, counted); a round of tiles adds 10 to 14 us of start, end and stores.  Four waves instead of the eight
// of 128 x 64 that stood here: a wave's fragments serve twice the products, and its sums fill the accumulation registers.  A wave that is
// alone on its SIMD covers nothing but by its own order: reads and requests stand one by one between the products (all of a row tile's in front of
// its eight products: 819 us at 8192 cubed, one behind each 778).  Steps of 64 with two slots: 802 us.  What it gives: gemm_plan.
template <typename T, int NT, bool AKC, bool BKC, bool F32>
__global__ __launch_bounds__(256, 1) void gemm_big_kernel(const bimamba2_gemm_params p, int mtiles, int ntiles, int kper) {
    typedef BigTile<NT> G;
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    constexpr int MT = G::MT, BM = G::BM, BN = G::BN, AL = G::AL, BL = G::BL;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[BRING * G::SLOT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4, wm = wave >> 1, wn = wave & 1;
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
    const bool ragged = K % GK != 0;

    // byte offset of this lane's 16 bytes of unit u in a k tile of which `left` k exist (what lies outside the matrix reads a valid neighbour)
    auto offset = [&](auto KC, auto ISB, unsigned ld, int valid, int u, int left) __attribute__((always_inline)) -> unsigned {
        if constexpr (decltype(KC)::value) {
            const int row = u * 16 + (lane >> 2), chunk = (lane & 3) ^ ((row >> 2) & 3);
            const int r = decltype(ISB)::value ? (row & ~31) + ((row & 12) << 1) + ((row & 16) >> 2) + (row & 3) : row;
            return __umul24(min(r, valid - 1), ld) + (unsigned)min(chunk * 8, (left - 1) & ~7) * 2;
        } else {
            const int row = (u & 3) * 8 + (lane >> 3), col = (u >> 2) * 64 + (((lane & 7) ^ tile64_swz(row)) << 3);
            return __umul24(min(row, left - 1), ld) + (unsigned)min(col, (valid - 1) & ~7) * 2;
        }
    };
    typedef std::integral_constant<bool, AKC> AKc;
    typedef std::integral_constant<bool, BKC> BKc;
    unsigned ao[AL], bo[BL];
    auto offsets = [&](int left) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < AL; ++i) ao[i] = offset(AKc(), std::false_type(), lda, mvalid, wave + 4 * i, left);
#pragma unroll
        for (int i = 0; i < BL; ++i) bo[i] = offset(BKc(), std::true_type(), ldb, nvalid, wave + 4 * i, left);
    };
    const unsigned astep = AKC ? GK * 2 : GK * lda, bstep = BKC ? GK * 2 : GK * ldb;
    // request i (0 .. AL + BL - 1) of step `it` into the slot at byte so
    auto request = [&](auto I, int it, unsigned so) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        if constexpr (i < AL) load16_to_lds_at(abase + (size_t)it * astep, ao[i], smem + so + (wave + 4 * i) * 1024);
        else load16_to_lds_at(bbase + (size_t)it * bstep, bo[i - AL], smem + so + G::A_B + (wave + 4 * (i - AL)) * 1024);
    };
    // The last step of a k that is no multiple of 32, once this wave's share of it has landed: the elements behind the end
    // become zero (what the loads found there may be an infinity, or no number at all).
    auto clear_tail = [&](unsigned so) __attribute__((always_inline)) {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        const int it = nk - 1, left = K - it * GK;
        const unsigned at = lds_addr(smem) + so + lane * 16;
#pragma unroll 1
        for (int u = wave; u < (BM + BN) / 16; u += 4) {
            const bool kc = u < BM / 16 ? AKC : BKC;
            const int k = kc ? ((lane & 3) ^ ((lane >> 4) & 3)) * 8 : (u & 3) * 8 + (lane >> 3);
            u32x4 v = raw_lds_read_at<u32x4, 0>(at + u * 1024);
            raw_lds_wait();
            raw_lds_use(v);
            if (kc) v &= u32x4{mask_from(k, left), mask_from(k + 2, left), mask_from(k + 4, left), mask_from(k + 6, left)};
            else if (k >= left) v = u32x4{0, 0, 0, 0};
            raw_lds_write128_at<0>(at + u * 1024, __builtin_bit_cast(f32x4, v));
        }
        raw_lds_wait();
    };

    const unsigned sb = lds_addr(smem);
    // fragment addresses in slot 0, k half 0
    unsigned a_l[4], b_l[4];
    if constexpr (AKC) {
        a_l[0] = sb + (wm * MT * 16 + lr) * 64 + ((lg ^ (lr >> 2)) << 4);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) a_l[j] = sb + (wm * 2) * 4096 + (tile64_tr_offset(8 * lg + (lr >> 2), 4 * (lr & 3)) ^ (j << 5));
    }
    if constexpr (BKC) {
        b_l[0] = sb + G::A_B + (wn * NT * 16 + lr) * 64 + ((lg ^ (lr >> 2)) << 4);
    } else {
        const unsigned b0 = sb + G::A_B + tile64_tr_offset(8 * lg + (lr >> 2), 8 * (lr & 3));
#pragma unroll
        for (int t = 0; t < NT / 2; ++t) {
            const int pair = wn * (NT / 2) + t;
            b_l[t] = (b0 ^ ((pair & 1) << 6)) + (pair >> 1) * 4096;
        }
    }
    struct Frags {
        Frag a[AKC ? MT : 1], b[BKC ? NT : 1];
        i16x4 al[AKC ? 1 : MT], ah[AKC ? 1 : MT], bl[BKC ? 1 : NT], bh[BKC ? 1 : NT];
    };
    // read i (B's first, then A's; two to a fragment whose k lies along the rows) of the slot at byte so
    constexpr int BR = BKC ? NT : 2 * NT, NR = BR + (AKC ? MT : 2 * MT);
    auto read1 = [&](auto I, Frags &f, unsigned so) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        if constexpr (i < BR) {
            if constexpr (BKC) f.b[i] = raw_lds_read_at<Frag, i * 1024>(b_l[0] + so);
            else {
                constexpr int j = i / 2, O = (j & 1) * 8;
                if constexpr (i % 2 == 0) f.bl[j] = raw_lds_tr16_read_at<O>(b_l[j >> 1] + so);
                else f.bh[j] = raw_lds_tr16_read_at<O + 512>((b_l[j >> 1] ^ 64u) + so);
            }
        } else {
            if constexpr (AKC) f.a[i - BR] = raw_lds_read_at<Frag, (i - BR) * 1024>(a_l[0] + so);
            else {
                constexpr int j = (i - BR) / 2, O = (j >> 2) * 4096;
                if constexpr (i % 2 == 0) f.al[j] = raw_lds_tr16_read_at<O>(a_l[j & 3] + so);
                else f.ah[j] = raw_lds_tr16_read_at<O + 512>(a_l[(j & 3) ^ 2] + so);
            }
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
    auto multiply1 = [&](auto I, Frags &f) __attribute__((always_inline)) {
        constexpr int mt = decltype(I)::value / NT, nt = decltype(I)::value % NT;
        Frag a, b;
        if constexpr (AKC) a = f.a[mt];
        else a = __builtin_bit_cast(Frag, __builtin_shufflevector(f.al[mt], f.ah[mt], 0, 1, 2, 3, 4, 5, 6, 7));
        if constexpr (BKC) b = f.b[nt];
        else b = __builtin_bit_cast(Frag, __builtin_shufflevector(f.bl[nt], f.bh[nt], 0, 1, 2, 3, 4, 5, 6, 7));
        big_mma<T>(b, a, acc[mt][nt]);
    };
    constexpr int NQ = AL + BL, NM = MT * NT;                 // requests and products of a step
    // Two steps' rows of 64 bytes make one cache line where k is contiguous: the requests of two steps go out side by side, every other step.
    constexpr bool PAIRS = AKC || BKC;
    constexpr int AHEAD = PAIRS ? 4 : BRING;
    const int last = nk - 1, left = K - last * GK;
    auto slot_of = [&](int it) __attribute__((always_inline)) { return (unsigned)(it % BRING) * G::SLOT; };
    auto next_slot = [&](unsigned so, int n) __attribute__((always_inline)) {
        const unsigned v = so + n * G::SLOT;
        return v >= BRING * G::SLOT ? v - BRING * G::SLOT : v;
    };
    big_settle<1>(acc);
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
        if (s < nk) {
            offsets(s == last ? left : GK);
            static_for<0, NQ>([&](auto I) __attribute__((always_inline)) { request(I, s, s * G::SLOT); });
        }
    if (last < AHEAD) wait_vmcnt<0>();
    else if constexpr (PAIRS) wait_vmcnt<(AHEAD - 2) * NQ>();
    else wait_vmcnt<(AHEAD - 1) * NQ>();
    if (ragged && last < AHEAD) clear_tail(slot_of(last));
    raw_lds_barrier();
    Frags fa, fb;
    static_for<0, NR>([&](auto I) __attribute__((always_inline)) { read1(I, fa, 0u); });
    unsigned so = 0;                                          // slot of step `it`
    auto step = [&](auto MORE, auto ODD, int it, Frags &cur, Frags &nxt) __attribute__((always_inline)) {
        constexpr bool more = decltype(MORE)::value, odd = decltype(ODD)::value;
        const unsigned sn = next_slot(so, 1);
        raw_lds_wait();
        if constexpr (!PAIRS || odd) {                        // the next step's tiles have landed
            constexpr int NEWER = PAIRS ? 1 : AHEAD - 2;
            if (more || (PAIRS ? it + 4 < last : it + 1 + NEWER < nk)) wait_vmcnt<NEWER * NQ>();
            else {
                wait_vmcnt<0>();
            }
        }
        if (!more && ragged && it == last - 1 && last >= AHEAD) clear_tail(sn);
        raw_lds_barrier();                                    // ... everybody's share of them; the slots of steps it and before are free
        use(cur);
        const unsigned s4 = next_slot(so, PAIRS ? (odd ? 3 : 4) : 0), s5 = PAIRS ? (odd ? next_slot(so, 4) : so) : so;
        const int i4 = it + (PAIRS ? (odd ? 3 : 4) : 5), i5 = it + (PAIRS && odd ? 4 : 5);
        // One read or request behind a product: the matrix unit is busy 16 cycles with it, and a wave alone on its SIMD has nothing else to cover them.
        static_for<0, NM>([&](auto J) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value;
            multiply1(J, cur);
            constexpr int SP = 3 * NM / 4, r = (j * NR + SP - 1) / SP;       // read r stands behind product r SP / NR
            if constexpr (r < NR && r * SP / NR == j) read1(std::integral_constant<int, r>(), nxt, sn);       // (behind the last step: not used)
            if constexpr (j % (NM / NQ) == NM / NQ - 1 && j / (NM / NQ) < NQ) {
                constexpr int i = j / (NM / NQ);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (PAIRS) {
                    constexpr int q = i + (odd ? NQ : 0);                    // of the pair's 2 NQ
                    if constexpr (q % 2 == 0) { if (more || i4 < last) request(std::integral_constant<int, q / 2>(), i4, s4); }
                    else if (more || i5 < last) request(std::integral_constant<int, q / 2>(), i5, s5);
                } else if (more || i4 < last) request(std::integral_constant<int, i>(), i4, s5);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        // the last step's requests, whose offsets differ where it is ragged (and whose place in the loop differs from tile to tile)
        if constexpr (!more && !(PAIRS && !odd)) {
            if ((PAIRS && i4 == last) || i5 == last) {
                offsets(left);
                static_for<0, NQ>([&](auto I) __attribute__((always_inline)) { request(I, last, PAIRS && i4 == last ? s4 : s5); });
            }
        }
        so = sn;
    };
    int it = 0;
    for (; it + 6 < last; it += 2) {
        step(std::true_type(), std::false_type(), it, fa, fb);
        step(std::true_type(), std::true_type(), it + 1, fb, fa);
    }
    for (; it < nk; it += 2) {
        step(std::false_type(), std::false_type(), it, fa, fb);
        if (it + 1 < nk) step(std::false_type(), std::true_type(), it + 1, fb, fa);
    }
    raw_lds_wait();
    use(fa);
    use(fb);
    big_settle<2>(acc);
    store_tile<T, MT, NT, F32, true, 4, BRING * G::SLOT>(p, acc, smem, wave, lane, m0 + wm * MT * 16, n0 + wn * NT * 16, split);
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
    int tile;        // 0: 256 x 256, 1: 256 x 192 (gemm_big_kernel), 2: 128 x 128, 3: 64 x 64 (gemm_kernel)
    int nsplit, kper;
};

struct GemmTileCost {
    int bm, bn, per_cu;
    double start_us, fixed_us, each_us;     // a round of workgroups: start and end, and per step fixed + each * (tiles that share the CU)
    double kcontig;                         // factor of a step where k is contiguous in an operand
    double slices_us;                       // the launch that adds the k slices up
    double crowd;                           // what c tiles that share a CU cost each other beyond that: factor 1 + crowd c (c - 1) of a step
};
// fitted to 360 products of layers of 128 to 1024 columns over 72 to 65536 rows with operands from memory, every tile and number of slices
// each.  Held against another 598 of layers of 128 to 4096 columns (weight gradients, and the input gradients and forward products that come here): the plan chosen
// takes 1.006 of the best one's time in the geometric mean, 1.08 at the 98th percentile, 1.21 at worst.  Against the plan with 128 x 128 tiles as the largest, 400
// weight gradients 0.85 (0.47 to 1.12, seven above 1.03: few columns over long sums, and 3000 rows where two slices more pay).  Without the crowd 64 x 64 tiles were
// taken for more of those: 1546 x 320 over 9110 rows 34.3 -> 29.3 us, 1286 x 192 over 19392 40.6 -> 36.1 (33.0 in eleven slices of 128 x 128).
constexpr GemmTileCost GEMM_TILES[4] = {{256, 256, 1, 3.1, 0.50, 0.12, 1.2, 8.5, 0.}, {256, 192, 1, 3.0, 0.40, 0.106, 1.4, 6.6, 0.},
                                        {128, 128, 2, 3.0, 0.22, 0.11, 1.4, 6.6, 0.}, {64, 64, 4, 3.3, 0.12, 0.08, 1.3, 3.5, 0.025}};

// Tile and number of k slices by the estimated time: per round of workgroups its start and end and its steps at the round's
// occupancy; for k slices the partial tiles that are written and read again (5 TB/s) and the launch that adds them.  us, with 128 x 128 tiles as
// the largest -> chosen now: 3224 x 768 over 16384 rows 111 (three slices) -> 88 (six of 256 x 256); 768 x 1536 60 (six) -> 54 (ten of
// 256 x 192); 4256 x 1024 over 65536 550 -> 493; 16384 x 768 from 3224 columns 105 (the library 82) -> 71, uncut in 256 x 192.
GemmPlan gemm_plan(const bimamba2_gemm_params *p) {
    const int64_t m = p->m, n = p->n, steps = (p->k + 31) / 32;
    GemmPlan best{3, 1, (int)steps * 32};
    double best_cost = 1e30;
    for (int t = 0; t < 4; ++t) {
        const GemmTileCost &c = GEMM_TILES[t];
        const double slow = p->a_kcontig ? c.kcontig : 1.0;
        const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn), slots = 256 * c.per_cu;
        for (int s = 1; s <= 16; ++s) {
            const int64_t per = (steps + s - 1) / s;
            if (s > 1 && (per < 8 || (steps + per - 1) / per != s)) continue;
            const int64_t full = tiles * s / slots, rest = tiles * s % slots;
            auto round = [&](int64_t wgs) {
                const int64_t share = (wgs + 255) / 256;
                return c.start_us + per * slow * (c.fixed_us + c.each_us * share) * (1. + c.crowd * (share * (share - 1)));
            };
            double cost = full * round(slots) + (rest ? round(rest) : 0.0);
            if (s > 1) cost += c.slices_us + (double)m * n * 8 * s / 5e6;
            if (cost < best_cost) { best_cost = cost; best = GemmPlan{t, s, (int)(per * 32)}; }
        }
    }
    return best;
}

template <typename T, int TILE, bool AKC, bool BKC, bool F32> int launch_gemm_tile(const bimamba2_gemm_params *p, const GemmPlan &g) {
    const GemmTileCost &c = GEMM_TILES[TILE];
    const int mt = (p->m + c.bm - 1) / c.bm, nt = (p->n + c.bn - 1) / c.bn;
    const dim3 grid((unsigned)(mt * nt * g.nsplit)), block(256);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
    if constexpr (TILE == 0) hipLaunchKernelGGL((gemm_big_kernel<T, 8, AKC, BKC, F32>), grid, block, 0, s, *p, mt, nt, g.kper);
    else if constexpr (TILE == 1) hipLaunchKernelGGL((gemm_big_kernel<T, 6, AKC, BKC, F32>), grid, block, 0, s, *p, mt, nt, g.kper);
    else if constexpr (TILE == 2) hipLaunchKernelGGL((gemm_kernel<T, 128, 128, 2, 2, AKC, BKC, F32>), grid, block, 0, s, *p, mt, nt, g.kper);
    else hipLaunchKernelGGL((gemm_kernel<T, 64, 64, 2, 2, AKC, BKC, F32>), grid, block, 0, s, *p, mt, nt, g.kper);
    return check_launch();
}

template <typename T, int TILE> int launch_gemm_form(const bimamba2_gemm_params *p, const GemmPlan &g) {
    const bool f32 = g.nsplit > 1;
    if (p->a_kcontig && p->b_kcontig) return f32 ? launch_gemm_tile<T, TILE, true, true, true>(p, g) : launch_gemm_tile<T, TILE, true, true, false>(p, g);
    if (p->a_kcontig) return f32 ? launch_gemm_tile<T, TILE, true, false, true>(p, g) : launch_gemm_tile<T, TILE, true, false, false>(p, g);
    if (!p->b_kcontig) return f32 ? launch_gemm_tile<T, TILE, false, false, true>(p, g) : launch_gemm_tile<T, TILE, false, false, false>(p, g);
    return BIMAMBA2_EUNSUPPORTED;
}

template <typename T> int launch_gemm_t(const bimamba2_gemm_params *p) {
    const GemmPlan g = gemm_plan(p);
    if (g.nsplit > 1 && !p->partial) return BIMAMBA2_EWORKSPACE;
    const int rc = g.tile == 0   ? launch_gemm_form<T, 0>(p, g)
                   : g.tile == 1 ? launch_gemm_form<T, 1>(p, g)
                   : g.tile == 2 ? launch_gemm_form<T, 2>(p, g)
                                 : launch_gemm_form<T, 3>(p, g);
    if (rc || g.nsplit == 1) return rc;
    const int64_t threads = (int64_t)p->m * ((p->n + 7) / 8);
    hipLaunchKernelGGL(gemm_reduce_kernel<T>, dim3((unsigned)((threads + NTHREADS - 1) / NTHREADS)), dim3(NTHREADS), 0,
                       reinterpret_cast<hipStream_t>(p->stream), *p, g.nsplit);
    return check_launch();
}

}  // namespace

void gemm_plan_of(const bimamba2_gemm_params *p, int *tile, int *slices) {
    const GemmPlan g = gemm_plan(p);
    *tile = g.tile;
    *slices = g.nsplit;
}

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
