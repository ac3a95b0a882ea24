// The work of one workgroup of the dCB kernel for 16-bit types with wide heads: a wave takes whole heads.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "dcb_body.hpp"
#include "launch.hpp"

namespace bm2 {

// What dcb_body.hpp describes, for headdim 64, chunk_size % 64 == 0 and aligned rows (16 bits): a wave has a whole 64x64 tile and takes
// every W-th head of its group by itself, so that between its start and its end there is no barrier and no exchange with other waves, the
// tile's sums over rows and columns end inside the wave (45 instructions a head and direction for 64 rows and columns), and a head's
// fixed costs - waits, reductions, stores - stand against 64 entries a lane.
//  * dCB (64 registers) and C.B^T (64) stay in registers over the heads, a head's G takes another 64 (253 in all: two waves a SIMD).
//  * A head's dout and x rows come by direct loads into the wave's own 16 KB of LDS and are asked for as soon as the head before them has
//    been read into registers.  Read from global memory straight into MFMA operands the same tiles took 44 us instead of 34 (512
//    tiles of 32 heads): there neighbouring lanes hold different rows, so each 16 bytes are a request of their own.
//  * Off the diagonal the decay is a row factor times a column factor about the tile's edge, so a position has one exponential.
// Bound by instruction issue: 480 vector instructions and 32 products (16 x 16 x 32) a head and wave off the diagonal, 1.25 us at two
// waves a SIMD, 1.45 with the loads.  (Counters of the launch with the state passing, 4 x 2048, 32 heads: vector units busy 58 % of the time, matrix
// units 11 %, LDS 22 %, 28 % of the waves' time waiting for an instruction; 8 groups of 4 heads, 4 x 4096: 46, 8, 23 and 25 %.)  16-row
// stripes of a tile to four waves, all of them on the same head with a barrier each (the kernel before this one): 51 us against 34 for 512 tiles of 32 heads, 134 against 88 for 8192 tiles of 4 (heads of 64, bfloat16).
// At headdim 128 a tile and head are 32 KB, and a wave waits for the second half of them: 88 us instead of 86 with the state passing (1024
// tiles of 16 heads), 70 without it; with 32 KB of LDS a wave, i.e. one workgroup a CU, 87 without it: such heads stay with that kernel.
// Errors against 64 bits are those of that kernel (the sums of a tile's heads are split over W waves and added up in wave order).
//
constexpr int DCB_HEADS_RESIDENT = 512;     // workgroups of the kernel that are on the chip at once: two a CU
// W waves share a 64x64 tile (t, s) of the (b, c, g) plane and take its heads in turn, so a workgroup of four waves has 4 / W tiles.
template <int W> struct DcbHeadsMap {
    static constexpr int TILES = 4 / W;
    static constexpr int TILE = 64 * 64 * 2, RING = 2 * TILE;         // per wave: a head's dout and x rows
    static constexpr int VEC = 4 * RING, VEC_WAVE = 10 * 64 * 4;      // per wave: vectors of the tile's 64 positions, the next head's decays and dt behind them
    static constexpr int LDS = VEC + 4 * VEC_WAVE;
    // over the rings at the end: stripes handed to their owners, then dCB and its transpose in 16 bits on their way out
    static constexpr int COMB = W == 1 ? 0 : 4 * (W - 1) * (4 / W) * 4096, IMG = W == 1 ? 0 : COMB;
    static_assert(IMG + TILES * 16384 <= VEC, "the way out lies over the rings");
};

// the lane's number, counted on the spot (a register that is held across a loop otherwise)
__device__ __forceinline__ int lane_number() {
    int n;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(n));
    return n;
}
template <int CTRL> __device__ __forceinline__ float dpp_of(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// One step of a sum over lanes that also picks: lanes with `second` set get the sums of b, the others those of a, over the lane and
// its partner (CTRL names the lane whose `second` is the other one).
template <int CTRL> __device__ __forceinline__ float dpp_fold(float a, float b, bool second) {
    return (second ? b : a) + dpp_of<CTRL>(second ? a : b);
}
// the four lanes l % 16, + 16, + 32, + 48 added up; lane group g gets the sum of v[g]
__device__ __forceinline__ float lanegroup_fold(const f32x4 &v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    auto fold32 = [](float a, float b) {
        const u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        const unsigned lo = r[0], hi = r[1];
        return __uint_as_float(lo) + __uint_as_float(hi);
    };
    const float a = fold32(v[0], v[2]), b = fold32(v[1], v[3]);
    const u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    const unsigned lo = r[0], hi = r[1];
    return __uint_as_float(lo) + __uint_as_float(hi);
}

// UNI: the single-direction operator - tiles above the diagonal are empty, tiles on it keep the forward half.
template <typename T, bool UNI, int W>
__device__ __forceinline__ void bwd_dcb_heads_body(const bimamba2_params &p, int nc, int nqt, BlockId bid, int gdx, int gdz, unsigned char *smem, bool out16) {
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    typedef DcbHeadsMap<W> L;
    static_assert(sizeof(T) == 2, "16-bit operands");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int hw = wave % W, ti = wave / W;
    // the tiles on the diagonal cost more: they come first in launch order, which spreads them over the compute units
    const int tid = bid.y * L::TILES + ti;
    const bool mine = tid < nqt * nqt;             // (else a place behind the last tile: with one tile a plane the division would be by zero)
    int tt = 0, st = 0;
    if (tid < nqt) tt = st = tid;
    else if (mine) {
        const int k = tid - nqt;
        tt = k / (nqt - 1);
        st = k % (nqt - 1);
        st += st >= tt;
    }
    const int tile = tt * nqt + st;
    const int g = bid.x % p.ngroups, bc = bid.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, P = p.headdim, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int t0 = tt * 64, s0 = st * 64;
    const int hps = (hpg + gdz - 1) / gdz;
    const int h_begin = bid.z * hps, h_end = min(hpg, h_begin + hps);
    const int nhs = max(h_end - h_begin, 0), nhw = nhs > hw ? (nhs - hw + W - 1) / W : 0;      // heads of the slice, of this wave
    const int h0 = g * hpg + h_begin + hw;
    const bool live = mine && t0 < limit && s0 < limit && !(UNI && st > tt);
    const int64_t tv_head = (int64_t)nc * nqt * nqt * DCB_VEC * W;
    float *tv = p.da_intra + ((((int64_t)b * H + h0) * nc + c) * nqt * nqt + tile) * DCB_VEC;
    f32x4 dcb[4][4] = {};
    if (mine && !live)
        for (int hh = 0; hh < nhw; ++hh) {
            tv[hh * tv_head + lane] = 0.f;
            tv[hh * tv_head + 64 + lane] = 0.f;
        }

    // ---- requests: a lane's rows of the two tiles are wave-uniform bases plus 32-bit offsets
    const int nit = live ? nhw : 0;
    const char *ybase, *xbase;
    unsigned y_bytes, x_bytes;                                 // of a row
    int64_t y_head;
    const char *c1, *c2, *c3;                                  // off the diagonal cs[t], cs[s], dt[s]; on it cs_f, cs_b, dt
    {
        const T *yp;
        int64_t y_row;
        if (p.has_z) { y_row = (int64_t)H * P; y_head = P; yp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * y_row + (int64_t)h0 * P; }
        else { y_row = p.dout_sl; y_head = p.dout_sh; yp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * y_row + h0 * p.dout_sh; }
        ybase = uniform_ptr(yp + t0 * y_row);
        xbase = uniform_ptr(reinterpret_cast<const T *>(p.x) + b * p.x_sb + ((int64_t)c * Q + s0) * p.x_sl + h0 * p.x_sh);
        y_bytes = (unsigned)(y_row * (int64_t)sizeof(T));
        x_bytes = (unsigned)(p.x_sl * (int64_t)sizeof(T));
        const int64_t o = (((int64_t)b * H + h0) * nc + c) * Q;
        const float *cs = st <= tt ? p.cs_f : p.cs_b;
        c1 = uniform_ptr(cs + o + t0);
        c2 = uniform_ptr((st == tt ? p.cs_b : cs) + o + s0);
        c3 = uniform_ptr(p.dt_out + o + s0);
    }
    const int64_t cs_head = (int64_t)nc * Q * W * 4;
    unsigned char *ring = smem + wave * L::RING, *vec = smem + L::VEC + wave * L::VEC_WAVE;
    const unsigned ring_a = lds_addr(ring), vec_a = lds_addr(vec);
    // 64 rows of 128 bytes from `base` (rows `stride` bytes apart, those from `valid` on are the last valid one again) by eight direct loads, 8
    // rows each, a row's 16 bytes to consecutive lanes; 16-byte unit u of row r lies at u ^ r % 8.
    auto request_rows = [&](const char *base, unsigned stride, int valid, unsigned char *to) __attribute__((always_inline)) {
        const int ln = lane_number();
        const unsigned r = ln >> 3, u = ((ln & 7) ^ r) * 16;
        if (valid >= 64) {
            const unsigned off = __umul24(r, stride) + u;
#pragma unroll
            for (int k = 0; k < 8; ++k) load16_to_lds_at(base + (size_t)k * 8 * stride, off, to + k * 1024);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) load16_to_lds_at(base, __umul24(min(k * 8 + r, (unsigned)valid - 1), stride) + u, to + k * 1024);
        }
    };
    // the same for C and B, whose row stride may be any; units: how many of a row's 16-byte units there are
    auto request_cb_rows = [&](const char *base, int64_t stride, int valid, unsigned char *to, int units) __attribute__((always_inline)) {
        const int ln = lane_number(), r = ln >> 3, u = min((ln & 7) ^ r, units - 1) * 16;
        for (int k = 0; k < 8; ++k) load16_to_lds(base + (min(k * 8 + r, valid - 1) * stride + u), to + k * 1024);
    };
    // the fragments' place: row r0 + l % 16, unit ks * 4 + l / 16
    auto frag_at = [&](int ln, int ks) __attribute__((always_inline)) { return ring_a + (ln & 15) * 128 + (((ks * 4 + (ln >> 4)) ^ (ln & 7)) << 4); };
    auto request = [&]() __attribute__((always_inline)) {
        request_rows(ybase, y_bytes, limit - t0, ring);
        request_rows(xbase, x_bytes, limit - s0, ring + L::TILE);
        const unsigned ln = lane_number() * 4;
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c1 + ln), (lds_ptr_t)(vec + 1792), 4, 0, 0);
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c2 + ln), (lds_ptr_t)(vec + 2048), 4, 0, 0);
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c3 + ln), (lds_ptr_t)(vec + 2304), 4, 0, 0);
        c1 += cs_head;
        c2 += cs_head;
        c3 += cs_head;
        ybase += y_head * W * (int64_t)sizeof(T);
        xbase += (int64_t)p.x_sh * W * (int64_t)sizeof(T);
    };
    // acc (+)= Y X^T over 64 columns in the ring
    auto ring_products = [&](f32x4 (&acc)[4][4], bool first, bool both) __attribute__((always_inline)) {
        const int ln = lane_number();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (ks == 1 && !both) break;
            const unsigned fa = frag_at(ln, ks);
            Frag xf0 = raw_lds_read_at<Frag, L::TILE>(fa), xf1 = raw_lds_read_at<Frag, L::TILE + 2048>(fa);
            Frag xf2 = raw_lds_read_at<Frag, L::TILE + 4096>(fa), xf3 = raw_lds_read_at<Frag, L::TILE + 6144>(fa);
            Frag y0 = raw_lds_read_at<Frag, 0>(fa), y1 = raw_lds_read_at<Frag, 2048>(fa), y2 = raw_lds_read_at<Frag, 4096>(fa), y3 = raw_lds_read_at<Frag, 6144>(fa);
            raw_lds_wait_n<3>();
            raw_lds_use(xf0); raw_lds_use(xf1); raw_lds_use(xf2); raw_lds_use(xf3); raw_lds_use(y0);
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            auto stripe = [&](f32x4 (&a)[4], const Frag &yf) __attribute__((always_inline)) {
                const bool z = ks == 0 && first;
                a[0] = M::mma(yf, xf0, z ? zero : a[0]);
                a[1] = M::mma(yf, xf1, z ? zero : a[1]);
                a[2] = M::mma(yf, xf2, z ? zero : a[2]);
                a[3] = M::mma(yf, xf3, z ? zero : a[3]);
            };
            stripe(acc[0], y0);
            raw_lds_wait();
            raw_lds_use(y1); raw_lds_use(y2); raw_lds_use(y3);
            stripe(acc[1], y1);
            stripe(acc[2], y2);
            stripe(acc[3], y3);
        }
    };

    // ---- C.B^T of the tile, every wave its own copy, in accumulator layout: 0 behind the end of the sequence
    f32x4 cbt[4][4] = {};
    if (nit > 0) {
        if (p.CB) {
            const float *cbg = p.CB + ((int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        cbt[q][j][i] = cbg[(int64_t)min(t0 + q * 16 + lg * 4 + i, limit - 1) * Q + min(s0 + j * 16 + lr, limit - 1)];
        } else {
            const char *cg = uniform_ptr(reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + t0) * p.C_sl + g * p.C_sg);
            const char *bg = uniform_ptr(reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + s0) * p.B_sl + g * p.B_sg);
            for (int n0 = 0; n0 < p.dstate; n0 += 64) {
                const int units = min(8, (p.dstate - n0) / 8);
                raw_lds_wait();
                request_cb_rows(cg + n0 * 2, p.C_sl * 2, limit - t0, ring, units);
                request_cb_rows(bg + n0 * 2, p.B_sl * 2, limit - s0, ring + L::TILE, units);
                wait_vmcnt<0>();
                ring_products(cbt, false, units > 4);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + q * 16 + lg * 4 + i >= limit || s0 + j * 16 + lr >= limit) cbt[q][j][i] = 0.f;
        raw_lds_wait();
        request();
    }

    f32x4 acc[4][4];
    // the products of a head; the next head's operands are requested into the ring as soon as the fragments have left it.  Younger than the
    // requests of the step in hand are the two stores of the head before it.
    auto all_products = [&](bool begin, bool more, float &d1, float &d2, float &d3) __attribute__((always_inline)) {
        if (begin) wait_vmcnt<0>();
        else wait_vmcnt<2>();
        const unsigned a = vec_a + lane_number() * 4;
        float e1 = raw_lds_read_at<float, 1792>(a), e2 = raw_lds_read_at<float, 2048>(a), e3 = raw_lds_read_at<float, 2304>(a);
        raw_lds_wait();
        raw_lds_use(e1); raw_lds_use(e2); raw_lds_use(e3);
        d1 = e1; d2 = e2; d3 = e3;
        ring_products(acc, true, true);
        if (more) request();
    };
    // sums over the 16 lanes of a row group: of a stripe's four rows i, then of the four stripes; the lane gets those of one row
    auto rows_of_stripe = [&](const float (&r)[4], int ln) __attribute__((always_inline)) {
        const bool b3 = ln & 8, b2 = ln & 4;
        return dpp_fold<0x141>(dpp_fold<0x128>(r[0], r[1], b3), dpp_fold<0x128>(r[2], r[3], b3), b2);      // row_half_mirror, row_ror:8
    };
    auto rows_of_tile = [&](const float (&u)[4], int ln) __attribute__((always_inline)) {
        const bool b1 = ln & 2, b0 = ln & 1;
        return dpp_fold<0xb1>(dpp_fold<0x4e>(u[0], u[1], b1), dpp_fold<0x4e>(u[2], u[3], b1), b0);         // quad_perm 1 0 3 2, 2 3 0 1
    };
    // which row that is
    auto row_of_lane = [&](int ln) __attribute__((always_inline)) { return 8 * (ln & 2) + 32 * (ln & 1) + 4 * (ln >> 4) + ((ln >> 3) & 1) + ((ln >> 1) & 2); };
    if (st != tt) {
        const int mref = st < tt ? 0 : min(63, limit - 1 - t0);
#pragma unroll 1
        for (int it = 0; it < nit; ++it) {
            float e1, e2, e3;
            all_products(it == 0, it + 1 < nit, e1, e2, e3);
            const int ln = lane_number();
            const int lr = ln & 15, lg = ln >> 4, row = row_of_lane(ln);
            const float ml = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e1), mref)) * LOG2E;
            const float el = t0 + ln < limit ? __builtin_amdgcn_exp2f(__builtin_fmaf(e1, LOG2E, -ml)) : 0.f;
            const float fl = s0 + ln < limit ? e3 * __builtin_amdgcn_exp2f(__builtin_fmaf(e2, -LOG2E, ml)) : 0.f;
            raw_lds_write_at<0>(vec_a + ln * 4, el);
            raw_lds_write_at<256>(vec_a + ln * 4, fl);
            const unsigned ra = vec_a + lg * 16, ca = vec_a + lr * 4;
            f32x4 E[4] = {raw_lds_read_at<f32x4, 0>(ra), raw_lds_read_at<f32x4, 64>(ra), raw_lds_read_at<f32x4, 128>(ra), raw_lds_read_at<f32x4, 192>(ra)};
            float F[4] = {raw_lds_read_at<float, 256>(ca), raw_lds_read_at<float, 320>(ca), raw_lds_read_at<float, 384>(ca), raw_lds_read_at<float, 448>(ca)};
            float erow = raw_lds_read_at<float, 0>(vec_a + row * 4);
            raw_lds_wait();
#pragma unroll
            for (int q = 0; q < 4; ++q) { raw_lds_use(E[q]); raw_lds_use(F[q]); }
            raw_lds_use(erow);
            float u[4];
            f32x4 col = {};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float rp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float a = acc[q][j][i], w = a * cbt[q][j][i];
                        col[j] = __builtin_fmaf(w, E[q][i], col[j]);
                        rp[i] = __builtin_fmaf(w, F[j], rp[i]);
                        dcb[q][j][i] = __builtin_fmaf(a * E[q][i], F[j], dcb[q][j][i]);
                    }
                u[q] = rows_of_stripe(rp, ln);
            }
            tv[ln] = lanegroup_fold(col) * fl;
            tv[64 + row] = rows_of_tile(u, ln) * erow;
            tv += tv_head;
        }
    } else {
#pragma unroll 1
        for (int it = 0; it < nit; ++it) {
            float e1, e2, e3;
            all_products(it == 0, it + 1 < nit, e1, e2, e3);
            const int ln = lane_number();
            const int lr = ln & 15, lg = ln >> 4, row = row_of_lane(ln);
            // Blocks off the tile's diagonal: the decay separates as above, about a reference point between columns and rows: the tile's
            // middle for its two quarters (half = 0), the middle of a half for the blocks beside the diagonal (1).  A position's factor is
            // a row factor on one side of the point and a column factor (with dt) on the other, so one vector holds both.
            const bool in_ = t0 + ln < limit;
            auto at = [&](float v, int l) __attribute__((always_inline)) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), min(l, limit - 1 - t0))); };
            const unsigned va = vec_a + ln * 4;
            const float dtl = in_ ? e3 : 0.f;
            raw_lds_write_at<0>(va, in_ ? e1 : 0.f);
            raw_lds_write_at<256>(va, in_ ? e2 : 0.f);
            raw_lds_write_at<512>(va, dtl);
            {
                const float mf = at(e1, 32) * LOG2E, mf1 = (ln < 32 ? at(e1, 16) : at(e1, 48)) * LOG2E;
                const float d0 = __builtin_fmaf(e1, LOG2E, -mf), d1 = __builtin_fmaf(e1, LOG2E, -mf1);
                raw_lds_write_at<768>(va, in_ ? (ln < 32 ? dtl * __builtin_amdgcn_exp2f(-d0) : __builtin_amdgcn_exp2f(d0)) : 0.f);
                raw_lds_write_at<1024>(va, in_ ? (!(ln & 16) ? dtl * __builtin_amdgcn_exp2f(-d1) : __builtin_amdgcn_exp2f(d1)) : 0.f);
                if (!UNI) {
                    const float mb = at(e2, 31) * LOG2E, mb1 = (ln < 32 ? at(e2, 15) : at(e2, 47)) * LOG2E;
                    const float r0 = __builtin_fmaf(e2, LOG2E, -mb), r1 = __builtin_fmaf(e2, LOG2E, -mb1);
                    raw_lds_write_at<1280>(va, in_ ? (ln >= 32 ? dtl * __builtin_amdgcn_exp2f(-r0) : __builtin_amdgcn_exp2f(r0)) : 0.f);
                    raw_lds_write_at<1536>(va, in_ ? (ln & 16 ? dtl * __builtin_amdgcn_exp2f(-r1) : __builtin_amdgcn_exp2f(r1)) : 0.f);
                }
            }
            const unsigned ra = vec_a + lg * 16, ca = vec_a + lr * 4;
            f32x4 colf = {}, colb = {};
            float uf[4], ub[4];
            static_for<0, 4>([&](auto QQ) __attribute__((always_inline)) {
                constexpr int q = decltype(QQ)::value;
                float df[4] = {0.f, 0.f, 0.f, 0.f}, db[4] = {0.f, 0.f, 0.f, 0.f};
                // the blocks of the other half of the columns (j0, j0 + 1), the one beside the diagonal in the same half (j2)
                constexpr bool FWD0 = q >= 2, FWD1 = q & 1;
                constexpr int j0 = FWD0 ? 0 : 2, j2 = q ^ 1, V0 = FWD0 ? 768 : 1280, V1 = (FWD1 ? 768 : 1280) + 256;
                f32x4 E0 = raw_lds_read_at<f32x4, V0 + q * 64>(ra), E1 = raw_lds_read_at<f32x4, V1 + q * 64>(ra);
                float F0 = raw_lds_read_at<float, V0 + j0 * 64>(ca), F1 = raw_lds_read_at<float, V0 + j0 * 64 + 64>(ca), F2 = raw_lds_read_at<float, V1 + j2 * 64>(ca);
                f32x4 tf = raw_lds_read_at<f32x4, q * 64>(ra), tb = raw_lds_read_at<f32x4, 256 + q * 64>(ra);
                float sf = raw_lds_read_at<float, q * 64>(ca), sb = raw_lds_read_at<float, 256 + q * 64>(ca), dts = raw_lds_read_at<float, 512 + q * 64>(ca);
                raw_lds_wait();
                raw_lds_use(E0); raw_lds_use(E1); raw_lds_use(F0); raw_lds_use(F1); raw_lds_use(F2);
                raw_lds_use(tf); raw_lds_use(tb); raw_lds_use(sf); raw_lds_use(sb); raw_lds_use(dts);
                auto block = [&](int j, const f32x4 &E, float F, f32x4 &col, float (&rp)[4]) __attribute__((always_inline)) {
                    float cp = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float a = acc[q][j][i], w = a * cbt[q][j][i];
                        cp = __builtin_fmaf(w, E[i], cp);
                        rp[i] = __builtin_fmaf(w, F, rp[i]);
                        dcb[q][j][i] = __builtin_fmaf(a * E[i], F, dcb[q][j][i]);
                    }
                    col[j] = __builtin_fmaf(cp, F, col[j]);
                };
                auto rows = [&](const f32x4 &E, const float (&rp)[4], float (&d)[4]) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) d[i] = __builtin_fmaf(rp[i], E[i], d[i]);
                };
                if constexpr (!UNI || FWD0) {
                    float rp[4] = {0.f, 0.f, 0.f, 0.f};
                    block(j0, E0, F0, FWD0 ? colf : colb, rp);
                    block(j0 + 1, E0, F1, FWD0 ? colf : colb, rp);
                    rows(E0, rp, FWD0 ? df : db);
                }
                if constexpr (!UNI || FWD1) {
                    float rp[4] = {0.f, 0.f, 0.f, 0.f};
                    block(j2, E1, F2, FWD1 ? colf : colb, rp);
                    rows(E1, rp, FWD1 ? df : db);
                }
                // the block on the diagonal: forward direction below it, reverse above it, both (factor 1) on it
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = lg * 4 + i;                 // row and column (lr) inside the block
                    float ex = __builtin_amdgcn_exp2f((lr < r ? tf[i] - sf : tb[i] - sb) * LOG2E);
                    if (lr == r) ex = UNI ? 1.f : 2.f;
                    if (UNI && lr > r) ex = 0.f;
                    if (t0 + q * 16 + r >= limit) ex = 0.f;
                    const float v = acc[q][q][i] * (ex * dts), w = v * cbt[q][q][i];
                    dcb[q][q][i] += v;
                    const float wf = lr < r ? w : 0.f, wb = lr > r ? w : 0.f;
                    df[i] += wf;
                    db[i] += wb;
                    colf[q] += wf;
                    colb[q] += wb;
                }
                uf[q] = rows_of_stripe(df, ln);
                if (!UNI) ub[q] = rows_of_stripe(db, ln);
            });
            const float rowf = rows_of_tile(uf, ln), rowb = UNI ? 0.f : rows_of_tile(ub, ln);
            raw_lds_write_at<0>(vec_a + row * 4, rowf);
            raw_lds_write_at<256>(vec_a + row * 4, rowb);
            float rwf = raw_lds_read_at<float, 0>(va), rwb = raw_lds_read_at<float, 256>(va);
            raw_lds_wait();
            raw_lds_use(rwf); raw_lds_use(rwb);
            tv[ln] = lanegroup_fold(colf) - rwf;
            tv[64 + ln] = UNI ? 0.f : lanegroup_fold(colb) - rwb;
            tv += tv_head;
        }
    }
    const int le = lane_number(), lre = le & 15, lge = le >> 4;
    // ---- the waves' shares of dCB are added up: wave hw owns the stripes q with q % W == hw
    if constexpr (W > 1) {
        __syncthreads();                           // (everybody is done with the C.B^T tiles)
        f32x4 *comb = reinterpret_cast<f32x4 *>(smem) + le;
        // stripe q of wave v: slot (v before q's owner ? v : v - 1) of that stripe
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q % W != hw) {
                const int sl = hw < q % W ? hw : hw - 1;
#pragma unroll
                for (int j = 0; j < 4; ++j) comb[(((ti * 4 + q) * (W - 1) + sl) * 4 + j) * 64] = dcb[q][j];
            }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q % W == hw) {
#pragma unroll
                for (int sl = 0; sl < W - 1; ++sl)
#pragma unroll
                    for (int j = 0; j < 4; ++j) dcb[q][j] += comb[(((ti * 4 + q) * (W - 1) + sl) * 4 + j) * 64];
            }
    }
    const int64_t oo = ((int64_t)bid.z * gdx + (int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
    if (!out16) {
        if (!mine) return;
        float *out = p.dCB + oo, *outT = p.dCBT + oo;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q % W != hw) continue;
            const int trow = t0 + q * 16 + lge * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int s = s0 + j * 16 + lre;
#pragma unroll
                for (int i = 0; i < 4; ++i) out[(int64_t)(trow + i) * Q + s] = dcb[q][j][i];
                *reinterpret_cast<f32x4 *>(outT + (int64_t)s * Q + trow) = dcb[q][j];
            }
        }
        return;
    }
    // dCB / dCBT in the element type of the inputs (inside bimamba2_bwd, one head slice: their one reader rounds them to that type
    // for its MFMA anyway, so nothing changes but the bytes moved), through LDS as whole rows of 128 bytes.  16-byte units of a row lie
    // at unit ^ (row / 4) % 8 (dCB, written four rows at a time) and unit ^ row % 8 (the transpose, where somebody reads it).
    T *img = reinterpret_cast<T *>(smem + L::IMG + ti * 16384), *imgT = img + 4096;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q % W != hw) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            T v4[4];
            const int t = q * 16 + lge * 4, s = j * 16 + lre;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v4[i] = from_f<T>(dcb[q][j][i]);
                img[(t + i) * 64 + (((s >> 3) ^ ((t >> 2) & 7)) << 3) + (s & 7)] = v4[i];
            }
            if (p.dCBT) *reinterpret_cast<uint2 *>(imgT + s * 64 + (((t >> 3) ^ (s & 7)) << 3) + (t & 7)) = *reinterpret_cast<const uint2 *>(v4);
        }
    }
    if constexpr (W > 1) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
    if (!mine) return;
    T *out = reinterpret_cast<T *>(p.dCB) + oo + (int64_t)t0 * Q + s0, *outT = reinterpret_cast<T *>(p.dCBT) + oo + (int64_t)s0 * Q + t0;
#pragma unroll
    for (int k = 0; k < 8 / W; ++k) {
        const int r = (hw * (8 / W) + k) * 8 + (le >> 3), u = le & 7;
        *reinterpret_cast<f32x4 *>(out + r * Q + u * 8) = *reinterpret_cast<const f32x4 *>(img + r * 64 + ((u ^ ((r >> 2) & 7)) << 3));
        if (p.dCBT) *reinterpret_cast<f32x4 *>(outT + r * Q + u * 8) = *reinterpret_cast<const f32x4 *>(imgT + r * 64 + ((u ^ (r & 7)) << 3));
    }
}

}  // namespace bm2
