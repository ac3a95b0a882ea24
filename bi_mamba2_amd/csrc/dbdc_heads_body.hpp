// The work of one workgroup of the dB / dC kernel (state parts) for 16-bit types, dstate 64 and headdim 64 or 128: a wave takes whole heads.
#pragma once
#include "common.hpp"
#include "dcb_heads_body.hpp"
#include "launch.hpp"

namespace bm2 {

// What dbdc_body.hpp describes, with the states in their 16-bit copies: a wave has 64 rows and takes every W-th head of its slice by itself, one
// direction after the other.  Its rows' B (C) values (64 registers) and the sums of dB (dC) (64) stay in registers over the heads, a product
// takes another 64; a head's x (dout) rows and a state tile come by direct loads into the wave's own 16 KB of LDS, the second direction's
// tile into the place of the first one's as soon as that has been read, the next head's operands behind them.  The waves' sums are added
// up in wave order at the end.  A wider head is taken 64 columns of it at a time: its pieces' products add up in the same registers.
// W waves share 64 rows, so a workgroup of four waves has 4 / W row tiles.
template <int W> struct DbdcHeadsMap {
    static constexpr int TILES = 4 / W, TILE = 64 * 64 * 2, RING = 2 * TILE;
    static constexpr int VEC = 4 * RING, VEC_WAVE = 7 * 64 * 4;       // per wave: row factors of both directions; cs_f, cs_b, dt of the head to come, cs_f and cs_b at the chunk's ends
    static constexpr int LDS = VEC + 4 * VEC_WAVE;
    static constexpr int COMB = W == 1 ? 0 : 4 * (W - 1) * (4 / W) * 4096;        // over the rings at the end, as in DcbHeadsMap
    static_assert(COMB <= VEC, "the exchange lies over the rings");
};

// PRODUCT: the part of dB (dC) inside the chunk, sum_t dCB[t, s] C[t, n] (sum_s dCB[t, s] B[s, n]), is formed here as well, the sums over the
// heads are added to it from their registers and the result leaves in its own type, with the bits that two launches give.  That takes one slice of heads,
// chunks of 256 and dCB in 16 bits, of which no transpose is needed: dC reads its tiles as they lie, dB by transpose reads.  The
// chunk's C (B) rows lie in the second halves of the four rings, 64 rows in each, for all waves; the 64 x 64 pieces of dCB in the first
// halves, W of a tile's four at a time, with one wave to a tile asked for under the last head and under the products.  Bound by
// memory with one wave to a tile (4 x 4096, 32 heads in 8 groups: 81 us, 71 without the product; 405 MB), by its waits else (16 x 1024, 24 heads: 40.9, 39.5 without).
// bid.x: (batch, chunk, group), bid.y: row tiles, bid.z: slice of hps heads
template <typename T, bool IS_DB, int W, bool PRODUCT>
__device__ __forceinline__ void bwd_dbdc_heads_body(const bimamba2_params &p, int nc, int nqt, int hps, BlockId bid, unsigned char *smem) {
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    typedef DbdcHeadsMap<W> L;
    static_assert(sizeof(T) == 2, "16-bit operands");
    constexpr int N = 64;
    const int P = p.headdim, np = P / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hw = wave % W, ti = wave / W;
    const int rt = bid.y * L::TILES + ti;
    const int g = bid.x % p.ngroups, bc = bid.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int r0 = rt * 64, valid = limit - r0;                       // rows of the tile inside the sequence
    const int hh0 = bid.z * hps, nhs = max(min(hpg, hh0 + hps) - hh0, 0), nhw = nhs > hw ? (nhs - hw + W - 1) / W : 0;
    const int h0 = g * hpg + hh0 + hw;
    const bool live = rt < nqt && valid > 0;
    const int nit = live ? nhw * np : 0;

    unsigned char *ring = smem + wave * L::RING, *vec = smem + L::VEC + wave * L::VEC_WAVE;
    const unsigned ring_a = lds_addr(ring), vec_a = lds_addr(vec);
    const int64_t cs_head = (int64_t)nc * Q * W;
    // ---- requests
    const char *xbase, *sf, *sb, *c1, *c2, *c3;
    unsigned x_bytes;
    int64_t x_head;
    {
        const T *xp;
        int64_t xs;
        if (IS_DB) { xs = p.x_sl; x_head = p.x_sh; xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * xs + h0 * x_head; }
        else if (p.has_z) { xs = (int64_t)H * P; x_head = P; xp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * xs + (int64_t)h0 * P; }
        else { xs = p.dout_sl; x_head = p.dout_sh; xp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * xs + h0 * x_head; }
        xbase = uniform_ptr(xp + r0 * xs);
        x_bytes = (unsigned)(xs * (int64_t)sizeof(T));
        const int64_t so = ((int64_t)(b * nc + c) * H + h0) * P * N;
        sf = uniform_ptr(reinterpret_cast<const T *>(IS_DB ? p.dstates16_f : p.states16_f) + so);
        sb = uniform_ptr(reinterpret_cast<const T *>(IS_DB ? p.dstates16_b : p.states16_b) + so);
        const int64_t o = (((int64_t)b * H + h0) * nc + c) * Q;
        c1 = uniform_ptr(p.cs_f + o);
        c2 = uniform_ptr(p.cs_b + o);
        c3 = uniform_ptr(p.dt_out + o);
    }
    // from a head's last piece to the first one of the wave's next head
    const int64_t x_wrap = (x_head * W - (np - 1) * 64) * (int64_t)sizeof(T), s_wrap = ((int64_t)P * W - (np - 1) * 64) * N * (int64_t)sizeof(T);
    int asked = 0, piece = 0;                      // of the head to come, of the one in hand
    // rows of 128 bytes to their place, 8 a request: 16-byte unit u of row r at u ^ r % 8
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
    // a state tile [p][n] for transpose reads: 16-byte unit u of row r at u ^ tile64_swz(r)
    auto request_state = [&](const char *base) __attribute__((always_inline)) {
        const int ln = lane_number(), r = ln >> 3;
#pragma unroll
        for (int k = 0; k < 8; ++k) load16_to_lds_at(base + k * 1024, r * 128 + (((ln & 7) ^ tile64_swz(k * 8 + r)) << 4), ring + L::TILE + k * 1024);
    };
    // the head's rows, its first state tile, the decays and dt of its rows
    auto request_head = [&]() __attribute__((always_inline)) {
        request_rows(xbase, x_bytes, valid, ring);
        request_state(sf);
        const unsigned ln = (unsigned)min(r0 + lane_number(), Q - 1) * 4;
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c1 + ln), (lds_ptr_t)(vec + 512), 4, 0, 0);
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c2 + ln), (lds_ptr_t)(vec + 768), 4, 0, 0);
        if (IS_DB) {
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c3 + ln), (lds_ptr_t)(vec + 1024), 4, 0, 0);
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(c1 + (Q - 1) * 4), (lds_ptr_t)(vec + 1280), 4, 0, 0);
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)c2, (lds_ptr_t)(vec + 1536), 4, 0, 0);
        }
        if (++asked < np) {
            xbase += 64 * sizeof(T);
            sf += 64 * N * sizeof(T);
        } else {
            asked = 0;
            c1 += cs_head * 4;
            c2 += cs_head * 4;
            c3 += cs_head * 4;
            xbase += x_wrap;
            sf += s_wrap;
        }
    };

    // ---- PRODUCT: this wave's 64 of the chunk's C (B) rows, and the piece of dCB at k rows (columns) that it brings
    const char *krows = nullptr, *cb = nullptr;
    if constexpr (PRODUCT) {
        const int k0 = min(wave * 64, limit - 1);
        krows = uniform_ptr(IS_DB ? reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + k0) * p.C_sl + g * p.C_sg
                                  : reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + k0) * p.B_sl + g * p.B_sg);
        cb = uniform_ptr(reinterpret_cast<const T *>(p.dCB) + (int64_t)bid.x * Q * Q + (IS_DB ? r0 : (int64_t)r0 * Q));
    }
    auto request_krows = [&]() __attribute__((always_inline)) {
        const int ln = lane_number(), r = ln >> 3, last = max(limit - 1 - wave * 64, 0);
        const unsigned stride = (unsigned)((IS_DB ? p.C_sl : p.B_sl) * (int64_t)sizeof(T));
#pragma unroll
        for (int k = 0; k < 8; ++k)
            load16_to_lds_at(krows, __umul24(min(k * 8 + r, last), stride) + (((ln & 7) ^ tile64_swz(k * 8 + r)) << 4), ring + L::TILE + k * 1024);
    };
    auto request_cb = [&](int piece) __attribute__((always_inline)) {      // (dB reads it transposed, dC as it lies)
        const int ln = lane_number(), r = ln >> 3;
        const char *base = cb + piece * (IS_DB ? 64 * 512 : 128);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            load16_to_lds_at(base + k * 8 * 512, r * 512 + (((ln & 7) ^ (IS_DB ? tile64_swz(k * 8 + r) : r)) << 4), ring + k * 1024);
    };

    // ---- this lane's B (C) values: row 16 q + 4 lg + i, column 16 j + lr; the rows pass through the ring
    f32x4 cr[4][4];
    f32x4 tot[4][4] = {};
    if (nit > 0) {
        const int64_t rs = (IS_DB ? p.B_sl : p.C_sl) * (int64_t)sizeof(T);
        const char *rows = uniform_ptr(IS_DB ? reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + ((int64_t)c * Q + r0) * p.B_sl + g * p.B_sg
                                             : reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + r0) * p.C_sl + g * p.C_sg);
        const int r = lane >> 3, u = ((lane & 7) ^ r) * 16;
        for (int k = 0; k < 8; ++k) load16_to_lds(rows + (min(k * 8 + r, valid - 1) * rs + u), ring + k * 1024);
        wait_vmcnt<0>();
        const int lr = lane & 15, lg = lane >> 4;
        const T *t = reinterpret_cast<const T *>(ring);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = q * 16 + lg * 4 + i, col = j * 16 + lr;
                    const float v = to_f(t[row * 64 + (((col >> 3) ^ (row & 7)) << 3) + (col & 7)]);
                    cr[q][j][i] = row < valid ? v : 0.f;
                }
        raw_lds_wait();
        request_head();
    }
    const int64_t uv0 = (((int64_t)b * H + h0) * nc + c) * Q + r0;
    float *uf = (IS_DB ? p.v_f : p.u_f) + uv0, *ub = (IS_DB ? p.v_b : p.u_b) + uv0;
    float part[2] = {0.f, 0.f};                    // of a row's sum: the head's pieces so far
#pragma unroll 1
    for (int it = 0; it < nit; ++it) {
        const int ln = lane_number(), lr = ln & 15, lg = ln >> 4;
        // what the head asked for has landed (younger is the store of the last sums of the head before it)
        if (it == 0) wait_vmcnt<0>();
        else wait_vmcnt<1>();
        {
            const unsigned a = vec_a + ln * 4;
            float f = raw_lds_read_at<float, 512>(a), r = raw_lds_read_at<float, 768>(a), d = 1.f, ef = 0.f, eb = 0.f;
            if (IS_DB) { d = raw_lds_read_at<float, 1024>(a); ef = raw_lds_read_at<float, 1280>(a); eb = raw_lds_read_at<float, 1536>(a); }
            raw_lds_wait();
            raw_lds_use(f); raw_lds_use(r);
            if (IS_DB) { raw_lds_use(d); raw_lds_use(ef); raw_lds_use(eb); }
            const bool in = ln < valid;
            raw_lds_write_at<0>(a, in ? (IS_DB ? d * __expf(ef - f) : __expf(f)) : 0.f);
            raw_lds_write_at<256>(a, in ? (IS_DB ? d * __expf(eb - r) : __expf(r)) : 0.f);
        }
        static_for<0, 2>([&](auto DIR) __attribute__((always_inline)) {
            constexpr int dir = decltype(DIR)::value;
            if (dir == 1) wait_vmcnt<1>();        // the second direction's tile (younger is the store of the first one's sums)
            const unsigned ta = ring_a + L::TILE, va = vec_a + dir * 256;
            const int kk = 8 * lg + (lr >> 2), nn = 4 * (lr & 3);
            float u[4];
            // 32 rows at a time (with 64 the product's registers are too many)
            static_for<0, 2>([&](auto HALF) __attribute__((always_inline)) {
                constexpr int q0 = 2 * decltype(HALF)::value;
                f32x4 acc[2][4];
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, 2>([&](auto KS) __attribute__((always_inline)) {
                    constexpr int ks = decltype(KS)::value;
                    const unsigned fa = ring_a + lr * 128 + (((ks * 4 + lg) ^ (ln & 7)) << 4);        // row 16 q + lr, unit 4 ks + lg
                    Frag x0 = raw_lds_read_at<Frag, q0 * 2048>(fa), x1 = raw_lds_read_at<Frag, q0 * 2048 + 2048>(fa);
                    // state fragments: rows (p) 32 ks + 8 lg .. + 7 of column 16 j + lr
                    i16x4 lo[4], hi[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        lo[j] = raw_lds_tr16_read_at<ks * 4096>(ta + tile64_tr_offset(kk, j * 16 + nn));
                        hi[j] = raw_lds_tr16_read_at<ks * 4096>(ta + tile64_tr_offset(kk + 4, j * 16 + nn));
                    }
                    raw_lds_wait();
                    raw_lds_use(x0); raw_lds_use(x1);
#pragma unroll
                    for (int j = 0; j < 4; ++j) { raw_lds_use(lo[j]); raw_lds_use(hi[j]); }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const Frag st = __builtin_bit_cast(Frag, __builtin_shufflevector(lo[j], hi[j], 0, 1, 2, 3, 4, 5, 6, 7));
                        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                        acc[0][j] = M::mma(x0, st, ks == 0 ? zero : acc[0][j]);
                        acc[1][j] = M::mma(x1, st, ks == 0 ? zero : acc[1][j]);
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
                // the tile has left the ring: the other direction's, or the next head's operands, take its place
                if (q0 == 2) {
                    if (dir == 0) {
                        request_state(sb);
                        sb += piece + 1 < np ? 64 * N * (int64_t)sizeof(T) : s_wrap;
                    } else if (it + 1 < nit) request_head();
                    else if (PRODUCT && W == 1) {                  // (nobody else's: the ring is this wave's until the barrier)
                        request_krows();
                        request_cb(0);
                    }
                }
                f32x4 s4[2] = {raw_lds_read_at<f32x4, q0 * 64>(va + lg * 16), raw_lds_read_at<f32x4, q0 * 64 + 64>(va + lg * 16)};
                raw_lds_wait();
                raw_lds_use(s4[0]); raw_lds_use(s4[1]);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    float w[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            w[i] = __builtin_fmaf(acc[k][j][i], cr[q0 + k][j][i], w[i]);
                            tot[q0 + k][j][i] = __builtin_fmaf(s4[k][i], acc[k][j][i], tot[q0 + k][j][i]);
                        }
                    // (pinned: the sums are not needed before the loop's end, and their additions would be moved there with the products they read)
#pragma unroll
                    for (int j = 0; j < 4; ++j) raw_lds_use(tot[q0 + k][j]);
                    u[q0 + k] = dpp_fold<0x141>(dpp_fold<0x128>(w[0], w[1], ln & 8), dpp_fold<0x128>(w[2], w[3], ln & 8), ln & 4);
                }
            });
            const int row = 8 * (ln & 2) + 32 * (ln & 1) + 4 * lg + ((ln >> 3) & 1) + ((ln >> 1) & 2);      // the row whose sum the folds leave here
            float srow = raw_lds_read_at<float, 0>(va + row * 4);
            raw_lds_wait();
            raw_lds_use(srow);
            const float v = dpp_fold<0xb1>(dpp_fold<0x4e>(u[0], u[1], ln & 2), dpp_fold<0x4e>(u[2], u[3], ln & 2), ln & 1) * srow;
            part[dir] = piece ? part[dir] + v : v;
            (dir ? ub : uf)[row] = row < valid ? part[dir] : 0.f;         // (without a branch: the waits count this store)
        });
        if (++piece == np) {
            piece = 0;
            uf += cs_head;
            ub += cs_head;
        }
    }
    // ---- the waves' shares are added up: wave hw owns the stripes q with q % W == hw
    const int le = lane_number(), lre = le & 15, lge = le >> 4;
    if constexpr (W > 1) {
        __syncthreads();
        f32x4 *comb = reinterpret_cast<f32x4 *>(smem) + le;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q % W != hw) {
                const int sl = hw < q % W ? hw : hw - 1;
#pragma unroll
                for (int j = 0; j < 4; ++j) comb[(((ti * 4 + q) * (W - 1) + sl) * 4 + j) * 64] = tot[q][j];
            }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q % W == hw) {
#pragma unroll
                for (int sl = 0; sl < W - 1; ++sl)
#pragma unroll
                    for (int j = 0; j < 4; ++j) tot[q][j] += comb[(((ti * 4 + q) * (W - 1) + sl) * 4 + j) * 64];
            }
    }
    if constexpr (PRODUCT) {
        if constexpr (W > 1) __syncthreads();      // (everybody has read the stripes)
        if (W > 1 || nit == 0) {
            request_krows();
            if (live) request_cb(hw);
        }
        const unsigned smem_a = lds_addr(smem);
        const int kk = 8 * lge + (lre >> 2), nn = 4 * (lre & 3);
        constexpr int NS = 4 / W;                  // this wave's stripes: 16 rows from 16 (W i + hw) on
        f32x4 inner[NS][4] = {};
#pragma unroll 1
        for (int step = 0; step < 4 / W; ++step) {
            wait_vmcnt<0>();
            if (W > 1 || step == 0) __syncthreads();
            if (live)
#pragma unroll 1
                for (int k = 0; k < W; ++k) {
                    const int kb = step * W + k;
                    const unsigned aa = smem_a + (ti * W + k) * L::RING, ka = smem_a + kb * L::RING + L::TILE;
                    static_for<0, 2>([&](auto KS) __attribute__((always_inline)) {
                        constexpr int ks = decltype(KS)::value;
                        Frag av[NS];
                        i16x4 alo[NS], ahi[NS], lo[4], hi[4];
#pragma unroll
                        for (int i = 0; i < NS; ++i) {
                            const int q = i * W + hw;
                            if constexpr (IS_DB) {
                                alo[i] = raw_lds_tr16_read_at<ks * 4096>(aa + tile64_tr_offset(kk, q * 16 + nn));
                                ahi[i] = raw_lds_tr16_read_at<ks * 4096>(aa + tile64_tr_offset(kk + 4, q * 16 + nn));
                            } else av[i] = raw_lds_read_at<Frag, 0>(aa + (q * 16 + lre) * 128 + (((ks * 4 + lge) ^ (le & 7)) << 4));
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            lo[j] = raw_lds_tr16_read_at<ks * 4096>(ka + tile64_tr_offset(kk, j * 16 + nn));
                            hi[j] = raw_lds_tr16_read_at<ks * 4096>(ka + tile64_tr_offset(kk + 4, j * 16 + nn));
                        }
                        raw_lds_wait();
#pragma unroll
                        for (int i = 0; i < NS; ++i)
                            if constexpr (IS_DB) { raw_lds_use(alo[i]); raw_lds_use(ahi[i]); }
                            else raw_lds_use(av[i]);
#pragma unroll
                        for (int j = 0; j < 4; ++j) { raw_lds_use(lo[j]); raw_lds_use(hi[j]); }
                        __builtin_amdgcn_sched_barrier(0);
                        if (W == 1 && ks == 1 && step + 1 < 4) request_cb(step + 1);       // (the piece has been read)
                        // rows behind the sequence hold its last one again
                        const int n = limit - kb * 64 - ks * 32 - 8 * lge;
                        if (kb * 64 + ks * 32 + 32 > limit)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    lo[j][i] = i < n ? lo[j][i] : (short)0;
                                    hi[j][i] = i + 4 < n ? hi[j][i] : (short)0;
                                }
#pragma unroll
                        for (int i = 0; i < NS; ++i) {
                            if constexpr (IS_DB) av[i] = __builtin_bit_cast(Frag, __builtin_shufflevector(alo[i], ahi[i], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                inner[i][j] = M::mma(av[i], __builtin_bit_cast(Frag, __builtin_shufflevector(lo[j], hi[j], 0, 1, 2, 3, 4, 5, 6, 7)), inner[i][j]);
                        }
                    });
                }
            if constexpr (W > 1) {
                __syncthreads();                   // (the tile's waves have read the pieces)
                if (live && step + 1 < 4 / W) request_cb((step + 1) * W + hw);
            }
        }
        if (!live) return;
        // out through this wave's piece of LDS as whole rows of 128 bytes; 16-byte unit u of row r at u ^ (r / 4) % 8
        const int64_t o_sl = (IS_DB ? p.dB_sl : p.dC_sl) ? (IS_DB ? p.dB_sl : p.dC_sl) : (int64_t)p.ngroups * N;
        const int64_t o_sb = (IS_DB ? p.dB_sl : p.dC_sl) ? (IS_DB ? p.dB_sb : p.dC_sb) : p.seqlen * o_sl;
        T *out = reinterpret_cast<T *>(IS_DB ? p.dB : p.dC) + b * o_sb + ((int64_t)c * Q + r0) * o_sl + (int64_t)g * N;
        T *img = reinterpret_cast<T *>(ring);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q % W == hw)
#pragma unroll
                for (int j = 0; j < 4; ++j) inner[q / W][j] += tot[q][j];
#pragma unroll
        for (int k = 0; k < NS; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = k * 16 + lge * 4 + i, s = j * 16 + lre;
                    img[t * 64 + (((s >> 3) ^ ((t >> 2) & 7)) << 3) + (s & 7)] = from_f<T>(inner[k][j][i]);
                }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 2 * NS; ++k) {
            const int t = k * 8 + (le >> 3), u = le & 7, r = ((k >> 1) * W + hw) * 16 + (k & 1) * 8 + (le >> 3);
            if (r < valid) *reinterpret_cast<f32x4 *>(out + r * o_sl + u * 8) = *reinterpret_cast<const f32x4 *>(img + t * 64 + ((u ^ ((t >> 2) & 7)) << 3));
        }
        return;
    }
    if (!live) return;
    float *out = (IS_DB ? p.dBs : p.dCs) + (int64_t)bid.z * p.batch * p.seqlen * p.ngroups * N;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q % W != hw) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = q * 16 + lge * 4 + i;
                if (r < valid) out[(((int64_t)b * p.seqlen + (int64_t)c * Q + r0 + r) * p.ngroups + g) * N + j * 16 + lre] = tot[q][j][i];
            }
    }
}

}  // namespace bm2
