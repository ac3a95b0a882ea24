// The work of one workgroup of the dCB kernels.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace bm2 {

// =========================================================================================================
// One workgroup owns one 64x64 tile (tt, st) of the chunk's (t, s) plane for one (b, c, g) and loops over the
// heads of the group; wave w owns rows 16w..16w+15 of the tile.  Per head, G[t,s] = dy_h[t,:] . x_h[s,:]
// (K = headdim; both operands are read from global memory straight into MFMA operand registers, the next
// K chunk being requested while the current one is multiplied), then
//   f[t,s] = 1[s<=t] G dt[s] e^{cs_f[t]-cs_f[s]},  b[t,s] = 1[s>=t] G dt[s] e^{cs_b[t]-cs_b[s]}
//   dCB[t,s] = sum_{h in group} (f + b)                       (kept in registers across the head loop)
//   W_f = 1[s<t] f CB,  W_b = 1[s>t] b CB                     (what the within-chunk gradient of dt*A is made of)
// The within-chunk gradient  da[i] = sum_{t>=i>s} W_f[t,s] + sum_{t<=i<s} W_b[t,s]  is assembled by the consumer
// (chunk_cumsum_bwd) from per-tile vectors written here to da_intra[b, h, c, tile, 2, 64]:
//   off-diagonal tile: [0] = column sums cw[s] = sum_t W,  [1] = row sums rw[t] = sum_s W
//   diagonal tile    : [0] = cw_f - rw_f, [1] = cw_b - rw_b of the tile's own W_f, W_b; the tile's contribution
//                      to da[i] is the exclusive prefix sum of [0] plus the exclusive suffix sum of [1]
//                      (da[i+1] - da[i] = cw_f[i] - rw_f[i] inside a tile; at most 64 terms, so the cancellation
//                      stays at float32 rounding level)
// One barrier per head (to combine the four waves' column sums); the decay vectors of up to DCB_HEADS heads are
// put into LDS beforehand.
// =========================================================================================================
constexpr int DCB_HEADS = 32;
constexpr int DCB_SLICE_HEADS = 32;     // heads per slice
constexpr int DCB_SLICES_MAX = 4;
constexpr int DCB_VEC = 2 * 64;      // floats per tile and head in da_intra

// Per head: turns the G tile (acc) into this head's share of dCB (added to dcb) and into the column / row sums of W that
// chunk_cumsum_bwd assembles.  cs = {cs_f[t], cs_b[t], cs_f[s], cs_b[s], dt[s]} of the tile (LDS), pb = exchange buffer
// of the four waves (LDS), tv = the (tile, head) slot of da_intra.  Contains one workgroup barrier.
template <typename T>
__device__ __forceinline__ void dcb_finish_head(f32x4 (&acc)[4], f32x4 (&dcb)[4], const f32x4 (&cbr)[4], const float (*cs)[64],
                                                float (*pb)[64], float *tv, const int (&tl)[4], int st, int tt) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15;
    float cft[4], cbt[4], dtv[4], cfs[4], cbs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        cft[i] = cs[0][tl[i]];
        cbt[i] = cs[1][tl[i]];
        cfs[i] = cs[2][i * 16 + lr];
        cbs[i] = cs[3][i * 16 + lr];
        dtv[i] = cs[4][i * 16 + lr];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
    }
    // column sums (this wave's 16 rows) and row sums of W; on the diagonal tile one pair per direction
    float cwa[4], cwb[4], rwa[4] = {0.f, 0.f, 0.f, 0.f}, rwb[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int sl = j * 16 + lr;
        float ca = 0.f, cb2 = 0.f;
        if (st != tt) {
            // one direction only: forward below the diagonal, reverse above it
            const float csv = st < tt ? cfs[j] : cbs[j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = acc[j][i] * dtv[j] * __expf((st < tt ? cft[i] : cbt[i]) - csv);
                dcb[j][i] += v;
                const float w = v * cbr[j][i];
                ca += w;
                rwa[i] += w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float gv = acc[j][i] * dtv[j];
                const float f = (sl <= tl[i]) ? gv * __expf(cft[i] - cfs[j]) : 0.f;
                const float r = (sl >= tl[i]) ? gv * __expf(cbt[i] - cbs[j]) : 0.f;
                dcb[j][i] += f + r;
                const float wf = (sl < tl[i]) ? f * cbr[j][i] : 0.f;
                const float wb = (sl > tl[i]) ? r * cbr[j][i] : 0.f;
                ca += wf; rwa[i] += wf;
                cb2 += wb; rwb[i] += wb;
            }
        }
        cwa[j] = ca;
        cwb[j] = cb2;
    }
    // hand the sums to the other waves through LDS (double-buffered by head parity)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float v = cwa[j];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (lane < 16) pb[wave][j * 16 + lane] = v;
        if (st == tt) {
            float u = cwb[j];
            u += __shfl_xor(u, 16, 64);
            u += __shfl_xor(u, 32, 64);
            if (lane < 16) pb[4 + wave][j * 16 + lane] = u;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float r = row16_sum(rwa[i]);
        if (lr == 0) pb[8][tl[i]] = r;
        if (st == tt) {
            const float u = row16_sum(rwb[i]);
            if (lr == 0) pb[9][tl[i]] = u;
        }
    }
    __syncthreads();
    // off-diagonal: [0] = column sums, [1] = row sums.  diagonal: [0] = cw_f - rw_f, [1] = cw_b - rw_b
    // (the consumer turns them into the tile's own contribution with a prefix resp. suffix sum)
    if (threadIdx.x < 128) {
        const int q = threadIdx.x & 63, which = threadIdx.x >> 6;
        const int base = (st != tt || which == 0) ? 0 : 4;
        float a0 = pb[base][q], a1 = pb[base + 1][q];
        float a2 = pb[base + 2][q], a3 = pb[base + 3][q];
        float r8 = pb[st != tt ? 8 : 8 + which][q];
            float v;
        if (st != tt) v = which == 0 ? a0 + a1 + a2 + a3 : r8;
        else v = a0 + a1 + a2 + a3 - r8;
        tv[which * 64 + q] = v;
    }
}

struct DcbMap {
    static constexpr int PART = 4 * DCB_HEADS * 5 * 64, LDS = PART + 4 * 2 * 10 * 64;
};
// lds: DcbMap::LDS bytes; bid / gdx / gdz: block index and grid extents (x: batch * chunks * groups, y: tiles, z: head slices)
template <typename T, bool FAST>
__device__ __forceinline__ void bwd_dcb_body(const bimamba2_params &p, int nc, int nqt, BlockId bid, int gdx, int gdz, char *lds) {
    typedef Mma<T> M;
    constexpr int KPL = M::KPL, KSTEP = M::KSTEP;
    constexpr int KC = sizeof(T) == 2 ? 64 : 16;          // K chunk held in registers
    constexpr int NKS = KC / KSTEP;
    float (*cst)[5][64] = reinterpret_cast<float (*)[5][64]>(lds);               // cs_f[t], cs_b[t], cs_f[s], cs_b[s], dt[s] per head
    float (*part)[10][64] = reinterpret_cast<float (*)[10][64]>(lds + DcbMap::PART);   // per-wave column sums (f: 0-3, b: 4-7), row sums (f: 8, b: 9)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    // bid.x = (b, c, g) varies fastest so that the tiles of one (b, c, g), which share x and dout rows, run on
    // the same XCD (workgroups are dealt round-robin to the 8 XCDs) and hit its L2
    const int tile = bid.y;
    const int tt = tile / nqt, st = tile % nqt;
    const int g = bid.x % p.ngroups, bc = bid.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, P = p.headdim, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int t0 = tt * 64, s0 = st * 64;
    const bool live = t0 < limit && s0 < limit;
    const float *cbg = p.CB + ((int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
    int tl[4];     // local row of this lane's accumulator elements
#pragma unroll
    for (int i = 0; i < 4; ++i) tl[i] = wave * 16 + lg * 4 + i;
    f32x4 cbr[4], dcb[4] = {};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + tl[i], s = s0 + j * 16 + lr;
            cbr[j][i] = (t < limit && s < limit) ? cbg[(int64_t)t * Q + s] : 0.f;   // 0 also masks rows / columns past the end
        }
    // operand rows of this lane: A = dy row t0 + 16 wave + lr; B = x rows s0 + 16 j + lr
    const int arow = min(t0 + wave * 16 + lr, limit - 1);
    int brow[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) brow[j] = min(s0 + j * 16 + lr, limit - 1);
    const int nkc = (P + KC - 1) / KC;
    // without FAST: whole vectors of the rows (unconditional loads from clamped addresses), or element by element
    const bool whole = !FAST && P % KPL == 0 && aligned16(reinterpret_cast<const T *>(p.x), p.x_sb | p.x_sl | p.x_sh) &&
                       (p.has_z ? aligned16(reinterpret_cast<const T *>(p.dout_x), P) : aligned16(reinterpret_cast<const T *>(p.dout), p.dout_sb | p.dout_sl | p.dout_sh));

    // bid.z selects a slice of the group's heads; its dCB partial sum goes to slice bid.z of the output
    const int hps = (hpg + gdz - 1) / gdz;
    const int h_begin = bid.z * hps, h_end = min(hpg, h_begin + hps);
    for (int hbase = h_begin; hbase < h_end; hbase += DCB_HEADS) {
        const int nh = min(DCB_HEADS, h_end - hbase);
        __syncthreads();
        for (int base = 0; base < nh * 5 * 64; base += NTHREADS * 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {                   // eight independent loads in flight per thread
                const int idx = base + u * NTHREADS + threadIdx.x;
                const int hh = idx / 320, which = (idx % 320) / 64, q = idx % 64;
                const int64_t o = (((int64_t)b * H + g * hpg + hbase + min(hh, nh - 1)) * nc + c) * Q;
                const int pos = min((which < 2 ? t0 : s0) + q, Q - 1);
                const float *src = which == 0 || which == 2 ? p.cs_f : (which == 4 ? p.dt_out : p.cs_b);
                v[u] = src[o + pos];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int idx = base + u * NTHREADS + threadIdx.x;
                if (idx < nh * 5 * 64) cst[idx / 320][(idx % 320) / 64][idx % 64] = v[u];
            }
        }
        __syncthreads();
        if (!live) {
            for (int hh = 0; hh < nh; ++hh) {
                const int64_t o = (((int64_t)b * H + g * hpg + hbase + hh) * nc + c);
                float *tv = p.da_intra + (o * nqt * nqt + tile) * DCB_VEC;
                for (int i = threadIdx.x; i < DCB_VEC; i += NTHREADS) tv[i] = 0.f;
            }
            continue;
        }
        // flattened loop over (head, K chunk) with two operand buffers
        typename M::Frag af[1][NKS], bf[1][4][NKS];        // operands in flight (next step)
        typename M::Frag afc[NKS], bfc[4][NKS];            // operands being multiplied
        const int nit = nh * nkc;
        auto issue = [&](int it) __attribute__((always_inline)) {
            constexpr int B_ = 0;
            const int hh = it / nkc, k0 = (it % nkc) * KC;
            const int h = g * hpg + hbase + hh;
            const T *yp;
            int64_t ys;
            if (p.has_z) { ys = (int64_t)H * P; yp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * ys + (int64_t)h * P; }
            else { ys = p.dout_sl; yp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * ys + h * p.dout_sh; }
            const T *xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * p.x_sl + h * p.x_sh;
            const T *ar = yp + (int64_t)arow * ys;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int kb = k0 + ks * KSTEP + lg * KPL;
                if (FAST) af[B_][ks] = M::load(ar + kb);
                else if (whole) {
                    af[B_][ks] = M::load(ar + min(kb, P - KPL));
                    if (kb >= P) af[B_][ks] = typename M::Frag{};
                } else {
                    float v[KPL];
#pragma unroll
                    for (int i = 0; i < KPL; ++i) v[i] = kb + i < P ? to_f(ar[kb + i]) : 0.f;
                    af[B_][ks] = M::pack(v);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const T *br = xp + (int64_t)brow[j] * p.x_sl;
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    const int kb = k0 + ks * KSTEP + lg * KPL;
                    if (FAST) bf[B_][j][ks] = M::load(br + kb);
                    else if (whole) {
                        bf[B_][j][ks] = M::load(br + min(kb, P - KPL));
                        if (kb >= P) bf[B_][j][ks] = typename M::Frag{};
                    } else {
                        float v[KPL];
#pragma unroll
                        for (int i = 0; i < KPL; ++i) v[i] = kb + i < P ? to_f(br[kb + i]) : 0.f;
                        bf[B_][j][ks] = M::pack(v);
                    }
                }
            }
        };
        f32x4 acc[4] = {};
        auto finish_head = [&](int hh) __attribute__((always_inline)) {
            const int64_t o = (((int64_t)b * H + g * hpg + hbase + hh) * nc + c);
            dcb_finish_head<T>(acc, dcb, cbr, cst[hh], part[hh & 1], p.da_intra + (o * nqt * nqt + tile) * DCB_VEC, tl, st, tt);
        };
        issue(0);
        for (int it = 0; it < nit; ++it) {
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                afc[ks] = af[0][ks];
#pragma unroll
                for (int j = 0; j < 4; ++j) bfc[j][ks] = bf[0][j][ks];
            }
            if (it + 1 < nit) issue(it + 1);                // requested now, needed in the next iteration
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                if (!FAST && (it % nkc) * KC + ks * KSTEP >= P) continue;      // (uniform) narrow heads
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = M::mma(afc[ks], bfc[j][ks], acc[j]);
            }
            if (it % nkc == nkc - 1) {
                // rows past the end of the sequence were read from a valid row: drop them
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + tl[i] >= limit) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[j][i] = 0.f;
                    }
                finish_head(it / nkc);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
    const int64_t oo = ((int64_t)bid.z * gdx + (int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
    float *out = p.dCB + oo, *outT = p.dCBT + oo;       // dCBT[s, t] = dCB[t, s], read by the dB product
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int s = s0 + j * 16 + lr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + tl[i];
            if (t < Q && s < Q) out[(int64_t)t * Q + s] = dcb[j][i];
        }
        if (s < Q) {
            if (t0 + tl[0] + 3 < Q && Q % 4 == 0) *reinterpret_cast<f32x4 *>(outT + (int64_t)s * Q + t0 + tl[0]) = dcb[j];
            else
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + tl[i] < Q) outT[(int64_t)s * Q + t0 + tl[i]] = dcb[j][i];
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// Variant for 16-bit types with headdim % 8 == 0, chunk_size % 64 == 0 and aligned operands (heads of 64: dcb_heads_body.hpp, but for the
// launches of several roles).
//
// The kernel is bound by its instruction count, not by memory, so everything per head is pared down:
//  * the dout tile, the x tile and the decay vectors of each (head, KC-wide headdim chunk) step travel from global memory
//    straight into a ring of LDS slots (global_load_lds, 16 bytes per lane, no registers, no address arithmetic beyond
//    one 64-bit add per request), one step ahead of the one being multiplied; 16-byte units are XOR-swizzled by the row
//    so that the fragment reads spread over the banks;
//  * a wave owns 16 rows t; against a block of 16 columns s that lies wholly below (s < t) or above (s > t) the diagonal
//    the decay factor separates, exp(cs[t] - cs[s]) = exp(cs[t] - m) * exp(m - cs[s]) with m taken at the edge of the
//    wave's rows nearest to the columns, so that both factors are <= 1 for A <= 0: 8 exponentials instead of 16 per
//    block and the factors move out of the row and column sums.  Only the 16x16 block on the diagonal takes the masked
//    two-direction path;
//  * the column sums over the four 16-lane groups come from one MFMA with a matrix of ones per column block.
// ---------------------------------------------------------------------------------------------------------
// sum of v over the four lanes l%16, l%16+16, l%16+32, l%16+48, delivered to all of them: D = ones(16x4) * B where lane l
// supplies B[k = l/16][n = l%16]
__device__ __forceinline__ float lanegroup_sum_mfma(float v) {
    const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x4f32(1.0f, v, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    return d[0];
}

// Slots of the ring.  Two (the step being multiplied and the one after it, requested right after the barrier that frees
// its slot) measured 60 us against 62 us for three slots requested two steps ahead.
constexpr int DCB_RING = 2;
constexpr int DCB_PART_B = 10 * 64 * 4;                   // per-wave column sums (f: 0-3, b: 4-7), row sums (f: 8, b: 9)


// UNI: the single-direction operator - tiles above the diagonal are empty, tiles on it keep the forward half.
// bid / gdx / gdz: block index and grid extents (x: batch * chunks * groups, y: tiles, z: head slices)
// Which (batch, chunk, group) and which tile the id-th workgroup of the dCB grid takes.  Workgroups are dealt round-robin to
// the 8 XCDs in id order, and the tiles of one (b, c, g) read the same dout and x rows (each row tile four times at chunk
// 256), so they belong on one XCD, close in time.  A grid that is resident all at once (up to
// `resident` workgroups) has (b, c, g) fastest: equal ids modulo 8 share an XCD, and all diagonal tiles, which cost more, come first and spread
// over the CUs.  A larger grid runs in several rounds, and with that order a row tile's readers are rounds apart and
// each fetches it from memory again (768 MB of reads at 8 groups of 4 heads, batch 4 x 4096; 172 -> 155 us): there
// eight (b, c, g) at a time, one per XCD, go through all their tiles before the next eight start.
__device__ __forceinline__ BlockId dcb_block_of(int id, int gdx, int ntiles, int nblocks, int resident = 1024) {
    if (nblocks <= resident || gdx % 8) return BlockId{id % gdx, id / gdx, 0};
    const int k = id >> 3;
    return BlockId{(k / ntiles) * 8 + (id & 7), k % ntiles, 0};
}

// KC: headdim columns per step, 64 (headdim above 32), or 32.  WHOLE: headdim is a multiple of it.  Otherwise (a multiple of 8) the
// rest of a row's units in LDS stays as it was cleared before the first request: a step with such a rest is always the same
// slot's (headdim <= 128, two slots), so nothing else is ever put there.
// smem: DcbRingMap<KC>::LDS bytes, 16-byte aligned
template <int KC> struct DcbRingMap {
    static constexpr int TILE = 64 * KC * 2;                   // one 64-row tile of 16-bit elements
    static constexpr int CS = 2 * TILE;                        // cs_f[t], cs_b[t], cs_f[s], cs_b[s], dt[s]: 5 x 64 floats
    static constexpr int SLOT = CS + 5 * 64 * 4, PART = DCB_RING * SLOT, LDS = PART + 2 * DCB_PART_B;
};
template <typename T, bool UNI, int KC, bool WHOLE>
__device__ __forceinline__ void bwd_dcb_ring_body(const bimamba2_params &p, int nc, int nqt, BlockId bid, int gdx, int gdz, unsigned char *smem, bool out16 = false) {
    typedef Mma<T> M;
    typedef typename M::Frag Frag;
    static_assert(sizeof(T) == 2 && DCB_RING == 2, "ring variant is for 16-bit operands");
    constexpr int NKS = KC / 32, UNITS = KC / 8;               // 16-byte units per row
    constexpr int DCB_TILE_B = DcbRingMap<KC>::TILE, DCB_CS_OFF = DcbRingMap<KC>::CS, DCB_SLOT_B = DcbRingMap<KC>::SLOT, DCB_PART_OFF = DcbRingMap<KC>::PART;
    // position of a row's unit among its units: neighbouring rows' accesses to one unit fall on different banks
    auto unit_at = [](int row, int unit) { return unit ^ (KC == 64 ? row & 7 : (row >> 1) & 3); };
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    // the tiles on the diagonal cost more: they come first in launch order, which spreads them over the compute units
    int tt, st;
    if (bid.y < nqt) tt = st = bid.y;
    else {
        const int k = bid.y - nqt;
        tt = k / (nqt - 1);
        st = k % (nqt - 1);
        st += st >= tt;
    }
    const int tile = tt * nqt + st;
    const int g = bid.x % p.ngroups, bc = bid.x / p.ngroups, c = bc % nc, b = bc / nc;
    const int Q = p.chunk_size, P = p.headdim, H = p.nheads, hpg = H / p.ngroups;
    const int limit = min(Q, p.seqlen - c * Q);
    const int t0 = tt * 64, s0 = st * 64;
    const int trow = wave * 16 + lg * 4;                       // first of this lane's four accumulator rows
    f32x4 cbr[4] = {}, dcb[4] = {};
    const int hps = (hpg + gdz - 1) / gdz;
    const int h_begin = bid.z * hps, h_end = min(hpg, h_begin + hps);
    const int nkc = (P + KC - 1) / KC, nhs = h_end - h_begin, nit = nhs * nkc;
    const int h0 = g * hpg + h_begin;
    // (a caller's dcb_slices may leave a slice without heads: it writes zeros and requests nothing, its h0 may lie behind the last head)
    const bool live = t0 < limit && s0 < limit && !(UNI && st > tt) && nhs > 0;
    const int64_t tv_head = (int64_t)nc * nqt * nqt * DCB_VEC;
    float *tv0 = p.da_intra + ((((int64_t)b * H + h0) * nc + c) * nqt * nqt + tile) * DCB_VEC;
    if (!live) {
        for (int hh = 0; hh < nhs; ++hh)
            for (int i = threadIdx.x; i < DCB_VEC; i += NTHREADS) tv0[hh * tv_head + i] = 0.f;
    } else {
        const unsigned sbase = lds_addr(smem);
        if constexpr (!WHOLE) {
            for (int i = threadIdx.x; i < DCB_PART_OFF / 16; i += NTHREADS) reinterpret_cast<f32x4 *>(smem)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            __syncthreads();
        }
        // ---- requests: unit u = i*256 + thread of a tile lies at position u % UNITS of row r = u / UNITS.
        // Addresses are a wave-uniform base (scalar registers, moved on from head to head) plus this lane's 32-bit byte offset
        // (the launcher checks that the rows of a chunk lie within 32 bits of each other): six vector registers less than
        // four per-lane pointers (126 registers instead of 138: four workgroups fit a CU where the grid has them).
        const char *ybase, *xbase;
        constexpr int NREQ = 64 * UNITS / NTHREADS;            // per thread and tile
        unsigned yoff[NREQ], xoff[NREQ];
        int ucol[NREQ];                                        // headdim column of the unit inside the step
        int64_t y_head, y_row;
        {
            const T *yp;
            if (p.has_z) { y_row = (int64_t)H * P; y_head = P; yp = reinterpret_cast<const T *>(p.dout_x) + ((int64_t)b * p.seqlen + (int64_t)c * Q) * y_row + (int64_t)h0 * P; }
            else { y_row = p.dout_sl; y_head = p.dout_sh; yp = reinterpret_cast<const T *>(p.dout) + b * p.dout_sb + (int64_t)c * Q * y_row + h0 * p.dout_sh; }
            const T *xp = reinterpret_cast<const T *>(p.x) + b * p.x_sb + (int64_t)c * Q * p.x_sl + h0 * p.x_sh;
            ybase = uniform_ptr(yp);
            xbase = uniform_ptr(xp);
#pragma unroll
            for (int i = 0; i < NREQ; ++i) {
                const int u = i * NTHREADS + threadIdx.x, r = u / UNITS, col = unit_at(r, u % UNITS) * 8;
                ucol[i] = col;
                yoff[i] = (unsigned)(((int64_t)min(t0 + r, limit - 1) * y_row + col) * (int64_t)sizeof(T));
                xoff[i] = (unsigned)(((int64_t)min(s0 + r, limit - 1) * p.x_sl + col) * (int64_t)sizeof(T));
            }
        }
        const float *csrc;                                     // threads 0..79: 16-byte unit of the five decay vectors
        {
            const int which = min((int)threadIdx.x >> 4, 4), j4 = (threadIdx.x & 15) * 4;
            const int64_t o = (((int64_t)b * H + h0) * nc + c) * Q + (which < 2 ? t0 : s0) + j4;
            csrc = (which == 0 || which == 2 ? p.cs_f : (which == 4 ? p.dt_out : p.cs_b)) + o;
        }
        const int64_t x_head = p.x_sh, cs_head = (int64_t)nc * Q;
        int ikc = 0;
        // requests one step into `slot` and moves the source pointers on to the next step
        auto issue = [&](int slot) __attribute__((always_inline)) {
            unsigned char *sl = smem + slot * DCB_SLOT_B + wave * 1024;
            if constexpr (WHOLE) {
#pragma unroll
                for (int i = 0; i < NREQ; ++i) load16_to_lds_at(ybase, yoff[i], sl + i * 4096);
#pragma unroll
                for (int i = 0; i < NREQ; ++i) load16_to_lds_at(xbase, xoff[i], sl + DCB_TILE_B + i * 4096);
            } else {
#pragma unroll
                for (int i = 0; i < NREQ; ++i)
                    if (ikc * KC + ucol[i] < P) {
                        load16_to_lds_at(ybase, yoff[i], sl + i * 4096);
                        load16_to_lds_at(xbase, xoff[i], sl + DCB_TILE_B + i * 4096);
                    }
            }
            if (threadIdx.x < 80) __builtin_amdgcn_global_load_lds((gbl_ptr_t)csrc, (lds_ptr_t)(sl + DCB_CS_OFF), 16, 0, 0);
            const bool last = ++ikc == nkc;
            if (last) ikc = 0;
            const int64_t dy = last ? y_head - (nkc - 1) * KC : KC, dx = last ? x_head - (nkc - 1) * KC : KC;
            ybase += dy * (int64_t)sizeof(T);
            xbase += dx * (int64_t)sizeof(T);
            if (last) csrc += cs_head;
        };
        // ---- per-lane LDS byte offsets inside a slot
        unsigned a_off[NKS], b_off[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int ch = unit_at(lr, ks * 4 + lg);
            a_off[ks] = ((wave * 16 + lr) * UNITS + ch) * 16;
            b_off[ks] = DCB_TILE_B + (lr * UNITS + ch) * 16;   // column block j adds j * 16 rows
        }
        const unsigned ct_off = DCB_CS_OFF + trow * 4, cc_off = DCB_CS_OFF + lr * 4, cm_off = DCB_CS_OFF + wave * 64;
        const int rows_left = limit - t0 - trow;               // accumulator rows i >= rows_left lie past the sequence end

        f32x4 acc[4] = {};
        issue(0);
        if (DCB_RING > 2 && nit > 1) issue(1);
        if (p.CB) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float *cbg = p.CB + ((int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = t0 + trow + i, s = s0 + j * 16 + lr;
                    cbr[j][i] = (t < limit && s < limit) ? cbg[(int64_t)t * Q + s] : 0.f;
                }
            }
        } else {
            // no CB given: the tile CB[t, s] = C_t . B_s is rebuilt here, once per workgroup; both operands are read from
            // global memory in MFMA layout (dstate is contiguous) and the product lands in the layout of cbr
            const T *crow = reinterpret_cast<const T *>(p.Cm) + b * p.C_sb + ((int64_t)c * Q + min(t0 + wave * 16 + lr, limit - 1)) * p.C_sl + g * p.C_sg + lg * 8;
            const T *brow = reinterpret_cast<const T *>(p.Bm) + b * p.B_sb + (int64_t)c * Q * p.B_sl + g * p.B_sg + lg * 8;
            for (int n0 = 0; n0 < p.dstate; n0 += 32) {
                const Frag cf = M::load(crow + n0);
#pragma unroll
                for (int j = 0; j < 4; ++j) cbr[j] = M::mma(cf, M::load(brow + (int64_t)min(s0 + j * 16 + lr, limit - 1) * p.B_sl + n0), cbr[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + trow + i >= limit || s0 + j * 16 + lr >= limit) cbr[j][i] = 0.f;
        }
        // settle these register loads here: inside the loop a wait for them would drain the ring's requests as well
        wait_vmcnt<0>();
        int slot = 0, slot2 = (DCB_RING - 1) % DCB_RING, kc = 0, par = 0;
        float *tv = tv0 + (wave & 1) * 64 + lane;
        // the sums of a head are written out one iteration later, after the barrier that the next step needs anyway
        // (waves 0 and 1; off-diagonal: [0] = column sums, [1] = row sums.  diagonal: [0] = cw_f - rw_f, [1] = cw_b - rw_b,
        // which the consumer turns into the tile's own contribution with a prefix resp. suffix sum)
        bool pending = false;
        auto write_out = [&](int pbuf) __attribute__((always_inline)) {
            if (wave < 2) {
                const unsigned pq = sbase + DCB_PART_OFF + pbuf * DCB_PART_B + lane * 4;
                float v;
                if (st != tt && wave == 1) {
                    v = raw_lds_read_at<float, 2048>(pq);
                    raw_lds_wait();
                    raw_lds_use(v);
                } else {
                    float a0, a1, a2, a3, r8 = 0.f;
                    if (wave == 0) {
                        a0 = raw_lds_read_at<float, 0>(pq); a1 = raw_lds_read_at<float, 256>(pq);
                        a2 = raw_lds_read_at<float, 512>(pq); a3 = raw_lds_read_at<float, 768>(pq);
                        if (st == tt) r8 = raw_lds_read_at<float, 2048>(pq);
                    } else {
                        a0 = raw_lds_read_at<float, 1024>(pq); a1 = raw_lds_read_at<float, 1024 + 256>(pq);
                        a2 = raw_lds_read_at<float, 1024 + 512>(pq); a3 = raw_lds_read_at<float, 1024 + 768>(pq);
                        r8 = raw_lds_read_at<float, 2048 + 256>(pq);
                    }
                    raw_lds_wait();
                    raw_lds_use(a0); raw_lds_use(a1); raw_lds_use(a2); raw_lds_use(a3); raw_lds_use(r8);
                    v = a0 + a1 + a2 + a3 - r8;
                }
                *tv = v;
            }
            tv += tv_head;
        };
        // The head loop is compiled once per kind of tile: off the diagonal (KIND = -1), and on it once per wave (KIND = the
        // wave's index, which decides for every column block whether it lies below, on or above the wave's rows), so that
        // none of these decisions is taken, and no register moved to a common place, inside the loop.
        auto run = [&](auto TILE_KIND) __attribute__((always_inline)) {
            constexpr int KIND = decltype(TILE_KIND)::value;
            constexpr bool DIAG = KIND >= 0;
            constexpr bool LOWER = KIND == -1;             // off the diagonal: -1 below it (forward direction), -2 above
        for (int it = 0; it < nit; ++it) {
            // with two slots nothing but step `it` is outstanding here; with more, the requests of step `it` went out before
            // those of the step after it (waves 0 and 1 make five requests per step, the others four)
            if (DCB_RING > 2 && it + 1 < nit) {
                if (wave < 2) wait_vmcnt<5>();
                else wait_vmcnt<4>();
            } else {
                wait_vmcnt<0>();
            }
            raw_lds_barrier();     // step `it` has landed for everybody; every wave is done with the slot and the sums of step it - 1
            // (the store of the sums goes out before the requests: the wait at the top of the next step counts on the
            // requests of the step after it being this wave's youngest operations)
            if (pending) {
                write_out(par ^ 1);
                pending = false;
            }
            if (it + DCB_RING - 1 < nit) issue(slot2);
            const unsigned sb = sbase + slot * DCB_SLOT_B;
            Frag af[NKS], bf[4][NKS];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                af[ks] = raw_lds_read_at<Frag, 0>(sb + a_off[ks]);
                bf[0][ks] = raw_lds_read_at<Frag, 0>(sb + b_off[ks]);
                bf[1][ks] = raw_lds_read_at<Frag, 256 * UNITS>(sb + b_off[ks]);
                bf[2][ks] = raw_lds_read_at<Frag, 512 * UNITS>(sb + b_off[ks]);
                bf[3][ks] = raw_lds_read_at<Frag, 768 * UNITS>(sb + b_off[ks]);
            }
            raw_lds_wait();
            // (the first product of a head starts from a literal zero: no registers to clear between heads)
            const bool first = kc == 0;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                raw_lds_use(af[ks]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    raw_lds_use(bf[j][ks]);
                    if (ks == 0 && first) acc[j] = M::mma(af[ks], bf[j][ks], f32x4{0.f, 0.f, 0.f, 0.f});
                    else acc[j] = M::mma(af[ks], bf[j][ks], acc[j]);
                }
            }
            if (++kc == nkc) {
                kc = 0;
                // ---- decay vectors of this head (off the diagonal only the ones of the tile's direction)
                f32x4 cft_, cbt_;
                float cfs[4], cbs[4], dts[4], mf, mb;
                if constexpr (DIAG || LOWER) {
                    cft_ = raw_lds_read_at<f32x4, 0>(sb + ct_off);
                    cfs[0] = raw_lds_read_at<float, 512>(sb + cc_off); cfs[1] = raw_lds_read_at<float, 512 + 64>(sb + cc_off);
                    cfs[2] = raw_lds_read_at<float, 512 + 128>(sb + cc_off); cfs[3] = raw_lds_read_at<float, 512 + 192>(sb + cc_off);
                    mf = raw_lds_read_at<float, 0>(sb + cm_off);           // reference point: cs_f at the first of the wave's 16 rows
                }
                if constexpr (DIAG || !LOWER) {
                    cbt_ = raw_lds_read_at<f32x4, 256>(sb + ct_off);
                    cbs[0] = raw_lds_read_at<float, 768>(sb + cc_off); cbs[1] = raw_lds_read_at<float, 768 + 64>(sb + cc_off);
                    cbs[2] = raw_lds_read_at<float, 768 + 128>(sb + cc_off); cbs[3] = raw_lds_read_at<float, 768 + 192>(sb + cc_off);
                    mb = raw_lds_read_at<float, 256 + 60>(sb + cm_off);    // cs_b at the last of them
                }
                dts[0] = raw_lds_read_at<float, 1024>(sb + cc_off); dts[1] = raw_lds_read_at<float, 1024 + 64>(sb + cc_off);
                dts[2] = raw_lds_read_at<float, 1024 + 128>(sb + cc_off); dts[3] = raw_lds_read_at<float, 1024 + 192>(sb + cc_off);
                raw_lds_wait();
                if constexpr (DIAG || LOWER) {
                    raw_lds_use(cft_); raw_lds_use(mf);
#pragma unroll
                    for (int j = 0; j < 4; ++j) raw_lds_use(cfs[j]);
                }
                if constexpr (DIAG || !LOWER) {
                    raw_lds_use(cbt_); raw_lds_use(mb);
#pragma unroll
                    for (int j = 0; j < 4; ++j) raw_lds_use(cbs[j]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) raw_lds_use(dts[j]);
                if (rows_left < 4) {
                    // rows past the end of the sequence were read from a valid row: drop them
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i >= rows_left) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) acc[j][i] = 0.f;
                        }
                }
                // W = dCB_h * CB; col*[j]: this lane's part of the column sums, row*[i]: of the row sums
                float colF[4], colB[4] = {0.f, 0.f, 0.f, 0.f}, rowF[4], rowB[4] = {0.f, 0.f, 0.f, 0.f};
                // one 16 x 16 block whose columns lie on one side of the wave's rows: factors E (rows) and Fd (columns)
                auto sep_block = [&](int j, const float (&E)[4], float Fd, float &col, float (&rp)[4]) __attribute__((always_inline)) {
                    float cp = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float a = acc[j][i], y = a * cbr[j][i];
                        cp = __builtin_fmaf(y, E[i], cp);
                        rp[i] = __builtin_fmaf(y, Fd, rp[i]);
                        dcb[j][i] = __builtin_fmaf(a * E[i], Fd, dcb[j][i]);
                    }
                    col = cp * Fd;
                };
                if constexpr (!DIAG) {
                    // forward direction below the diagonal, reverse above it
                    float E[4], rp[4] = {0.f, 0.f, 0.f, 0.f};
                    const float ml = (LOWER ? mf : mb) * LOG2E;
#pragma unroll
                    for (int i = 0; i < 4; ++i) E[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(LOWER ? cft_[i] : cbt_[i], LOG2E, -ml));
#pragma unroll
                    for (int j = 0; j < 4; ++j) sep_block(j, E, dts[j] * __builtin_amdgcn_exp2f(__builtin_fmaf(LOWER ? cfs[j] : cbs[j], -LOG2E, ml)), colF[j], rp);
#pragma unroll
                    for (int i = 0; i < 4; ++i) rowF[i] = rp[i] * E[i];
                } else {
                    float Ef[4], Eb[4], rpf[4] = {0.f, 0.f, 0.f, 0.f}, rpb[4] = {0.f, 0.f, 0.f, 0.f};
                    float df[4] = {0.f, 0.f, 0.f, 0.f}, db[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < 4; ++i) { Ef[i] = __expf(cft_[i] - mf); Eb[i] = __expf(cbt_[i] - mb); }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (j < KIND) { sep_block(j, Ef, dts[j] * __expf(mf - cfs[j]), colF[j], rpf); }
                        else if (j > KIND) { colF[j] = 0.f; if (!UNI) sep_block(j, Eb, dts[j] * __expf(mb - cbs[j]), colB[j], rpb); }
                        else {
                            // the block on the diagonal: both directions, masked element by element
                            float ca = 0.f, cb2 = 0.f;
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const int ti = lg * 4 + i;     // row and column (lr) inside the block
                                const float gv = acc[j][i] * dts[j];
                                const float f = (lr <= ti) ? gv * __expf(cft_[i] - cfs[j]) : 0.f;
                                const float r = (!UNI && lr >= ti) ? gv * __expf(cbt_[i] - cbs[j]) : 0.f;
                                dcb[j][i] += f + r;
                                const float wf = (lr < ti) ? f * cbr[j][i] : 0.f;
                                const float wb = (lr > ti) ? r * cbr[j][i] : 0.f;
                                ca += wf; df[i] += wf;
                                cb2 += wb; db[i] += wb;
                            }
                            colF[j] = ca;
                            colB[j] = cb2;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) { rowF[i] = __builtin_fmaf(rpf[i], Ef[i], df[i]); rowB[i] = __builtin_fmaf(rpb[i], Eb[i], db[i]); }
                }
                // ---- hand the sums to the other waves through LDS (double-buffered by head parity)
                const unsigned pb = sbase + DCB_PART_OFF + par * DCB_PART_B;
                {
                    float cs4[4], cs4b[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) cs4[j] = lanegroup_sum_mfma(colF[j]);
                    if constexpr (DIAG) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) cs4b[j] = lanegroup_sum_mfma(colB[j]);
                    }
                    f32x4 rs, rsb;
#pragma unroll
                    for (int i = 0; i < 4; ++i) rs[i] = row16_sum(rowF[i]);
                    if constexpr (DIAG) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) rsb[i] = row16_sum(rowB[i]);
                    }
                    const unsigned pw = pb + wave * 256 + lr * 4;
                    if (lane < 16) {
                        raw_lds_write_at<0>(pw, cs4[0]); raw_lds_write_at<64>(pw, cs4[1]);
                        raw_lds_write_at<128>(pw, cs4[2]); raw_lds_write_at<192>(pw, cs4[3]);
                        if constexpr (DIAG) {
                            raw_lds_write_at<1024>(pw, cs4b[0]); raw_lds_write_at<1024 + 64>(pw, cs4b[1]);
                            raw_lds_write_at<1024 + 128>(pw, cs4b[2]); raw_lds_write_at<1024 + 192>(pw, cs4b[3]);
                        }
                    }
                    if (lr == 0) {
                        raw_lds_write128_at<2048>(pb + trow * 4, rs);
                        if constexpr (DIAG) raw_lds_write128_at<2048 + 256>(pb + trow * 4, rsb);
                    }
                }
                raw_lds_wait();
                pending = true;            // written out after the next barrier (or after the loop)
                par ^= 1;
            }
            slot = slot + 1 == DCB_RING ? 0 : slot + 1;
            slot2 = slot2 + 1 == DCB_RING ? 0 : slot2 + 1;
        }
        };
        if (st < tt) run(std::integral_constant<int, -1>());
        else if (st > tt) run(std::integral_constant<int, -2>());
        else if (wave == 0) run(std::integral_constant<int, 0>());
        else if (wave == 1) run(std::integral_constant<int, 1>());
        else if (wave == 2) run(std::integral_constant<int, 2>());
        else run(std::integral_constant<int, 3>());
        if (pending) {
            raw_lds_barrier();
            write_out(par ^ 1);
        }
    }
    const int64_t oo = ((int64_t)bid.z * gdx + (int64_t)(b * nc + c) * p.ngroups + g) * Q * Q;
    if (out16) {
        // dCB / dCBT in the element type of the inputs (inside bimamba2_bwd, one head slice: their one reader rounds them to
        // that type for its MFMA anyway, so nothing changes but the bytes moved)
        T *out = reinterpret_cast<T *>(p.dCB) + oo, *outT = reinterpret_cast<T *>(p.dCBT) + oo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int s = s0 + j * 16 + lr;
            T v4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v4[i] = from_f<T>(dcb[j][i]);
                out[(int64_t)(t0 + trow + i) * Q + s] = v4[i];
            }
            if (p.dCBT) *reinterpret_cast<uint2 *>(outT + (int64_t)s * Q + t0 + trow) = *reinterpret_cast<const uint2 *>(v4);
        }
        return;
    }
    float *out = p.dCB + oo, *outT = p.dCBT + oo;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int s = s0 + j * 16 + lr;
#pragma unroll
        for (int i = 0; i < 4; ++i) out[(int64_t)(t0 + trow + i) * Q + s] = dcb[j][i];
        *reinterpret_cast<f32x4 *>(outT + (int64_t)s * Q + t0 + trow) = dcb[j];
    }
}

}  // namespace bm2
