// Launches of the backward pass whose workgroups have different roles, for chunks of up to 128 positions and float32 state tensors
// (float32, narrow heads or states): kernels that depend on the same earlier launches and not on each other.  At usual sizes none
// of them fills the chip, and each alone ends with a wait for its slowest workgroup and a launch of 3 to 5 us.
// One element type a translation unit (kernels_roles_*.hip).
#pragma once
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"
#include "chunk_state_body.hpp"
#include "dbdc_body.hpp"
#include "dcb_body.hpp"
#include "scan_body.hpp"

namespace bm2 {

static inline bool roles_al16(const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

// ---- dCB and the gradients of the states entering the chunks ----
// RING: columns per step of the ring variant (16-bit types; WHOLE: headdim a multiple of 64), 0: the variant through registers
// DFAST, CFAST: unconditional loads in that one and in the kernel of the states' gradients (16 bits: the one with direct loads)
template <typename T, int RING, bool WHOLE, bool DFAST, bool CFAST>
__global__ __launch_bounds__(NTHREADS) void bwd_dcb_dstates_kernel(const bimamba2_params p, int nc, int nqt, int gdx, int gdz, int nnt, int npt, int ndcb) {
    constexpr int DCB_LDS = RING ? DcbRingMap<RING ? RING : 64>::LDS : DcbMap::LDS;
    constexpr bool NARROW = sizeof(T) == 2 && CFAST;
    constexpr int STATE_LDS = NARROW ? ChunkStateNarrowMap::LDS : ChunkStateMap<T>::LDS;
    __shared__ __attribute__((aligned(16))) char lds[DCB_LDS > STATE_LDS ? DCB_LDS : STATE_LDS];
    const int id = blockIdx.x;
    if (id < ndcb) {
        const int per = gdx * nqt * nqt;
        if constexpr (RING > 0) {
            BlockId bid = dcb_block_of(id % per, gdx, nqt * nqt, per);
            bid.z = id / per;
            bwd_dcb_ring_body<T, false, RING, WHOLE>(p, nc, nqt, bid, gdx, gdz, reinterpret_cast<unsigned char *>(lds));
        } else {
            bwd_dcb_body<T, DFAST>(p, nc, nqt, BlockId{id % gdx, id / gdx % (nqt * nqt), id / per}, gdx, gdz, lds);
        }
    } else {
        const int k = id - ndcb;
        if constexpr (NARROW) chunk_state_narrow_body<T, true>(p, nc, k % nnt, k / nnt % npt, k / (nnt * npt), lds);
        else chunk_state_body<T, true, CFAST>(p, nc, k % nnt, k / nnt % npt, k / (nnt * npt), lds);
    }
}

// ---- dx, dB and dC (state parts) ----
// NJS: 16-column tiles of headdim a dx workgroup; NT, NJ, FAST: see bwd_dbdc_body
template <typename T, int NJS, int NT, int NJ, bool FAST>
__global__ __launch_bounds__(DBDC_THREADS, NJ < 4 ? 4 : 2) void bwd_dx_db_dc_kernel(const bimamba2_params p, int nc, int npt, int ndx, int ndb, int gdx, int hps) {
    static_assert(DBDC_THREADS == SCAN_THREADS, "roles of one launch");
    constexpr int A = ScanMap<T, 1, NJS, true, 0>::LDS, B = DbdcMap<T, 1>::LDS;
    __shared__ __attribute__((aligned(16))) char lds[A > B ? A : B];
    const int id = blockIdx.x;
    if (id < ndx) {
        chunk_scan_body<T, 1, NJS, true, true, 0>(p, nc, npt, id, lds);
    } else {
        const int k = id - ndx;
        if (k < ndb) bwd_dbdc_body<T, NT, 1, true, FAST, false, NJ>(p, nc, hps, BlockId{k % gdx, 0, k / gdx}, lds);
        else bwd_dbdc_body<T, NT, 1, false, FAST, false, NJ>(p, nc, hps, BlockId{(k - ndb) % gdx, 0, (k - ndb) / gdx}, lds);
    }
}

template <typename T> int launch_dcb_dstates_t(const bimamba2_params *p, const RolesShape &r) {
    const int nc = r.nchunks, nqt = (p->chunk_size + 63) / 64, gdx = p->batch * nc * p->ngroups, gdz = r.dcb_slices;
    const int nnt = (p->dstate + 63) / 64, npt = (p->headdim + 63) / 64, ndcb = gdx * nqt * nqt * gdz;
    const dim3 grid(ndcb + nnt * npt * p->batch * nc * p->nheads);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
#define BM2_R(RING, WHOLE, DFAST, CFAST) hipLaunchKernelGGL((bwd_dcb_dstates_kernel<T, RING, WHOLE, DFAST, CFAST>), grid, dim3(NTHREADS), 0, s, *p, nc, nqt, gdx, gdz, nnt, npt, ndcb)
    if constexpr (sizeof(T) == 2) {
        if (!r.dcb_ring) return BIMAMBA2_EINVAL;
        if (r.dstates_narrow) {
            if (p->headdim <= 32) BM2_R(32, false, false, true);
            else if (p->headdim % 64) BM2_R(64, false, false, true);
            else BM2_R(64, true, false, true);
        } else if (p->headdim <= 32) BM2_R(32, false, false, false);
        else if (p->headdim % 64) BM2_R(64, false, false, false);
        else BM2_R(64, true, false, false);
    } else {
        if (r.dcb_fast && r.dstates_fast) BM2_R(0, false, true, true);
        else if (r.dcb_fast) BM2_R(0, false, true, false);
        else BM2_R(0, false, false, false);
    }
#undef BM2_R
    return check_launch();
}

template <typename T> int launch_dx_db_dc_t(const bimamba2_params *p, const RolesShape &r) {
    const int nc = r.nchunks, pw = scan_col_tile_of(p->headdim, p->dtype), npt = (p->headdim + pw - 1) / pw;
    const int gdx = p->batch * nc * p->ngroups, ndx = r.dx ? p->batch * nc * p->nheads * npt : 0, ndb = gdx * r.dbdc_slices;
    const dim3 grid(ndx + 2 * ndb);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
#define BM2_R(NJS, NT, NJ, FAST) hipLaunchKernelGGL((bwd_dx_db_dc_kernel<T, NJS, NT, NJ, FAST>), grid, dim3(DBDC_THREADS), 0, s, *p, nc, npt, ndx, ndb, gdx, r.dbdc_heads)
#define BM2_RN(NJS)                                           \
    do {                                                      \
        if (p->dstate <= 16) BM2_R(NJS, 1, 1, false);         \
        else if (p->dstate <= 32) BM2_R(NJS, 1, 2, false);    \
        else if (p->dstate <= 64) BM2_R(NJS, 1, 4, false);    \
        else BM2_R(NJS, 2, 4, false);                         \
    } while (0)
    if (pw == 16) BM2_RN(1);
    else if (pw == 32) {
        if constexpr (sizeof(T) == 4) {
            if (r.dbdc_fast && p->dstate == 64) { BM2_R(2, 1, 4, true); return check_launch(); }
            if (r.dbdc_fast && p->dstate == 128) { BM2_R(2, 2, 4, true); return check_launch(); }
        }
        BM2_RN(2);
    } else if constexpr (sizeof(T) == 2) BM2_RN(4);
#undef BM2_RN
#undef BM2_R
    return check_launch();
}

}  // namespace bm2
