// Launches of the chunk-scan kernel (forward output) and its mirror (dx in the backward pass) for gfx950; see scan_body.hpp.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "scan_body.hpp"

namespace bm2 {

static inline int nchunks(const bimamba2_params *p) { return (p->seqlen + p->chunk_size - 1) / p->chunk_size; }
static inline hipStream_t stream_of(const bimamba2_params *p) { return reinterpret_cast<hipStream_t>(p->stream); }


// Waves that a SIMD holds, two for every workgroup of a CU; it bounds the registers (512 / waves).  The kernel is a chain of memory
// phases and products that only other workgroups cover: where a few registers less make room for another, they are worth it.
constexpr int scan_waves_per_simd(int bytes, int qt, int nj, int nf) { return nf > 0 || qt > 1 || bytes == 2 ? 4 : 8; }

// (what a workgroup does: scan_body.hpp)
template <typename T, int QT, int NJ, bool BWD, bool FAST, int NF, bool UNI = false, bool STATES = true>
__global__ __launch_bounds__(SCAN_THREADS, scan_waves_per_simd(sizeof(T), QT, NJ, NF)) void chunk_scan_kernel(const bimamba2_params p, int nc, int npt) {
    __shared__ __attribute__((aligned(16))) char lds[ScanMap<T, QT, NJ, BWD, NF>::LDS];
    chunk_scan_body<T, QT, NJ, BWD, FAST, NF, UNI, STATES>(p, nc, npt, blockIdx.x, lds);
}

static inline bool al16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

static inline int scan_col_tile(const bimamba2_params *p) {
    return scan_col_tile_of(p->headdim, p->dtype);
}

// whether the kernels without guarded fallbacks apply (vs = elements per 16 bytes)
static bool scan_fast(const bimamba2_params *p, bool bwd, int pw, int vs) {
    auto mult = [vs](int64_t a, int64_t b, int64_t c) { return a % vs == 0 && b % vs == 0 && c % vs == 0; };
    bool fast = p->chunk_size % 32 == 0 && p->headdim % pw == 0 && p->dstate % vs == 0 && al16(p->x) && mult(p->x_sb, p->x_sl, p->x_sh);
    if (bwd) {
        fast = fast && al16(p->Bm) && mult(p->B_sb, p->B_sl, p->B_sg) && al16(p->dx) && mult(p->dx_sb, p->dx_sl, 0);
        fast = fast && (p->has_z ? al16(p->dout_x) : (al16(p->dout) && mult(p->dout_sb, p->dout_sl, p->dout_sh)));
    } else {
        fast = fast && al16(p->Cm) && mult(p->C_sb, p->C_sl, p->C_sg) && al16(p->out);
        if (p->has_z) fast = fast && al16(p->z) && mult(p->z_sb, p->z_sl, p->z_sh) && (!p->out_x || al16(p->out_x));
    }
    return fast;
}

bool scan_is_fast(const bimamba2_params *p, bool bwd) { return scan_fast(p, bwd, scan_col_tile(p), p->dtype == BIMAMBA2_F32 ? 4 : 8); }

// the conditions of the kernels that rebuild C.B^T, apart from the state dimension
static bool scan_rebuild_shape(const bimamba2_params *p, bool bwd) {
    if (p->dtype == BIMAMBA2_F32 || scan_col_tile(p) != 64) return false;
    auto mult = [](int64_t a, int64_t b, int64_t c) { return a % 8 == 0 && b % 8 == 0 && c % 8 == 0; };
    if (p->B_sl <= 0 || p->C_sl <= 0 || p->B_sl > (1 << 21) || p->C_sl > (1 << 21)) return false;   // 256 rows in 32-bit byte offsets
    if (!(bwd ? al16(p->dstates_f) && al16(p->dstates_b) : al16(p->states_f) && al16(p->states_b))) return false;
    return p->dstate % 64 == 0 && scan_fast(p, bwd, 64, 8) && al16(p->Bm) && mult(p->B_sb, p->B_sl, p->B_sg) && al16(p->Cm) && mult(p->C_sb, p->C_sl, p->C_sg);
}

bool scan_recomputes_cb(const bimamba2_params *p, bool bwd) { return p->dstate == 64 && scan_rebuild_shape(p, bwd); }

bool chunk_scan_uses_scan16(const bimamba2_params *p, bool bwd) {
    // state dimension 64, or 128 in the forward kernel
    return scan_rebuild_shape(p, bwd) && (p->headdim == 64 || p->headdim == 128) && (p->dstate == 64 || (p->dstate == 128 && !bwd));
}

template <typename T, bool BWD>
static int launch_scan_t(const bimamba2_params *p, bool free16) {
    const int nc = nchunks(p);
    const int P = p->headdim, Q = p->chunk_size, N = p->dstate;
    constexpr int VS = 16 / (int)sizeof(T);
    const int pw = scan_col_tile(p);
    const int npt = (P + pw - 1) / pw;
    dim3 grid(p->batch * nc * p->nheads * npt);
    hipStream_t s = reinterpret_cast<hipStream_t>(p->stream);
    const bool fast = scan_fast(p, BWD, pw, VS);
    const bool states = BWD ? p->dstates_f || p->dstates16_f : p->states_f || p->states16_f;       // (else one_chunk())
#define BM2_SCAN_K(QTV, NJV, FAST, NF)                                                                                                          \
    do {                                                                                                                                        \
        if (states) hipLaunchKernelGGL((chunk_scan_kernel<T, QTV, NJV, BWD, FAST, NF>), grid, dim3(SCAN_THREADS), 0, s, *p, nc, npt);             \
        else hipLaunchKernelGGL((chunk_scan_kernel<T, QTV, NJV, BWD, FAST, NF, false, false>), grid, dim3(SCAN_THREADS), 0, s, *p, nc, npt);      \
    } while (0)
#define BM2_SCAN(QTV, NJV)                          \
    do {                                            \
        if (fast) BM2_SCAN_K(QTV, NJV, true, 0);    \
        else BM2_SCAN_K(QTV, NJV, false, 0);        \
    } while (0)
    const int qt = Q <= 128 ? 1 : 2;             // 16-row tiles per wave (8 waves)
    // 16-bit copies of the entering states: known to the kernels that rebuild CB only
    const void *c16f = BWD ? p->dstates16_f : p->states16_f, *c16b = BWD ? p->dstates16_b : p->states16_b;
    if (c16f && (!al16(c16f) || !al16(c16b) || !(p->causal || c16b))) return BIMAMBA2_EINVAL;
    if constexpr (sizeof(T) == 2) {
        // the shapes of the 16-bit kernel with transposed products and a raw operand tile: it needs the 16-bit copies of the
        // entering states (the composites keep them at these shapes) and no CB
        if ((free16 || (c16f && (p->causal || c16b))) && (BWD ? p->CBT : p->CB) == nullptr && chunk_scan_uses_scan16(p, BWD))
            return launch_chunk_scan16(p, BWD);
        if (p->causal) {                                // single-direction comparator: the fused kernels only
            if (!states) return BIMAMBA2_EINVAL;
            if (!scan_recomputes_cb(p, BWD)) return BIMAMBA2_EUNSUPPORTED;
            if (qt == 1) hipLaunchKernelGGL((chunk_scan_kernel<T, 1, 4, BWD, true, 2, true>), grid, dim3(SCAN_THREADS), 0, s, *p, nc, npt);
            else hipLaunchKernelGGL((chunk_scan_kernel<T, 2, 4, BWD, true, 2, true>), grid, dim3(SCAN_THREADS), 0, s, *p, nc, npt);
            return check_launch();
        }
        if ((BWD ? p->CBT : p->CB) == nullptr) {
            if (!scan_recomputes_cb(p, BWD)) return BIMAMBA2_EINVAL;   // (the kernels below rebuild C.B^T at state dimension 64 only)
            if (qt == 1) BM2_SCAN_K(1, 4, true, 2);
            else BM2_SCAN_K(2, 4, true, 2);
            return check_launch();
        }
    }
    // (the kernels below read the forward pass's 16-bit copies of the entering states too, but not the mirror's)
    if (p->causal || (c16f && (BWD || sizeof(T) != 2))) return BIMAMBA2_EUNSUPPORTED;
    if ((BWD ? p->CBT : p->CB) == nullptr) return BIMAMBA2_EINVAL;
    if (pw == 16) { if (qt == 1) BM2_SCAN(1, 1); else BM2_SCAN(2, 1); }
    else if (pw == 32) { if (qt == 1) BM2_SCAN(1, 2); else BM2_SCAN(2, 2); }
    else if constexpr (sizeof(T) == 2) { if (qt == 1) BM2_SCAN(1, 4); else BM2_SCAN(2, 4); }   // (float32: 32 columns at most)
#undef BM2_SCAN
#undef BM2_SCAN_K
    return check_launch();
}

// free16: the entering states are zero and have no tensors (one_chunk()), at a shape where they would travel as 16-bit copies
int launch_chunk_scan(const bimamba2_params *p, bool bwd, bool free16) {
    switch (p->dtype) {
        case BIMAMBA2_F32: return bwd ? launch_scan_t<float, true>(p, free16) : launch_scan_t<float, false>(p, free16);
        case BIMAMBA2_BF16: return bwd ? launch_scan_t<bf16_t, true>(p, free16) : launch_scan_t<bf16_t, false>(p, free16);
        case BIMAMBA2_F16: return bwd ? launch_scan_t<f16_t, true>(p, free16) : launch_scan_t<f16_t, false>(p, free16);
        default: return BIMAMBA2_EUNSUPPORTED;
    }
}

}  // namespace bm2
