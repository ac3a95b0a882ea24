// C ABI of libbimamba2_hip.so: argument checks, workspace carving and the forward / backward pipelines.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>

#include "../../include/bimamba2.h"
#include "launch.hpp"

using namespace bm2;

namespace {

inline int nchunks(const bimamba2_params *p) { return (p->seqlen + p->chunk_size - 1) / p->chunk_size; }
inline hipStream_t stream_of(const bimamba2_params *p) { return reinterpret_cast<hipStream_t>(p->stream); }
inline size_t elem_size(int dtype) { return dtype == BIMAMBA2_F32 ? 4 : 2; }
inline int sp_nsplit(const bimamba2_params *p) { return (p->headdim * p->dstate + 1023) / 1024; }

// the forward scan kernel that rebuilds C.B^T from the 16-bit copies' side: it exists beyond state dimension 64 (128) and
// runs where the entering states are given as copies
inline bool fwd_scan_rebuilds_cb(const bimamba2_params *p) {
    return chunk_scan_uses_scan16(p, false) && p->states16_f && (p->causal || p->states16_b);
}

int check_problem(const bimamba2_params *p) {
    if (!p) return BIMAMBA2_EINVAL;
    if (p->batch <= 0 || p->seqlen <= 0 || p->nheads <= 0 || p->headdim <= 0 || p->ngroups <= 0 || p->dstate <= 0)
        return BIMAMBA2_EINVAL;
    if (p->nheads % p->ngroups) return BIMAMBA2_EINVAL;
    if (p->dtype < BIMAMBA2_F32 || p->dtype > BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
    if (p->dt_dtype < BIMAMBA2_F32 || p->dt_dtype > BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
    if (p->chunk_size < BIMAMBA2_MIN_CHUNK || p->chunk_size > BIMAMBA2_MAX_CHUNK) return BIMAMBA2_EUNSUPPORTED;
    if (p->headdim > BIMAMBA2_MAX_HEADDIM || p->dstate > BIMAMBA2_MAX_DSTATE) return BIMAMBA2_EUNSUPPORTED;
    // grid.z = batch * nchunks * nheads must fit the launch limits
    const int64_t z = (int64_t)p->batch * nchunks(p) * p->nheads;
    if (z > 2147483647LL / 2) return BIMAMBA2_EUNSUPPORTED;
    return BIMAMBA2_OK;
}

// A sequence that one chunk holds, without states going in or out and without tensors for the states entering the chunks: these are
// zero, nothing crosses a chunk boundary, and neither the chunk states and their passing nor the state parts of the backward pass are
// formed (the sums are the same but for terms of zero).  us of kernels a pass, bfloat16, heads of 64, z gate: 1 x 197, 12 heads, dstate 64 25 -> 17
// forward, 91 -> 60 in training (10 -> 7 launches); 8 x 250, 24 heads, dstate 128 48 -> 27, 168 -> 90; layer 16 x 200, d_model 768 109 -> 95,
// 363 -> 303.  What follows from it is which pointers are NULL: the scan kernels' states, the last launch's state parts.
inline bool one_chunk(const bimamba2_params *p) {
    return p->seqlen <= p->chunk_size && !p->causal && !p->initial_f && !p->initial_b && !p->final_f && !p->final_b && !p->dfinal_f && !p->dfinal_b &&
           !p->dinitial_f && !p->dinitial_b && !p->states_f && !p->states_b && !p->states16_f && !p->states16_b && !p->dstates_f && !p->dstates_b &&
           !p->dstates16_f && !p->dstates16_b;
}
// whether such a problem's entering states would travel as 16-bit copies, i.e. which scan kernel is the one to run without any
// (a forward pass that a backward pass follows keeps them in float32 at other shapes than bimamba2_state_copies()'s)
inline bool one_chunk_free16(const bimamba2_params *p, bool is_bwd) {
    if (p->dtype == BIMAMBA2_F32) return false;
    return bimamba2_state_copies(p) != 0 || (!is_bwd && !(p->fwd_saved & 4) && (p->headdim * p->dstate) % 4 == 0);
}

#define REQUIRE(ptr)                        \
    do {                                    \
        if (!(ptr)) return BIMAMBA2_EINVAL; \
    } while (0)
#define TRY(expr)              \
    do {                       \
        int rc_ = (expr);      \
        if (rc_) return rc_;   \
    } while (0)

struct Carver {
    char *base;
    size_t off = 0;
    explicit Carver(void *b) : base(static_cast<char *>(b)) {}
    template <typename T> T *take(size_t n) {
        off = (off + 255) & ~size_t(255);
        T *r = base ? reinterpret_cast<T *>(base + off) : nullptr;
        off += n * sizeof(T);
        return r;
    }
};

inline bool al16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// What the tensors of states that a caller brings, or leaves out, decide about a pass
struct StateForm {
    bool one;           // one_chunk()
    bool by_heads;      // dbdc_both_by_heads() will hold (what is carved is aligned)
    bool together;      // db_dc_roles()
};
StateForm state_form(const bimamba2_params *q, int is_bwd) {
    StateForm f{one_chunk(q), false, false};
    if (!is_bwd) return f;
    const bool copies = bimamba2_state_copies(q) != 0, brought = q->states16_f && q->states16_b && al16(q->states16_f) && al16(q->states16_b);
    f.by_heads = copies && !q->dstates_f && dbdc_by_heads(q) && (q->states16_f ? brought : !q->states_f) &&
                 (!q->dstates16_f || (q->dstates16_b && al16(q->dstates16_f) && al16(q->dstates16_b)));
    f.together = db_dc_roles(q, copies || q->states16_f || q->dstates16_f);
    return f;
}

// Assigns every intermediate that is NULL in `q` from the workspace; returns the bytes used.
size_t carve(bimamba2_params *q, int is_bwd, void *ws, const StateForm &form) {
    Carver cv(ws);
    const bool one = form.one;
    const size_t nc = nchunks(q), Q = q->chunk_size;
    const size_t bhcq = (size_t)q->batch * q->nheads * nc * Q;
    const size_t cbn = (size_t)q->batch * nc * q->ngroups * Q * Q;
    const size_t stn = (size_t)q->batch * nc * q->nheads * q->headdim * q->dstate;
    auto need_f = [&](float *&ptr, size_t n) { if (!ptr) ptr = cv.take<float>(n); };
    need_f(q->dt_out, bhcq);
    need_f(q->cs_f, bhcq);
    need_f(q->cs_b, bhcq);
    // 16-bit copies of the entering states (see states16_f in the header): used where the kernels know them and the
    // caller does not ask for the float32 entering states; a backward pass that got the copies from the forward pass
    // needs no float32 states at all
    const bool copies = bimamba2_state_copies(q) != 0;
    const bool saved_copies = is_bwd && q->fwd_saved && q->states16_f;
    // a forward pass whose caller keeps no states (no pointer given for them) has one reader of the entering states, the scan
    // kernel, and every 16-bit scan kernel reads the copies: the state passing then writes half the bytes, the scan reads half
    // (under the conditions of the state-passing kernel that writes them)
    const bool fwd_only_copies = !is_bwd && !q->causal && (q->dtype == BIMAMBA2_BF16 || q->dtype == BIMAMBA2_F16) &&
                                 (q->headdim * q->dstate) % 4 == 0 && al16(q->final_f) && al16(q->final_b) &&
                                 al16(q->initial_f) && al16(q->initial_b) && !q->states_b && !q->states16_b;
    const bool carve16 = !one && (copies || fwd_only_copies) && !q->states_f && !q->states16_f;
    // CB: read by the forward scan and by the dCB kernel unless they rebuild it; CB^T: by the dx kernel, likewise.  (The
    // forward scan kernel for state dimension 128 rebuilds it as well, and runs where the entering states travel as copies.)
    const bool fwd_scan16 = !is_bwd && chunk_scan_uses_scan16(q, false) &&
                            (one ? one_chunk_free16(q, false) : (carve16 || q->states16_f) && (q->causal || carve16 || q->states16_b));
    if (is_bwd ? !(scan_recomputes_cb(q, true) && dcb_recomputes_cb(q)) : !(scan_recomputes_cb(q, false) || fwd_scan16)) need_f(q->CB, cbn);
    if (carve16) {
        q->states16_f = cv.take<char>(stn * 2);
        q->states16_b = cv.take<char>(stn * 2);
    }
    // a forward pass whose caller asks for no float32 states at all keeps the per-chunk states in the 16-bit copies' place
    // too (the chunk-state kernel writes them there, the inter-chunk scan replaces them by the entering states)
    const bool states16_only = !is_bwd && !q->states_f && !q->states_b && (carve16 || (q->states16_f && q->states16_b)) &&
                               chunk_states_in_16bit(q);
    if (!saved_copies && !states16_only && !one) {
        need_f(q->states_f, stn);
        need_f(q->states_b, stn);
    }
    if (is_bwd && copies && !q->dstates_f && !q->dstates16_f && !one) {
        q->dstates16_f = cv.take<char>(stn * 2);
        q->dstates16_b = cv.take<char>(stn * 2);
    }
    if (is_bwd) {
        const size_t nqt = (Q + 63) / 64;
        if (!q->dBs && !q->dCs) q->dbdc_heads = choose_dbdc_heads(q, !one && form.by_heads, form.together);
        if (!q->dCB && !q->dCBT) q->dcb_slices = choose_dcb_slices(q);      // (which asks about the last launch, and that about the slices of dB and dC)
        need_f(q->dCB, cbn * dcb_slices(q));
        need_f(q->dCBT, cbn * dcb_slices(q));
        if (!scan_recomputes_cb(q, true)) need_f(q->CBT, cbn);
        // where the 16-bit copies of the gradients exist and the caller asks for no float32 tensors, the per-chunk gradients
        // live in the copies' place as well (written there by the dstates kernels, replaced in place by the backward
        // inter-chunk scan): no float32 tensors at all
        // (the in-place kernel of the backward inter-chunk scan reads the entering states from their copies as well)
        const bool dstates16_only = copies && !q->dstates_f && !q->dstates_b && (carve16 || q->states16_f);
        if (!dstates16_only && !one) {
            need_f(q->dstates_f, stn);
            need_f(q->dstates_b, stn);
        }
        if (q->has_z && !q->dout_x)
            q->dout_x = cv.take<char>((size_t)q->batch * q->seqlen * q->nheads * q->headdim * elem_size(q->dtype));
        need_f(q->ddt_direct, bhcq * ddt_direct_planes(*q));
        need_f(q->da_intra, (size_t)q->batch * q->nheads * nc * nqt * nqt * 128);
        if (one) {
            q->u_f = q->u_b = q->v_f = q->v_b = q->ddA_chunk_f = q->ddA_chunk_b = q->dBs = q->dCs = nullptr;
        } else {
            need_f(q->u_f, bhcq);
            need_f(q->u_b, bhcq);
            need_f(q->v_f, bhcq);
            need_f(q->v_b, bhcq);
            need_f(q->ddA_chunk_f, (size_t)q->batch * q->nheads * nc * sp_nsplit(q));
            need_f(q->ddA_chunk_b, (size_t)q->batch * q->nheads * nc * sp_nsplit(q));
            const int hps = q->dbdc_heads > 0 ? q->dbdc_heads : 8;
            const size_t slices = (q->nheads / q->ngroups + hps - 1) / hps;   // head slices of the dB / dC partial sums
            const size_t bn = slices * q->batch * q->seqlen * q->ngroups * q->dstate;
            need_f(q->dBs, bn);
            need_f(q->dCs, bn);
        }
        // partial sums of dD, then those of dA and ddt_bias (the composite reduces all three in one launch at the end)
        need_f(q->red, (size_t)q->batch * nc * q->nheads * q->headdim + (size_t)2 * q->batch * nc * q->nheads);
    }
    return (cv.off + 255) & ~size_t(255);
}
size_t carve(bimamba2_params *q, int is_bwd, void *ws) { return carve(q, is_bwd, ws, state_form(q, is_bwd)); }

// Device memory that lives as long as the process: the workspace of bimamba2_fwd_static.  Every GPU the library runs on
// holds its own copy at its own address; in host code the array's name is not a device address, so the address is asked
// for once per device (hipGetSymbolAddress, with that device current) and kept.
static __device__ __align__(256) unsigned char scratch[BIMAMBA2_STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::atomic<void *> scratch_of_device[MAX_DEVICES];

int static_scratch(void **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return BIMAMBA2_ELAUNCH;
    void *ptr = scratch_of_device[dev].load(std::memory_order_acquire);
    if (!ptr) {
        // two host threads may both get here: they are given the same address
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return BIMAMBA2_ELAUNCH;
        scratch_of_device[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return BIMAMBA2_OK;
}

}  // namespace

extern "C" {

const char *bimamba2_strerror(int code) {
    switch (code) {
        case BIMAMBA2_OK: return "ok";
        case BIMAMBA2_EINVAL: return "invalid argument (null pointer or inconsistent dimensions)";
        case BIMAMBA2_EUNSUPPORTED:
            return "unsupported problem (need 32 <= chunk_size <= 256, headdim <= 128, dstate <= 256, dtype f32/bf16/f16)";
        case BIMAMBA2_EWORKSPACE: return "workspace missing or too small";
        case BIMAMBA2_ELAUNCH: return "HIP kernel launch failed";
        case BIMAMBA2_ESCRATCH: return "the problem needs more intermediate memory than the static scratch buffer holds";
        default: return "unknown error";
    }
}

int bimamba2_version(void) { return 100; }
size_t bimamba2_params_size(void) { return sizeof(bimamba2_params); }

size_t bimamba2_workspace_bytes(const bimamba2_params *p, int is_bwd) {
    if (check_problem(p)) return 0;
    bimamba2_params asked = *p;
    if (is_bwd) asked.final_f = asked.final_b = nullptr;      // (as the pass does)
    // the most that any form takes which tensors of states set after the question can lead to
    const StateForm now = state_form(&asked, is_bwd);
    size_t most = 0;
    for (int k = 0; k < 8; ++k) {
        if (((k & 1) && !now.one) || ((k & 2) && !now.by_heads) || ((k & 4) && !now.together)) continue;
        bimamba2_params q = asked;
        most = std::max(most, carve(&q, is_bwd, nullptr, StateForm{now.one && !(k & 1), now.by_heads && !(k & 2), now.together && !(k & 4)}));
    }
    if (!is_bwd && !asked.states_f && !asked.states16_f) {
        // float32 states of the caller's: no copies, and a scan kernel that reads CB where the one for copies would not (dstate 128, few heads)
        asked.states_f = asked.states_b = reinterpret_cast<float *>(256);
        most = std::max(most, carve(&asked, is_bwd, nullptr));
    }
    return most;
}

int bimamba2_state_copies(const bimamba2_params *p) {
    if (check_problem(p)) return 0;
    if (p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return 0;
    if (p->dstate != 64 || p->headdim % 64 || p->chunk_size % 64) return 0;
    auto al = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    // the vector kernels of the two state-passing stages, the scan kernels that rebuild CB, the dB / dC kernels with the
    // ring of state tiles: every one of them must be the one that runs
    if (!(al(p->states_f) && al(p->states_b) && al(p->dstates_f) && al(p->dstates_b) && al(p->final_f) && al(p->final_b) &&
          al(p->initial_f) && al(p->initial_b) && al(p->dfinal_f) && al(p->dfinal_b) && al(p->dinitial_f) && al(p->dinitial_b)))
        return 0;
    if (!al(p->states16_f) || !al(p->states16_b) || !al(p->dstates16_f) || !al(p->dstates16_b)) return 0;
    return scan_recomputes_cb(p, false) && scan_recomputes_cb(p, true) && dcb_recomputes_cb(p) ? 1 : 0;
}

int bimamba2_chunk_scan_reads_cb(const bimamba2_params *p, int which) {
    if (check_problem(p)) return 1;
    if (which == 2) return dcb_recomputes_cb(p) ? 0 : 1;
    if (which == 3) return chunk_state_does_cumsum(p) ? 0 : 1;
    if (which == 0 && fwd_scan_rebuilds_cb(p)) return 0;
    return scan_recomputes_cb(p, which != 0) ? 0 : 1;
}

int bimamba2_chunk_scan_heads_per_workgroup(const bimamba2_params *p, int bwd) {
    if (check_problem(p)) return 1;
    return chunk_scan_uses_scan16(p, bwd != 0) ? chunk_scan16_heads_per_workgroup(p) : 1;
}

int bimamba2_fwd_one_launch(const bimamba2_params *p) { return check_problem(p) || !scan_once_applies(p) ? 0 : scan_once_walks(p) ? 2 : 1; }

// A chunk costs its pairs of positions (they grow with the chunk) and its states (which do not); small calls want many workgroups, i.e. small
// chunks.  The lines follow the length, the heads and the operands of a row but not the number of rows, so that a row's result is the same
// alone and in any batch; where they lie is therefore between what one row and what many rows want.  us a pass with chunks of 64 / 128 / 256
// (z gate, D, one group; forward alone and, second, with the backward pass; workgroups: of one row in chunks of 128, for wide heads
// 256, as counted below):
//  * float32: pairs run at the float32 matrix rate.  Heads of 64, dstate 64: 1024 positions, 8 heads (128 workgroups) 30 / 33, 98 / 101, four
//    rows 52 / 45, 171 / 150; 2048, 8 heads (256) 41 / 37, 131 / 118; 512, 8 heads (64) 27 / 32, 80 / 91, four rows 39 / 36, 126 / 118, sixteen 79 / 65,
//    270 / 235.  Heads of 32, dstate 16: 2048, 24 heads (384) 37 / 36, 133 / 136; 1024, 8 heads (64) 23 / 27, 74 / 83, four rows 30 / 30, 106 / 108.
//    Chunks of 256: 118, 477 where 128 takes 99, 384 (4 x 2048, 16 heads of 64).  Never above the caller's: the result is off by the
//    resolution of sums over a chunk (1.6 times as much in chunks twice as long).
//  * 16 bits, heads of 64 or 128 with dstate 64 or 128; heads of 64, dstate 64: 2048, 24 heads (192)
//    43 / 37 / 35, 119 / 112 / 120, four rows 87 / 64 / 56, 280 / 215 / 201; 1024, 24 heads (96) 34 / 28 / 32, 101 / 96 / 112; 8192, 8 heads (256) 58 / 44 / 40,
//    168 / 130 / 124; 512, 8 heads (16; 32 in chunks of 128) 24 / 25 / 30, 72 / 75 / 89, sixteen rows 43 / 37 / 36, 128 / 117 / 119; 200, 8 heads 23 / 24 / 29,
//    71 / 73 / 84.  dstate 128: 2048, 24 heads 55 / 49 / 49, 197 / 154 / 160, four rows 122 / 91 / 85, 657 / 394 / 348.  Never below the caller's, where small
//    calls would be faster: their result is 0.4 % (128) and 1.5 % (64) further from float64 in bfloat16 (1 x 197, 12 heads:
//    2.013e-3 / 2.023e-3 / 2.048e-3), most of it from the states in 16 bits (float16, 520 positions, 16 heads: 3.03e-4 / 3.02e-4 / 3.01e-4).
//    A pass with gradients grows to 128 at most: the last launch of chunks of 256 takes dCB rounded to 16 bits, that of up to 128 in two
//    parts, and dB and dC are 14 to 21 % further off in 256 (2.40e-3 against 2.89e-3 at any number of heads, groups and both state
//    dimensions), for 3 to 8 % of the time at dstate 64 and 3 to 21 % at 128 (4 x 4096, 32 heads in 8 groups 617 / 584; dstate 128, 2 x 2048,
//    8 heads of 128 177 / 172, 2 x 7236, 42 heads of 64 1334 / 1102).  In chunks that are no multiples of 64 its states stay in float32 at dstate 64: they are kept (float16, 640
//    positions, 16 heads: out 2.58e-4 in chunks of 160, 3.08e-4 in 128).
//  * other 16-bit shapes, 64 / 128, heads of 32, dstate 32: 1024, 8 heads (64) 22 / 24, 61 / 67, four rows 26 / 25, 89 / 84; 2048, 8 heads (128) 25 / 25,
//    79 / 79; 2048, 24 heads (384) 34 / 29, 114 / 106; 512, 8 heads (32) 21 / 23, 57 / 64, sixteen rows 38 / 31, 116 / 101.  128 and 256: 41 / 45, 145 / 194 (4 x
//    2048, 16 heads); 8 groups, 4 x 4096, 32 heads 149 / 178, 580 / 784; 4 x 1024, 8 heads 20 / 34, 117 / 136; 2 x 512 19 / 32.  Below the
//    caller's chunk only where the chunk states take their weighted operand in two 16-bit parts: with one, dA was 5 to 32 % further from
//    float64 in chunks of 128 than of 256 (900 positions, 8 heads, 400 inputs); with two no output is (dA -0.3 to -7 %, out -0.4 to
//    -0.8 %, dB and dC -18 to -28 %).  Nor in training without a gate where one chunk, or little more, holds the sequence: dA is made of
//    products of the operands themselves within a chunk, and only what crosses a boundary has been rounded (200 positions, 64 heads of 64 in 8 groups,
//    dstate 32, bfloat16: 1.2e-6 in chunks of 256, 7.3e-4 in 128; 257 three times as far off in 128, 270 1.3, 288 1.1, 320 and 384 1.0, 512 1.1, 900 0.84
//    times; with a gate, whose product with the gradient is rounded, 1.0 at all of them).  128 / 256 there, heads of 32, dstate 16: 200 positions, 8
//    heads 63 / 106, sixteen rows 78 / 132; 24 heads of 64, dstate 32 142 / 188.
int bimamba2_chunk_for(const bimamba2_params *p, int training) {
    if (check_problem(p)) return p ? p->chunk_size : 0;
    const int Q = p->chunk_size, P = p->headdim, N = p->dstate;
    // (packed sequences that need no count of their boundaries keep their size: counting them synchronises)
    if (p->causal || Q % 32 || (p->seq_idx && Q <= BIMAMBA2_MAX_SEQ_BOUNDARIES)) return Q;
    // of one row in one launch over (chunk, head, headdim tile), in whole chunks' worth of positions: the rest of a sequence is a workgroup
    // that fills nothing (4 x 136, 8 heads of 128, dstate 128: 30.5 us in chunks of 64, 31.2 in a whole chunk of 128 and one of 8 positions)
    auto workgroups = [&](int q, int columns) { return (int64_t)p->seqlen * p->nheads * ((P + columns - 1) / columns) / q; };
    constexpr int CUS = 256;
    if (p->dtype == BIMAMBA2_F32) return Q > 64 ? std::min(Q, workgroups(128, 32) >= CUS / 2 ? 128 : 64) : Q;
    const bool wide = (P == 64 || P == 128) && (N == 64 || N == 128);
    if (wide && !training) {
        // the kernel that rebuilds C.B^T takes aligned rows; others run the generic one, which is among the other shapes below (x at an odd
        // element, a pass with gradients: 4 x 2048, 16 heads of 64, dstate 64 444 / 416 / 555, dstate 128 672 / 543 / 677)
        bimamba2_params q = *p;
        // (an operand that is not named yet will be contiguous)
        auto rows = [&](const void *t, int64_t &sb, int64_t &sl, int64_t &si, int heads, int width) {
            if (!t && !sb && !sl && !si) sb = (int64_t)p->seqlen * (sl = (int64_t)heads * (si = width));
        };
        rows(q.x, q.x_sb, q.x_sl, q.x_sh, p->nheads, P);
        rows(q.Bm, q.B_sb, q.B_sl, q.B_sg, p->ngroups, N);
        rows(q.Cm, q.C_sb, q.C_sl, q.C_sg, p->ngroups, N);
        if (chunk_scan_uses_scan16(&q, false))
            return std::max(Q, workgroups(256, 64) >= CUS / 2 ? 256 : workgroups(128, 64) >= CUS / 8 ? 128 : Q);
    }
    // (in chunks that are no multiples of 64 such a pass keeps its states in float32)
    if (training && N == 64 && P % 64 == 0 && Q % 64) return Q;
    if (Q <= 128) return workgroups(128, 64) >= (wide ? CUS / 8 : CUS / 4) ? 128 : Q;
    // (a sequence that one chunk holds, or little more, in training without a gate: see above)
    if (training && !p->has_z && p->seqlen > 128 && 4 * (int64_t)p->seqlen < 5 * (int64_t)Q) return Q;
    bimamba2_params q = *p;
    q.chunk_size = 128;
    const bool exact_states = !(P % 64 == 0 && N % 64 == 0) && chunk_state_narrow(&q, false) && chunk_state_narrow(&q, true);
    return exact_states ? 128 : Q;
}

int bimamba2_ddt_direct_planes(const bimamba2_params *p) {
    if (check_problem(p)) return 1;
    return ddt_direct_planes(*p);
}

int bimamba2_seq_boundaries(const bimamba2_params *p, int32_t *counts) {
    TRY(check_problem(p));
    REQUIRE(p->seq_idx); REQUIRE(counts);
    if (p->batch > 65535) return BIMAMBA2_EUNSUPPORTED;
    return launch_seq_boundaries(p, counts);
}

int bimamba2_chunk_cumsum_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->dt); REQUIRE(p->A); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (p->has_dt_bias) REQUIRE(p->dt_bias);
    return launch_chunk_cumsum_fwd(p);
}

int bimamba2_bmm_chunk_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->Bm); REQUIRE(p->Cm); REQUIRE(p->CB);
    return launch_bmm_chunk_fwd(p);
}

int bimamba2_chunk_state_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->x); REQUIRE(p->Bm); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (p->states_f || !p->states16_f) { REQUIRE(p->states_f); REQUIRE(p->states_b); }   // (else: 16-bit per-chunk states in states16_*)
    return launch_chunk_state(p, false);
}

int bimamba2_state_passing_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (p->states_f || !p->states16_f) { REQUIRE(p->states_f); REQUIRE(p->states_b); }
    return launch_state_passing_fwd(p);
}

int bimamba2_chunk_scan_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->x); REQUIRE(p->Cm); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->CB && !(p->Bm && (scan_recomputes_cb(p, false) || fwd_scan_rebuilds_cb(p)))) return BIMAMBA2_EINVAL;   // without CB the kernel rebuilds it from Cm, Bm
    if (!p->states16_f) { REQUIRE(p->states_f); REQUIRE(p->states_b); }
    REQUIRE(p->out);
    if (p->has_D) REQUIRE(p->D);
    if (p->has_z) REQUIRE(p->z);
    return launch_chunk_scan(p, false);
}

int bimamba2_chunk_scan_bwd_dz(const bimamba2_params *p) {
    TRY(check_problem(p));
    if (!p->has_z) return BIMAMBA2_EINVAL;
    REQUIRE(p->z); REQUIRE(p->dout); REQUIRE(p->out_x); REQUIRE(p->dz); REQUIRE(p->dout_x);
    return launch_bwd_dz(p);
}

int bimamba2_chunk_scan_bwd_dstates(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->Cm); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (p->dstates_f || !p->dstates16_f) { REQUIRE(p->dstates_f); REQUIRE(p->dstates_b); }   // (else: 16-bit per-chunk gradients in dstates16_*)
    if (p->has_z) REQUIRE(p->dout_x); else REQUIRE(p->dout);
    return launch_chunk_state(p, true);
}

int bimamba2_chunk_scan_bwd_dz_dstates(const bimamba2_params *p) {
    TRY(check_problem(p));
    if (!p->has_z) return BIMAMBA2_EINVAL;
    REQUIRE(p->z); REQUIRE(p->dout); REQUIRE(p->out_x); REQUIRE(p->dz); REQUIRE(p->dout_x);
    REQUIRE(p->Cm); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (p->dstates_f || !p->dstates16_f) { REQUIRE(p->dstates_f); REQUIRE(p->dstates_b); }
    return launch_bwd_dz_dstates(p);       // BIMAMBA2_EUNSUPPORTED where only the two separate kernels exist
}

int bimamba2_state_passing_bwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->states16_f) { REQUIRE(p->states_f); REQUIRE(p->states_b); }
    if (p->dstates_f || !p->dstates16_f) { REQUIRE(p->dstates_f); REQUIRE(p->dstates_b); }
    REQUIRE(p->ddA_chunk_f); REQUIRE(p->ddA_chunk_b);
    return launch_state_passing_bwd(p);
}

int bimamba2_chunk_scan_bwd_dx(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->x); REQUIRE(p->Bm); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->CBT && !(p->Cm && scan_recomputes_cb(p, true))) return BIMAMBA2_EINVAL;   // without CBT the kernel rebuilds it from Cm, Bm
    if (!p->dstates16_f) { REQUIRE(p->dstates_f); REQUIRE(p->dstates_b); }
    REQUIRE(p->dx); REQUIRE(p->ddt_direct);
    if (p->has_z) REQUIRE(p->dout_x); else REQUIRE(p->dout);
    if (p->has_D) { REQUIRE(p->D); REQUIRE(p->dD); REQUIRE(p->red); }
    const int nc = nchunks(p);
    TRY(launch_chunk_scan(p, true));
    if (p->has_D) {
        if (p->D_has_hdim) return launch_reduce(p->red, p->dD, p->batch * nc, p->nheads * p->headdim, 1, stream_of(p));
        return launch_reduce(p->red, p->dD, p->batch * nc, p->nheads, p->headdim, stream_of(p));
    }
    return BIMAMBA2_OK;
}

int bimamba2_chunk_state_bwd_db(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->x); REQUIRE(p->Bm); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->dstates16_f) { REQUIRE(p->dstates_f); REQUIRE(p->dstates_b); }
    REQUIRE(p->dBs); REQUIRE(p->v_f); REQUIRE(p->v_b);
    return launch_bwd_dbdc(p, true);
}

int bimamba2_chunk_scan_bwd_dc(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->Cm); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->states16_f) { REQUIRE(p->states_f); REQUIRE(p->states_b); }
    REQUIRE(p->dCs); REQUIRE(p->u_f); REQUIRE(p->u_b);
    if (p->has_z) REQUIRE(p->dout_x); else REQUIRE(p->dout);
    return launch_bwd_dbdc(p, false);
}

static int check_bwd_dcb(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->x); REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
    if (!p->CB && !(p->Cm && p->Bm && dcb_recomputes_cb(p))) return BIMAMBA2_EINVAL;   // without CB the kernel rebuilds it from Cm, Bm
    REQUIRE(p->dCB); REQUIRE(p->dCBT); REQUIRE(p->da_intra);
    if (p->has_z) REQUIRE(p->dout_x); else REQUIRE(p->dout);
    return BIMAMBA2_OK;
}

int bimamba2_chunk_scan_bwd_dcb(const bimamba2_params *p) {
    TRY(check_bwd_dcb(p));
    return launch_bwd_dcb(p);
}

int bimamba2_bmm_chunk_bwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->Bm); REQUIRE(p->Cm); REQUIRE(p->dCB); REQUIRE(p->dCBT); REQUIRE(p->dBs); REQUIRE(p->dCs); REQUIRE(p->dB); REQUIRE(p->dC);
    return launch_bmm_chunk_bwd(p);
}

int bimamba2_chunk_cumsum_bwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    REQUIRE(p->dt); REQUIRE(p->A); REQUIRE(p->da_intra); REQUIRE(p->u_f); REQUIRE(p->u_b); REQUIRE(p->v_f); REQUIRE(p->v_b);
    REQUIRE(p->ddA_chunk_f); REQUIRE(p->ddA_chunk_b); REQUIRE(p->ddt_direct); REQUIRE(p->ddt); REQUIRE(p->dA); REQUIRE(p->red);
    if (p->has_dt_bias) REQUIRE(p->dt_bias);
    return launch_chunk_cumsum_bwd(p);
}

// chunk cumsum + chunk states: one launch where the chunk-state kernel does both, else the two stages
static int forward_cumsum_and_states(const bimamba2_params *q) {
    if (chunk_state_does_cumsum(q)) {
        REQUIRE(q->dt); REQUIRE(q->A); REQUIRE(q->x); REQUIRE(q->Bm);
        if (q->has_dt_bias) REQUIRE(q->dt_bias);
        return launch_chunk_state(q, false, true);
    }
    TRY(bimamba2_chunk_cumsum_fwd(q));
    return bimamba2_chunk_state_fwd(q);
}

int bimamba2_fwd(const bimamba2_params *p) {
    TRY(check_problem(p));
    if (p->causal && p->final_b) return BIMAMBA2_EINVAL;
    bimamba2_params q = *p;
    const size_t need = carve(&q, 0, p->workspace);
    if (need > 256 && (!p->workspace || p->workspace_bytes < need)) return BIMAMBA2_EWORKSPACE;
    if (scan_once_applies(p)) {
        REQUIRE(p->dt); REQUIRE(p->A); REQUIRE(p->x); REQUIRE(p->Bm); REQUIRE(p->Cm); REQUIRE(p->out);
        if (p->has_dt_bias) REQUIRE(p->dt_bias);
        if (p->has_D) REQUIRE(p->D);
        if (p->has_z) REQUIRE(p->z);
        if (q.final_f || q.final_b) {
            // (the result of such a call is the same in bits whether or not the final states are asked for)
            if (fwd_front_merged(&q)) {
                bimamba2_params qs = q;
                qs.CB = nullptr;      // (nobody reads it; float32, 1 x 256 positions, 4 heads of 32, us a call: chunked launches 17.1, cumsum and states apart 17.7, so 16.0)
                TRY(launch_fwd_front(&qs));
            } else TRY(forward_cumsum_and_states(&q));
            TRY(bimamba2_state_passing_fwd(&q));
        }
        return launch_scan_once(p);
    }
    if (one_chunk(&q)) {
        REQUIRE(q.dt); REQUIRE(q.A); REQUIRE(q.x); REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.out);
        if (q.has_dt_bias) REQUIRE(q.dt_bias);
        if (q.has_D) REQUIRE(q.D);
        if (q.has_z) REQUIRE(q.z);
        const bool free16 = one_chunk_free16(&q, false);
        TRY(launch_fwd_cumsum_cb(&q, free16));
        if (scan_recomputes_cb(&q, false) || (free16 && chunk_scan_uses_scan16(&q, false))) q.CB = nullptr;
        return launch_chunk_scan(&q, false, free16);
    }
    if (fwd_front_merged(&q)) {
        REQUIRE(q.dt); REQUIRE(q.A); REQUIRE(q.x); REQUIRE(q.Bm); REQUIRE(q.Cm);
        if (q.has_dt_bias) REQUIRE(q.dt_bias);
        TRY(launch_fwd_front(&q));
    } else {
        TRY(forward_cumsum_and_states(&q));
        if (q.CB) TRY(bimamba2_bmm_chunk_fwd(&q));     // given by the caller, or carved because the scan kernel reads it
    }
    TRY(bimamba2_state_passing_fwd(&q));
    if (scan_recomputes_cb(&q, false) || fwd_scan_rebuilds_cb(&q)) q.CB = nullptr;
    TRY(bimamba2_chunk_scan_fwd(&q));
    return BIMAMBA2_OK;
}

int bimamba2_fwd_static(const bimamba2_params *p) {
    TRY(check_problem(p));
    bimamba2_params q = *p;
    q.workspace = nullptr;
    q.workspace_bytes = 0;
    {
        bimamba2_params sized = q;
        if (carve(&sized, 0, nullptr) > BIMAMBA2_STATIC_SCRATCH_BYTES) return BIMAMBA2_ESCRATCH;
    }
    // nothing in the forward pipeline accumulates into its intermediates: every one is written in full before it is
    // read, so what the last call left in the buffer does not matter
    TRY(static_scratch(&q.workspace));
    q.workspace_bytes = BIMAMBA2_STATIC_SCRATCH_BYTES;
    return bimamba2_fwd(&q);
}

// Which launches of a backward pass are there in a merged form; q: the caller's p with what it leaves to the pass carved
struct BwdForm {
    bool one;           // one chunk without states (a forward pass over one chunk leaves none: its caller says so)
    bool own_dcb;       // dCB and dCB^T are the pass's own
    bool dcb_sp;        // dCB with the backward state passing (one chunk: dCB's alone, with its place for 16-bit results)
    bool dcb16;         // dCB in the 16-bit element type: the two launches that write and read it are the merged ones (their reader rounds it to that type for its MFMA anyway)
    bool dx_db_dc;      // dx, dB and dC in one launch at the end
    bool by_heads;      // dB and dC in one launch, heads in turn
    bool product;       // and the part of both inside the chunks with them, where nobody asked for the partial sums
};
static BwdForm bwd_form(const bimamba2_params *p, const bimamba2_params *q) {
    BwdForm f;
    f.one = one_chunk(q) && (!p->fwd_saved || (p->fwd_saved & 4));
    f.own_dcb = !p->dCB && !p->dCBT;
    f.dcb_sp = (f.one ? dcb_recomputes_cb(q) && (q->headdim * q->dstate) % 4 == 0 : bwd_dcb_sp_merged(q)) && (f.own_dcb || dcb_slices(q) == 1);
    f.dcb16 = f.own_dcb && f.dcb_sp && dcb_slices(q) == 1 && bwd_tail_merged(q);
    f.dx_db_dc = !f.one && dx_db_dc_merged(q);
    f.by_heads = !f.one && !f.dx_db_dc && dbdc_both_by_heads(q);
    f.product = f.by_heads && f.dcb16 && !p->dBs && !p->dCs && dbdc_with_product(q);
    return f;
}

int bimamba2_bwd_db_dc_complete(const bimamba2_params *p) {
    if (check_problem(p)) return 0;
    bimamba2_params q = *p;
    q.final_f = q.final_b = nullptr;
    carve(&q, 1, reinterpret_cast<void *>(256));      // (a place to count from: nothing is read or written)
    return bwd_form(p, &q).product ? 1 : 0;
}

// leave: the final sums are appended to it instead of being launched
static int backward(const bimamba2_params *p, ReduceJobs *leave) {
    TRY(check_problem(p));
    bimamba2_params q = *p;
    q.final_f = q.final_b = nullptr;
    const size_t need = carve(&q, 1, p->workspace);
    if (need > 256 && (!p->workspace || p->workspace_bytes < need)) return BIMAMBA2_EWORKSPACE;
    if ((p->dBs || p->dCs) && p->dbdc_heads > 8) return BIMAMBA2_EINVAL;      // (a caller's slices; this call's own may be longer)
    // what a caller has to bring, before any launch: which stages run, and with them whose checks, depends on the problem
    REQUIRE(q.x); REQUIRE(q.dt); REQUIRE(q.A); REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.dout);
    REQUIRE(q.dx); REQUIRE(q.ddt); REQUIRE(q.dA); REQUIRE(q.dB); REQUIRE(q.dC);
    if (q.has_dt_bias) REQUIRE(q.dt_bias);
    if (q.has_D) { REQUIRE(q.D); REQUIRE(q.dD); }
    if (q.has_z) { REQUIRE(q.z); REQUIRE(q.out_x); REQUIRE(q.dz); }
    const BwdForm form = bwd_form(p, &q);
    const bool one = form.one, own_dcb = form.own_dcb, dcb_sp = form.dcb_sp, dcb16 = form.dcb16;
    if (p->fwd_saved) {
        REQUIRE(p->dt_out); REQUIRE(p->cs_f); REQUIRE(p->cs_b);
        if (!p->states16_f && !one) { REQUIRE(p->states_f); REQUIRE(p->states_b); }
    } else if (one) {
        bimamba2_params qs = q;
        qs.CB = nullptr;
        TRY(launch_fwd_cumsum_cb(&qs, one_chunk_free16(&q, true)));
    } else {
        // recompute the forward intermediates (the reference does the same, src/ssd/bi/ssd_combined.py:373-380)
        TRY(forward_cumsum_and_states(&q));
        TRY(bimamba2_state_passing_fwd(&q));
    }
    if (one) {
        // state parts that the caller has places for (the pass itself neither forms nor reads them): nothing crosses a chunk boundary
        const size_t rows = (size_t)q.batch * q.nheads * q.chunk_size, heads = q.nheads / q.ngroups, hps = p->dbdc_heads > 0 ? p->dbdc_heads : 8;
        const size_t sums = (heads + hps - 1) / hps * q.batch * q.seqlen * q.ngroups * q.dstate;
        for (float *t : {p->u_f, p->u_b, p->v_f, p->v_b})
            if (t) TRY(launch_fill(t, rows, 0.f, stream_of(&q)));
        for (float *t : {p->ddA_chunk_f, p->ddA_chunk_b})
            if (t) TRY(launch_fill(t, (size_t)q.batch * q.nheads * sp_nsplit(&q), 0.f, stream_of(&q)));
        for (float *t : {p->dBs, p->dCs})
            if (t) TRY(launch_fill(t, sums, 0.f, stream_of(&q)));
    }
    const bool need_cbt = !scan_recomputes_cb(&q, true), need_cb = need_cbt || !dcb_recomputes_cb(&q);
    const bool saved_cb = (p->fwd_saved & 2) && p->CB && p->CBT;
    const bool form_cb = need_cb && !saved_cb;     // (else left there by the forward pass)
    if (!need_cb) q.CB = nullptr;
    // dz and dstates as one launch where the kernel for it exists (dout_x goes from the first to the second inside the workgroup)
    const bool dz_dstates = q.has_z && !one && bwd_dz_dstates_fused(&q), dz_bmm = q.has_z && !dz_dstates && form_cb;
    if (form_cb && !dz_bmm) TRY(bimamba2_bmm_chunk_fwd(&q));  // CB for the dCB kernel, CB^T for the dx kernel, unless they rebuild it
    if (dz_dstates) TRY(bimamba2_chunk_scan_bwd_dz_dstates(&q));
    else if (dz_bmm) {
        REQUIRE(q.z); REQUIRE(q.dout); REQUIRE(q.out_x); REQUIRE(q.dz); REQUIRE(q.dout_x); REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.CB);
        TRY(launch_bwd_dz_bmm(&q));
    } else if (q.has_z) TRY(bimamba2_chunk_scan_bwd_dz(&q));
    // the last launch adds up the head slices of dCB
    const bool tail_small = !bwd_tail_merged(&q) && bwd_tail_small(&q);
    const int ncb = own_dcb && (tail_small || bwd_tail_merged(&q)) ? dcb_slices(&q) : 1;
    // the dCB kernel is bound by instruction issue and moves little data: right behind dz it runs while the memory system
    // still writes back dz's output, which the memory-bound kernels after it would otherwise wait behind
    const bool dx_db_dc = form.dx_db_dc, by_heads = form.by_heads, product = form.product;
    const bool both = by_heads || (!one && !dx_db_dc && db_dc_merged(&q));      // dC with dB
    if (dcb_sp && (ncb == dcb_slices(&q))) {
        // the backward state passing (streams, few instructions) rides along with the dCB kernel in one launch
        if (!dx_db_dc && !one && !both) TRY(bimamba2_chunk_scan_bwd_dc(&q));
        if (!dz_dstates && !one) TRY(bimamba2_chunk_scan_bwd_dstates(&q));
        REQUIRE(q.x); REQUIRE(q.dt_out); REQUIRE(q.cs_f); REQUIRE(q.cs_b); REQUIRE(q.dCB); REQUIRE(q.dCBT); REQUIRE(q.da_intra);
        if (!one) {
            if (!q.dstates16_f) REQUIRE(q.dstates_f);
            REQUIRE(q.ddA_chunk_f); REQUIRE(q.ddA_chunk_b);
        }
        if (q.has_z) REQUIRE(q.dout_x); else REQUIRE(q.dout);
        bimamba2_params qd = q;
        if (product) qd.dCBT = nullptr;      // (nobody reads it)
        TRY(launch_bwd_dcb_sp(&qd, dcb16));
    } else {
        TRY(check_bwd_dcb(&q));
        if (one) TRY(launch_bwd_dcb(&q, ncb == 1));
        else if (!dz_dstates && ncb == dcb_slices(&q) && dcb_dstates_merged(&q)) {
            REQUIRE(q.Cm);
            TRY(launch_dcb_dstates(&q));
        } else {
            TRY(launch_bwd_dcb(&q, ncb == 1));
            if (!dz_dstates) TRY(bimamba2_chunk_scan_bwd_dstates(&q));
        }
        if (!one) {
            if (!dx_db_dc && !both) TRY(bimamba2_chunk_scan_bwd_dc(&q));           // (between the two memory-bound state kernels: measured best)
            TRY(bimamba2_state_passing_bwd(&q));
        }
    }
    if (dx_db_dc) {
        REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.dBs); REQUIRE(q.dCs); REQUIRE(q.u_f); REQUIRE(q.u_b); REQUIRE(q.v_f); REQUIRE(q.v_b);
        REQUIRE(q.states_f); REQUIRE(q.states_b); REQUIRE(q.dstates_f); REQUIRE(q.dstates_b);
    } else if (both) {
        REQUIRE(q.x); REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.dBs); REQUIRE(q.dCs); REQUIRE(q.u_f); REQUIRE(q.u_b); REQUIRE(q.v_f); REQUIRE(q.v_b);
        if (!by_heads) { REQUIRE(q.states_f); REQUIRE(q.states_b); REQUIRE(q.dstates_f); REQUIRE(q.dstates_b); }
        TRY(by_heads ? launch_dbdc_both(&q, product) : launch_db_dc(&q));
    } else if (!one) TRY(bimamba2_chunk_state_bwd_db(&q));
    ReduceJobs jobs;
    {
        // as bimamba2_chunk_scan_bwd_dx, with the reduction of the dD partial sums left for the end
        bimamba2_params qx = q;
        if (scan_recomputes_cb(&q, true)) qx.CBT = nullptr;
        REQUIRE(qx.dx); REQUIRE(qx.ddt_direct);
        if (qx.has_D) { REQUIRE(qx.D); REQUIRE(qx.dD); }
        const int nc = nchunks(&q);
        TRY(dx_db_dc ? launch_dx_db_dc(&qx) : launch_chunk_scan(&qx, true, one && one_chunk_free16(&q, true)));
        if (q.has_D) {
            if (q.D_has_hdim) jobs.job[jobs.n++] = ReduceJob{q.red, q.dD, q.batch * nc, q.nheads * q.headdim, 1};
            else jobs.job[jobs.n++] = ReduceJob{q.red, q.dD, q.batch * nc, q.nheads, q.headdim};
        }
    }
    {
        // as bimamba2_bmm_chunk_bwd and bimamba2_chunk_cumsum_bwd (its partial sums behind those of dD): one launch for
        // both where the kernel for it exists
        bimamba2_params qc = q;
        qc.red = q.red + (size_t)q.batch * nchunks(&q) * q.nheads * q.headdim;
        REQUIRE(q.ddt); REQUIRE(q.dA); REQUIRE(q.dB); REQUIRE(q.dC);
        if (product) {
            TRY(launch_chunk_cumsum_bwd(&qc, &jobs));
        } else if (bwd_tail_merged(&q)) {
            TRY(launch_bwd_tail(&qc, &jobs, dcb16, ncb));
        } else if (tail_small) {
            REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.dt); REQUIRE(q.A);
            if (q.has_dt_bias) REQUIRE(q.dt_bias);
            TRY(launch_bwd_tail_small(&qc, &jobs, ncb));
        } else if (one) {
            REQUIRE(q.Bm); REQUIRE(q.Cm); REQUIRE(q.dt); REQUIRE(q.A);
            if (q.has_dt_bias) REQUIRE(q.dt_bias);
            TRY(launch_bmm_chunk_bwd(&q));
            TRY(launch_chunk_cumsum_bwd(&qc, &jobs));
        } else {
            TRY(bimamba2_bmm_chunk_bwd(&q));
            TRY(launch_chunk_cumsum_bwd(&qc, &jobs));
        }
    }
    if (leave) *leave = jobs;
    else TRY(launch_reduce_jobs(jobs, stream_of(&q)));
    return BIMAMBA2_OK;
}

int bimamba2_bwd(const bimamba2_params *p) { return backward(p, nullptr); }

size_t bimamba2_norm_params_size(void) { return sizeof(bimamba2_norm_params); }

static int check_norm(const bimamba2_norm_params *p) {
    if (!p) return BIMAMBA2_EINVAL;
    if (p->rows < 0 || p->cols <= 0 || p->group_size <= 0 || p->cols % p->group_size) return BIMAMBA2_EINVAL;
    if (p->dtype != BIMAMBA2_F32 && p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
    if (p->group_size > 32768) return BIMAMBA2_EUNSUPPORTED;
    if (!p->x || !p->weight || (p->has_z && !p->z) || (p->has_bias && !p->bias)) return BIMAMBA2_EINVAL;
    return BIMAMBA2_OK;
}

size_t bimamba2_rmsnorm_gated_workspace_bytes(const bimamba2_norm_params *p) {
    if (check_norm(p)) return 0;
    return norm_workspace_bytes(p);
}

int bimamba2_rmsnorm_gated_fwd(const bimamba2_norm_params *p) {
    TRY(check_norm(p));
    REQUIRE(p->out);
    if (p->rows == 0) return BIMAMBA2_OK;
    return launch_rmsnorm_gated(p, false);
}

static int check_norm_bwd(const bimamba2_norm_params *p) {
    TRY(check_norm(p));
    REQUIRE(p->dout); REQUIRE(p->rstd); REQUIRE(p->dx); REQUIRE(p->dweight);
    if (p->layer_norm) REQUIRE(p->mean);
    if (p->has_z) REQUIRE(p->dz);
    if (p->has_bias) REQUIRE(p->dbias);
    if (!p->workspace || p->workspace_bytes < norm_workspace_bytes(p)) return BIMAMBA2_EWORKSPACE;
    return BIMAMBA2_OK;
}

int bimamba2_rmsnorm_gated_bwd(const bimamba2_norm_params *p) {
    TRY(check_norm_bwd(p));
    return launch_rmsnorm_gated(p, true);
}

size_t bimamba2_conv_params_size(void) { return sizeof(bimamba2_conv_params); }

size_t bimamba2_cast_params_size(void) { return sizeof(bimamba2_cast_params); }

static int check_cast(const bimamba2_cast_params *p) {
    if (!p || p->count < 0 || p->count > BIMAMBA2_CAST_MAX) return BIMAMBA2_EINVAL;
    auto known = [](int d) { return d == BIMAMBA2_F32 || d == BIMAMBA2_BF16 || d == BIMAMBA2_F16; };
    for (int k = 0; k < p->count; ++k) {
        const bimamba2_cast_item &it = p->item[k];
        if (it.n < 0 || (it.n > 0 && (!it.src || !it.dst))) return BIMAMBA2_EINVAL;
        if (!known(it.src_dtype) || !known(it.dst_dtype)) return BIMAMBA2_EUNSUPPORTED;
        if (it.op < BIMAMBA2_CAST_COPY || it.op > BIMAMBA2_CAST_MUL) return BIMAMBA2_EINVAL;
        if (it.op == BIMAMBA2_CAST_MUL && it.n > 0 && !it.aux) return BIMAMBA2_EINVAL;
    }
    return BIMAMBA2_OK;
}

int bimamba2_cast_many(const bimamba2_cast_params *p) {
    TRY(check_cast(p));
    return launch_cast_many(p);
}

static int check_conv(const bimamba2_conv_params *p) {
    if (!p) return BIMAMBA2_EINVAL;
    if (p->batch < 0 || p->seqlen < 0 || p->channels <= 0) return BIMAMBA2_EINVAL;
    if (p->dtype != BIMAMBA2_F32 && p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
    if (p->width < 1 || p->width > 9 || p->width % 2 == 0) return BIMAMBA2_EUNSUPPORTED;
    if (p->seqlen > (1 << 30)) return BIMAMBA2_EUNSUPPORTED;
    if (!p->x || !p->weight || (p->has_bias && !p->bias)) return BIMAMBA2_EINVAL;
    return BIMAMBA2_OK;
}

size_t bimamba2_conv1d_silu_workspace_bytes(const bimamba2_conv_params *p) {
    if (check_conv(p)) return 0;
    return conv_workspace_bytes(p);
}

int bimamba2_conv1d_silu_fwd(const bimamba2_conv_params *p) {
    TRY(check_conv(p));
    REQUIRE(p->out);
    if (p->batch == 0 || p->seqlen == 0) return BIMAMBA2_OK;
    return launch_conv1d_silu(p, false);
}

static int check_conv_bwd(const bimamba2_conv_params *p) {
    TRY(check_conv(p));
    REQUIRE(p->dout); REQUIRE(p->dx); REQUIRE(p->dweight);
    if (p->has_bias) REQUIRE(p->dbias);
    if (!p->workspace || p->workspace_bytes < conv_workspace_bytes(p)) return BIMAMBA2_EWORKSPACE;
    return BIMAMBA2_OK;
}

int bimamba2_conv1d_silu_bwd(const bimamba2_conv_params *p) {
    TRY(check_conv_bwd(p));
    if (p->batch == 0 || p->seqlen == 0) {
        TRY(launch_fill(p->dweight, (size_t)p->channels * p->width, 0.f, reinterpret_cast<hipStream_t>(p->stream)));
        if (p->has_bias) TRY(launch_fill(p->dbias, (size_t)p->channels, 0.f, reinterpret_cast<hipStream_t>(p->stream)));
        return BIMAMBA2_OK;
    }
    return launch_conv1d_silu(p, true);
}

int bimamba2_norm_scan_conv_bwd(const bimamba2_norm_params *norm, const bimamba2_params *scan, const bimamba2_conv_params *conv,
                                const bimamba2_cast_params *casts) {
    TRY(check_norm_bwd(norm));
    TRY(check_problem(scan));
    TRY(check_conv_bwd(conv));
    TRY(check_cast(casts));
    if (norm->rows == 0 || conv->batch == 0 || conv->seqlen == 0) return BIMAMBA2_EINVAL;
    if (norm->stream != scan->stream || conv->stream != scan->stream) return BIMAMBA2_EINVAL;
    LayerSums sums;
    TRY(launch_rmsnorm_gated(norm, true, &sums));
    TRY(backward(scan, &sums.jobs));
    TRY(launch_conv1d_silu(conv, true, &sums));
    return launch_layer_sums(sums, casts, stream_of(scan));
}

size_t bimamba2_gemm_params_size(void) { return sizeof(bimamba2_gemm_params); }

static int check_gemm(const bimamba2_gemm_params *p) {
    if (!p || p->m <= 0 || p->n <= 0 || p->k <= 0 || !p->a || !p->b || !p->c) return BIMAMBA2_EINVAL;
    if (p->dtype != BIMAMBA2_BF16 && p->dtype != BIMAMBA2_F16) return BIMAMBA2_EUNSUPPORTED;
    auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (!al16(p->a) || !al16(p->b) || !al16(p->c) || p->lda % 8 || p->ldb % 8 || p->ldc < p->n) return BIMAMBA2_EUNSUPPORTED;
    auto up8 = [](int64_t v) { return (v + 7) / 8 * 8; };
    if (p->lda < up8(p->a_kcontig ? p->k : p->m) || p->ldb < up8(p->b_kcontig ? p->k : p->n)) return BIMAMBA2_EUNSUPPORTED;
    // offsets inside a tile are 32-bit products of 24-bit factors: 256 rows of k, or the whole k range of rows
    if (p->lda >= (1 << 23) || p->ldb >= (1 << 23) || p->k >= (1 << 24)) return BIMAMBA2_EUNSUPPORTED;
    const int64_t most = int64_t(1) << 31;
    if ((p->a_kcontig ? 256 : (int64_t)p->k) * p->lda * 2 + 2 * (int64_t)p->k >= 2 * most) return BIMAMBA2_EUNSUPPORTED;
    if ((p->b_kcontig ? 256 : (int64_t)p->k) * p->ldb * 2 + 2 * (int64_t)p->k >= 2 * most) return BIMAMBA2_EUNSUPPORTED;
    if (!p->a_kcontig && p->b_kcontig) return BIMAMBA2_EUNSUPPORTED;
    if (p->b_kcontig && p->k % 8) return BIMAMBA2_EUNSUPPORTED;   // (no caller has such rows of B)
    return BIMAMBA2_OK;
}

int bimamba2_gemm_plan(const bimamba2_gemm_params *p, int *slices) {
    if (!p || !slices || p->m <= 0 || p->n <= 0 || p->k <= 0) return BIMAMBA2_EINVAL;
    int tile;
    gemm_plan_of(p, &tile, slices);
    return tile;
}

size_t bimamba2_gemm_workspace_bytes(const bimamba2_gemm_params *p) { return check_gemm(p) ? 0 : gemm_workspace_bytes(p); }

int bimamba2_gemm(const bimamba2_gemm_params *p) {
    TRY(check_gemm(p));
    const size_t need = gemm_workspace_bytes(p);
    if (need && (!p->partial || p->partial_bytes < need)) return BIMAMBA2_EWORKSPACE;
    return launch_gemm(p);
}

}  // extern "C"
