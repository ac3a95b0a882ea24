// Host-side declarations shared by the kernel files and the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/bimamba2.h"

namespace bm2 {

struct BlockId { int x, y, z; };      // a workgroup's place in the grid of its kernel, or of its role in a launch of several

static inline int check_launch() { return hipGetLastError() == hipSuccess ? BIMAMBA2_OK : BIMAMBA2_ELAUNCH; }

// Width of the headdim column tile of the chunk-scan kernels (64 columns for 16-bit types, 32 for float32, less for narrow
// heads), and with it the number of planes of ddt_direct: every column tile of the dx kernel writes the row sums of its own
// columns to its own (batch, nheads, nchunks, chunk_size) plane, and the reader adds the planes in order (no atomics).
__host__ __device__ inline int scan_col_tile_of(int headdim, int dtype) {
    return headdim <= 16 ? 16 : (headdim <= 32 || dtype == BIMAMBA2_F32) ? 32 : 64;
}
__host__ __device__ inline int ddt_direct_planes(const bimamba2_params &p) {
    const int pw = scan_col_tile_of(p.headdim, p.dtype);
    return (p.headdim + pw - 1) / pw;
}

int launch_chunk_cumsum_fwd(const bimamba2_params *p);
int launch_seq_boundaries(const bimamba2_params *p, int32_t *counts);
int launch_bmm_chunk_fwd(const bimamba2_params *p);
int launch_fwd_cumsum_cb(const bimamba2_params *p, bool states16);     // chunk cumsum and, with p->CB, C.B^T in one launch
int launch_chunk_state(const bimamba2_params *p, bool dstates, bool cumsum = false);   // cumsum: also does the chunk cumsum
bool chunk_state_does_cumsum(const bimamba2_params *p);
bool chunk_state_narrow(const bimamba2_params *p, bool dstates);
// chunk cumsum, chunk states and C.B^T (left out where CB is NULL) as one launch, where fwd_front_merged() says it exists
bool fwd_front_merged(const bimamba2_params *p);
int launch_fwd_front(const bimamba2_params *p);
// the forward pass may keep its per-chunk states in states16_f/b only (16-bit type, no float32 state tensors)
bool chunk_states_in_16bit(const bimamba2_params *p);
// the chunk-state kernel whose workgroups walk through several heads of one (batch, chunk): where it is used, and its launch
bool chunk_state_uses_heads_kernel(const bimamba2_params *p);
int launch_chunk_state_heads(const bimamba2_params *p);
int launch_state_passing_fwd(const bimamba2_params *p);
int launch_chunk_scan(const bimamba2_params *p, bool bwd, bool free16 = false);
// a forward pass over a short sequence in one launch (kernels_scan_once.hip), and where it is the one to run
bool scan_once_applies(const bimamba2_params *p);
bool scan_once_walks(const bimamba2_params *p);       // ... by workgroups that own whole sequences
int launch_scan_once(const bimamba2_params *p);
// the 16-bit kernel of kernels_scan16.hip (launch_chunk_scan picks it where it applies)
int launch_chunk_scan16(const bimamba2_params *p, bool bwd);
// heads of one group that a workgroup of that kernel walks through (they share one C.B^T product)
int chunk_scan16_heads_per_workgroup(const bimamba2_params *p);
// whether launch_chunk_scan() would pick that kernel for this problem (the 16-bit copies of the entering states given)
bool chunk_scan_uses_scan16(const bimamba2_params *p, bool bwd);
// true when that launch recomputes CB (bwd: CB^T) from the C and B rows instead of reading it
bool scan_recomputes_cb(const bimamba2_params *p, bool bwd);
// true when the dCB launch can rebuild its CB tiles from the C and B rows (then CB may be NULL)
bool dcb_recomputes_cb(const bimamba2_params *p);

int launch_bwd_dz(const bimamba2_params *p);
int launch_bwd_dz_bmm(const bimamba2_params *p);       // dz and C.B^T in one launch
bool bwd_dz_dstates_fused(const bimamba2_params *p);   // dz and dstates as one launch
int launch_bwd_dz_dstates(const bimamba2_params *p);
int launch_state_passing_bwd(const bimamba2_params *p);
int choose_dbdc_heads(const bimamba2_params *p, bool by_heads, bool together);   // heads per slice of the dB / dC partial sums; by_heads: for the next three; together: db_dc_roles()
bool dbdc_by_heads(const bimamba2_params *p);       // dB and dC by waves that take whole heads, given 16-bit copies of the states
bool dbdc_both_by_heads(const bimamba2_params *p);  // with them given
bool dbdc_with_product(const bimamba2_params *p);   // and one slice of heads, chunks of 256: with dCB in 16 bits it can write dB and dC themselves
int launch_dbdc_both(const bimamba2_params *p, bool product);     // both in one launch
int launch_bwd_dbdc(const bimamba2_params *p, bool is_db);
int launch_bwd_dcb(const bimamba2_params *p, bool add_up = true);   // add_up: also the launch that adds several head slices up
int choose_dcb_slices(const bimamba2_params *p);
int dcb_slices(const bimamba2_params *p);   // head slices whose dCB partial sums the kernel keeps apart
int launch_bmm_chunk_bwd(const bimamba2_params *p);
// out[j] = sum_i sum_k in[(i*nj + j)*nk + k]
struct ReduceJob { const float *in; float *out; int ni, nj, nk; };
struct ReduceJobs { ReduceJob job[4]; int n = 0; };
int launch_reduce_jobs(const ReduceJobs &jobs, hipStream_t stream);
// out[j] = sum_i in[i*nj + j]; width > 0: columns are rows of width + 1, whose last goes to extra (NULL: nowhere) and the others to out
struct ColumnSums { const float *in; float *out, *extra; int ni, nj, width; };
// the final sums that several backward stages leave to one launch
struct LayerSums { ReduceJobs jobs; ColumnSums cols[3]; int ncols = 0; };
// casts: which of the sums leave in another type or multiplied (the item's source is the float32 place, which is not written then);
// BIMAMBA2_EINVAL where an item is none of the sums
int launch_layer_sums(const LayerSums &sums, const bimamba2_cast_params *casts, hipStream_t stream);
// defer != NULL: the final reductions of dA and ddt_bias are appended to *defer instead of being launched
int launch_chunk_cumsum_bwd(const bimamba2_params *p, ReduceJobs *defer = nullptr);
// bmm_chunk_bwd and chunk_cumsum_bwd as one launch, where bwd_tail_merged() says it exists
// the dCB kernel and the backward state passing as one launch, where bwd_dcb_sp_merged() says it exists
bool bwd_dcb_sp_merged(const bimamba2_params *p);
// out16 / in16: dCB and dCBT in the element type of the inputs between the two launches (one head slice: the reader rounds
// them to that type anyway)
int launch_bwd_dcb_sp(const bimamba2_params *p, bool out16 = false);
bool bwd_tail_merged(const bimamba2_params *p);
int launch_bwd_tail(const bimamba2_params *p, ReduceJobs *defer, bool in16 = false, int ncb = 1);
// the same for chunks of up to 128 positions, any type and shape (ncb: head slices of dCB still to be added up)
bool bwd_tail_small(const bimamba2_params *p);
int launch_bwd_tail_small(const bimamba2_params *p, ReduceJobs *defer, int ncb);
// launches of several roles (roles.hpp), with what their kernels' own launches know about the problem
struct RolesShape {
    int nchunks, dcb_slices, dbdc_slices, dbdc_heads;
    bool dcb_ring, dcb_fast, dstates_fast, dstates_narrow, dbdc_fast, dx;
};
bool dcb_dstates_merged(const bimamba2_params *p);      // dCB and dstates in one launch
int launch_dcb_dstates(const bimamba2_params *p);
bool dx_db_dc_merged(const bimamba2_params *p);         // dx, dB and dC in one launch
int launch_dx_db_dc(const bimamba2_params *p);
bool db_dc_roles(const bimamba2_params *p, bool states16);      // dB and dC in one launch, with dx or without; states16: the states in 16-bit copies
bool db_dc_merged(const bimamba2_params *p);
int launch_db_dc(const bimamba2_params *p);
int launch_dcb_dstates_f32(const bimamba2_params *p, const RolesShape &r);
int launch_dcb_dstates_bf16(const bimamba2_params *p, const RolesShape &r);
int launch_dcb_dstates_f16(const bimamba2_params *p, const RolesShape &r);
int launch_dx_db_dc_f32(const bimamba2_params *p, const RolesShape &r);
int launch_dx_db_dc_bf16(const bimamba2_params *p, const RolesShape &r);
int launch_dx_db_dc_f16(const bimamba2_params *p, const RolesShape &r);
bool scan_is_fast(const bimamba2_params *p, bool bwd);  // the scan kernel without guarded fallbacks applies
int launch_fill(float *ptr, size_t n, float value, hipStream_t stream);
// out[j] = sum_{i<ni} sum_{k<nk} in[(i*nj + j)*nk + k]
int launch_reduce(const float *in, float *out, int ni, int nj, int nk, hipStream_t stream);

// gated RMSNorm (kernels_norm.hip)
int launch_rmsnorm_gated(const bimamba2_norm_params *p, bool bwd, LayerSums *leave = nullptr);   // leave: the sums are appended instead of launched
size_t norm_workspace_bytes(const bimamba2_norm_params *p);

// depthwise conv1d + SiLU (kernels_conv.hip)
int launch_conv1d_silu(const bimamba2_conv_params *p, bool bwd, LayerSums *leave = nullptr);
size_t conv_workspace_bytes(const bimamba2_conv_params *p);
// several small element-wise conversions in one launch (kernels_conv.hip)
int launch_cast_many(const bimamba2_cast_params *p);

// matrix products of the layer's projections (kernels_gemm.hip)
int launch_gemm(const bimamba2_gemm_params *p);
size_t gemm_workspace_bytes(const bimamba2_gemm_params *p);
void gemm_plan_of(const bimamba2_gemm_params *p, int *tile, int *slices);     // tile 0: 256 x 256, 1: 256 x 192, 2: 128 x 128, 3: 64 x 64

}  // namespace bm2
