// The launches of roles.hpp for bf16.
#include "roles.hpp"

namespace bm2 {

int launch_dcb_dstates_bf16(const bimamba2_params *p, const RolesShape &r) { return launch_dcb_dstates_t<bf16_t>(p, r); }
int launch_dx_db_dc_bf16(const bimamba2_params *p, const RolesShape &r) { return launch_dx_db_dc_t<bf16_t>(p, r); }

}  // namespace bm2
