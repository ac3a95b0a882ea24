// The launches of roles.hpp for f16.
#include "roles.hpp"

namespace bm2 {

int launch_dcb_dstates_f16(const bimamba2_params *p, const RolesShape &r) { return launch_dcb_dstates_t<f16_t>(p, r); }
int launch_dx_db_dc_f16(const bimamba2_params *p, const RolesShape &r) { return launch_dx_db_dc_t<f16_t>(p, r); }

}  // namespace bm2
