// The launches of roles.hpp for f32.
#include "roles.hpp"

namespace bm2 {

int launch_dcb_dstates_f32(const bimamba2_params *p, const RolesShape &r) { return launch_dcb_dstates_t<float>(p, r); }
int launch_dx_db_dc_f32(const bimamba2_params *p, const RolesShape &r) { return launch_dx_db_dc_t<float>(p, r); }

}  // namespace bm2
