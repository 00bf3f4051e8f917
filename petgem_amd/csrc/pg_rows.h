// Element matrices and numeric assembly (kernels in pg_rows.hip), launched by the
// entry points in pg_element.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/petgem_amd.h"

namespace pg {

// M, K (E, n, n) row-major of E elements of order p from the geometry workspace
void launch_element_matrices(int p, int64_t E, const double* coef, const int32_t* orient,
                             double* M, double* K, hipStream_t st);

// CSR values of the plan's system: K_e - i omega_mu M_e into `values` (complex), or,
// with Kout, K_e and M_e into Kout and Mout
void launch_assembly(const pg_plan_dev& pl, const double* coef, const int32_t* orient,
                     double omega_mu, const uint8_t* ent_bc, double2* values, double* Kout,
                     double* Mout, hipStream_t st);

}  // namespace pg
