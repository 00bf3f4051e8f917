// Adjoint gradient contraction (kernel in pg_adjoint.hip), launched by the entry
// points in pg_element.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pg {

// g[e] += sum_r -omega_mu[r] Im(lam_r,e^T M_e x_r,e) for E elements of order p;
// column r of x and lam holds DOF d < ndof at d * sd + r * sr.  coef, orient: the
// geometry workspace; omega_mu: host array (nrhs), read before the call returns.
void launch_adjoint_grad(int p, int64_t E, const double* coef, const int32_t* orient,
                         const int32_t* dofs, int64_t ndof, int nrhs, int64_t sd, int64_t sr,
                         const double2* x, const double2* lam, const double* omega_mu, double* g, hipStream_t st);

}  // namespace pg
