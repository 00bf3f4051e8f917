// Adjoint gradient contraction: g_e = sum_r -omega_r mu0 Im(lam_e^T M_e x_e).
#include <hip/hip_runtime.h>

#include "pg_adjoint.h"
#include "pg_common.h"
#include "pg_factor.h"

namespace pg {
namespace {

constexpr int kBS = 256;

// the value of the neighbouring lane (lane ^ 1)
__device__ inline double swap_pair(double v) {
  constexpr int kQuad = 0xB1;  // quad_perm [1, 0, 3, 2]
  return __hiloint2double(
      __builtin_amdgcn_mov_dpp(__double2hiint(v), kQuad, 0xF, 0xF, true),
      __builtin_amdgcn_mov_dpp(__double2loint(v), kQuad, 0xF, 0xF, true));
}

// omega_r mu0 of the columns of one launch, passed with the launch
constexpr int kCols = 32;
struct Omegas {
  double v[kCols];
};

// DOF offsets within a column: bytes in 32 bits where a column ends below 4 GiB
// (one add per gather), 64-bit otherwise
template <typename O>
__device__ inline double at(const double* __restrict__ col, O off) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(col) + off);
}

// Two neighbouring lanes per element, the real and the imaginary part of x: each
// forms M_e of its real vector (factored, pg_factor.h) and its product with the
// other part of lam: Im(lam^T M x) = lam_im M x_re + lam_re M x_im.
// Bound: FP64 issue and the gathers of x and lam.  93 750 elements, p = 2, two
// columns: 19 us (the bytes alone 11 us) against 485 us with one thread per
// element, every entry of M_e contracted from a gathered table row; p = 2, eight
// columns on arbitrary numbering 5.3 -> 0.18 ms, p = 3 (10 368 elements, nine
// columns) 7.7 -> 0.10 ms.  At p = 2 two waves per SIMD with lam in flight during
// the product beat three without (74 against 89 us a call before the 32-bit
// offsets); at p = 3 the same would spill.
template <int P, typename O>
__global__ void __launch_bounds__(kBS, (P == 1 ? 3 : (P == 2 ? 2 : 1))) k_adjoint_grad(
    int64_t E, const double* __restrict__ coef, const int32_t* __restrict__ orient,
    const int32_t* __restrict__ dofs, int nrhs, int64_t sd, int64_t sr,
    const double* __restrict__ x, const double* __restrict__ lam, const Omegas om,
    double* __restrict__ g) {
  constexpr int N = fac::n_dofs<P>();
  __shared__ double faces[fac::face_table_size<P>()];
  if constexpr (P > 1) {
    constexpr auto t = fac::kFaces<P>;
    for (int i = threadIdx.x; i < fac::face_table_size<P>(); i += kBS) faces[i] = t.v[i];
    __syncthreads();
  }
  const int64_t nb = gridDim.x;
  int64_t b = blockIdx.x;
  if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;  // XCD-contiguous ranges of elements
  const int64_t e = b * (kBS / 2) + threadIdx.x / 2;
  const int part = threadIdx.x & 1;
  if (e >= E) return;  // both lanes of a pair
  O off[N];
#pragma unroll
  for (int i = 0; i < N; ++i) off[i] = (O)dofs[e * N + i] * (O)(16 * sd);
  const int pk = orient[e];
  double cf[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) cf[c] = coef[12 * e + c];
  double acc = 0.0;
  for (int r = 0; r < nrhs; ++r) {
    const double* xr = x + 2 * r * sr + part;
    const double* lr = lam + 2 * r * sr + (1 - part);
    double xv[N], m[N];
#pragma unroll
    for (int i = 0; i < N; ++i) xv[i] = at(xr, off[i]);
    fac::orient_in<P>(pk, faces, xv);
    fac::mass_product<P, double>(xv, cf, [&](int i, double v) { m[i] = v; });
    // p = 3: lam is loaded once the intermediates are gone (it would spill);
    // p = 2: during them
    if (P == 3) __builtin_amdgcn_sched_barrier(0);
    fac::orient_out<P>(pk, faces, m);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) s += at(lr, off[i]) * m[i];
    acc += -om.v[r] * (s + swap_pair(s));
  }
  if (part == 0) g[e] += acc;
}

}  // namespace

void launch_adjoint_grad(int p, int64_t E, const double* coef, const int32_t* orient,
                         const int32_t* dofs, int64_t ndof, int nrhs, int64_t sd, int64_t sr,
                         const double2* x, const double2* lam, const double* omega_mu, double* g,
                         hipStream_t st) {
  int64_t nb = (2 * E + kBS - 1) / kBS;
  if (nb >= 64) nb = (nb + 7) / 8 * 8;
  const dim3 gr((unsigned)nb), bl(kBS);
  const bool small = ndof * sd < (1LL << 28);  // of 16 bytes
  for (int r0 = 0; r0 < nrhs; r0 += kCols) {
    const int nr = nrhs - r0 < kCols ? nrhs - r0 : kCols;
    Omegas om{};
    for (int r = 0; r < nr; ++r) om.v[r] = omega_mu[r0 + r];
    const double* xr = reinterpret_cast<const double*>(x + r0 * sr);
    const double* lr = reinterpret_cast<const double*>(lam + r0 * sr);
#define PG_GRAD(P, O)                                                                         \
  hipLaunchKernelGGL((k_adjoint_grad<P, O>), gr, bl, 0, st, E, coef, orient, dofs, nr, sd, sr, \
                     xr, lr, om, g)
    if (p == 1 && small) PG_GRAD(1, uint32_t);
    else if (p == 1) PG_GRAD(1, int64_t);
    else if (p == 2 && small) PG_GRAD(2, uint32_t);
    else if (p == 2) PG_GRAD(2, int64_t);
    else if (small) PG_GRAD(3, uint32_t);
    else PG_GRAD(3, int64_t);
#undef PG_GRAD
  }
}

}  // namespace pg
