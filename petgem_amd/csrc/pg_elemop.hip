// Element-by-element ("matrix-free") application of the assembled operator
//     A = sum_e P_e^T (K_e - i omega mu0 M_e) P_e,   PEC rows and columns -> identity,
// for gfx950, as an alternative to the CSR SpMV inside the Krylov solver.
//
// The element matrices are never stored: two lanes take one element (real and
// imaginary part), any orientation, and form K_e x and M_e x from 12 geometric
// coefficients by expanding field and curl in Bernstein monomials (pg_factor.h).
// Two forms:
//
//  k_eop_blk    p <= 2: one kernel; a workgroup owns a cluster of entities,
//               computes every element around them and sums their results in LDS.
//  k_eop_fac    the element products alone, writing the elements' n local results
//               (slot layout [group][i][element of 64]), and
//  k_eop_sum    one thread per mesh entity (edge, face), in the entity
//               schedule: sums the entity's local results over its elements
//               in a fixed order (atomic-free, bitwise reproducible), and
//               fuses the COCG dot product or the residual (k_eop_sum_dof: one
//               thread per DOF, small p = 3 operators).
//
// Orders p = 1, 2 and 3 (n = 6, 20, 45), complex128 and complex64.  The summation
// order differs from the assembled CSR's, so results agree with the CSR SpMV to
// rounding.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

#include "pg_basis.h"
#include "pg_common.h"
#include "pg_eop.h"
#include "pg_factor.h"

namespace pg {

namespace eop {

constexpr int kBS = 256;
constexpr int kMaxGrid = 2048;
// waves per SIMD the element products are compiled for
template <int P, typename R>
constexpr int fac_waves() {
  return P == 3 ? (sizeof(R) == 8 ? 1 : 2) : (sizeof(R) == 8 ? 3 : 5);
}
constexpr double kMu0 = 4.0 * 3.14159265358979323846 * 1e-7;  // petgem/solver.py:175

template <typename R>
struct Cx;
template <>
struct Cx<double> {
  using T = double2;
};
template <>
struct Cx<float> {
  using T = float2;
};

// local entities carrying DOFs (edges; faces from p = 2; the volume at p = 3),
// their first local DOF and their number of DOFs
template <int P>
constexpr int n_local_entities() {
  return P == 1 ? 6 : (P == 2 ? 10 : 11);
}
template <int P>
constexpr int loc_off(int la) {
  return la < 6 ? la * P : (la < 10 ? 6 * P + (la - 6) * P * (P - 1) : 6 * P + 4 * P * (P - 1));
}
template <int P>
constexpr int loc_nd(int la) {
  return la < 6 ? P : (la < 10 ? P * (P - 1) : P * (P - 1) * (P - 2) / 2);
}

__device__ inline double2 to_d(double2 v) { return v; }
__device__ inline double2 to_d(float2 v) { return make_double2(v.x, v.y); }
__device__ inline void store(double2* p, double2 v) { *p = v; }
__device__ inline void store(float2* p, double2 v) { *p = make_float2((float)v.x, (float)v.y); }

// the value of the neighbouring lane (lane ^ 1)
__device__ inline int swap_pair(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);  // quad_perm [1, 0, 3, 2]
}
__device__ inline float swap_pair(float v) { return __int_as_float(swap_pair(__float_as_int(v))); }
__device__ inline double swap_pair(double v) {
  return __hiloint2double(swap_pair(__double2hiint(v)), swap_pair(__double2loint(v)));
}

// the face coefficients of the factored products, to LDS; all threads
template <int P, typename R>
__device__ inline void fac_fill(R* faces) {
  if constexpr (P > 1) {
    constexpr auto t = fac::kFaces<P>;
    for (int i = threadIdx.x; i < fac::face_table_size<P>(); i += blockDim.x) faces[i] = (R)t.v[i];
    __syncthreads();
  }
}

template <int NV>
__device__ inline void write_partials(double (&v)[NV], double* part) {
  __shared__ double sm[NV][kBS / kWave];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) sm[k][w] = v[k];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
      for (int i = 0; i < kBS / kWave; ++i) s += sm[k][i];
      part[(int64_t)k * gridDim.x + blockIdx.x] = s;
    }
}

// ---------------------------------------------------------------------------
// local products in factored form (pg_factor.h).  Slots: group w of 64 elements,
// element l of the group; edofs[w][la][l] = first global DOF of local entity la, -1 for a PEC entity or an empty slot (its x is taken as 0);
// ocode[w][l] the packed orientation; coef[w][c][l]: c < 6 the mass
// coefficients times -omega mu0, c >= 6 the curl-curl coefficients.  Two
// neighbouring lanes take one element: lane 2 i the real part of x, lane
// 2 i + 1 the imaginary part, each forming K x and M x of its real vector and
// giving the other M x (y_re = K x_re - M' x_im, y_im = K x_im + M' x_re), so
// a wave holds 32 elements and the registers of one real vector each.
// Bound: memory, about 220 MB of indices, coefficients, x and local results in
// 48 us at 384 000 elements, p = 2, complex128 (4.6 TB/s; a copy reaches 5.1).
// One lane per element of one orientation combination per wave, entries formed
// from scalar table loads (two waves per SIMD, waiting for the scalar cache),
// took 107 us; on a mesh of 55 566 elements with arbitrary orientations, one
// element per wave, 420 us against 12 us now.  p = 3, 82 944 elements: 20 us in
// complex64 against 151 us from tables, 34 us in complex128 (302 registers, one
// wave per SIMD; two waves with 256 are no faster) against 326 us as a dense
// product with the tables on the FP64 matrix cores.
// ---------------------------------------------------------------------------
template <int P, typename R>
__global__ void __launch_bounds__(kBS, (fac_waves<P, R>())) k_eop_fac(
    int64_t nw, const int32_t* __restrict__ done, const int32_t* __restrict__ wseg, int dstride,
    const int32_t* __restrict__ edofs, const int32_t* __restrict__ ocode,
    const R* __restrict__ coef, const R* __restrict__ x, R* __restrict__ ye) {
  constexpr int N = fac::n_dofs<P>();
  constexpr int NLE = n_local_entities<P>();
  __shared__ R faces[fac::face_table_size<P>()];
  fac_fill<P>(faces);
  // looked at below, with the first loads under way
  const int32_t stop = done && !wseg ? *done : 0;
  // XCD-contiguous ranges of slot groups (workgroup b runs on XCD b % 8)
  const int64_t nb = gridDim.x;
  int64_t b = blockIdx.x;
  if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;
  const int64_t hw = b * (kBS / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t w = hw >> 1;
  if (w >= nw) return;
  // segmented operator: the group's mesh has converged
  if (wseg && done[(int64_t)__builtin_amdgcn_readfirstlane(wseg[w]) * dstride]) return;
  const int lane = threadIdx.x % kWave, part = lane & 1;
  const int l = (int)(hw & 1) * (kWave / 2) + (lane >> 1);
  // all index and coefficient loads first, then all gathers, unconditionally
  // (a masked entity reads x[0] and is zeroed after), so that the wave waits
  // for memory twice rather than once per DOF
  int f[NLE];
#pragma unroll
  for (int la = 0; la < NLE; ++la) f[la] = edofs[(w * NLE + la) * kWave + l];
  int code = ocode[w * kWave + l];
  R g[6], h[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    g[c] = coef[(w * 12 + c) * kWave + l];
    h[c] = coef[(w * 12 + 6 + c) * kWave + l];
  }
  if (stop) return;
  R xv[N], y[N];
#pragma unroll
  for (int la = 0; la < NLE; ++la) {
    const R* xe = x + 2 * (int64_t)(f[la] >= 0 ? f[la] : 0) + part;
#pragma unroll
    for (int k = 0; k < loc_nd<P>(la); ++k) xv[loc_off<P>(la) + k] = xe[2 * k];
  }
#pragma unroll
  for (int la = 0; la < NLE; ++la)
#pragma unroll
    for (int k = 0; k < loc_nd<P>(la); ++k)
      xv[loc_off<P>(la) + k] = f[la] >= 0 ? xv[loc_off<P>(la) + k] : R(0);
  fac::orient_in<P>(code, faces, xv);
  const R sg = part ? R(1) : R(-1);
  fac::mass_product<P, R>(xv, g, [&](int i, R v) { y[i] = sg * swap_pair(v); });
  __builtin_amdgcn_sched_barrier(0);  // one product's intermediates at a time
  fac::curl_product<P, R>(xv, h, [&](int i, R v) { y[i] += v; });
  asm("" : "+v"(code));  // the coefficients again, not kept through the products
  fac::orient_out<P>(code, faces, y);
#pragma unroll
  for (int i = 0; i < N; ++i) ye[((w * N + i) * kWave + l) * 2 + part] = y[i];
}

// ---------------------------------------------------------------------------
// per-entity sums.  gm[i] = {r0, d, s0, s1} for the i-th scheduled entity:
// rows r0 .. r0+d, local results at gslot[s0 .. s1) (+ t * 64 for DOF t);
// s0 == s1 marks a PEC entity (identity rows).  MODE as in the CSR SpMV.
// XCD x (workgroup b runs on XCD b % 8) sweeps the x-th eighth of the schedule.
// ---------------------------------------------------------------------------
template <int D, int MODE, typename C>
__global__ void __launch_bounds__(kBS) k_eop_sum(int64_t nent, const int32_t* __restrict__ done,
                                                 const int4* __restrict__ gm,
                                                 const int32_t* __restrict__ gslot,
                                                 const C* __restrict__ ye, const C* __restrict__ x,
                                                 C* __restrict__ y, const double2* __restrict__ b,
                                                 double* part) {
  const int32_t stop = done ? *done : 0;
  const int64_t blk = blockIdx.x, nb = gridDim.x;
  int64_t first = blk * kBS, end = nent, stride = nb * kBS;
  if (nb % 8 == 0) {
    const int64_t xc = blk % 8, nbx = nb / 8;
    first = nent * xc / 8 + (blk / 8) * kBS;
    end = nent * (xc + 1) / 8;
    stride = nbx * kBS;
  }
  double red[2] = {0.0, 0.0};
  int64_t ent = first + threadIdx.x;
  int4 mn = make_int4(0, 0, 0, 0);
  if (ent < end) mn = gm[ent];
  if (stop) return;
  for (; ent < end; ent += stride) {
    const int4 m = mn;
    if (ent + stride < end) mn = gm[ent + stride];
    const int r0 = m.x, d = m.y, s0 = m.z, s1 = m.w;
    // x at the entity's rows (identity rows; the MODE 1 dot product), loaded
    // before the sums so that its latency overlaps theirs
    C xr[D];
    const bool need_x = MODE == 1 || s0 == s1;
#pragma unroll
    for (int t = 0; t < D; ++t) xr[t] = (need_x && t < d) ? x[r0 + t] : C{0, 0};
    C acc[D];
#pragma unroll
    for (int t = 0; t < D; ++t) acc[t] = C{0, 0};
    if (s0 == s1) {
#pragma unroll
      for (int t = 0; t < D; ++t) acc[t] = xr[t];
    } else {
      // two incidences per step (their loads in flight together), summed in
      // ascending slot order
      int k = s0;
      for (; k + 2 <= s1; k += 2) {
        const int b0 = gslot[k], b1 = gslot[k + 1];
        C v0[D], v1[D];
#pragma unroll
        for (int t = 0; t < D; ++t)
          if (t < d) {
            v0[t] = ye[b0 + t * kWave];
            v1[t] = ye[b1 + t * kWave];
          }
#pragma unroll
        for (int t = 0; t < D; ++t)
          if (t < d) {
            acc[t].x += v0[t].x;
            acc[t].y += v0[t].y;
            acc[t].x += v1[t].x;
            acc[t].y += v1[t].y;
          }
      }
      if (k < s1) {
        const int b0 = gslot[k];
#pragma unroll
        for (int t = 0; t < D; ++t)
          if (t < d) {
            const C v = ye[b0 + t * kWave];
            acc[t].x += v.x;
            acc[t].y += v.y;
          }
      }
    }
#pragma unroll
    for (int t = 0; t < D; ++t)
      if (t < d) {
        const int row = r0 + t;
        if (MODE == 2) {
          const double2 bb = b[row];
          const double2 rr = make_double2(bb.x - (double)acc[t].x, bb.y - (double)acc[t].y);
          store(y + row, rr);
          red[0] += rr.x * rr.x + rr.y * rr.y;
        } else {
          y[row] = acc[t];
          if (MODE == 1) {
            const double2 pv = to_d(xr[t]), qv = to_d(acc[t]);
            red[0] += pv.x * qv.x - pv.y * qv.y;
            red[1] += pv.x * qv.y + pv.y * qv.x;
          }
        }
      }
  }
  if (MODE == 1) write_partials<2>(red, part);
  if (MODE == 2) {
    double r1[1] = {red[0]};
    write_partials<1>(r1, part);
  }
}

// The same with a thread per (entity, DOF) and eight slots at a time: small p = 3
// operators, where a thread's chain of slots is the time of the call and six times
// the threads still fit the chip at once (product of 20 250 elements 23.0 -> 17.4 us; from
// kDofSumEntities on the entity's lane, which reads descriptors and slots once for its
// DOFs, is the faster: 82 944 elements in complex64 37 us, here 39).
constexpr int64_t kDofSumEntities = 1 << 17;
template <int D, int MODE, typename C>
__global__ void __launch_bounds__(kBS) k_eop_sum_dof(int64_t nent, const int32_t* __restrict__ done,
                                                     const int4* __restrict__ gm,
                                                     const int32_t* __restrict__ gslot,
                                                     const C* __restrict__ ye,
                                                     const C* __restrict__ x, C* __restrict__ y,
                                                     const double2* __restrict__ b, double* part) {
  constexpr int U = 8;
  const int32_t stop = done ? *done : 0;
  const int64_t blk = blockIdx.x, nb = gridDim.x;
  int64_t first = blk * kBS, end = nent * D, stride = nb * kBS;
  if (nb % 8 == 0) {
    const int64_t xc = blk % 8, nbx = nb / 8;
    first = nent * xc / 8 * D + (blk / 8) * kBS;
    end = nent * (xc + 1) / 8 * D;
    stride = nbx * kBS;
  }
  double red[2] = {0.0, 0.0};
  if (stop) return;
  for (int64_t i = first + threadIdx.x; i < end; i += stride) {
    const int4 m = gm[i / D];
    const int t = (int)(i % D);
    if (t >= m.y) continue;
    const int row = m.x + t;
    const bool pec = m.z == m.w;
    C xr = C{0, 0}, acc = C{0, 0};
    if (MODE == 1 || pec) xr = x[row];
    if (pec) acc = xr;
    for (int k = m.z; k < m.w; k += U) {  // ascending slot order
      int g[U];
      C v[U];
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (k + j < m.w) g[j] = gslot[k + j];
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (k + j < m.w) v[j] = ye[g[j] + t * kWave];
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (k + j < m.w) {
          acc.x += v[j].x;
          acc.y += v[j].y;
        }
    }
    if (MODE == 2) {
      const double2 bb = b[row];
      const double2 rr = make_double2(bb.x - (double)acc.x, bb.y - (double)acc.y);
      store(y + row, rr);
      red[0] += rr.x * rr.x + rr.y * rr.y;
    } else {
      y[row] = acc;
      if (MODE == 1) {
        const double2 pv = to_d(xr), qv = to_d(acc);
        red[0] += pv.x * qv.x - pv.y * qv.y;
        red[1] += pv.x * qv.y + pv.y * qv.x;
      }
    }
  }
  if (MODE == 1) write_partials<2>(red, part);
  if (MODE == 2) {
    double r1[1] = {red[0]};
    write_partials<1>(r1, part);
  }
}

// ---------------------------------------------------------------------------
// The whole product in one kernel: a workgroup owns a run of scheduled entities
// (a spatial cluster when the schedule is spatial), computes every element that
// touches them (128 elements, two lanes each, as k_eop_fac), keeps the local
// results of its own entities in LDS and sums each entity there in the slot
// order of k_eop_sum (bitwise the two-kernel result), so the local results never
// reach memory.  Elements on the border of a cluster are computed by every
// workgroup that owns one of their entities.
//   bmeta[b]      {first schedule position, entities, first element group, groups}
//   bslot[g][l]   slot of element l < 128 of group g, -1 empty
//   bcode, bdofs  its orientation and entities (as ocode, edofs)
//   bpos[g][q][l] LDS places of its local entities 2 q and 2 q + 1 (16 bits each,
//                 in complex values; 0xFFFF = not owned here)
//   em[i]         {first DOF, place | incidences << 16 | DOFs << 28} of entity i
// MODE as k_eop_sum.
// Bound: FP64 / FP32 issue (900 vector instructions per wave of 32 elements, each
// element 1.8 to 2.1 times) next to 180 MB of indices, coefficients, x and y.
// Against the two kernels: 384 000 elements, p = 2: 71 us (complex128, 98 before)
// and 53 us (complex64, 54; 85 against 105 inside the solve, where nothing of the
// local results is in cache); 13 182 elements 10.9 against 13.2 us, one launch
// less.  Loading the next block's indices ahead of the sums was slower (the
// registers spill or cost a wave per SIMD).
// ---------------------------------------------------------------------------
constexpr int kGroup = kBS / 2;  // elements per pass of a workgroup

template <int P, typename R, int MODE>
__global__ void __launch_bounds__(kBS, (fac_waves<P, R>())) k_eop_blk(
    int64_t nblk, const int32_t* __restrict__ done, const int4* __restrict__ bmeta,
    const int32_t* __restrict__ bslot, const int32_t* __restrict__ bcode,
    const int32_t* __restrict__ bdofs, const uint32_t* __restrict__ bpos,
    const int2* __restrict__ em, const R* __restrict__ coef, const R* __restrict__ x,
    typename Cx<R>::T* __restrict__ y, const double2* __restrict__ rhs, double* part) {
  using C = typename Cx<R>::T;
  constexpr int N = fac::n_dofs<P>();
  constexpr int NLE = n_local_entities<P>();
  constexpr int NQ = (NLE + 1) / 2;
  static_assert(P <= 2, "entities of up to two DOFs");
  constexpr int D = P;  // DOFs of an entity
  extern __shared__ __align__(16) char smem[];
  __shared__ R faces[fac::face_table_size<P>()];
  const int32_t stop = done ? *done : 0;
  const int tid = threadIdx.x, el = tid >> 1, part_ = tid & 1;
  // XCD x (workgroup b runs on XCD b % 8) takes the x-th eighth of the blocks
  const int64_t nb = gridDim.x;
  int64_t b = blockIdx.x, end = nblk, stride = nb;
  if (nb % 8 == 0) {
    const int64_t xc = b % 8;
    b = nblk * xc / 8 + b / 8;
    end = nblk * (xc + 1) / 8;
    stride = nb / 8;
  }
  int4 bm{0, 0, 0, 0};
  if (b < end) bm = bmeta[b];
  fac_fill<P>(faces);
  if (stop) return;
  double red[2] = {0.0, 0.0};
  while (b < end) {
    R* acc = reinterpret_cast<R*>(smem);
    for (int64_t g = bm.z; g < bm.z + bm.w; ++g) {
      const int slot = bslot[g * kGroup + el];
      int code = bcode[g * kGroup + el];
      int f[NLE];
#pragma unroll
      for (int la = 0; la < NLE; ++la) f[la] = bdofs[(g * NLE + la) * kGroup + el];
      uint32_t pos[NQ];
#pragma unroll
      for (int q = 0; q < NQ; ++q) pos[q] = bpos[(g * NQ + q) * kGroup + el];
      const R* cf = coef + 12 * (int64_t)(slot >= 0 ? slot : 0);
      R gm[6], h[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        gm[c] = cf[c];
        h[c] = cf[6 + c];
      }
      R xv[N], yv[N];
      bool pec = false;
#pragma unroll
      for (int la = 0; la < NLE; ++la) {
        pec |= f[la] < 0;
        const R* xe = x + 2 * (int64_t)(f[la] >= 0 ? f[la] : 0) + part_;
#pragma unroll
        for (int k = 0; k < loc_nd<P>(la); ++k) xv[loc_off<P>(la) + k] = xe[2 * k];
      }
      if (__any(pec)) {  // few waves hold a PEC entity or an empty place
#pragma unroll
        for (int la = 0; la < NLE; ++la)
#pragma unroll
          for (int k = 0; k < loc_nd<P>(la); ++k)
            xv[loc_off<P>(la) + k] = f[la] >= 0 ? xv[loc_off<P>(la) + k] : R(0);
      }
      fac::orient_in<P>(code, faces, xv);
      const R sg = part_ ? R(1) : R(-1);
      fac::mass_product<P, R>(xv, gm, [&](int i, R v) { yv[i] = sg * swap_pair(v); });
      __builtin_amdgcn_sched_barrier(0);  // one product's intermediates at a time
      fac::curl_product<P, R>(xv, h, [&](int i, R v) { yv[i] += v; });
      asm("" : "+v"(code));  // the coefficients again, not kept through the products
      fac::orient_out<P>(code, faces, yv);
#pragma unroll
      for (int la = 0; la < NLE; ++la) {
        const uint32_t at = (la & 1) ? pos[la / 2] >> 16 : pos[la / 2] & 0xFFFFu;
        if (at != 0xFFFFu)
#pragma unroll
          for (int k = 0; k < loc_nd<P>(la); ++k)
            acc[2 * (at + k) + part_] = yv[loc_off<P>(la) + k];
      }
    }
    const int4 cm = bm;
    b += stride;
    if (b < end) bm = bmeta[b];
    __syncthreads();
    for (int i = tid; i < cm.y * D; i += kBS) {
      const int2 e = em[cm.x + i / D];
      const int t = i % D, d = (uint32_t)e.y >> 28, n = (e.y >> 16) & 0xFFF, row = e.x + t;
      if (t >= d) continue;
      C s{0, 0}, xr{0, 0};
      if (MODE == 1 || n == 0) xr = reinterpret_cast<const C*>(x)[row];
      if (n == 0) s = xr;  // PEC: identity row
      const C* v = reinterpret_cast<const C*>(smem) + (e.y & 0xFFFF) + t;
      for (int q = 0; q < n; ++q) {
        s.x += v[q * d].x;
        s.y += v[q * d].y;
      }
      if (MODE == 2) {
        const double2 bb = rhs[row];
        const double2 rr = make_double2(bb.x - (double)s.x, bb.y - (double)s.y);
        store(y + row, rr);
        red[0] += rr.x * rr.x + rr.y * rr.y;
      } else {
        y[row] = s;
        if (MODE == 1) {
          const double2 pv = to_d(xr), qv = to_d(s);
          red[0] += pv.x * qv.x - pv.y * qv.y;
          red[1] += pv.x * qv.y + pv.y * qv.x;
        }
      }
    }
    __syncthreads();
  }
  if (MODE == 1) write_partials<2>(red, part);
  if (MODE == 2) {
    double r1[1] = {red[0]};
    write_partials<1>(r1, part);
  }
}

// ---------------------------------------------------------------------------
// multi-right-hand-side local products for the batched solver: column r of the
// (ndof, R) row-major block x gets y_e,r = (K_e - i omega_r mu0 M_e) x_e,r.
// One workgroup of 2 R threads (thread 2 r + part = the real or imaginary part
// of column r; R = 64 .. 256) per part of a slot group w of the single-RHS
// layout (64 elements, split into `split` parts), which takes its elements one
// after another.  The element is the same for the whole workgroup, so its
// entities, orientation and coefficients are scalars, and each of its DOFs is
// one contiguous load of 2 R values; K x_e and M x_e of the thread's real
// vector are formed without the element matrix (pg_factor.h), in FP64 for
// complex64 columns too (the same issue rate), and the two parts of a column
// exchange M x_e across neighbouring lanes.  Local results
// ye[((w N + i) 64 + l) R + r]: the single-RHS slot numbering times R, so the
// per-entity summation reuses the slot lists.
// With `dpart` each thread also sums its share of x_e,r^T y_e,r over its
// elements (FP64): dpart[(k R + r) gridDim + block], k = 0 real, 1 imaginary
// part, the element share of x_r^T A_r x_r (PEC DOFs are zero in x_e and add
// nothing here).
// Bound: FP64 issue on small meshes, the traffic of x and ye on large ones.
// Forming the 210 entry pairs of an element in LDS and applying them, one
// thread per column, 16 elements per workgroup, took 177, 281 and 1479 us at
// 2 058, 24 576 and 162 000 elements (64 complex128 columns); this takes 19, 184
// and 1261 us.  The first pays for filling the chip (140 workgroups then, 2 200
// now), the last is within 1.5 of the copy rate.  At most 168 registers (three
// waves per SIMD): M x_e is finished before K x_e begins.
// ---------------------------------------------------------------------------
template <int P, typename R>
__global__ void __launch_bounds__(512, 3) k_meop_local(
    int64_t nw, int nrhs, int split, const int32_t* __restrict__ done,
    const int32_t* __restrict__ edofs, const int32_t* __restrict__ ocode,
    const double* __restrict__ coefm, const double* __restrict__ omu, const R* __restrict__ x,
    R* __restrict__ ye, double* __restrict__ dpart) {
  constexpr int N = fac::n_dofs<P>();
  constexpr int NLE = n_local_entities<P>();
  __shared__ double faces[fac::face_table_size<P>()];
  fac_fill<P>(faces);
  if (done && *done) return;
  const int64_t nb = gridDim.x;
  int64_t b = blockIdx.x;
  if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;  // XCD-contiguous ranges of slot groups
  const int64_t w = b / split;
  if (w >= nw) return;
  const int per = kWave / split, l0 = (int)(b - w * split) * per;
  const int t = threadIdx.x, r = t >> 1;
  // y_re = K x_re + omega mu0 M x_im, y_im = K x_im - omega mu0 M x_re
  const double om = (t & 1) ? -omu[r] : omu[r];
  const int64_t ld = 2 * (int64_t)nrhs;
  double dre = 0.0, dim = 0.0;  // this part's share of x^T y over the elements
  for (int l = l0; l < l0 + per; ++l) {
    int f[NLE];
    bool any = false;
#pragma unroll
    for (int la = 0; la < NLE; ++la) {
      f[la] = edofs[(w * NLE + la) * kWave + l];
      any |= f[la] >= 0;
    }
    if (!any) continue;  // empty slot (or every entity PEC): no products; uniform branch
    double g[6], h[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      g[c] = coefm[(w * 12 + c) * kWave + l];
      h[c] = coefm[(w * 12 + 6 + c) * kWave + l];
    }
    double xv[N], y[N];
#pragma unroll
    for (int la = 0; la < NLE; ++la)
#pragma unroll
      for (int k = 0; k < loc_nd<P>(la); ++k)
        xv[loc_off<P>(la) + k] = f[la] >= 0 ? (double)x[(f[la] + k) * ld + t] : 0.0;
    int code = ocode[w * kWave + l];
    fac::orient_in<P>(code, faces, xv);
    fac::mass_product<P, double>(xv, g, [&](int i, double v) { y[i] = om * swap_pair(v); });
    __builtin_amdgcn_sched_barrier(0);  // one product's intermediates at a time
    fac::curl_product<P, double>(xv, h, [&](int i, double v) { y[i] += v; });
    // x^T y is the same in the code-0 functions
#pragma unroll
    for (int i = 0; i < N; ++i) {
      dre += xv[i] * y[i];
      dim += xv[i] * swap_pair(y[i]);
    }
    asm("" : "+s"(code));  // the coefficients again, not kept through the products
    fac::orient_out<P>(code, faces, y);
#pragma unroll
    for (int i = 0; i < N; ++i) ye[((w * N + i) * kWave + l) * ld + t] = (R)y[i];
  }
  if (dpart) {
    // real: re re - im im; imaginary: re im + im re
    dre -= swap_pair(dre);
    dim += swap_pair(dim);
    dpart[((t & 1) * (int64_t)nrhs + r) * gridDim.x + blockIdx.x] = (t & 1) ? dim : dre;
  }
}

// coefficients in slot order: mass part times -omega mu0, then curl-curl part
// (multi-mesh operator: omega mu0 of the wave's segment, womu[wseg[w]]); the 12 of
// a slot together (by_slot) or [group][c][element of 64]
template <typename R>
__global__ void k_eop_coef(int64_t nslot, const int32_t* __restrict__ perm,
                           const double* __restrict__ wscoef, double omega_mu,
                           const int32_t* __restrict__ wseg, const double* __restrict__ womu,
                           int by_slot, R* __restrict__ coef) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslot) return;
  const int64_t w = s / kWave, lane = s % kWave;
  const int64_t e = perm[s];
  const double om = womu ? womu[wseg[w]] : omega_mu;
#pragma unroll
  for (int c = 0; c < 12; ++c) {
    double v = e >= 0 ? wscoef[12 * e + c] : 0.0;
    if (c < 6) v = -(om * v);
    coef[by_slot ? s * 12 + c : (w * 12 + c) * kWave + lane] = (R)v;
  }
}

// k_eop_blk's orientations and entities from its slots
__global__ void __launch_bounds__(kBS) k_eop_blk_elements(int64_t n, int nle,
                                                          const int32_t* __restrict__ bslot,
                                                          const int32_t* __restrict__ ocode,
                                                          const int32_t* __restrict__ edofs,
                                                          int32_t* __restrict__ bcode,
                                                          int32_t* __restrict__ bdofs) {
  const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (i >= n) return;
  const int64_t s = bslot[i], g = i / kGroup, l = i % kGroup;
  bcode[i] = s >= 0 ? ocode[s] : 0;
  for (int la = 0; la < nle; ++la)
    bdofs[(g * nle + la) * kGroup + l] =
        s >= 0 ? edofs[(s / kWave * nle + la) * kWave + s % kWave] : -1;
}

template <typename R>
__global__ void __launch_bounds__(kBS) k_eop_copy(int64_t n, const R* __restrict__ x,
                                                  R* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (i < n) y[i] = x[i];
}

}  // namespace eop

struct ElemOp {
  int p = 0, N = 0, D = 1;
  int64_t E = 0, ndof = 0, nent = 0, nw = 0;
  int grid = 1;
  int32_t* edofs = nullptr;
  int32_t* perm = nullptr;
  int4* gm = nullptr;
  int32_t* gslot = nullptr;
  double* coef64 = nullptr;
  float* coef32 = nullptr;
  double2* ye64 = nullptr;
  float2* ye32 = nullptr;
  // packed element orientation per slot (orient_of)
  int32_t* ocode = nullptr;
  // multi-right-hand-side products (eop_multi_prepare): raw coefficients in
  // slot order (mass part without -omega mu0)
  double* coefm = nullptr;
  // one-kernel product (k_eop_blk) of a one-mesh operator, p <= 2; nblk = 0: the
  // two kernels (p = 3, multi-mesh operators, and meshes with an entity of more
  // elements than a workgroup takes)
  int64_t nblk = 0;
  int lds_values = 0;  // complex values of LDS per workgroup
  int4* bmeta = nullptr;
  int32_t *bslot = nullptr, *bcode = nullptr, *bdofs = nullptr;
  uint32_t* bpos = nullptr;
  int2* em = nullptr;
  // its x where the caller's y overlaps it (2 ndof reals)
  double* xcopy = nullptr;
  // multi-mesh operator (pg_eop_create_multi): segment of every wave, omega mu0
  // of every segment, first schedule position of every segment (nseg + 1)
  int nseg = 0;
  int32_t* wseg = nullptr;
  double* womu = nullptr;
  std::vector<int64_t> seg_pos, seg_wave;  // + first wave of every segment (nseg + 1)
  std::vector<void*> owned;

  template <typename T>
  int alloc(T** ptr, size_t count) {
    void* v = nullptr;
    hipError_t e = hipMalloc(&v, std::max<size_t>(count, 1) * sizeof(T));
    if (e != hipSuccess)
      PG_FAIL(PG_ERR_HIP, "hipMalloc(%zu): %s", count * sizeof(T), hipGetErrorString(e));
    owned.push_back(v);
    *ptr = static_cast<T*>(v);
    return PG_OK;
  }
  ~ElemOp() {  // release errors cannot be reported from here
    for (void* v : owned) (void)hipFree(v);
  }
};

int eop_grid(const ElemOp* op) { return op->grid; }
int64_t eop_ndof(const ElemOp* op) { return op->ndof; }

// element products of slot groups [w0, w0 + nwr) (all groups: 0, op->nw)
template <typename R>
static void launch_local(const ElemOp* op, const int32_t* done, const int32_t* wseg, int dstride,
                         const typename eop::Cx<R>::T* x, typename eop::Cx<R>::T* ye,
                         const R* coef, hipStream_t st, int64_t w0 = 0, int64_t nwr = -1) {
  if (nwr < 0) nwr = op->nw;
  if (nwr <= 0) return;
  const int nle = op->p == 1 ? 6 : (op->p == 2 ? 10 : 11);
  const int gpb = eop::kBS / (2 * kWave);  // slot groups per workgroup, two waves each
  int64_t nbl = (nwr + gpb - 1) / gpb;
  if (nbl >= 64) nbl = (nbl + 7) / 8 * 8;
  const dim3 g((unsigned)nbl), b(eop::kBS);
  const int32_t* ed = op->edofs + w0 * nle * kWave;
  const int32_t* oc = op->ocode + w0 * kWave;
  const int32_t* ws = wseg ? wseg + w0 : nullptr;
  const R* xr = reinterpret_cast<const R*>(x);
  R* yr = reinterpret_cast<R*>(ye + w0 * op->N * kWave);
  coef += w0 * 12 * kWave;
#define PG_FAC(P)                                                                               \
  hipLaunchKernelGGL((eop::k_eop_fac<P, R>), g, b, 0, st, nwr, done, ws, dstride, ed, oc, coef, \
                     xr, yr)
  if (op->p == 1) PG_FAC(1);
  else if (op->p == 2) PG_FAC(2);
  else PG_FAC(3);
#undef PG_FAC
}

template <typename R>
static void launch_impl(const ElemOp* op, int mode, const int32_t* done,
                        const typename eop::Cx<R>::T* x, typename eop::Cx<R>::T* y,
                        const double2* b, double* part, hipStream_t st, hipEvent_t mid,
                        typename eop::Cx<R>::T* ye, const R* coef) {
  using C = typename eop::Cx<R>::T;
  const dim3 g(op->grid), bl(eop::kBS);
#define PG_MODES(CALL) \
  if (mode == 0) {     \
    CALL(0);           \
  } else if (mode == 1) { \
    CALL(1);           \
  } else {             \
    CALL(2);           \
  }
  if (op->nblk > 0) {
    const R* xr = reinterpret_cast<const R*>(x);
#define PG_BLK(P, MM)                                                                           \
  hipLaunchKernelGGL((eop::k_eop_blk<P, R, MM>), g, bl, op->lds_values * sizeof(C), st, op->nblk, \
                     done, op->bmeta, op->bslot, op->bcode, op->bdofs, op->bpos, op->em, coef, xr, \
                     y, b, part)
#define PG_BLK1(MM) PG_BLK(1, MM)
#define PG_BLK2(MM) PG_BLK(2, MM)
    if (op->p == 1) {
      PG_MODES(PG_BLK1)
    } else {
      PG_MODES(PG_BLK2)
    }
#undef PG_BLK1
#undef PG_BLK2
#undef PG_BLK
    // a failed record only loses this timing sample (the elapsed-time query fails)
    if (mid) (void)hipEventRecord(mid, st);
    return;
  }
  launch_local<R>(op, done, nullptr, 0, x, ye, coef, st);
  if (mid) (void)hipEventRecord(mid, st);
#define PG_SUM(DD, MM)                                                                        \
  hipLaunchKernelGGL((eop::k_eop_sum<DD, MM, C>), g, bl, 0, st, op->nent, done, op->gm,       \
                     op->gslot, (const C*)ye, x, y, b, part)
#define PG_SUM1(MM) PG_SUM(1, MM)
#define PG_SUM2(MM) PG_SUM(2, MM)
#define PG_SUM6(MM) PG_SUM(6, MM)
#define PG_SUM_DOF(MM)                                                                        \
  hipLaunchKernelGGL((eop::k_eop_sum_dof<6, MM, C>), g, bl, 0, st, op->nent, done, op->gm,    \
                     op->gslot, (const C*)ye, x, y, b, part)
  if (op->D == 1) {
    PG_MODES(PG_SUM1)
  } else if (op->D == 2) {
    PG_MODES(PG_SUM2)
  } else if (op->nent < eop::kDofSumEntities) {
    PG_MODES(PG_SUM_DOF)
  } else {
    PG_MODES(PG_SUM6)
  }
#undef PG_SUM1
#undef PG_SUM2
#undef PG_SUM6
#undef PG_SUM_DOF
#undef PG_SUM
#undef PG_MODES
}

void eop_launch(const ElemOp* op, int mode, const int32_t* done, const double2* x, double2* y,
                const double2* b, double* part, hipStream_t st, hipEvent_t mid) {
  launch_impl<double>(op, mode, done, x, y, b, part, st, mid, op->ye64, op->coef64);
}
void eop_launch(const ElemOp* op, int mode, const int32_t* done, const float2* x, float2* y,
                const double2* b, double* part, hipStream_t st, hipEvent_t mid) {
  launch_impl<float>(op, mode, done, x, y, b, part, st, mid, op->ye32, op->coef32);
}

static int eop_refresh(ElemOp* op, const void* ws, double omega, hipStream_t st) {
  const double* wscoef = reinterpret_cast<const double*>(ws);
  const int64_t nslot = op->nw * kWave;
  const double om = omega * eop::kMu0;
  const dim3 g((unsigned)((nslot + 255) / 256)), b(256);
  hipLaunchKernelGGL(eop::k_eop_coef<double>, g, b, 0, st, nslot, op->perm, wscoef, om,
                     op->wseg, op->womu, op->nblk > 0, op->coef64);
  hipLaunchKernelGGL(eop::k_eop_coef<float>, g, b, 0, st, nslot, op->perm, wscoef, om,
                     op->wseg, op->womu, op->nblk > 0, op->coef32);
  // raw coefficients: -(-1 * v) = v exactly
  if (op->coefm)
    hipLaunchKernelGGL(eop::k_eop_coef<double>, g, b, 0, st, nslot, op->perm, wscoef, -1.0,
                       nullptr, nullptr, 0, op->coefm);
  PG_CHECK_LAUNCH();
  return PG_OK;
}

int eop_multi_prepare(ElemOp* op, const void* ws, hipStream_t st) {
  if (op->nseg > 0)
    PG_FAIL(PG_ERR_UNSUPPORTED, "multi-right-hand-side products of a multi-mesh operator");
  if (op->p > 2)
    PG_FAIL(PG_ERR_UNSUPPORTED, "multi-right-hand-side element products: p <= 2 only");
  if (op->coefm) return PG_OK;
  int rc;
  if ((rc = op->alloc(&op->coefm, op->nw * kWave * 12)) != PG_OK) return rc;
  const int64_t nslot = op->nw * kWave;
  const dim3 g((unsigned)((nslot + 255) / 256)), b(256);
  hipLaunchKernelGGL(eop::k_eop_coef<double>, g, b, 0, st, nslot, op->perm,
                     reinterpret_cast<const double*>(ws), -1.0, nullptr, nullptr, 0, op->coefm);
  PG_CHECK_LAUNCH();
  return PG_OK;
}

EopSchedule eop_schedule(const ElemOp* op) {
  return EopSchedule{op->gm, op->gslot, op->nent, op->nw, op->p, op->N, op->D};
}

int eop_segments(const ElemOp* op, const int64_t** seg_pos, const int64_t** seg_wave) {
  if (seg_pos) *seg_pos = op->seg_pos.data();
  if (seg_wave) *seg_wave = op->seg_wave.data();
  return op->nseg;
}

const double2* eop_local_segments(const ElemOp* op, const int32_t* done, int dstride,
                                  const double2* x, hipStream_t st, int64_t w0, int64_t w1) {
  if (w1 < 0) w1 = op->nw;
  launch_local<double>(op, done, op->wseg, dstride, x, op->ye64, op->coef64, st, w0,
                       w1 - w0);
  return op->ye64;
}
const float2* eop_local_segments(const ElemOp* op, const int32_t* done, int dstride,
                                 const float2* x, hipStream_t st, int64_t w0, int64_t w1) {
  if (w1 < 0) w1 = op->nw;
  launch_local<float>(op, done, op->wseg, dstride, x, op->ye32, op->coef32, st, w0,
                      w1 - w0);
  return op->ye32;
}

// workgroups per slot group: 16 elements each on large meshes, fewer (down to
// one) while the launch has under eight waves per SIMD of the chip
static int multi_split(const ElemOp* op, int R) {
  int split = 4;
  while (split < kWave && op->nw * split * (R / 32) < 8192) split *= 2;
  return split;
}
int64_t eop_multi_parts(const ElemOp* op, int R) { return op->nw * multi_split(op, R); }

template <typename RT>
static void multi_local(const ElemOp* op, int R, const int32_t* done, const double* omu,
                        const typename eop::Cx<RT>::T* x, typename eop::Cx<RT>::T* ye,
                        double* part, hipStream_t st) {
  const int split = multi_split(op, R);
  const dim3 g((unsigned)(op->nw * split)), b(2 * R);
  const RT* xr = reinterpret_cast<const RT*>(x);
  RT* yr = reinterpret_cast<RT*>(ye);
  if (op->p == 1)
    hipLaunchKernelGGL((eop::k_meop_local<1, RT>), g, b, 0, st, op->nw, R, split, done,
                       op->edofs, op->ocode, op->coefm, omu, xr, yr, part);
  else
    hipLaunchKernelGGL((eop::k_meop_local<2, RT>), g, b, 0, st, op->nw, R, split, done,
                       op->edofs, op->ocode, op->coefm, omu, xr, yr, part);
}
void eop_multi_local(const ElemOp* op, int R, const int32_t* done, const double* omu,
                     const double2* x, double2* ye, double* part, hipStream_t st) {
  multi_local<double>(op, R, done, omu, x, ye, part, st);
}
void eop_multi_local(const ElemOp* op, int R, const int32_t* done, const double* omu,
                     const float2* x, float2* ye, double* part, hipStream_t st) {
  multi_local<float>(op, R, done, omu, x, ye, part, st);
}

// Operator set-up from host copies of the element DOFs (hd, E x n), element
// orientation codes (hor), entity DOF ranges (bp), schedule (order, may be
// null) and PEC entities (hbc); ws = the device geometry coefficients.  With
// seg (a multi-mesh operator) the elements are grouped by segment first, so
// that no wave of 64 elements spans two segments, and each segment gets its
// own frequency.
struct SegInfo {
  int nseg = 0;
  std::vector<int64_t> pos;  // first schedule position of each segment (nseg + 1)
  std::vector<double> omega;
};

// host checks of the entity DOF ranges (before any device work)
static int check_block_ptr(int p, const int32_t* bp, int64_t nblocks, int64_t ndof) {
  const int maxd = p == 1 ? 1 : (p == 2 ? 2 : 6);
  if (bp[0] != 0 || bp[nblocks] != ndof)
    PG_FAIL(PG_ERR_ARG, "block_ptr must start at 0 and end at ndof");
  for (int64_t g = 0; g < nblocks; ++g)
    if (bp[g + 1] - bp[g] < 1 || bp[g + 1] - bp[g] > maxd)
      PG_FAIL(PG_ERR_ARG, "entity sizes must be in 1..%d at p=%d", maxd, p);
  return PG_OK;
}

// Blocks of k_eop_blk from the schedule (gm, and per incidence its slot * NLE + local
// entity): entities are taken in schedule order while the elements around them fit
// `passes` groups and their local results the LDS budget.  False when one entity alone
// does not fit.
struct Blocks {
  std::vector<int4> meta;
  std::vector<int32_t> slot;
  std::vector<uint16_t> pos;  // (two to a word of bpos)
  std::vector<int2> em;
  int lds_values = 1;
};
template <int NLE>
static bool make_blocks(int passes, int64_t nslot, const std::vector<int4>& gm,
                        const std::vector<int32_t>& inc, Blocks* B) {
  constexpr int G = eop::kGroup;
  constexpr int kMaxEnt = 1024;     // entities per block (PEC entities have no elements)
  constexpr int kMaxValues = 3072;  // complex128 values of LDS: 48 KB, three workgroups
  constexpr int NQ = (NLE + 1) / 2;
  const int64_t nent = (int64_t)gm.size();
  struct Mark {
    int32_t block, place;  // block that last took the slot, its element number there
  };
  std::vector<Mark> mark(nslot, Mark{-1, 0});
  const size_t ng0 = nslot / G * 5 / 2 + 1;  // each element about twice
  B->slot.reserve(ng0 * G);
  B->pos.reserve(ng0 * G * 2 * NQ);
  B->em.resize(nent);
  for (int64_t i = 0; i < nent;) {
    const int32_t b = (int32_t)B->meta.size();
    const int64_t i0 = i, g0 = (int64_t)B->slot.size() / G;
    int ne = 0, nv = 0;
    for (; i < nent && i - i0 < kMaxEnt; ++i) {
      const int4 m = gm[i];
      const int n = m.w - m.z;
      int fresh = n;  // at most; counted where that matters
      if (ne + n > passes * G) {
        fresh = 0;
        for (int k = m.z; k < m.w; ++k) fresh += mark[inc[k] / NLE].block != b;
      }
      if (n > 0xFFF || ne + fresh > passes * G || nv + n * m.y > kMaxValues) break;
      B->em[i] = make_int2(m.x, (int)((uint32_t)nv | (uint32_t)n << 16 | (uint32_t)m.y << 28));
      for (int k = m.z; k < m.w; ++k) {
        const int s = inc[k] / NLE, la = inc[k] % NLE;
        Mark& mk = mark[s];
        if (mk.block != b) {
          mk = Mark{b, ne++};
          const int64_t g = g0 + mk.place / G, e = mk.place % G;
          if (e == 0) {
            B->slot.resize((g + 1) * G, -1);
            B->pos.resize((g + 1) * G * 2 * NQ, 0xFFFF);
          }
          B->slot[g * G + e] = s;
        }
        B->pos[(((g0 + mk.place / G) * NQ + la / 2) * G + mk.place % G) * 2 + la % 2] =
            (uint16_t)nv;
        nv += m.y;
      }
    }
    if (i == i0) return false;
    B->meta.push_back(make_int4((int)i0, (int)(i - i0), (int)g0, (ne + G - 1) / G));
    B->lds_values = std::max(B->lds_values, nv);
  }
  return true;
}

// slot * (local entities) + local entity -> its first local result, (group * N + first
// local DOF) * 64 + element of the group
template <int P>
static void local_results(std::vector<int32_t>& list) {
  constexpr int NLE = eop::n_local_entities<P>(), N = fac::n_dofs<P>();
  for (int32_t& v : list) {
    const int s = v / NLE;
    v = (s / kWave * N + entity_local_offset(v % NLE, P)) * kWave + s % kWave;
  }
}

static int eop_build(int p, int64_t E, const void* ws, int64_t ndof, const int32_t* bp,
                     int64_t nblocks, const int32_t* order, const std::vector<int32_t>& hd,
                     const std::vector<int32_t>& hor, const std::vector<uint8_t>& hbc,
                     double omega, const SegInfo* seg, ElemOp** out, hipStream_t st) {
  const int N = ndof_element(p);
  const int nle = p == 1 ? 6 : (p == 2 ? 10 : 11);  // local entities carrying DOFs
  const int maxd = p == 1 ? 1 : (p == 2 ? 2 : 6);
  int rc0 = check_block_ptr(p, bp, nblocks, ndof);
  if (rc0 != PG_OK) return rc0;
  std::vector<int32_t> ent_of(ndof);
  for (int64_t g = 0; g < nblocks; ++g)
    for (int d = bp[g]; d < bp[g + 1]; ++d) ent_of[d] = (int32_t)g;
  // each local entity's global entity; its DOFs must be that entity's range in order
  std::vector<int32_t> eg((size_t)E * nle);
  std::vector<int32_t> cnt(nblocks, 0);
  for (int64_t e = 0; e < E; ++e)
    for (int la = 0; la < nle; ++la) {
      const int off = entity_local_offset(la, p), nd = entity_ndof(la, p);
      const int d0 = hd[e * N + off];
      if (d0 < 0 || d0 >= ndof) PG_FAIL(PG_ERR_ARG, "element %lld: DOF out of range", (long long)e);
      const int g = ent_of[d0];
      if (bp[g + 1] - bp[g] != nd || bp[g] != d0)
        PG_FAIL(PG_ERR_ARG, "element %lld: local entity %d does not match a block_ptr range",
                (long long)e, la);
      for (int k = 1; k < nd; ++k)
        if (hd[e * N + off + k] != d0 + k)
          PG_FAIL(PG_ERR_ARG, "element %lld: entity DOFs out of order", (long long)e);
      eg[e * nle + la] = g;
      if (!hbc[g]) cnt[g]++;
    }
  for (int64_t g = 0; g < nblocks; ++g)
    if (!hbc[g] && cnt[g] == 0)
      PG_FAIL(PG_ERR_ARG, "entity %lld belongs to no element", (long long)g);
  std::vector<int32_t> pos(nblocks);
  if (order) {
    std::vector<char> seen(nblocks, 0);
    for (int64_t i = 0; i < nblocks; ++i) {
      if (order[i] < 0 || order[i] >= nblocks || seen[order[i]])
        PG_FAIL(PG_ERR_ARG, "entity_order must be a permutation of 0..nblocks-1");
      seen[order[i]] = 1;
      pos[order[i]] = (int32_t)i;
    }
  } else {
    std::iota(pos.begin(), pos.end(), 0);
  }
  // element order: by segment (multi-mesh operator), then by the earliest schedule
  // position of the element's entities (spatial order when the schedule is)
  // (from here on an element's entities are known by their schedule positions, so that
  // what follows, element after element in that order, finds an entity's data near the
  // last one's)
  std::vector<int32_t> key(E);
  std::vector<int32_t> es(E, 0);
  for (int64_t e = 0; e < E; ++e) {
    int32_t* ep = &eg[e * nle];
    int32_t m = ep[0] = pos[ep[0]], mx = m;
    for (int la = 1; la < nle; ++la) {
      ep[la] = pos[ep[la]];
      m = std::min(m, ep[la]);
      mx = std::max(mx, ep[la]);
    }
    key[e] = m;
    if (seg) {
      const auto& sp = seg->pos;
      const int sm = (int)(std::upper_bound(sp.begin(), sp.end(), (int64_t)m) - sp.begin()) - 1;
      if (sm < 0 || sm >= seg->nseg || mx >= sp[sm + 1])
        PG_FAIL(PG_ERR_ARG, "element %lld has entities of two meshes", (long long)e);
      es[e] = sm;
    }
  }
  // (stable counting sort; a segment's schedule positions are consecutive, so the
  // position alone also orders the segments)
  std::vector<int32_t> first(nblocks + 1, 0), sorted(E);
  for (int64_t e = 0; e < E; ++e) first[key[e] + 1]++;
  for (int64_t i = 0; i < nblocks; ++i) first[i + 1] += first[i];
  for (int64_t e = 0; e < E; ++e) sorted[first[key[e]]++] = (int32_t)e;
  // slot groups of 64 elements of one segment
  std::vector<int32_t> perm, wsg;
  for (int64_t k = 0; k < E;) {
    const int sg = es[sorted[k]];
    int64_t k1 = k;
    while (k1 < E && es[sorted[k1]] == sg) ++k1;
    for (int64_t a = k; a < k1; a += kWave) {
      wsg.push_back(sg);
      for (int l = 0; l < kWave; ++l) perm.push_back(a + l < k1 ? sorted[a + l] : -1);
    }
    k = k1;
  }
  const int64_t nw = (int64_t)wsg.size(), nslot = nw * kWave;
  if (nslot * N >= (1LL << 31)) PG_FAIL(PG_ERR_UNSUPPORTED, "too many elements");
  // scheduled entities with their lists of local results (in schedule order; the list's
  // end counts up as it is filled, -1: PEC)
  std::vector<int4> gm(nblocks);
  int64_t total = 0;
  for (int64_t i = 0; i < nblocks; ++i) {
    const int64_t g = order ? order[i] : i;
    gm[i] = make_int4(bp[g], bp[g + 1] - bp[g], (int)total, hbc[g] ? -1 : (int)total);
    total += hbc[g] ? 0 : cnt[g];
    if (total >= (1LL << 31)) PG_FAIL(PG_ERR_UNSUPPORTED, "too many incidences");
  }
  // per slot its orientation, per slot and local entity the entity's first DOF (-1: PEC
  // or empty), and the lists: slot * nle + local entity, within an entity in ascending
  // slot order (a fixed summation order)
  std::vector<int32_t> hoc(nslot, 0), hed((size_t)nslot * nle, -1), inc(total);
  for (int64_t s = 0; s < nslot; ++s) {
    const int64_t e = perm[s];
    if (e < 0) continue;
    const int64_t w = s / kWave, l = s % kWave;
    hoc[s] = hor[e];
    for (int la = 0; la < nle; ++la) {
      int4& m = gm[eg[e * nle + la]];
      if (m.w < 0) continue;
      hed[(w * nle + la) * kWave + l] = m.x;
      inc[m.w++] = (int32_t)(s * nle + la);
    }
  }
  for (int4& m : gm)
    if (m.w < 0) m.w = m.z;
  // The one-kernel product at p <= 2.  Two groups per block from 131 072 elements:
  // fewer elements are computed twice (1.8 against 2.1 times each, p = 2), but a
  // block takes two passes, which pays once the blocks fill the chip several
  // times (us per FP64 iteration with one / two: 40.4 / 46.8 at 48 000 elements,
  // 66.7 / 64.6 at 105 000, 92 / 90 at 162 000, 196 / 182 at 384 000; mixed
  // precision 50.2 / 53.8 at 105 000, 73 / 70 at 162 000, 116 / 106 at 384 000).
  // At p = 3 an element costs four times as much and the two kernels are faster
  // (product at 82 944 elements 58 against 80 us, at 10 000 the same).
  Blocks B;
  const int passes = E >= (1 << 17) ? 2 : 1;
  if (seg || p > 2 ||
      !(p == 1 ? make_blocks<6>(passes, nslot, gm, inc, &B)
               : make_blocks<10>(passes, nslot, gm, inc, &B)))
    B = Blocks();
  std::vector<int32_t>& gslot = inc;
  if (p == 1) local_results<1>(gslot);
  else if (p == 2) local_results<2>(gslot);
  else local_results<3>(gslot);
  int rc = PG_OK;
  ElemOp* op = new ElemOp();
  op->p = p;
  op->N = N;
  op->D = maxd;
  op->E = E;
  op->ndof = ndof;
  op->nent = nblocks;
  op->nw = nw;
  {
    op->nblk = (int64_t)B.meta.size();
    op->lds_values = B.lds_values;
    const int64_t sums = maxd == 6 && nblocks < eop::kDofSumEntities ? 6 * nblocks : nblocks;
    int64_t g = op->nblk > 0 ? op->nblk : (sums + eop::kBS - 1) / eop::kBS;
    g = std::min<int64_t>(g, eop::kMaxGrid);
    if (g >= 64) g = (g / 8) * 8;
    op->grid = (int)std::max<int64_t>(g, 1);
  }
#define PG_A(ptr, cnt)                            \
  if ((rc = op->alloc(&(ptr), (cnt))) != PG_OK) { \
    delete op;                                    \
    return rc;                                    \
  }
  PG_A(op->edofs, hed.size());
  PG_A(op->perm, nslot);
  PG_A(op->ocode, nslot);
  PG_A(op->gm, nblocks);
  PG_A(op->gslot, gslot.size());
  PG_A(op->coef64, nslot * 12);
  PG_A(op->coef32, nslot * 12);
  if (op->nblk > 0) {
    PG_A(op->bmeta, B.meta.size());
    PG_A(op->bslot, B.slot.size());
    PG_A(op->bcode, B.slot.size());
    PG_A(op->bdofs, B.slot.size() * nle);
    PG_A(op->bpos, B.pos.size() / 2);
    PG_A(op->em, B.em.size());
    PG_A(op->xcopy, 2 * ndof);
  } else {
    PG_A(op->ye64, nslot * N);
    PG_A(op->ye32, nslot * N);
  }
  std::vector<double> womu;
  if (seg) {
    op->nseg = seg->nseg;
    op->seg_pos = seg->pos;
    op->seg_wave.assign(seg->nseg + 1, nw);
    for (int64_t w = nw - 1; w >= 0; --w) op->seg_wave[wsg[w]] = w;
    for (int sg = seg->nseg - 1; sg >= 0; --sg)  // a segment without waves starts where the next does
      op->seg_wave[sg] = std::min(op->seg_wave[sg], op->seg_wave[sg + 1]);
    for (double om : seg->omega) womu.push_back(om * eop::kMu0);
    PG_A(op->wseg, nw);
    PG_A(op->womu, womu.size());
  }
#undef PG_A
  const struct {
    void* dst;
    const void* src;
    size_t bytes;
  } up[] = {{op->edofs, hed.data(), hed.size() * sizeof(int32_t)},
            {op->perm, perm.data(), perm.size() * sizeof(int32_t)},
            {op->ocode, hoc.data(), hoc.size() * sizeof(int32_t)},
            {op->gm, gm.data(), gm.size() * sizeof(int4)},
            {op->gslot, gslot.data(), gslot.size() * sizeof(int32_t)},
            {op->bmeta, B.meta.data(), B.meta.size() * sizeof(int4)},
            {op->bslot, B.slot.data(), op->nblk ? B.slot.size() * sizeof(int32_t) : 0},
            {op->bpos, B.pos.data(), op->nblk ? B.pos.size() * sizeof(uint16_t) : 0},
            {op->em, B.em.data(), op->nblk ? B.em.size() * sizeof(int2) : 0},
            {op->wseg, wsg.data(), op->wseg ? wsg.size() * sizeof(int32_t) : 0},
            {op->womu, womu.data(), womu.size() * sizeof(double)}};
  for (const auto& u : up)
    if (u.bytes && hipMemcpy(u.dst, u.src, u.bytes, hipMemcpyHostToDevice) != hipSuccess) {
      delete op;
      PG_FAIL(PG_ERR_HIP, "element operator upload failed");
    }
  if (op->nblk > 0) {
    const int64_t n = (int64_t)B.slot.size();
    hipLaunchKernelGGL(eop::k_eop_blk_elements, dim3((unsigned)((n + eop::kBS - 1) / eop::kBS)),
                       dim3(eop::kBS), 0, st, n, nle, op->bslot, op->ocode, op->edofs, op->bcode,
                       op->bdofs);
  }
  if ((rc = eop_refresh(op, ws, omega, st)) != PG_OK) {
    delete op;
    return rc;
  }
  if (hipStreamSynchronize(st) != hipSuccess) {
    delete op;
    PG_FAIL(PG_ERR_HIP, "element operator setup failed");
  }
  *out = op;
  return PG_OK;
}

// y = A x.  y may be x or overlap it: the one-kernel product stores y while other
// workgroups still gather x, so it then reads a copy (the two kernels finish the
// gathers before the first store).
template <typename R>
static int apply(const void* handle, const R* x, R* y, void* stream) {
  if (!handle || !x || !y) PG_FAIL(PG_ERR_ARG, "bad arguments");
  using C = typename eop::Cx<R>::T;
  const ElemOp* op = static_cast<const ElemOp*>(handle);
  hipStream_t st = as_stream(stream);
  const int64_t n = 2 * op->ndof;
  const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(y);
  if (op->xcopy && xa < ya + n * sizeof(R) && ya < xa + n * sizeof(R)) {
    R* copy = reinterpret_cast<R*>(op->xcopy);
    hipLaunchKernelGGL(eop::k_eop_copy<R>, dim3((unsigned)((n + eop::kBS - 1) / eop::kBS)),
                       dim3(eop::kBS), 0, st, n, x, copy);
    x = copy;
  }
  eop_launch(op, 0, nullptr, reinterpret_cast<const C*>(x), reinterpret_cast<C*>(y), nullptr,
             nullptr, st);
  PG_CHECK_LAUNCH();
  return PG_OK;
}

}  // namespace pg

using namespace pg;

extern "C" {

int pg_eop_create(int p, int64_t E, const void* ws, const int32_t* dofs, int64_t ndof,
                  const int32_t* block_ptr, int64_t nblocks, const int32_t* order,
                  const uint8_t* ent_bc, double omega, void** out, void* stream) {
  if (!out || !ws || !dofs || !block_ptr || E <= 0 || ndof <= 0 || nblocks <= 0)
    PG_FAIL(PG_ERR_ARG, "bad arguments");
  if (p < 1 || p > 3)
    PG_FAIL(PG_ERR_UNSUPPORTED, "element-by-element operator: order p=%d not supported (1..3)", p);
  const int N = ndof_element(p);
  hipStream_t st = as_stream(stream);
  int rc0 = check_block_ptr(p, block_ptr, nblocks, ndof);
  if (rc0 != PG_OK) return rc0;
  // host copies of the element DOFs, orientations and PEC entities
  std::vector<int32_t> hd((size_t)E * N), hor(E);
  std::vector<uint8_t> hbc(nblocks, 0);
  const int32_t* dor = reinterpret_cast<const int32_t*>(reinterpret_cast<const double*>(ws) + 12 * E);
  PG_HIP(hipMemcpyAsync(hd.data(), dofs, hd.size() * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  PG_HIP(hipMemcpyAsync(hor.data(), dor, E * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  if (ent_bc)
    PG_HIP(hipMemcpyAsync(hbc.data(), ent_bc, nblocks, hipMemcpyDeviceToHost, st));
  PG_HIP(hipStreamSynchronize(st));
  ElemOp* op = nullptr;
  const int rc = eop_build(p, E, ws, ndof, block_ptr, nblocks, order, hd, hor, hbc, omega,
                           nullptr, &op, st);
  if (rc != PG_OK) return rc;
  *out = op;
  return PG_OK;
}

int pg_eop_create_multi(int p, int nseg, const int64_t* n_elems, const void* const* ws,
                        const int32_t* const* dofs, const int64_t* ndof,
                        const int32_t* const* block_ptr, const int64_t* nblocks,
                        const int32_t* const* order, const uint8_t* const* ent_bc,
                        const double* omega, void** out, void* stream) {
  if (!out || nseg <= 0 || !n_elems || !ws || !dofs || !ndof || !block_ptr || !nblocks || !omega)
    PG_FAIL(PG_ERR_ARG, "bad arguments");
  if (p < 1 || p > 3)
    PG_FAIL(PG_ERR_UNSUPPORTED, "element-by-element operator: order p=%d not supported (1..3)", p);
  const int N = ndof_element(p);
  hipStream_t st = as_stream(stream);
  // the union: mesh s's elements, DOFs and entities follow those of meshes < s
  int64_t E = 0, nd = 0, nb = 0;
  SegInfo seg;
  seg.nseg = nseg;
  seg.pos.push_back(0);
  for (int s = 0; s < nseg; ++s) {
    if (n_elems[s] <= 0 || ndof[s] <= 0 || nblocks[s] <= 0 || !ws[s] || !dofs[s] ||
        !block_ptr[s])
      PG_FAIL(PG_ERR_ARG, "mesh %d: bad arguments", s);
    int rc0 = check_block_ptr(p, block_ptr[s], nblocks[s], ndof[s]);
    if (rc0 != PG_OK) return rc0;
    E += n_elems[s];
    nd += ndof[s];
    nb += nblocks[s];
    seg.pos.push_back(nb);
    seg.omega.push_back(omega[s]);
  }
  if (nd >= (1LL << 31) || nb >= (1LL << 31) || E * N >= (1LL << 31))
    PG_FAIL(PG_ERR_UNSUPPORTED, "the meshes together are too large for 32-bit indices");
  std::vector<int32_t> hd((size_t)E * N), hor(E), bp(nb + 1), ord(nb);
  std::vector<uint8_t> hbc(nb, 0);
  double* wsu = nullptr;
  if (hipMalloc(&wsu, (size_t)E * 12 * sizeof(double)) != hipSuccess)
    PG_FAIL(PG_ERR_HIP, "hipMalloc(%lld) failed", (long long)(E * 12 * sizeof(double)));
  int64_t e0 = 0, d0 = 0, b0 = 0;
  int rc = PG_OK;
  for (int s = 0; s < nseg && rc == PG_OK; ++s) {
    const int64_t Es = n_elems[s];
    const double* wss = reinterpret_cast<const double*>(ws[s]);
    if (hipMemcpyAsync(wsu + 12 * e0, wss, Es * 12 * sizeof(double), hipMemcpyDeviceToDevice,
                       st) != hipSuccess ||
        hipMemcpyAsync(hd.data() + e0 * N, dofs[s], Es * N * sizeof(int32_t),
                       hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(hor.data() + e0, reinterpret_cast<const int32_t*>(wss + 12 * Es),
                       Es * sizeof(int32_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
        (ent_bc && ent_bc[s] &&
         hipMemcpyAsync(hbc.data() + b0, ent_bc[s], nblocks[s], hipMemcpyDeviceToHost, st) !=
             hipSuccess) ||
        hipStreamSynchronize(st) != hipSuccess) {
      rc = PG_ERR_HIP;
      break;
    }
    for (int64_t k = e0 * N; k < (e0 + Es) * N; ++k) hd[k] += (int32_t)d0;
    for (int64_t g = 0; g < nblocks[s]; ++g) {
      bp[b0 + g] = (int32_t)(block_ptr[s][g] + d0);
      const int32_t o = order && order[s] ? order[s][g] : (int32_t)g;
      if (o < 0 || o >= nblocks[s]) {
        rc = PG_ERR_ARG;
        break;
      }
      ord[b0 + g] = (int32_t)(o + b0);
    }
    e0 += Es;
    d0 += ndof[s];
    b0 += nblocks[s];
  }
  bp[nb] = (int32_t)nd;
  ElemOp* op = nullptr;
  if (rc == PG_OK)
    rc = eop_build(p, E, wsu, nd, bp.data(), nb, ord.data(), hd, hor, hbc, 0.0, &seg, &op, st);
  else
    set_error("multi-mesh element operator: copies failed or an entity order out of range");
  if (rc != PG_OK) {
    (void)hipFree(wsu);
    return rc;
  }
  op->owned.push_back(wsu);  // the union's coefficients, read by no refresh
  *out = op;
  return PG_OK;
}

int pg_eop_refresh(void* op, const void* ws, double omega, void* stream) {
  if (!op || !ws) PG_FAIL(PG_ERR_ARG, "bad arguments");
  if (static_cast<ElemOp*>(op)->nseg > 0)
    PG_FAIL(PG_ERR_UNSUPPORTED, "a multi-mesh element operator keeps its creation coefficients");
  return eop_refresh(static_cast<ElemOp*>(op), ws, omega, as_stream(stream));
}

int pg_eop_apply_z(const void* op, const double* x, double* y, void* stream) {
  return apply<double>(op, x, y, stream);
}

int pg_eop_apply_c(const void* op, const float* x, float* y, void* stream) {
  return apply<float>(op, x, y, stream);
}

int pg_eop_destroy(void* op) {
  delete static_cast<ElemOp*>(op);
  return PG_OK;
}

}  // extern "C"
