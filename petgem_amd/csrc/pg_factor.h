// Factored element products on the unit tetrahedron, p = 1 and 2.
//
// K_e x and M_e x of one element without its matrices or any table.  The
// field of the DOF vector x is expanded in Bernstein monomials of the
// barycentric coordinates times the constant gradients e_1, e_2, e_3 of
// lambda_1..lambda_3 (grad lambda_0 = -(e_1 + e_2 + e_3)); in that basis the
// geometry tensor acts on every monomial by itself, and the integral of two
// monomials is gamma! / (3 + |gamma|)!, whose sums over all pairs collapse to
// a few running sums.  The transposed expansion then gives the moments against
// the basis functions.  The curl-curl part does the same with the curl, which
// is linear (p = 2) or constant (p = 1) in the barycentric coordinates.
// About 700 multiply-adds per real vector and element at p = 2 for K x and M x
// together, against 1600 for forming the 210 entries once from the reference
// tables plus 750 for applying them, and no table to load.  The results are
// those of the order-2p quadrature (exact for these polynomials) to rounding.
//
// Orientation: every element is computed with edge flags and face codes 0; the
// functions of another flag or code are combinations of those with
// coefficients 0 and +-1 (Orient below), applied to x on the way in and, as
// the transpose, to the moments on the way out.
//
// Sums start from -0.0, which the compiler drops (x + -0.0 = x for every x),
// so the first contribution to a coefficient costs nothing.
#pragma once

#include "pg_basis.h"

namespace pg {
namespace fac {

template <int P>
constexpr int n_dofs() {
  return P * (P + 2) * (P + 3) / 2;
}

// v += s * (integer c in -3..3), c known at compile time
template <typename R>
PG_HD void acc(R& v, int c, R s) {
  if (c == 1) v = v + s;
  else if (c == -1) v = v - s;
  else if (c != 0) v = v + R(c) * s;
}
// component k of grad lambda_a, and of grad lambda_a x grad lambda_b
PG_HD constexpr int grad(int a, int k) { return a == 0 ? -1 : (a == k + 1 ? 1 : 0); }
PG_HD constexpr int gradx(int a, int b, int k) {
  return grad(a, (k + 1) % 3) * grad(b, (k + 2) % 3) - grad(a, (k + 2) % 3) * grad(b, (k + 1) % 3);
}
// local entities as constant expressions (edge_vert, face_vert)
PG_HD constexpr int ev(int e, int k) {
  constexpr int t[12] = {0, 1, 1, 2, 0, 2, 0, 3, 1, 3, 2, 3};
  return t[2 * e + k];
}
PG_HD constexpr int fv(int f, int k) {
  constexpr int t[12] = {0, 1, 2, 0, 1, 3, 1, 2, 3, 0, 2, 3};
  return t[3 * f + k];
}
// index of the product lambda_i lambda_j among the six mixed monomials
PG_HD constexpr int mono(int i, int j) {
  constexpr int t[16] = {0, 0, 1, 2, 0, 0, 3, 4, 1, 3, 0, 5, 2, 4, 5, 0};
  return t[4 * i + j];
}

// ---------------------------------------------------------------------------
// orientation of one element (packed as orient_of reads it) as coefficients:
// edge functions of degree 0 change sign with the edge's flag, those of degree
// 1 do not; the two functions of a face with code o are t[m][0], t[m][1] times
// the two of code 0 (the functions of a face span one space for every code)
// ---------------------------------------------------------------------------
template <int P, typename R>
struct Orient {
  R s[6];
  R t[P >= 2 ? 4 : 1][4];
  PG_HD explicit Orient(int packed) {
#pragma unroll
    for (int e = 0; e < 6; ++e) s[e] = (packed >> e) & 1 ? R(-1) : R(1);
    if constexpr (P >= 2) {
      // codes 0..5, two bits each (two's complement)
      constexpr int v[4][6] = {
          {1, 0, -1, 1, -1, 0}, {0, 1, -1, 1, 0, -1}, {0, -1, 1, 0, 1, -1}, {1, -1, 0, -1, 1, 0}};
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int sh = 30 - 2 * ((packed >> (6 + 3 * f)) & 7);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          unsigned pk = 0;
#pragma unroll
          for (int o = 0; o < 6; ++o) pk |= (unsigned)(v[k][o] & 3) << (2 * o);
          t[f][k] = R((int)(pk << sh) >> 30);
        }
      }
    }
  }
  // coefficients of the code-0 functions
  PG_HD void in(R* x) const {
#pragma unroll
    for (int e = 0; e < 6; ++e) x[P * e] = s[e] * x[P * e];
    if constexpr (P >= 2) {
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const R a = x[12 + 2 * f], b = x[13 + 2 * f];
        x[12 + 2 * f] = t[f][0] * a + t[f][2] * b;
        x[13 + 2 * f] = t[f][1] * a + t[f][3] * b;
      }
    }
  }
  // moments against the element's own functions
  PG_HD void out(R* y) const {
#pragma unroll
    for (int e = 0; e < 6; ++e) y[P * e] = s[e] * y[P * e];
    if constexpr (P >= 2) {
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const R a = y[12 + 2 * f], b = y[13 + 2 * f];
        y[12 + 2 * f] = t[f][0] * a + t[f][1] * b;
        y[13 + 2 * f] = t[f][2] * a + t[f][3] * b;
      }
    }
  }
};

// symmetric 3 x 3 product in place; g = (00, 11, 22, 01, 02, 12)
template <typename R>
PG_HD void sym3(const R (&g)[6], R (&v)[3]) {
  const R a = v[0], b = v[1], c = v[2];
  v[0] = g[0] * a + (g[3] * b + g[4] * c);
  v[1] = g[1] * b + (g[3] * a + g[5] * c);
  v[2] = g[2] * c + (g[4] * a + g[5] * b);
}

// y = K x, h the curl-curl coefficients H / det
template <int P, typename R>
PG_HD void curl_product(const R* x, const R (&h)[6], R* y) {
  if constexpr (P == 1) {
    // curl of the edge (a, b): 2 grad_a x grad_b, constant: 4 * volume 1/6
    R c[3] = {R(-0.0), R(-0.0), R(-0.0)};
#pragma unroll
    for (int e = 0; e < 6; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) acc(c[k], gradx(ev(e, 0), ev(e, 1), k), x[e]);
    sym3(h, c);
#pragma unroll
    for (int k = 0; k < 3; ++k) c[k] = c[k] * R(2.0 / 3.0);
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      R s = R(-0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) acc(s, gradx(ev(e, 0), ev(e, 1), k), c[k]);
      y[e] = s;
    }
  } else {
    // curl = sum_i lambda_i c[i]; a constant is the same value at every i
    R k0[3], c[4][3];
#pragma unroll
    for (int k = 0; k < 3; ++k) k0[k] = R(-0.0);
#pragma unroll
    for (int e = 0; e < 6; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) acc(k0[k], gradx(ev(e, 0), ev(e, 1), k), x[2 * e]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) c[i][k] = R(2) * k0[k];
    // edge functions (lambda_b - lambda_a) w: curl 3 (lambda_b - lambda_a) grad_a x grad_b
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const R s = R(3) * x[2 * e + 1];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(c[ev(e, 1)][k], gradx(ev(e, 0), ev(e, 1), k), s);
        acc(c[ev(e, 0)][k], -gradx(ev(e, 0), ev(e, 1), k), s);
      }
    }
    // face functions lambda_c (lambda_a grad_b - lambda_b grad_a):
    // curl 2 lambda_c grad_a x grad_b + lambda_a grad_c x grad_b - lambda_b grad_c x grad_a
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        const R s = x[12 + 2 * f + m];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(c[vc][k], 2 * gradx(va, vb, k), s);
          acc(c[va][k], gradx(vc, vb, k), s);
          acc(c[vb][k], -gradx(vc, va, k), s);
        }
      }
    // geometry, then the mass matrix (1 + delta_ij) / 120 of the lambda_i
#pragma unroll
    for (int i = 0; i < 4; ++i) sym3(h, c[i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const R s = ((c[0][k] + c[1][k]) + (c[2][k] + c[3][k]));
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i][k] = R(1.0 / 120.0) * (c[i][k] + s);
      k0[k] = R(2) * ((c[0][k] + c[1][k]) + (c[2][k] + c[3][k]));
    }
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      R s = R(-0.0), d = R(-0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(s, gradx(ev(e, 0), ev(e, 1), k), k0[k]);
        acc(d, gradx(ev(e, 0), ev(e, 1), k), c[ev(e, 1)][k]);
        acc(d, -gradx(ev(e, 0), ev(e, 1), k), c[ev(e, 0)][k]);
      }
      y[2 * e] = s;
      y[2 * e + 1] = R(3) * d;
    }
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        R s = R(-0.0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(s, 2 * gradx(va, vb, k), c[vc][k]);
          acc(s, gradx(vc, vb, k), c[va][k]);
          acc(s, -gradx(vc, va, k), c[vb][k]);
        }
        y[12 + 2 * f + m] = s;
      }
  }
}

// y = M x, g the mass coefficients (det G, times any factor)
template <int P, typename R>
PG_HD void mass_product(const R* x, const R (&g)[6], R* y) {
  // linear fields: u = sum_i lambda_i a[i], the Whitney functions
  // lambda_a grad_b - lambda_b grad_a
  R a[4][3];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) a[i][k] = R(-0.0);
#pragma unroll
  for (int e = 0; e < 6; ++e)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      acc(a[ev(e, 0)][k], grad(ev(e, 1), k), x[P * e]);
      acc(a[ev(e, 1)][k], -grad(ev(e, 0), k), x[P * e]);
    }
  if constexpr (P == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sym3(g, a[i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const R s = ((a[0][k] + a[1][k]) + (a[2][k] + a[3][k]));
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i][k] = R(1.0 / 120.0) * (a[i][k] + s);
    }
  } else {
    // quadratic: u = sum_i lambda_i^2 a[i] + sum_{i<j} lambda_i lambda_j b[ij]
    // (the linear part times sum_j lambda_j = 1)
    R b[6][3];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i + 1; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) b[mono(i, j)][k] = a[i][k] + a[j][k];
    // (lambda_b - lambda_a)(lambda_a grad_b - lambda_b grad_a)
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const int va = ev(e, 0), vb = ev(e, 1);
      const R s = x[2 * e + 1];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(b[mono(va, vb)][k], grad(va, k) + grad(vb, k), s);
        acc(a[va][k], -grad(vb, k), s);
        acc(a[vb][k], -grad(va, k), s);
      }
    }
    // lambda_c (lambda_a grad_b - lambda_b grad_a)
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        const R s = x[12 + 2 * f + m];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(b[mono(vc, va)][k], grad(vb, k), s);
          acc(b[mono(vc, vb)][k], -grad(va, k), s);
        }
      }
    R gs[6];  // 1 / 7!, the weight of every quartic monomial's gamma!
#pragma unroll
    for (int k = 0; k < 6; ++k) gs[k] = R(1.0 / 5040.0) * g[k];
#pragma unroll
    for (int i = 0; i < 4; ++i) sym3(gs, a[i]);
#pragma unroll
    for (int i = 0; i < 6; ++i) sym3(gs, b[i]);
    // moments: with B_i = sum_j b_ij, c_i = 4 a_i + B_i, S = 2 sum a + sum b
    //   lambda_i^2        24 a_i + 4 sum_{j/=i} a_j + 6 B_i + 2 (sum b - B_i)
    //                     = 2 S + 4 c_i + 4 a_i
    //   lambda_i lambda_j 6 (a_i + a_j) + 2 sum_{k/=i,j} a_k + 4 b_ij + 2 (..) + ..
    //                     = S + c_i + c_j + b_ij
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      R B[4], c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        B[i] = R(-0.0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j != i) B[i] = B[i] + b[mono(i, j)][k];
        c[i] = R(4) * a[i][k] + B[i];
      }
      // sum c = 4 sum a + 2 sum b = 2 S
      const R S2 = (c[0] + c[1]) + (c[2] + c[3]);
      const R S = R(0.5) * S2;
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i][k] = R(4) * (c[i] + a[i][k]) + S2;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i + 1; j < 4; ++j)
          b[mono(i, j)][k] = (S + b[mono(i, j)][k]) + (c[i] + c[j]);
    }
    // transposed expansion
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        R s = R(-0.0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(s, grad(vb, k), b[mono(vc, va)][k]);
          acc(s, -grad(va, k), b[mono(vc, vb)][k]);
        }
        y[12 + 2 * f + m] = s;
      }
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const int va = ev(e, 0), vb = ev(e, 1);
      R s = R(-0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(s, grad(va, k) + grad(vb, k), b[mono(va, vb)][k]);
        acc(s, -grad(vb, k), a[va][k]);
        acc(s, -grad(va, k), a[vb][k]);
      }
      y[2 * e + 1] = s;
    }
    // moments of lambda_i = lambda_i sum_j lambda_j
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j != i)
#pragma unroll
          for (int k = 0; k < 3; ++k) a[i][k] = a[i][k] + b[mono(i, j)][k];
  }
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    R s = R(-0.0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      acc(s, grad(ev(e, 1), k), a[ev(e, 0)][k]);
      acc(s, -grad(ev(e, 0), k), a[ev(e, 1)][k]);
    }
    y[P * e] = s;
  }
}

}  // namespace fac
}  // namespace pg
