// Factored element products on the unit tetrahedron, p = 1, 2 and 3.
//
// K_e x and M_e x of one element without its matrices or any table.  The
// field of the DOF vector x is expanded in Bernstein monomials of the
// barycentric coordinates times the constant gradients e_1, e_2, e_3 of
// lambda_1..lambda_3 (grad lambda_0 = -(e_1 + e_2 + e_3)); in that basis the
// geometry tensor acts on every monomial by itself, and the integral of two
// monomials is gamma! / (3 + |gamma|)!, whose sums over all pairs collapse to
// a few running sums.  The transposed expansion then gives the moments against
// the basis functions.  The curl-curl part does the same with the curl, one
// degree lower.  Every basis function is a polynomial phi in the lambda times
// a Whitney function w_ab = lambda_a grad_b - lambda_b grad_a, of degree 0, 1
// or 2: functions of one degree are expanded together and their sum is raised
// to the next degree (times sum_i lambda_i = 1) before the next ones join.
// About 800 operations per real vector and element at p = 2 for K x and M x
// together, against 1600 multiply-adds for forming the 210 entries once from
// the reference tables plus 750 for applying them, and no table to load (p = 3:
// 3 200 operations per real vector, against 17 600 instructions per element).  The results are those of the order-2p
// quadrature (exact for these polynomials) to rounding.
//
// Orientation: every element is computed with edge flags and face codes 0; the
// functions of another flag or code are combinations of those (orient_in,
// orient_out below), applied to x on the way in and, as the transpose, to the
// moments on the way out.
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

// v += s * c, c known at compile time
template <typename R>
PG_HD void acc(R& v, double c, R s) {
  if (c == 1.0) v = v + s;
  else if (c == -1.0) v = v - s;
  else if (c != 0.0) v = v + R(c) * s;
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
// Orientation of one element (packed as orient_of reads it).  Edge functions of
// even degree change sign with the edge's flag, those of odd degree do not.
// The functions of a face come in pairs f_0, f_1 (families 0 and 1); with the
// third, f_2, of the same kind (the family that starts at the face's third
// vertex) a code permutes the three, with a change of sign for codes 3..5 where
// phi is symmetric in a and b.  f_2 itself is a combination of the others:
//   phi = lambda_c                     f_2 = -f_0 - f_1
//   phi = lambda_c^2 / 2 - lambda_c (lambda_a + lambda_b), and
//   phi = (lambda_b - lambda_a) lambda_c (p = 3; no change of sign)
//                                      f_2 by face_third: all six functions of
//                                      the face and the volume's
// so with c the coefficients of f_0, f_1, f_2 from the pair's two, c_j =
// sum_m e[j][m] x_m, the code-0 coefficients are c_0, c_1 plus c_2 times f_2's.
// ---------------------------------------------------------------------------
// The coefficients by code are read from a table of face_entries<P>() values per
// code, which a kernel keeps in LDS (fill_faces): they differ from lane to lane,
// and forming them from the code took a fifth of the instructions at p = 2.
//   p = 2: c_0, c_1 after f_2 = -f_0 - f_1: t[m][j] = e[j][m] - e[2][m]
//   p = 3: e[j][m], and the sign -1 for codes 3..5
PG_HD constexpr int face_perm_entry(int o, int j, int m) {
  // f_m of code o is +-f_j of code 0
  constexpr int v[6][3][2] = {{{1, 0}, {0, 1}, {0, 0}},   {{0, 0}, {1, 0}, {0, 1}},
                              {{0, 1}, {0, 0}, {1, 0}},   {{0, 0}, {0, -1}, {-1, 0}},
                              {{-1, 0}, {0, 0}, {0, -1}}, {{0, -1}, {-1, 0}, {0, 0}}};
  return v[o][j][m];
}
template <int P>
PG_HD constexpr int face_entries() {
  return P == 3 ? 8 : 4;
}
template <int P>
PG_HD constexpr int face_table_size() {
  return P == 1 ? 1 : 8 * face_entries<P>();  // codes 6, 7 do not occur
}
template <int P>
PG_HD constexpr int face_table(int i) {
  const int o = i / face_entries<P>(), k = i % face_entries<P>();
  if (P == 1 || o > 5) return 0;
  if (P == 2) return face_perm_entry(o, k % 2, k / 2) - face_perm_entry(o, 2, k / 2);
  return k < 6 ? face_perm_entry(o, k / 2, k % 2) : (k == 6 ? (o > 2 ? -1 : 1) : 0);
}
template <int P>
struct FaceTable {
  int v[face_table_size<P>()];
};
template <int P>
constexpr FaceTable<P> make_face_table() {
  FaceTable<P> t{};
  for (int i = 0; i < face_table_size<P>(); ++i) t.v[i] = face_table<P>(i);
  return t;
}
template <int P>
inline constexpr FaceTable<P> kFaces = make_face_table<P>();
template <int P, typename R>
PG_HD const R* face_row(const R* tab, int packed, int f) {
  return tab + ((packed >> (6 + 3 * f)) & 7) * face_entries<P>();
}
// f_2 of face f, kind t (0: phi = lambda_c^2 / 2 - .., 1: phi = (lambda_b -
// lambda_a) lambda_c): coefficient of function k < 6 of the face, k - 6 of the volume
PG_HD constexpr double face_third(int f, int t, int k) {
  constexpr double c[2][6] = {{0.75, 0.75, 0.5, 0.5, -0.75, 0.75}, {0.5, -0.5, 1, -1, 0.5, 0.5}};
  constexpr double b[4][2][3] = {{{-0.75, -0.75, 0}, {-0.5, 0.5, 0}},
                                 {{-0.75, -0.75, -0.75}, {-0.5, 0.5, 0.5}},
                                 {{0, -0.75, -0.75}, {0, -0.5, 0.5}},
                                 {{-0.75, -0.75, -0.75}, {-0.5, -0.5, 0.5}}};
  return k < 6 ? c[t][k] : b[f][t][k - 6];
}
// x -> coefficients of the code-0 functions; tab = the table of face coefficients
template <int P, typename R>
PG_HD void orient_in(int packed, const R* tab, R* x) {
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    const R s = (packed >> e) & 1 ? R(-1) : R(1);
    x[P * e] = s * x[P * e];
    if constexpr (P >= 3) x[P * e + 2] = s * x[P * e + 2];
  }
  if constexpr (P >= 2)
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const R* q = face_row<P>(tab, packed, f);
      R* xf = x + 6 * P + f * P * (P - 1);
      if constexpr (P == 2) {
        const R a = xf[0], b = xf[1];
        xf[0] = q[0] * a + q[2] * b;
        xf[1] = q[1] * a + q[3] * b;
      } else {
        R c[3][3];  // [pair][j]
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          R a = xf[2 * t], b = xf[2 * t + 1];
          if (t == 2) a = q[6] * a, b = q[6] * b;
#pragma unroll
          for (int j = 0; j < 3; ++j) c[t][j] = q[2 * j] * a + q[2 * j + 1] * b;
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) xf[k] = c[k / 2][k % 2];
        xf[0] = xf[0] - c[0][2];
        xf[1] = xf[1] - c[0][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int k = 0; k < 9; ++k)
            acc(k < 6 ? xf[k] : x[36 + k], face_third(f, t, k), c[t + 1][2]);
      }
    }
}
// moments against the code-0 functions -> against the element's own
template <int P, typename R>
PG_HD void orient_out(int packed, const R* tab, R* y) {
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    const R s = (packed >> e) & 1 ? R(-1) : R(1);
    y[P * e] = s * y[P * e];
    if constexpr (P >= 3) y[P * e + 2] = s * y[P * e + 2];
  }
  if constexpr (P >= 2)
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const R* q = face_row<P>(tab, packed, f);
      R* yf = y + 6 * P + f * P * (P - 1);
      if constexpr (P == 2) {
        const R a = yf[0], b = yf[1];
        yf[0] = q[0] * a + q[1] * b;
        yf[1] = q[2] * a + q[3] * b;
      } else {
        R d[3][3];
#pragma unroll
        for (int k = 0; k < 6; ++k) d[k / 2][k % 2] = yf[k];
        d[0][2] = R(0) - (yf[0] + yf[1]);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          R v = R(-0.0);
#pragma unroll
          for (int k = 0; k < 9; ++k) acc(v, face_third(f, t, k), k < 6 ? yf[k] : y[36 + k]);
          d[t + 1][2] = v;
        }
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const R v = q[m] * d[t][0] + (q[2 + m] * d[t][1] + q[4 + m] * d[t][2]);
            yf[2 * t + m] = t == 2 ? q[6] * v : v;
          }
      }
    }
}

// ---------------------------------------------------------------------------
// p = 3: the 25 functions with quadratic phi (edges, the last four of each
// face, the volume), as coefficients on the 20 cubic monomials (field) and on
// the 10 quadratic ones (curl)
// ---------------------------------------------------------------------------
// quadratic monomial lambda_i lambda_j: i = j first, then the mixed ones
PG_HD constexpr int quad(int i, int j) { return i == j ? i : 4 + mono(i, j); }
// cubic monomial by its exponents: lambda_i^3 (0..3), lambda_i^2 lambda_j
// (4 + 3 i + ..), lambda_i lambda_j lambda_k (16 + the absent index)
PG_HD constexpr int cubic(int i, int j, int k) {
  if (i == j && j == k) return i;
  if (i == j) return 4 + 3 * i + (k > i ? k - 1 : k);
  if (i == k) return 4 + 3 * i + (j > i ? j - 1 : j);
  if (j == k) return 4 + 3 * j + (i > j ? i - 1 : i);
  return 16 + (6 - i - j - k);
}
constexpr int kCubicFns = 25;
struct CubicFns {
  int dof[kCubicFns];
  double field[kCubicFns][20][3];
  double curl[kCubicFns][10][3];
};
constexpr CubicFns make_cubic() {
  CubicFns r{};
  for (int n = 0; n < kCubicFns; ++n) {
    double phi[4][4] = {};  // phi = sum_{i <= j} phi[i][j] lambda_i lambda_j
    int a = 0, b = 0;
    const auto add = [&phi](int i, int j, double v) { phi[i < j ? i : j][i < j ? j : i] += v; };
    if (n < 6) {
      a = ev(n, 0);
      b = ev(n, 1);
      add(a, a, 1.0);
      add(b, b, 1.0);
      add(a, b, -4.0);
      r.dof[n] = 3 * n + 2;
    } else if (n < 22) {
      const int f = (n - 6) / 4, m = (n - 6) % 2, kind = (n - 6) % 4 / 2;
      a = fv(f, m);
      b = fv(f, (m + 1) % 3);
      const int c = fv(f, (m + 2) % 3);
      if (kind == 0) {
        add(c, c, 0.5);
        add(c, a, -1.0);
        add(c, b, -1.0);
      } else {
        add(b, c, 1.0);
        add(a, c, -1.0);
      }
      r.dof[n] = 18 + 6 * f + 2 + (n - 6) % 4;
    } else {
      const int m = n - 22;
      a = m % 4;
      b = (m + 1) % 4;
      add((m + 2) % 4, (m + 3) % 4, 1.0);
      r.dof[n] = 42 + m;
    }
    for (int i = 0; i < 4; ++i)
      for (int j = i; j < 4; ++j) {
        const double v = phi[i][j];
        if (v == 0.0) continue;
        for (int k = 0; k < 3; ++k) {
          // phi (lambda_a grad_b - lambda_b grad_a)
          r.field[n][cubic(i, j, a)][k] += v * grad(b, k);
          r.field[n][cubic(i, j, b)][k] -= v * grad(a, k);
          // 2 phi grad_a x grad_b + grad phi x w_ab
          r.curl[n][quad(i, j)][k] += 2.0 * v * gradx(a, b, k);
          r.curl[n][quad(j, a)][k] += v * gradx(i, b, k);
          r.curl[n][quad(j, b)][k] -= v * gradx(i, a, k);
          r.curl[n][quad(i, a)][k] += v * gradx(j, b, k);
          r.curl[n][quad(i, b)][k] -= v * gradx(j, a, k);
        }
      }
  }
  return r;
}
inline constexpr CubicFns kCubic = make_cubic();

// symmetric 3 x 3 product in place; g = (00, 11, 22, 01, 02, 12)
template <typename R>
PG_HD void sym3(const R (&g)[6], R (&v)[3]) {
  const R a = v[0], b = v[1], c = v[2];
  v[0] = g[0] * a + (g[3] * b + g[4] * c);
  v[1] = g[1] * b + (g[3] * a + g[5] * c);
  v[2] = g[2] * c + (g[4] * a + g[5] * b);
}

// ---------------------------------------------------------------------------
// scalar mass matrices of the Bernstein monomials of one component, in place
// ---------------------------------------------------------------------------
// degree 1: (1 + delta_ij) / 5!, without the factor
template <typename R>
PG_HD void mass1(R& a, R& b, R& c, R& d) {
  const R s = (a + b) + (c + d);
  a = a + s;
  b = b + s;
  c = c + s;
  d = d + s;
}
// degree 2 (q[0..3] the squares, q[4..9] the mixed), without the factor 1 / 7!:
// with B_i = sum_j q_ij, c_i = 4 q_ii + B_i, S = 2 sum q_ii + sum q_ij the moments
// are  24 q_ii + 4 sum_{j/=i} q_jj + 6 B_i + 2 (sum q_ij - B_i) = 2 S + 4 c_i + 4 q_ii
// and  S + c_i + c_j + q_ij
template <typename R>
PG_HD void mass2(R (*q)[3], int k) {
  R c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    R B = R(-0.0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j != i) B = B + q[quad(i, j)][k];
    c[i] = R(4) * q[i][k] + B;
  }
  const R S2 = (c[0] + c[1]) + (c[2] + c[3]);  // 2 S
  const R S = R(0.5) * S2;
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i][k] = R(4) * (c[i] + q[i][k]) + S2;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = i + 1; j < 4; ++j)
      q[quad(i, j)][k] = (S + q[quad(i, j)][k]) + (c[i] + c[j]);
}
// degree 3, without the factor 1 / 9!: (alpha + beta)! = alpha! beta! sum_kappa
// C(alpha, kappa) C(beta, kappa), so with v = beta! u the sums t_kappa = sum_beta
// C(beta, kappa) v_beta are formed degree by degree ((3 - |kappa|) t_kappa =
// sum_i (kappa_i + 1) t_{kappa + e_i}) and brought back up by the transpose
template <typename R>
PG_HD void mass3(R (*u)[3], int k) {
  R v[20];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = R(6) * u[i][k];
#pragma unroll
  for (int m = 4; m < 16; ++m) v[m] = R(2) * u[m][k];
#pragma unroll
  for (int m = 16; m < 20; ++m) v[m] = u[m][k];
  R t2[10], t1[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // kappa = 2 e_i: 3 v_iii + sum_j v_iij
    R s = R(-0.0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j != i) s = s + v[cubic(i, i, j)];
    t2[i] = R(3) * v[i] + s;
#pragma unroll
    for (int j = i + 1; j < 4; ++j) {
      // kappa = e_i + e_j: 2 v_iij + 2 v_ijj + sum_k v_ijk
      R w = R(-0.0);
#pragma unroll
      for (int l = 0; l < 4; ++l)
        if (l != i && l != j) w = w + v[cubic(i, j, l)];
      t2[quad(i, j)] = R(2) * (v[cubic(i, i, j)] + v[cubic(i, j, j)]) + w;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // (2 t_ii + sum_j t_ij) / 2
    R s = R(-0.0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j != i) s = s + t2[quad(i, j)];
    t1[i] = t2[i] + R(0.5) * s;
  }
  // t_0 = sum t_i / 3, and back up: t1 + t_0 / 3
  const R t0 = R(1.0 / 9.0) * ((t1[0] + t1[1]) + (t1[2] + t1[3]));
#pragma unroll
  for (int i = 0; i < 4; ++i) t1[i] = R(0.5) * (t1[i] + t0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    t2[i] = t2[i] + R(2) * t1[i];
#pragma unroll
    for (int j = i + 1; j < 4; ++j) t2[quad(i, j)] = t2[quad(i, j)] + (t1[i] + t1[j]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u[i][k] = R(6) * (v[i] + R(3) * t2[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j != i) {
        const int m = cubic(i, i, j);
        u[m][k] = R(2) * (v[m] + (R(2) * t2[quad(i, j)] + t2[i]));
      }
  }
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const int i = l == 0 ? 1 : 0, j = l <= 1 ? 2 : 1, n = l == 3 ? 2 : 3;
    u[16 + l][k] = v[16 + l] + (t2[quad(i, j)] + (t2[quad(i, n)] + t2[quad(j, n)]));
  }
}

// K x, h the curl-curl coefficients H / det; sink(i, (K x)_i)
template <int P, typename R, typename Sink>
PG_HD void curl_product(const R* x, const R (&h)[6], Sink sink) {
  // degree 0: Whitney functions of the edges, curl 2 grad_a x grad_b
  R k0[3] = {R(-0.0), R(-0.0), R(-0.0)};
#pragma unroll
  for (int e = 0; e < 6; ++e)
#pragma unroll
    for (int k = 0; k < 3; ++k) acc(k0[k], gradx(ev(e, 0), ev(e, 1), k), x[P * e]);
  if constexpr (P == 1) {
    sym3(h, k0);
#pragma unroll
    for (int k = 0; k < 3; ++k) k0[k] = R(2.0 / 3.0) * k0[k];  // 2 * 2 / 3!
  } else {
    // curl = sum_i lambda_i c[i]; a constant is the same value at every i
    R c[4][3];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) c[i][k] = R(2) * k0[k];
    // edge functions (lambda_b - lambda_a) w: curl 3 (lambda_b - lambda_a) grad_a x grad_b
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const R s = R(3) * x[P * e + 1];
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
        const R s = x[6 * P + f * P * (P - 1) + m];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(c[vc][k], 2 * gradx(va, vb, k), s);
          acc(c[va][k], gradx(vc, vb, k), s);
          acc(c[vb][k], -gradx(vc, va, k), s);
        }
      }
    if constexpr (P == 2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sym3(h, c[i]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        mass1(c[0][k], c[1][k], c[2][k], c[3][k]);
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i][k] = R(1.0 / 120.0) * c[i][k];
      }
    } else {
      R q[10][3];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i; j < 4; ++j)
#pragma unroll
          for (int k = 0; k < 3; ++k) q[quad(i, j)][k] = i == j ? c[i][k] : c[i][k] + c[j][k];
#pragma unroll
      for (int n = 0; n < kCubicFns; ++n)
#pragma unroll
        for (int m = 0; m < 10; ++m)
#pragma unroll
          for (int k = 0; k < 3; ++k) acc(q[m][k], kCubic.curl[n][m][k], x[kCubic.dof[n]]);
      R hs[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) hs[k] = R(1.0 / 5040.0) * h[k];
#pragma unroll
      for (int m = 0; m < 10; ++m) sym3(hs, q[m]);
#pragma unroll
      for (int k = 0; k < 3; ++k) mass2(q, k);
#pragma unroll
      for (int n = 0; n < kCubicFns; ++n) {
        R s = R(-0.0);
#pragma unroll
        for (int m = 0; m < 10; ++m)
#pragma unroll
          for (int k = 0; k < 3; ++k) acc(s, kCubic.curl[n][m][k], q[m][k]);
        sink(kCubic.dof[n], s);
      }
      // moments of lambda_i = lambda_i sum_j lambda_j
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          R s = R(-0.0);
#pragma unroll
          for (int j = 0; j < 4; ++j) s = s + q[quad(i, j)][k];
          c[i][k] = s;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) k0[k] = R(2) * ((c[0][k] + c[1][k]) + (c[2][k] + c[3][k]));
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      R d = R(-0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(d, gradx(ev(e, 0), ev(e, 1), k), c[ev(e, 1)][k]);
        acc(d, -gradx(ev(e, 0), ev(e, 1), k), c[ev(e, 0)][k]);
      }
      sink(P * e + 1, R(3) * d);
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
        sink(6 * P + f * P * (P - 1) + m, s);
      }
  }
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    R s = R(-0.0);
#pragma unroll
    for (int k = 0; k < 3; ++k) acc(s, gradx(ev(e, 0), ev(e, 1), k), k0[k]);
    sink(P * e, s);
  }
}

// M x, g the mass coefficients (det G, times any factor); sink(i, (M x)_i)
template <int P, typename R, typename Sink>
PG_HD void mass_product(const R* x, const R (&g)[6], Sink sink) {
  // degree 1: u = sum_i lambda_i a[i], the Whitney functions
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
      mass1(a[0][k], a[1][k], a[2][k], a[3][k]);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i][k] = R(1.0 / 120.0) * a[i][k];
    }
  } else {
    // degree 2: u = sum_{i <= j} lambda_i lambda_j q[ij]
    R q[10][3];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) q[quad(i, j)][k] = i == j ? a[i][k] : a[i][k] + a[j][k];
    // (lambda_b - lambda_a)(lambda_a grad_b - lambda_b grad_a)
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const int va = ev(e, 0), vb = ev(e, 1);
      const R s = x[P * e + 1];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(q[quad(va, vb)][k], grad(va, k) + grad(vb, k), s);
        acc(q[va][k], -grad(vb, k), s);
        acc(q[vb][k], -grad(va, k), s);
      }
    }
    // lambda_c (lambda_a grad_b - lambda_b grad_a)
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        const R s = x[6 * P + f * P * (P - 1) + m];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(q[quad(vc, va)][k], grad(vb, k), s);
          acc(q[quad(vc, vb)][k], -grad(va, k), s);
        }
      }
    R gs[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) gs[k] = R(P == 2 ? 1.0 / 5040.0 : 1.0 / 362880.0) * g[k];
    if constexpr (P == 2) {
#pragma unroll
      for (int m = 0; m < 10; ++m) sym3(gs, q[m]);
#pragma unroll
      for (int k = 0; k < 3; ++k) mass2(q, k);
    } else {
      // degree 3
      R u[20][3];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          u[i][k] = q[i][k];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (j != i) u[cubic(i, i, j)][k] = q[i][k] + q[quad(i, j)][k];
        }
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        const int i = l == 0 ? 1 : 0, j = l <= 1 ? 2 : 1, n = l == 3 ? 2 : 3;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          u[16 + l][k] = q[quad(i, j)][k] + (q[quad(i, n)][k] + q[quad(j, n)][k]);
      }
#pragma unroll
      for (int n = 0; n < kCubicFns; ++n)
#pragma unroll
        for (int m = 0; m < 20; ++m)
#pragma unroll
          for (int k = 0; k < 3; ++k) acc(u[m][k], kCubic.field[n][m][k], x[kCubic.dof[n]]);
#pragma unroll
      for (int m = 0; m < 20; ++m) sym3(gs, u[m]);
#pragma unroll
      for (int k = 0; k < 3; ++k) mass3(u, k);
#pragma unroll
      for (int n = 0; n < kCubicFns; ++n) {
        R s = R(-0.0);
#pragma unroll
        for (int m = 0; m < 20; ++m)
#pragma unroll
          for (int k = 0; k < 3; ++k) acc(s, kCubic.field[n][m][k], u[m][k]);
        sink(kCubic.dof[n], s);
      }
      // moments of lambda_i lambda_j = lambda_i lambda_j sum_l lambda_l
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i; j < 4; ++j)
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            R s = R(-0.0);
#pragma unroll
            for (int l = 0; l < 4; ++l) s = s + u[cubic(i, j, l)][k];
            q[quad(i, j)][k] = s;
          }
    }
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int va = fv(f, m), vb = fv(f, (m + 1) % 3), vc = fv(f, (m + 2) % 3);
        R s = R(-0.0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          acc(s, grad(vb, k), q[quad(vc, va)][k]);
          acc(s, -grad(va, k), q[quad(vc, vb)][k]);
        }
        sink(6 * P + f * P * (P - 1) + m, s);
      }
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const int va = ev(e, 0), vb = ev(e, 1);
      R s = R(-0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc(s, grad(va, k) + grad(vb, k), q[quad(va, vb)][k]);
        acc(s, -grad(vb, k), q[va][k]);
        acc(s, -grad(va, k), q[vb][k]);
      }
      sink(P * e + 1, s);
    }
    // moments of lambda_i = lambda_i sum_j lambda_j
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        R s = R(-0.0);
#pragma unroll
        for (int j = 0; j < 4; ++j) s = s + q[quad(i, j)][k];
        a[i][k] = s;
      }
  }
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    R s = R(-0.0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      acc(s, grad(ev(e, 1), k), a[ev(e, 0)][k]);
      acc(s, -grad(ev(e, 0), k), a[ev(e, 1)][k]);
    }
    sink(P * e, s);
  }
}

}  // namespace fac
}  // namespace pg
