// Element matrices and numeric assembly, a row of an element matrix per thread.
//
// Row i of K_e and M_e is the product with the i-th unit vector, formed without
// tables (pg_factor.h).  The element matrices and the assembled values have to agree
// bit for bit (every CSR slot is the sum of its element entries in ascending element
// order), so multiplications and additions are contracted within an expression of the
// source only: the same expressions round alike in every kernel.
#pragma clang fp contract(on)

#include <hip/hip_runtime.h>

#include <algorithm>

#include "pg_common.h"
#include "pg_factor.h"
#include "pg_rows.h"

namespace pg {
namespace {

constexpr int kRows = kWave;  // element rows of one wave

template <int P>
constexpr int n_vol() {
  return P * (P - 1) * (P - 2) / 2;
}
template <int P>
__device__ inline int first_dof(int la) {
  return la < 6 ? la * P : (la < 10 ? 6 * P + (la - 6) * P * (P - 1) : 6 * P + 4 * P * (P - 1));
}
template <int P, typename R>
__device__ inline void fill_faces(R* faces) {
  if constexpr (P > 1) {
    constexpr auto t = fac::kFaces<P>;
    for (int i = threadIdx.x; i < fac::face_table_size<P>(); i += blockDim.x) faces[i] = (R)t.v[i];
  }
}

// nothing that needs the orientation moves up across this: its face combinations, 4
// to 72 doubles from LDS, are not held beside the product's own values
__device__ inline void settle(int& code) {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" : "+v"(code));
}
// row i of M_e and of K_e
template <int P>
__device__ inline void unit_vector(int i, int code, const double* faces, double* x) {
#pragma unroll
  for (int j = 0; j < fac::n_dofs<P>(); ++j) x[j] = j == i ? 1.0 : 0.0;
  fac::orient_in<P>(code, faces, x);
  __builtin_amdgcn_sched_barrier(0);
}
template <int P>
__device__ inline void mass_row(int i, int code, const double* faces,
                                const double (&g)[6], double* m) {
  double x[fac::n_dofs<P>()];
  unit_vector<P>(i, code, faces, x);
  fac::mass_product<P, double>(x, g, [&](int j, double v) { m[j] = v; });
  settle(code);
  fac::orient_out<P>(code, faces, m);
}
template <int P>
__device__ inline void curl_row(int i, int code, const double* faces,
                                const double (&h)[6], double* k) {
  double x[fac::n_dofs<P>()];
  unit_vector<P>(i, code, faces, x);
  fac::curl_product<P, double>(x, h, [&](int j, double v) { k[j] = v; });
  settle(code);
  fac::orient_out<P>(code, faces, k);
}

// ---------------------------------------------------------------------------
// Element matrices: a wave takes 64 consecutive rows, which it stores through LDS in
// contiguous runs.  Bound: the stores (16 n^2 bytes per element).  41 154 elements,
// p = 2: 52 us, what the bytes alone take; a thread per entry, contracting 12 table
// values gathered from L2 for each, took 160 us.
// ---------------------------------------------------------------------------
template <int P>
__global__ void __launch_bounds__(kWave, (P == 3 ? 1 : 3)) k_element_matrices(
    int64_t E, const double* __restrict__ coef, const int32_t* __restrict__ orient,
    double* __restrict__ M, double* __restrict__ K) {
  constexpr int N = fac::n_dofs<P>();
  constexpr int LD = N | 1;  // odd: a column of rows spreads over the banks
  __shared__ double buf[kRows * LD];
  __shared__ double faces[fac::face_table_size<P>()];
  fill_faces<P>(faces);
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * kRows, rows = E * N, r = r0 + threadIdx.x;
  double mrow[N];
  if (r < rows) {
    const int64_t e = r / N;
    const int i = (int)(r - e * N);
    const int code = orient[e];
    double g[6], h[6], krow[N];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      g[c] = coef[12 * e + c];
      h[c] = coef[12 * e + 6 + c];
    }
    mass_row<P>(i, code, faces, g, mrow);
    __builtin_amdgcn_sched_barrier(0);
    curl_row<P>(i, code, faces, h, krow);
#pragma unroll
    for (int j = 0; j < N; ++j) buf[threadIdx.x * LD + j] = krow[j];
  }
  const int n = (int)(rows - r0 < kRows ? rows - r0 : kRows) * N;
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += kWave) K[r0 * N + q] = buf[q / N * LD + q % N];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (r < rows) buf[threadIdx.x * LD + j] = mrow[j];
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += kWave) M[r0 * N + q] = buf[q / N * LD + q % N];
}

// ---------------------------------------------------------------------------
// Assembly.  A wave takes a few batches of consecutive entities of one class (edges,
// faces, volumes).  A batch is the entities whose d rows of the matrices of the
// elements around them are 64 rows at most.  The rows of K_e are formed into LDS, a
// row per thread; a thread per pair (A, B) (p <= 2) or per column (p = 3) adds the
// contributors in ascending element order; the rows of M_e follow through the same LDS.
// Pairs are consecutive in the CSR rows, so the stores of a wave are contiguous.  A
// batch's contributors are read in one go: an element contributes to one pair per
// local entity, so they are counted by the elements, and the diagonal ones, in order,
// are the batch's (entity, element) items.  An entity with more than 64 rows is taken
// in pieces, its slots read back in between.
// One wave per workgroup: no barriers, and nine workgroups fit into a CU's LDS at
// p = 2.  What bounds it is latency at two waves per SIMD: the matrix cores have no
// work here (a row is some 800 FP64 operations on 12 coefficients), and bytes (1 GB at
// 162 000 elements, p = 2: 200 us), VALU (160 us) and LDS (110 us) add up to 417 us
// because too few waves overlap them.  What took most of the time at first was the
// wait of a batch's first loads for the stores of the batch before (loads and stores
// return in order): contributors, pairs, orientations and coefficients are now asked
// for a batch ahead and are there before the stores (546 -> 468 us, then 436 -> 428),
// which bypass the caches' reuse (467 -> 436).  At p <= 2 the sums of K_e stay in
// registers until those of M_e are there, so that a slot is written once: written in two
// halves, 1.25 GB went to HBM in place of 0.7.  p = 3 keeps two passes: its columns
// do not fit into registers.
// The whole call, against a wave per entity that gathered 12 table values for every
// entry: 162 000 elements p = 2 724 -> 417 us; 10 368 elements
// p = 3 261 -> 250, 63 888 elements 1533 -> 1206; 162 000 elements p = 1 253 -> 102.
// ---------------------------------------------------------------------------
constexpr int kAsmPairs = 256;  // pairs staged at a time: the batches of usual meshes have fewer
constexpr int kDiagonal = 1 << 24, kEliminated = 2 << 24, kTwo = 4 << 24, kMore = 8 << 24;

template <int P>
constexpr int class_dofs(int cls) {
  return cls == 0 ? P : (cls == 1 ? P * (P - 1) : n_vol<P>());
}
template <int P>
constexpr int n_local() {
  return P == 1 ? 6 : (P == 2 ? 10 : 11);
}
// entities of four batches, on meshes with five elements per edge (at most 63)
template <int P>
constexpr int class_entities(int cls) {
  return cls == 0 ? (P == 1 ? 48 : (P == 2 ? 24 : 16)) : (cls == 1 ? (P == 2 ? 60 : 20) : 60);
}

template <int P>
__host__ __device__ inline int wave_entities(int cls, int share) {
  const int n = class_entities<P>(cls) * share / 16;
  return n > 0 ? n : 1;
}

struct AsmArgs {
  int64_t nE, nF, nV, npairs;
  const int32_t *epair, *rowptr, *slot0, *cbeg, *ab;
  const uint32_t* contrib;
  const double* coef;
  const int32_t* orient;
  double omega_mu;
  const uint8_t* bc;
  double *K, *M;  // of slot z: K[stride * z]
  int stride;
  int share;  // a wave's entities: class_entities() * share / 16, one at least
  int64_t waves;
  int split;  // 2: K_e and M_e by different waves, else 1
};

template <int P>
struct AsmShared {
  static constexpr int LD = fac::n_dofs<P>() | 1;
  static constexpr int kContrib = kRows * n_local<P>() / P;
  double rows[kRows * LD];
  double faces[fac::face_table_size<P>()];
  uint16_t u[kContrib];  // places in `rows` of the contributors' rows
  // a pair's first slot; place of its first two contributors' rows | kind << 24; length
  // of its rows; its first contributor
  int4 pairs[kAsmPairs + 1];
  int32_t len[kWave], dslot[kWave];  // of an entity: its rows' length, its diagonal slot
  int32_t row0[kWave];               // its first slot less the columns before it
  // of an item (this batch's, the next one's): its element and local entity there; its
  // entity's items: first | end << 8
  int32_t it_e[2][kRows];
  uint8_t it_l[2][kRows];
  uint16_t it_f[kRows];
  uint16_t col[P > 2 ? kAsmPairs * P * (P - 1) : 1];  // of a column: its pair, DOF of it
  uint16_t ent[kWave];  // an entity's items: first | end << 8
  uint8_t dbc[kWave];
  int32_t ncol;
};

__device__ inline int lane_value(int x, int lane) { return __builtin_amdgcn_readlane(x, lane); }

template <int P, int CLS>
__device__ inline void assemble_class(const AsmArgs& a, int64_t block, AsmShared<P>& s) {
  constexpr int N = fac::n_dofs<P>(), LD = AsmShared<P>::LD, L = n_local<P>();
  constexpr int D = class_dofs<P>(CLS);
  constexpr int DE = P, DF = P * (P - 1), DV = n_vol<P>(), MAXD = P == 1 ? 1 : DF;
  constexpr int CL = P <= 2 ? MAXD : 1;  // columns summed by one thread
  constexpr int kPer = kRows / D;     // elements of a batch
  constexpr int CT = (kPer * L + kWave - 1) / kWave, PT = kAsmPairs / kWave;  // per thread
  const int t = threadIdx.x;
  const int ME = wave_entities<P>(CLS, a.share);
  const int pass0 = a.split == 2 ? (int)((blockIdx.x >> 3) & 1) : 0, pass1 = a.split == 2 ? pass0 + 1 : 2;
  const int64_t base = CLS == 0 ? 0 : (CLS == 1 ? a.nE : a.nE + a.nF);
  const int64_t cnt = CLS == 0 ? a.nE : (CLS == 1 ? a.nF : a.nV);
  const int64_t A0 = block * ME;  // within the class
  const int nA = (int)(cnt - A0 < ME ? cnt - A0 : ME);
  // thread i: first pair and contributor of entity i (of the end, thread nA)
  int pair = 0, cs = 0, row_first = 0, len = 0;
  if (t <= nA) {
    int64_t lo = 0, hi = a.npairs;
    if (a.epair) {
      lo = a.epair[base + A0 + t];
    } else {  // a plan without its entities' first pairs: pairs ascend in A
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (a.ab[2 * mid] < base + A0 + t) lo = mid + 1;
        else hi = mid;
      }
    }
    pair = (int32_t)lo;
    cs = a.cbeg[lo];
    if (t < nA) {
      const int64_t r0 = (CLS == 0 ? 0 : (CLS == 1 ? a.nE * DE : a.nE * DE + a.nF * DF)) + (A0 + t) * D;
      row_first = a.rowptr[r0];
      s.len[t] = len = a.rowptr[r0 + 1] - row_first;
    }
  }
  if constexpr (P > 2) {  // columns are counted through the wave's entities
    int before = len;
    for (int d = 1; d < kWave; d <<= 1) {
      const int x = __shfl_up(before, d);
      if (t >= d) before += x;
    }
    s.row0[t] = row_first - (before - len);
  }
  fill_faces<P>(s.faces);
  const int cs_next = __shfl(cs, t + 1);
  auto diagonal = [](uint32_t v) { return ((v >> 4) & 15) == (v & 15); };
  // a batch: entities [i0, i1), one in pieces if i1 == i0, and its first contributors
  // and pairs.  They are asked for a batch ahead and there before the stores of the
  // current one: a wait for a load is a wait for all stores before it.
  uint32_t u[CT];
  int2 ab[PT];
  int sl[PT], cb[PT], ce[PT];
  auto batch_end = [&](int i) {
    return i + (int)__popcll(__ballot(t >= i && t < nA && cs_next - lane_value(cs, i) <= kPer * L));
  };
  auto load_batch = [&](int i0, int i1) {
    const int c0 = lane_value(cs, i0), c1 = lane_value(cs, i1);
    const int p0 = lane_value(pair, i0), p1 = lane_value(pair, i1 > i0 ? i1 : i0 + 1);
#pragma unroll
    for (int j = 0; j < CT; ++j)
      if (c0 + t + j * kWave < c1) u[j] = a.contrib[c0 + t + j * kWave];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int p = p0 + t + j * kWave;
      if (p < p1) {
        ab[j] = reinterpret_cast<const int2*>(a.ab)[p];
        sl[j] = a.slot0[p];
        cb[j] = a.cbeg[p];
        ce[j] = a.cbeg[p + 1];
      }
    }
  };
  auto arrived = [&] {
#pragma unroll
    for (int j = 0; j < CT; ++j) asm volatile("" : "+v"(u[j]));
#pragma unroll
    for (int j = 0; j < PT; ++j)
      asm volatile("" : "+v"(ab[j].x), "+v"(ab[j].y), "+v"(sl[j]), "+v"(cb[j]), "+v"(ce[j]));
  };
  // a row per thread: its function, its element's orientation and coefficients
  struct Row {
    int r = 0, code = 0;
    double h[6];
    const double* e;
  } rw;
  rw.e = a.coef;
  uint8_t ba[PT], bb[PT];
  auto load_row = [&](int nit, int buf) {
    if (t < nit * D) {
      const int e = s.it_e[buf][t / D];
      rw.r = first_dof<P>(s.it_l[buf][t / D]) + t % D;
      rw.code = a.orient[e];
      rw.e = a.coef + 12 * (int64_t)e;
#pragma unroll
      for (int c = 0; c < 6; ++c) rw.h[c] = rw.e[6 + c];
    }
  };
  auto load_bc = [&](int p0, int p1) {
    if (a.bc)
#pragma unroll
      for (int j = 0; j < PT; ++j)
        if (p0 + t + j * kWave < p1) {
          ba[j] = a.bc[ab[j].x];
          bb[j] = a.bc[ab[j].y];
        }
  };
  int steps = 0;  // of a bisection in an entity's items
  auto prepare = [&](int i0, int i1, int buf) {
    const int c0 = lane_value(cs, i0), c1 = lane_value(cs, i1);
    const int f0 = (cs - c0) / L, f1 = (cs_next - c0) / L;
    const bool mine = t >= i0 && t < i1;
    if (mine) {
      s.ent[t] = (uint16_t)(f0 | f1 << 8);
      for (int f = f0; f < f1; ++f) s.it_f[f] = (uint16_t)(f0 | f1 << 8);
    }
    steps = 0;
    while (__ballot(mine && f1 - f0 > 1 << steps)) ++steps;
    int before = 0;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const bool d = c0 + t + j * kWave < c1 && diagonal(u[j]);
      const uint64_t m = __ballot(d);
      if (d) {
        const int it = before + (int)__popcll(m & ((1ull << t) - 1));
        s.it_e[buf][it] = (int)(u[j] >> 8);
        s.it_l[buf][it] = (uint8_t)(u[j] & 15);
      }
      before += (int)__popcll(m);
    }
    __syncthreads();
    load_row((c1 - c0) / L, buf);
    load_bc(lane_value(pair, i0), lane_value(pair, i1));
  };
  auto prepared = [&] {
    asm volatile("" : "+v"(rw.code));
#pragma unroll
    for (int c = 0; c < 6; ++c) asm volatile("" : "+v"(rw.h[c]));
    if (a.bc)
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        int x = ba[j] | bb[j];
        asm volatile("" : "+v"(x));
        ba[j] = bb[j] = (uint8_t)x;
      }
  };
  int i1 = batch_end(0), next = 0, buf = 0;
  load_batch(0, i1);
  if (i1 > 0) prepare(0, i1, 0);
  for (int i0 = 0; i0 < nA; i0 = i1, i1 = next, buf ^= 1) {
    const bool pieces = i1 == i0;
    if (pieces) i1 = i0 + 1;
    else if (a.split == 2 && i0 > 0) prepare(i0, i1, buf);
    const int c0 = lane_value(cs, i0), p0 = lane_value(pair, i0);
    const int c1 = lane_value(cs, i1), p1 = lane_value(pair, i1);
    const int total = (c1 - c0) / L;
    next = i1 < nA ? batch_end(i1) : i1;
    int diag0 = 0;
    if (pieces) {
      for (int p = p0 + t; p < p1; p += kWave)
        if (a.ab[2 * (int64_t)p] == a.ab[2 * (int64_t)p + 1]) s.it_e[buf][0] = a.cbeg[p];
      __syncthreads();
      diag0 = s.it_e[buf][0];
      __syncthreads();
    }
    int col0 = P > 2 ? lane_value(row_first, i0) - s.row0[i0] : 0;  // first staged column
    auto stage = [&](int q, int last, int A, int B, int z, int c, int end, bool elim) {
      const int i = (int)(A - base - A0), n = end - c;
      int y = (A == B ? kDiagonal : 0) | (elim ? kEliminated : 0) | (n > 1 ? kTwo : 0) |
              (n > 2 ? kMore : 0);
      if (!pieces) y |= s.u[c - c0] | (n > 1 ? s.u[c - c0 + 1] << 12 : 0);
      s.pairs[q] = make_int4(z, y, s.len[i], c);
      s.pairs[q + 1].w = end;  // (or the next one's, the same)
      if constexpr (P > 2) {
        const int col = z - s.row0[i] - col0, d = B < a.nE ? DE : (B < a.nE + a.nF ? DF : DV);
        for (int l = 0; l < d; ++l) s.col[col + l] = (uint16_t)(q << 3 | l);
        if (q == last) s.ncol = col + d;
      }
      if (A == B) {
        s.dslot[i] = z;
        s.dbc[i] = elim;
      }
    };
    int nit = total;
    auto load_piece = [&](int e0) {
      nit = total - e0 < kPer ? total - e0 : kPer;
      if (t < nit) {
        const uint32_t v = a.contrib[diag0 + e0 + t];
        s.it_e[buf][t] = (int)(v >> 8);
        s.it_l[buf][t] = (uint8_t)(v & 15);
      }
      if (t == 0) s.ent[i0] = (uint16_t)(nit << 8);
      __syncthreads();
      load_row(nit, buf);
    };
    if (pieces) {
      load_piece(0);
      load_bc(p0, p1);
    }
    int code = rw.code, r = rw.r;
    double cf[6], cg[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      cf[c] = rw.h[c];
      cg[c] = rw.e[c];
    }
    if (!pieces) {
      int at[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j)
        at[j] = c0 + t + j * kWave < c1 ? s.it_f[(t + j * kWave) / L] : 0;
      for (int b = steps - 1; b >= 0; --b)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const int mid = (at[j] & 255) + (1 << b);
          if (mid < at[j] >> 8 && s.it_e[buf][mid] <= (int)(u[j] >> 8)) at[j] += 1 << b;
        }
#pragma unroll
      for (int j = 0; j < CT; ++j)
        if (c0 + t + j * kWave < c1)
          s.u[t + j * kWave] = (uint16_t)((at[j] & 255) * D * LD + first_dof<P>((int)(u[j] & 15)));
      __syncthreads();
    }
    const int last = (p1 - p0 < kAsmPairs ? p1 - p0 : kAsmPairs) - 1;
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (p0 + t + j * kWave < p1)
        stage(t + j * kWave, last, ab[j].x, ab[j].y, sl[j], cb[j], ce[j], a.bc && (ba[j] | bb[j]));
    for (int e0 = 0;;) {
      const bool row = t < nit * D;
      double* out = a.K;
      const bool sums = P <= 2 && a.split == 1 && !pieces && p1 - p0 <= kAsmPairs;
      constexpr int SR = P <= 2 ? kAsmPairs / kWave : 1;
      double ks[SR][D][CL];
#pragma unroll
      for (int pass = 0; pass < 2; ++pass, out = a.M) {
        if (pass < pass0 || pass >= pass1) continue;
        const bool ahead = e0 + kPer >= total && i1 < nA;
        if (ahead && pass == pass0) load_batch(i1, next);
        if (ahead && pass == 1 && pass0 == 0 && next > i1) prepare(i1, next, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        if (row) {
          double x[N];
          asm volatile("" : "+v"(r));  // (else the unit vector stays in registers)
          settle(code);
          if (pass == 0) {
            curl_row<P>(r, code, s.faces, cf, x);
          } else {
            mass_row<P>(r, code, s.faces, cg, x);
            // the product with omega mu0 is rounded by itself, as the reference forms
            // i*w*mu0*M_e before adding
            if (a.stride == 2)
#pragma unroll
              for (int j = 0; j < N; ++j) x[j] = -(a.omega_mu * x[j]);
          }
#pragma unroll
          for (int j = 0; j < N; ++j) s.rows[t * LD + j] = x[j];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ahead && pass == pass0) arrived();
        if (ahead && pass == 1 && pass0 == 0) prepared();
        __syncthreads();
        const double one = pass == 0 ? 1.0 : 0.0;  // of an eliminated diagonal
        if (sums) {
          // all columns of the batch, their sums of K_e kept until those of M_e are there
#pragma unroll
          for (int j = 0; j < (P <= 2 ? SR : 0); ++j) {
            const int w = t + j * kWave;
            if (w < p1 - p0) {
              const int4 pr = s.pairs[w];
              double v[D][CL] = {};
              auto add = [&](int at) {
#pragma unroll
                for (int k = 0; k < D; ++k)
#pragma unroll
                  for (int l = 0; l < CL; ++l) v[k][l] += s.rows[at + k * LD + l];
              };
              add(pr.y & 4095);
              if (pr.y & kTwo) add((pr.y >> 12) & 4095);
              if ((pr.y & kMore) && !(pr.y & kDiagonal))
                for (int c = pr.w + 2; c < s.pairs[w + 1].w; ++c) add(s.u[c - c0]);
              if (pass == 0) {
#pragma unroll
                for (int k = 0; k < D; ++k)
#pragma unroll
                  for (int l = 0; l < CL; ++l) ks[j][k][l] = v[k][l];
              } else if (!(pr.y & kDiagonal)) {
#pragma unroll
                for (int k = 0; k < D; ++k)
#pragma unroll
                  for (int l = 0; l < CL; ++l) {
                    const int64_t z = pr.x + l + (int64_t)k * pr.z;
                    const double2 y = pr.y & kEliminated ? make_double2(0.0, 0.0)
                                                         : make_double2(ks[j][k][l], v[k][l]);
                    if (a.stride == 2) {
                      typedef double dv2 __attribute__((ext_vector_type(2)));
                      dv2 yy = {y.x, y.y};
                      __builtin_nontemporal_store(yy, reinterpret_cast<dv2*>(a.K) + z);
                    } else {
                      a.K[z] = y.x;
                      a.M[z] = y.y;
                    }
                  }
              }
            }
          }
        }
        for (int pc = sums ? p1 : p0; pc < p1; pc += kAsmPairs) {
          const int np = p1 - pc < kAsmPairs ? p1 - pc : kAsmPairs;
          if (p1 - p0 > kAsmPairs && (pc > p0 || e0 > 0 || pass > pass0)) {  // else they are there
            if constexpr (P > 2) col0 = a.slot0[pc] - s.row0[a.ab[2 * (int64_t)pc] - base - A0];
            for (int q = t; q < np; q += kWave) {
              const int A = a.ab[2 * (int64_t)(pc + q)], B = a.ab[2 * (int64_t)(pc + q) + 1];
              stage(q, np - 1, A, B, a.slot0[pc + q], a.cbeg[pc + q], a.cbeg[pc + q + 1],
                    a.bc && (a.bc[A] | a.bc[B]));
            }
            __syncthreads();
          }
          const int ncol = P <= 2 ? np : s.ncol;  // (column groups)
          for (int w = t; w < ncol; w += kWave) {
            const int x = P <= 2 ? 0 : s.col[w];
            const int q = P <= 2 ? w : x >> 3, l0 = P <= 2 ? 0 : x & 7;
            const int4 pr = s.pairs[q];
            if (pr.y & kDiagonal) continue;  // the diagonal blocks come below
            const int64_t z0 = pr.x + l0, len = pr.z;
            double v[D][CL] = {};
            auto add = [&](int at) {
#pragma unroll
              for (int k = 0; k < D; ++k)
#pragma unroll
                for (int l = 0; l < CL; ++l) v[k][l] += s.rows[at + k * LD + l0 + l];
            };
            if (pieces) {
              if (e0 > 0)
#pragma unroll
                for (int k = 0; k < D; ++k)
#pragma unroll
                  for (int l = 0; l < CL; ++l) v[k][l] = out[a.stride * (z0 + k * len + l)];
              for (int c = pr.w; c < s.pairs[q + 1].w; ++c) {
                const uint32_t y = a.contrib[c];
                int lo = 0, hi = nit - 1;
                while (lo < hi) {
                  const int mid = (lo + hi) >> 1;
                  if (s.it_e[buf][mid] < (int)(y >> 8)) lo = mid + 1;
                  else hi = mid;
                }
                if (s.it_e[buf][lo] == (int)(y >> 8)) add(lo * D * LD + first_dof<P>((int)(y & 15)));
              }
            } else {
              // one or two elements on a conforming mesh
              add(pr.y & 4095);
              if (pr.y & kTwo) add((pr.y >> 12) & 4095);
              if (pr.y & kMore)
                for (int c = pr.w + 2; c < s.pairs[q + 1].w; ++c) add(s.u[c - c0]);
            }
#pragma unroll
            for (int k = 0; k < D; ++k)
#pragma unroll
              for (int l = 0; l < CL; ++l)
                out[a.stride * (z0 + k * len + l)] = pr.y & kEliminated ? 0.0 : v[k][l];
          }
          __syncthreads();
        }
        // diagonal blocks: all elements of an entity
        for (int w = t; w < (i1 - i0) * D * D; w += kWave) {
          const int i = i0 + w / (D * D), k = w / D % D, l = w % D;
          const int range = s.ent[i];
          double* z = out + a.stride * (s.dslot[i] + (int64_t)k * s.len[i] + l);
          double v = e0 > 0 ? *z : 0.0;
          for (int f = range & 255; f < range >> 8; ++f)
            v += s.rows[(f * D + k) * LD + first_dof<P>(s.it_l[buf][f]) + l];
          *z = s.dbc[i] ? (k == l ? one : 0.0) : v;
        }
        __syncthreads();
      }
      e0 += kPer;
      if (e0 >= total) break;
      load_piece(e0);
      code = rw.code;
      r = rw.r;
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        cf[c] = rw.h[c];
        cg[c] = rw.e[c];
      }
    }
  }
}

template <int P>
__host__ __device__ inline int64_t asm_blocks(int cls, int64_t count, int share) {
  const int me = wave_entities<P>(cls, share);
  return class_dofs<P>(cls) ? (count + me - 1) / me : 0;
}

template <int P>
__global__ void __launch_bounds__(kWave, (P == 3 ? 1 : 2)) k_asm_rows(const AsmArgs a) {
  __shared__ AsmShared<P> s;
  // (the two waves of the same entities on the same XCD: their halves of a slot meet in
  // its L2)
  int64_t b = a.split == 2 ? (blockIdx.x >> 4) * 8 + (blockIdx.x & 7) : blockIdx.x;
  if (b >= a.waves) return;
  const int64_t nbE = asm_blocks<P>(0, a.nE, a.share),
                nbF = asm_blocks<P>(1, a.nF, a.share);
  if (b < nbE) {
    assemble_class<P, 0>(a, b, s);
    return;
  }
  b -= nbE;
  if constexpr (P > 1) {
    if (b < nbF) {
      assemble_class<P, 1>(a, b, s);
      return;
    }
    b -= nbF;
  }
  if constexpr (P > 2) assemble_class<P, 2>(a, b, s);
}

template <int P>
void launch_asm(AsmArgs& a, hipStream_t st) {
  auto blocks = [&](int share) {
    return asm_blocks<P>(0, a.nE, share) + asm_blocks<P>(1, a.nF, share) +
           asm_blocks<P>(2, a.nV, share);
  };
  // several batches a wave while they leave every CU several rounds of waves; on an
  // empty chip, where a wave's own time is the call's, less than a batch, and K_e and
  // M_e by different waves (p = 1: 384 elements 9.9 -> 7.9 us, 2058 10.1 -> 7.7; p = 2:
  // 2058 elements 13.7 -> 12.5, 3072, the same either way, 14.9)
  a.share = 16;
  while (a.share > 4 && blocks(a.share) < 10240) a.share /= 2;
  while (a.share > 1 && blocks(a.share) < 512) a.share /= 2;
  a.split = blocks(a.share) < 1024 ? 2 : 1;
  a.waves = blocks(a.share);
  const int64_t nb = a.split == 2 ? (a.waves + 7) / 8 * 16 : a.waves;
  if (nb > 0) hipLaunchKernelGGL(k_asm_rows<P>, dim3((unsigned)nb), dim3(kWave), 0, st, a);
}

}  // namespace

void launch_element_matrices(int p, int64_t E, const double* coef, const int32_t* orient,
                             double* M, double* K, hipStream_t st) {
  const int n = ndof_element(p);
  const dim3 g((unsigned)((E * n + kRows - 1) / kRows)), b(kWave);
  if (p == 1)
    hipLaunchKernelGGL(k_element_matrices<1>, g, b, 0, st, E, coef, orient, M, K);
  else if (p == 2)
    hipLaunchKernelGGL(k_element_matrices<2>, g, b, 0, st, E, coef, orient, M, K);
  else
    hipLaunchKernelGGL(k_element_matrices<3>, g, b, 0, st, E, coef, orient, M, K);
}

void launch_assembly(const pg_plan_dev& pl, const double* coef, const int32_t* orient,
                     double omega_mu, const uint8_t* ent_bc, double2* values, double* Kout,
                     double* Mout, hipStream_t st) {
  double* v = reinterpret_cast<double*>(values);
  AsmArgs a{pl.n_edges,    pl.n_faces,       pl.n_elems,    pl.npairs, pl.entity_pair, pl.rowptr,
            pl.pair_slot0, pl.pair_cbeg,     pl.pair_ab,    pl.contrib, coef,          orient,
            omega_mu,      ent_bc,           Kout ? Kout : v, Kout ? Mout : v + 1, Kout ? 1 : 2,
            16, 0, 1};
  if (pl.p == 1)
    launch_asm<1>(a, st);
  else if (pl.p == 2)
    launch_asm<2>(a, st);
  else
    launch_asm<3>(a, st);
}

}  // namespace pg
