"""Generate ``csrc/pg_eop_mask.h``: the structural zeros of the element tables.

For order p, an element entry of the pair (i, j >= i) of local DOFs is a sum of
the 12 table components T_c[v_i][v_j] (6 mass, 6 curl-curl) of the two DOFs'
orientation variants.  Some components vanish for every orientation of the
element (the quadrature sums cancel exactly; the computed values are rounding
noise below 1e-16 of the largest entry).  This script evaluates the tables of
the built library (``pg_tables_host``) over all 2^6 * 6^4 orientation
combinations and writes, per pair, a 12-bit mask of the components that are
zero in every one of them: the terms that an entry formed from the tables can
leave out.  (The element products form no entries, csrc/pg_factor.h; the masks
pin the tables' structure in the tests.)

Usage (after ``python -m petgem_amd.build``)::

    python -m petgem_amd.gen_eop_mask        # rewrites petgem_amd/csrc/pg_eop_mask.h
"""
import itertools
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "csrc", "pg_eop_mask.h")
REL_ZERO = 1e-15  # a component counts as zero below this fraction of max|T|


def structural_zeros(p):
    from . import _native as nat
    nvol = p * (p - 1) * (p - 2) // 2
    nv = 12 * p + 24 * p * (p - 1) + nvol
    n = 6 * p + 4 * p * (p - 1) + nvol
    T = np.zeros(nv * nv * 12)
    nat.check(nat.lib().pg_tables_host(p, T.ctypes.data, T.size))
    T = T.reshape(nv, nv, 12)
    tol = REL_ZERO * np.abs(T).max()
    iu, ju = np.triu_indices(n)
    zero = None
    faces = itertools.product(range(6), repeat=4) if p >= 2 else [(0, 0, 0, 0)]
    for fos in faces:
        for eos in itertools.product((0, 1), repeat=6):
            v = [(la * 2 + eos[la]) * p + k for la in range(6) for k in range(p)]
            if p >= 2:
                nf = p * (p - 1)
                v += [12 * p + (f * 6 + fos[f]) * nf + k for f in range(4) for k in range(nf)]
            v += [12 * p + 24 * p * (p - 1) + k for k in range(nvol)]
            v = np.asarray(v)
            z = np.abs(T[v[iu], v[ju]]) <= tol  # (pairs, 12), pairs row-major upper triangle
            zero = z if zero is None else (zero & z)
    return (zero * (1 << np.arange(12))).sum(axis=1).astype(np.int64)


def main():
    lines = ["// Generated by `python -m petgem_amd.gen_eop_mask` from the element tables: per",
             "// pair k = (i, j >= i) of local DOFs (row-major upper triangle), bit c set when",
             "// table component c (0..5 mass, 6..11 curl-curl) vanishes for every orientation.",
             "#pragma once", "", "#include <cstdint>", "", "namespace pg {", "namespace eop {", ""]
    for p in (1, 2, 3):
        m = structural_zeros(p)
        lines.append(f"constexpr uint16_t kZero{p}[{m.size}] = {{")
        for a in range(0, m.size, 12):
            lines.append("    " + ", ".join(f"0x{int(x):03x}" for x in m[a:a + 12]) + ",")
        lines.append("};")
        lines.append("")
    lines += ["template <int P>", "constexpr uint16_t zero_mask(int k) {",
              "  return P == 1 ? kZero1[k] : (P == 2 ? kZero2[k] : kZero3[k]);", "}", "",
              "}  // namespace eop",
              "}  // namespace pg", ""]
    with open(OUT, "w") as f:
        f.write("\n".join(lines))
    print(OUT)


if __name__ == "__main__":
    main()
