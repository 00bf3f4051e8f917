"""Performance cases: the calls a user of petgem_amd makes, over the sizes they make them at.

A case names a mesh (n^3 hexahedra of 6 tetrahedra with displaced nodes), a basis
order p and one call.  ``order`` says how the mesh is numbered: "grid" is the
structured numbering of the synthetic workloads; "free" numbers nodes, elements
and each element's vertices at random, as a mesh generator's files do (on the
test mesh of this repository two consecutive elements lie 0.29 mesh diameters
apart, against 0.37 for two random ones, and its 9 453 elements have 1 510
different edge and face orientations).

``exact`` recomputes each result in 64 bits with torch alone: its own basis,
quadrature, assembly and Krylov solve.
"""
import functools
import math

import numpy as np
import torch

from petgem_amd import _native as nat
from petgem_amd import core
from petgem_amd.mesh import Topology
from petgem_amd.synthetic import kuhn_grid, layered_sigma

MU0 = 4.0 * math.pi * 1e-7
LENGTH = 10000.0


def listed():
    return [
        # the smallest whole forward step a user runs (a p = 1 trial mesh): geometry,
        # assembly, source, preconditioner, COCG, receivers; hundreds of iterations of
        # kernels that take less time than their launches
        dict(name="solve_p1_small", kind="solve", p=1, n=8, order="grid", precision="fp64",
             pc="jacobi", frequency=1.0, receivers=21),
        # the default forward step (p = 2, FP64, entity-block Jacobi) at an ordinary size
        dict(name="solve_p2_fp64", kind="solve", p=2, n=13, order="grid", precision="fp64",
             pc="bjacobi", frequency=1.0, receivers=41),
        # the same in mixed precision on a mesh generator's numbering
        dict(name="solve_p2_mixed_free", kind="solve", p=2, n=16, order="free",
             precision="mixed", pc="bjacobi", frequency=1.0, receivers=101),
        # many sources and frequencies at once: 64 columns
        dict(name="batch_p2_64", kind="batch", p=2, n=7, order="grid", nrhs=64, frequency=0.5),
        # one product with the system at the size of the headline benchmark: what a
        # Krylov iteration spends most of its time on, also for a user's own iteration
        dict(name="apply_p2_c128_large", kind="apply", p=2, n=40, order="grid",
             dtype="complex128", frequency=1.0),
        # a product on a mesh generator's numbering
        dict(name="apply_p2_c128_free", kind="apply", p=2, n=21, order="free",
             dtype="complex128", frequency=1.0),
        # the complex64 product of the mixed-precision rounds at the highest order
        dict(name="apply_p3_c64", kind="apply", p=3, n=15, order="grid", dtype="complex64",
             frequency=1.0),
        # reassembly for a new model or frequency (each step of an inversion)
        dict(name="assemble_p2", kind="assemble", p=2, n=30, order="grid", frequency=0.25),
        dict(name="assemble_p3_free", kind="assemble", p=3, n=12, order="free", frequency=1.0),
        # the element matrices themselves (the reference's computeElementalMatrices)
        dict(name="matrices_p2", kind="matrices", p=2, n=19, order="grid"),
        # the backward direction: gradient of a misfit with respect to every element's
        # conductivity from two forward and adjoint solutions
        dict(name="gradient_p2", kind="gradient", p=2, n=25, order="grid", nrhs=2,
             frequency=1.0),
        # the calls around a solve: locate a receiver line, source vector, fields at the
        # receivers, adjoint source
        dict(name="points_p2", kind="points", p=2, n=17, order="free", receivers=101,
             frequency=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# largest n of a drawn case by kind and order p (no dearer than the listed ones); a
# free p = 3 mesh keeps tables per element orientation, so it stays small
_MOST = {"solve": (16, 13, 6), "batch": (10, 7, 0), "apply": (40, 34, 18),
         "assemble": (40, 30, 14), "matrices": (30, 19, 9), "gradient": (40, 25, 12),
         "points": (24, 20, 12)}


def draw(rng):
    kind = rng.choice(("solve", "batch", "apply", "apply", "assemble", "matrices", "gradient",
                       "points"))
    p = rng.choice((1, 2)) if kind == "batch" else rng.choice((1, 2, 2, 3))
    order = rng.choice(("grid", "free"))
    hi = _MOST[kind][p - 1]
    if p == 3 and order == "free" and kind == "apply":
        hi = 7
    if p == 3 and order == "free" and kind == "solve":
        hi = 5
    c = dict(kind=kind, p=p, n=_log_int(rng, 4, hi), order=order)
    if kind != "matrices":
        c["frequency"] = round(math.exp(rng.uniform(math.log(0.25), math.log(2.0))), 3)
    if kind == "solve":
        c["precision"] = rng.choice(("fp64", "mixed"))
        c["pc"] = rng.choice(("jacobi", "bjacobi"))
        c["receivers"] = rng.randint(5, 101)
    elif kind == "apply":
        c["dtype"] = rng.choice(("complex128", "complex64"))
    elif kind == "batch":
        c["nrhs"] = rng.choice((8, 16, 64))
    elif kind == "gradient":
        c["nrhs"] = rng.randint(1, 9)
    elif kind == "points":
        c["receivers"] = _log_int(rng, 1, 400)
    return c


# --------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=4)
def _topology(n, p, order):
    """Numbered mesh of the case (the program's mesh file, without its coordinates)."""
    pts, tets = kuhn_grid(n, LENGTH)
    if order == "free":
        r = np.random.default_rng(7919 * n + p)
        new = r.permutation(len(pts))
        q = np.empty_like(pts)
        q[new] = pts
        even = np.array([(0, 1, 2, 3), (0, 2, 3, 1), (0, 3, 1, 2), (1, 0, 3, 2), (1, 2, 0, 3),
                         (1, 3, 2, 0), (2, 0, 1, 3), (2, 1, 3, 0), (2, 3, 0, 1), (3, 0, 2, 1),
                         (3, 1, 0, 2), (3, 2, 1, 0)])
        tets = new[tets][r.permutation(len(tets))]
        tets = np.take_along_axis(tets, even[r.integers(0, 12, len(tets))], axis=1)
        pts = q
    return Topology(pts, tets, p)


def _model(case, seed):
    """Displaced node coordinates per element and layered conductivities with 10 % noise."""
    t = _topology(case["n"], case["p"], case["order"])
    r = np.random.default_rng(seed)
    h = LENGTH / case["n"]
    inner = (np.abs(t.points) < 0.5 * LENGTH - 0.5 * h).all(1)
    pts = t.points + np.where(inner[:, None], r.uniform(-0.1 * h, 0.1 * h, t.points.shape), 0.0)
    coords = pts[t.elems_nodes]
    sigma = layered_sigma(coords.mean(1), block=True, noise=0.1, seed=seed)
    return t, coords, sigma, r


def _device_mesh(t, coords):
    return core.DeviceMesh(t.p, coords, t.elems_nodes, t.elems_edges, t.elem_edges_nodes,
                           t.elem_faces_edges, t.dofs, t.n_edges, t.n_faces, t.elems_faces)


@functools.lru_cache(maxsize=4)
def _plan(n, p, order):
    t = _topology(n, p, order)
    return core.Plan(_device_mesh(t, t.coords))


def _vectors(seed, shape, dtype=torch.float64, zero=None):
    """Random vectors; a solution or search direction is zero on the PEC DOFs (``zero``)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    v = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
    if zero is not None:
        v[..., torch.from_numpy(zero).cuda(), :] = 0.0
    return v.to(dtype)


def _source_of(coords, r):
    """A point inside an element near the sea floor, as survey sources lie."""
    cen = coords.mean(1)
    near = np.argsort(np.abs(cen[:, 2] + 950.0) + 0.1 * np.abs(cen[:, :2]).max(1))
    e = int(near[r.integers(0, max(1, min(20, len(near) // 4)))])
    return e, r.dirichlet(np.full(4, 2.0)) @ coords[e]


def _line(count, r):
    x = np.linspace(-4000.0, 4000.0, count) + r.uniform(-20.0, 20.0, count)
    return np.stack([x, r.uniform(-50.0, 50.0, count), -1000.0 + r.uniform(-20.0, 20.0, count)], 1)


RTOL = 1e-12  # tight enough that a solution is the system's and not the stopping point's


def prepare(case, seed):
    t, coords, sigma, r = _model(case, seed)
    kind = case["kind"]
    om = core.omega_of(case.get("frequency", 1.0))
    mesh = _device_mesh(t, coords)
    s = dict(kind=kind, mesh=mesh, omega=om, case=case)
    sig = torch.from_numpy(sigma).cuda()
    s["sigma"] = sig
    if kind == "points":
        el, pos = _source_of(coords, r)
        s.update(rx=_line(case["receivers"], r), source=pos, moment=r.standard_normal(3),
                 x=_vectors(seed, (t.ndof, 2)), coef=_vectors(seed + 1, (case["receivers"], 3, 2)))
        return s
    plan = _plan(case["n"], case["p"], case["order"])
    asm = core.Assembler(mesh, plan=plan)
    s["asm"] = asm
    if kind in ("assemble", "matrices"):
        if kind == "assemble":
            s["ent_bc"], _ = mesh.entity_mask(t.boundary_dofs)
            s["out"] = torch.empty((plan.nnz, 2), dtype=torch.float64, device="cuda")
        else:
            asm.geometry(sig)
        return s
    asm.geometry(sig)
    if kind == "gradient":
        s["x"] = _vectors(seed, (case["nrhs"], t.ndof, 2), zero=t.boundary_dofs)
        s["lam"] = _vectors(seed + 1, (case["nrhs"], t.ndof, 2), zero=t.boundary_dofs)
        s["omegas"] = om * np.linspace(1.0, 2.0, case["nrhs"])
        return s
    s["ent_bc"], s["dof_bc"] = mesh.entity_mask(t.boundary_dofs)
    order = mesh.entity_order()
    if kind == "apply":
        s["eop"] = core.ElementOperator(asm, om, s["ent_bc"], order)
        s["x"] = _vectors(seed, (t.ndof, 2),
                          torch.float64 if case["dtype"] == "complex128" else torch.float32,
                          t.boundary_dofs)
        return s
    if kind == "solve":
        s["values"] = asm.assemble(om, ent_bc=s["ent_bc"])
        s["eop"] = core.ElementOperator(asm, om, s["ent_bc"], order)
        s["solver"] = core.KrylovSolver(plan, s["values"], precision=case["precision"],
                                        pc=case["pc"], rtol=RTOL, block_ptr=mesh.block_ptr(),
                                        entity_order=order, eop=s["eop"])
        el, pos = _source_of(coords, r)
        s.update(source_element=el, source=pos, moment=np.array([1.0, 0.0, 0.0]))
        s["rx"] = _line(case["receivers"], r)
        s["rx_element"] = core.locate_points(mesh, s["rx"])
        return s
    # batch: columns cycle through four frequencies
    K, M = core.assemble_km(asm, s["ent_bc"])
    eop = (core.ElementOperator(asm, om, s["ent_bc"], order) if case["nrhs"] % 64 == 0 else None)
    s["batch"] = core.BatchSolver(plan, K, M, _frequencies(case), rtol=RTOL,
                                  block_ptr=mesh.block_ptr(), entity_order=order, pc="bjacobi",
                                  eop=eop)
    s["B"] = _batch_rhs(t, coords, case, r, s["dof_bc"])
    return s


def _frequencies(case):
    return [case["frequency"] * (1.0 + 0.5 * (c % 4)) for c in range(case["nrhs"])]


def _batch_rhs(t, coords, case, r, dof_bc):
    """Right-hand sides of dipole-like sources: values on one element's DOFs each."""
    B = torch.zeros((t.ndof, case["nrhs"], 2), dtype=torch.float64, device="cuda")
    free = torch.from_numpy(t.dofs).cuda()
    for c in range(case["nrhs"]):
        e, _ = _source_of(coords, r)
        v = torch.from_numpy(r.standard_normal(t.dofs.shape[1])).cuda()
        B[free[e], c, 1] = v
    B[dof_bc.bool()] = 0.0
    return B


# --------------------------------------------------------------------------- the calls
def run(s):
    kind, m = s["kind"], s["mesh"]
    if kind == "apply":
        return {"y": s["eop"].apply(s["x"])}
    if kind == "assemble":
        s["asm"].geometry(s["sigma"])
        return {"values": s["asm"].assemble(s["omega"], ent_bc=s["ent_bc"], out=s["out"])}
    if kind == "matrices":
        M, K = s["asm"].element_matrices()
        return {"M": M, "K": K}
    if kind == "gradient":
        g = torch.zeros(m.n_elems, dtype=torch.float64, device="cuda")
        nat.check(nat.lib().pg_adjoint_gradient(
            s["asm"].tables.handle, m.n_elems, nat.ptr(s["asm"].workspace), nat.ptr(m.dofs),
            len(s["omegas"]), m.ndof, nat.ptr(s["x"]), nat.ptr(s["lam"]), nat.ptr(s["omegas"]),
            nat.ptr(g), nat.stream_handle()))
        return {"gradient": g}
    if kind == "points":
        el = core.locate_points(m, s["rx"])
        src = core.locate_points(m, s["source"])
        b = core.source_vector(m, int(src[0]), s["source"], s["moment"], s["omega"])
        fields = core.receiver_fields(m, s["rx"], el, s["x"], s["omega"])
        f = torch.zeros((m.ndof, 2), dtype=torch.float64, device="cuda")
        pts = torch.from_numpy(s["rx"]).cuda()
        nat.check(nat.lib().pg_adjoint_rhs(
            m.p, len(s["rx"]), nat.ptr(pts), nat.ptr(el), nat.ptr(m.coords),
            nat.ptr(m.elems_nodes), nat.ptr(m.elems_edges), nat.ptr(m.edges_nodes),
            nat.ptr(m.faces_edges), nat.ptr(m.dofs), nat.ptr(s["coef"]), nat.ptr(f),
            nat.stream_handle()))
        return {"elements": el, "b": b, "fields": fields, "f": f}
    if kind == "batch":
        return {"X": s["batch"].solve(s["B"])[0]}
    asm = s["asm"]
    asm.geometry(s["sigma"])
    asm.assemble(s["omega"], ent_bc=s["ent_bc"], out=s["values"])
    b = core.source_vector(m, s["source_element"], s["source"], s["moment"], s["omega"])
    core.apply_dirichlet(asm.plan, None, s["dof_bc"], b)
    s["eop"].refresh(s["omega"])
    s["solver"].refresh()
    x, info = s["solver"].solve(b)
    if info["status"] != 0:
        raise RuntimeError(f"the solve did not converge: {info}")
    return {"x": x, "fields": core.receiver_fields(m, s["rx"], s["rx_element"], x, s["omega"])}


# --------------------------------------------------------------------------- least work
def work(case):
    """Inputs read once, outputs written once.  A solve counts the iterations COCG needs
    (about 18 n, 55 n and 71 n at p = 1, 2, 3 and 1 Hz to 1e-8 on these meshes, half as many
    again to 1e-12), each with one product and one read and write of its four vectors."""
    n, p, kind = case["n"], case["p"], case["kind"]
    E, edges, faces = 6 * n ** 3, 7 * n ** 3 + 9 * n ** 2 + 3 * n, 12 * n ** 3 + 6 * n ** 2
    nd = p * (p + 2) * (p + 3) // 2
    N = edges * p + faces * p * (p - 1) + E * p * (p - 1) * (p - 2) // 2
    ents = 6 if p == 1 else 10 if p == 2 else 11
    nnz = {1: 16.3, 2: 43.1, 3: 83.0}[p] * N  # per row on these meshes
    wide = 8 if case.get("dtype") == "complex64" else 16
    product = dict(bytes=E * (4 * ents + 4 + 12 * wide / 2) + 2 * N * wide,
                   flops=E * (nd * (nd + 1) // 2 * 24 + nd * nd * 8))
    entries = E * nd * (nd + 1) // 2 * 24
    if kind == "apply":
        return product
    if kind == "assemble":
        return dict(bytes=E * 248 + 16 * nnz, flops=entries)
    if kind == "matrices":
        return dict(bytes=E * (100 + 16 * nd * nd), flops=entries)
    if kind == "gradient":
        r = case["nrhs"]
        return dict(bytes=E * (100 + 4 * nd + 16) + 32 * N * r,
                    flops=E * (nd * (nd + 1) // 2 * 12 + r * nd * nd * 4))
    if kind == "points":
        return dict(bytes=E * 96 + 48 * N + case["receivers"] * 200, flops=E * 20)
    its = {1: 18, 2: 55, 3: 71}[p] * n * 1.5 / math.sqrt(case["frequency"])
    r = case.get("nrhs", 1)
    v = 8 if case.get("precision") == "mixed" else 16
    return dict(bytes=E * 248 + 16 * nnz + its * r * 8 * N * v, flops=its * r * product["flops"])


# --------------------------------------------------------------------------- 64-bit results
EDGES = ((0, 1), (1, 2), (0, 2), (0, 3), (1, 3), (2, 3))
FACES = ((0, 1, 2), (0, 1, 3), (1, 2, 3), (0, 2, 3))
FACE_EDGES = ((0, 1, 2), (0, 4, 3), (1, 5, 4), (2, 5, 3))
PERMS = ((0, 1, 2), (1, 2, 0), (2, 0, 1), (0, 2, 1), (1, 0, 2), (2, 1, 0))
CODES = {12: 0, 31: 1, 23: 2, 32: 3, 13: 4, 21: 5}


def _edge_family(a, b, ga, gb, p):
    """Legendre-weighted Whitney functions of an edge, and their curls (points, p, 3)."""
    w = a[:, None] * gb - b[:, None] * ga
    c = np.broadcast_to(np.cross(ga, gb), w.shape)
    s, t = b - a, a + b
    leg = [np.ones_like(a), s, 0.5 * (3.0 * s * s - t * t)]
    return [leg[i][:, None] * w for i in range(p)], [(i + 2.0) * leg[i][:, None] * c
                                                    for i in range(p)]


def _face_family(lam, g, verts, p):
    """Functions of one family on the face (v0, v1, v2): edge functions of (v0, v1) times
    integrated Jacobi polynomials of v2, by total degree."""
    a, b, c = (lam[v] for v in verts)
    ga, gb, gc = (g[v] for v in verts)
    E, C = _edge_family(a, b, ga, gb, p - 1)
    t, gt = a + b + c, ga + gb + gc
    L = {(r, 1): c for r in range(p - 1)}
    D = {(r, 1): np.broadcast_to(gc, (len(c), 3)) for r in range(p - 1)}
    if p == 3:  # second integrated Jacobi polynomial, weight 1: c (3 c - 2 t) / 2 scaled
        # P_0 = 1, P_1 = 3 c - t, P_2 = (10 c^2 - 8 c t + t^2) in the scaled variable
        p1, p2 = 3.0 * c - t, 10.0 * c * c - 8.0 * c * t + t * t
        al = 1.0
        a2, b2, c2 = (2 + al) / ((3 + al) * (4 + al)), al / ((2 + al) * (4 + al)), 1.0 / (
            (2 + al) * (3 + al))
        L[(0, 2)] = a2 * p2 + b2 * t * p1 - c2 * t * t
        R = -(p1 + t) / (2 + al)
        D[(0, 2)] = p1[:, None] * gc + R[:, None] * gt
    S, K = [], []
    for k in range(1, p):
        for r in range(k):
            l, d = L[(r, k - r)], D[(r, k - r)]
            S.append(E[r] * l[:, None])
            K.append(l[:, None] * C[r] + np.cross(d, E[r]))
    return S, K


def _variants(X, p):
    """Shape functions and curls at reference points for every orientation: lists by
    (edge, flag), (face, code) and the volume, stacked (V, points, 3)."""
    X = np.atleast_2d(X)
    lam = [1.0 - X.sum(1), X[:, 0], X[:, 1], X[:, 2]]
    g = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    S, C = [], []
    for a, b in EDGES:
        for i, j in ((a, b), (b, a)):
            s, c = _edge_family(lam[i], lam[j], g[i], g[j], p)
            S += s
            C += c
    for f in FACES if p > 1 else ():
        for q in PERMS:
            v = [f[k] for k in q]
            fam = [_face_family(lam, g, [v[m], v[(m + 1) % 3], v[(m + 2) % 3]], p)
                   for m in range(2)]
            for k in range(len(fam[0][0])):
                for m in range(2):
                    S.append(fam[m][0][k])
                    C.append(fam[m][1][k])
    for m in range(3 if p == 3 else 0):
        v, d = [(m + k) % 4 for k in range(3)], (m + 3) % 4
        s, c = _face_family(lam, g, v, 2)
        S.append(lam[d][:, None] * s[0])
        C.append(lam[d][:, None] * c[0] + np.cross(np.broadcast_to(g[d], s[0].shape), s[0]))
    return np.stack(S), np.stack(C)


def _orientations(t):
    """(E, n) variant index of every local DOF."""
    p, en = t.p, t.elems_nodes
    nf = p * (p - 1)
    cols = []
    ends = t.edges_nodes[t.elems_edges]
    for e, (a, b) in enumerate(EDGES):
        o = (en[:, a] == ends[:, e, 1]) & (en[:, b] == ends[:, e, 0])
        cols.append(((2 * e + o) * p)[:, None] + np.arange(p))
    if nf:
        owner = t.faces_edges[t.elems_faces]
        code = np.zeros(100, np.int64)
        for k, v in CODES.items():
            code[k] = v
        for f, (a, b, _) in enumerate(FACE_EDGES):
            k1 = (owner[:, f] == t.elems_edges[:, a, None]).argmax(1) + 1
            k2 = (owner[:, f] == t.elems_edges[:, b, None]).argmax(1) + 1
            cols.append((12 * p + (6 * f + code[10 * k1 + k2]) * nf)[:, None] + np.arange(nf))
    nv = p * (p - 1) * (p - 2) // 2
    cols.append(np.broadcast_to(12 * p + 24 * nf + np.arange(nv), (len(en), nv)))
    return np.concatenate(cols, 1)


def _points(p):
    x, w = np.polynomial.legendre.leggauss(p + 2)
    x, w = 0.5 * (x + 1), 0.5 * w
    a, b, c = (v.ravel() for v in np.meshgrid(x, x, x, indexing="ij"))
    wa, wb, wc = (v.ravel() for v in np.meshgrid(w, w, w, indexing="ij"))
    return np.stack([a, b * (1 - a), c * (1 - a) * (1 - b)], 1), wa * wb * wc * (1 - a) ** 2 * (
        1 - b)


class _Exact:
    """Element matrices of the case in 64 bits, a part of the elements at a time."""

    def __init__(self, t, coords, sigma, dev):
        self.t, self.dev = t, dev
        X, w = _points(t.p)
        S, C = _variants(X, t.p)
        tab = lambda F: torch.from_numpy(np.einsum("q,aqi,bqj->abij", w, F, F)).to(dev)  # noqa
        self.TS, self.TC = tab(S), tab(C)
        J = torch.from_numpy(coords[:, 1:] - coords[:, :1]).to(dev)      # rows x_k - x_0
        det, iJ = torch.linalg.det(J), torch.linalg.inv(J)
        sg = torch.from_numpy(sigma[:, (0, 0, 1)]).to(dev)
        self.G = det[:, None, None] * torch.einsum("eka,ek,ekb->eab", iJ, sg, iJ)
        self.H = torch.einsum("eak,ebk->eab", J, J) / det[:, None, None]
        self.var = torch.from_numpy(_orientations(t)).to(dev)
        self.dofs = torch.from_numpy(t.dofs).to(dev)
        self.step = {1: 60000, 2: 20000, 3: 3000}[t.p]

    def parts(self):
        for e in range(0, self.t.n_elems, self.step):
            k = slice(e, e + self.step)
            v = self.var[k]
            M = torch.zeros((len(v),) + 2 * (v.shape[1],), dtype=torch.float64, device=self.dev)
            K = torch.zeros_like(M)
            for a in range(3):
                for b in range(3):
                    M += self.G[k, a, b, None, None] * self.TS[:, :, a, b][v[:, :, None],
                                                                           v[:, None, :]]
                    K += self.H[k, a, b, None, None] * self.TC[:, :, a, b][v[:, :, None],
                                                                           v[:, None, :]]
            yield k, self.dofs[k], M, K

    def pattern(self):
        N = self.t.ndof
        keys = [torch.empty(0, dtype=torch.int64, device=self.dev)]
        for e in range(0, self.t.n_elems, self.step):
            d = self.dofs[e:e + self.step]
            keys = [torch.unique(torch.cat([keys[0], (d[:, :, None] * N + d[:, None, :]).ravel()]))]
        return keys[0]

    def km(self):
        """CSR keys (row * ndof + column, ascending) and the PEC-constrained K and M."""
        N, key = self.t.ndof, self.pattern()
        Kv = torch.zeros(len(key), dtype=torch.float64, device=self.dev)
        Mv = torch.zeros_like(Kv)
        for _, d, M, K in self.parts():
            at = torch.searchsorted(key, (d[:, :, None] * N + d[:, None, :]).ravel())
            Kv.index_add_(0, at, K.ravel())
            Mv.index_add_(0, at, M.ravel())
        bc = torch.zeros(N, dtype=torch.bool, device=self.dev)
        bc[torch.from_numpy(self.t.boundary_dofs).to(self.dev)] = True
        row, col = key // N, key % N
        fixed = bc[row] | bc[col]
        Kv[fixed] = (row == col)[fixed].double()
        Mv[fixed] = 0.0
        return row, col, Kv, Mv, bc


def _csr(row, col, v, N):
    crow = torch.zeros(N + 1, dtype=torch.int64, device=row.device)
    crow[1:] = torch.cumsum(torch.bincount(row, minlength=N), 0)
    return torch.sparse_csr_tensor(crow, col, v, (N, N), check_invariants=False)


def _cocg(row, col, Kv, Mv, om, B):
    """(N, R) solutions of (K - i om_r mu0 M) x_r = b_r by COCG with a diagonal
    preconditioner, restarted from the true residual until it is at 3e-14 or stays."""
    N = B.shape[0]
    wm = torch.as_tensor(om, dtype=torch.float64, device=B.device) * MU0
    K, M = _csr(row, col, Kv, N), _csr(row, col, Mv, N)
    dk, dm = Kv[row == col], Mv[row == col]
    dinv = 1.0 / torch.complex(dk[:, None].expand(B.shape), -dm[:, None] * wm)

    def mul(v):
        z = torch.view_as_real(v).reshape(N, -1)
        k, m = (K @ z).reshape(v.shape + (2,)), (M @ z).reshape(v.shape + (2,))
        return torch.complex(k[..., 0] + m[..., 1] * wm, k[..., 1] - m[..., 0] * wm)

    bn = B.abs().square().sum(0).sqrt()
    bn = torch.where(bn > 0, bn, torch.ones_like(bn))
    x = torch.zeros_like(B)
    last = math.inf
    for _ in range(8):
        r = B - mul(x)
        now = float((r.abs().square().sum(0).sqrt() / bn).max())
        if now < 3e-14 or now > 0.5 * last:
            break
        last, goal = now, max(1e-14, now * 1e-7)
        c, p, rho = torch.zeros_like(B), torch.zeros_like(B), None
        for k in range(20000):
            z = dinv * r
            new = (r * z).sum(0)
            live = new.abs() > 0
            p = z if rho is None else z + torch.where(live, new / rho, 0) * p
            rho = torch.where(live, new, torch.ones_like(new))
            q = mul(p)
            mu = (p * q).sum(0)
            al = torch.where(live & (mu.abs() > 0), rho / mu, torch.zeros_like(mu))
            c, r = c + al * p, r - al * q
            if k % 50 == 49 and float((r.abs().square().sum(0).sqrt() / bn).max()) < goal:
                break
        x = x + c
    return x


def _basis_at(t, coords, elements, pts):
    """Physical basis functions and curls (points, n, 3) of the located elements."""
    var = _orientations(t)[elements]
    c = coords[elements]
    J = c[:, 1:] - c[:, :1]
    iJ, det = np.linalg.inv(J), np.linalg.det(J)
    X = np.einsum("qk,qka->qa", pts - c[:, 0], iJ)
    S, C = _variants(X, t.p)
    k = np.arange(len(pts))[:, None]
    S, C = S[var, k], C[var, k]
    return np.einsum("qka,qna->qnk", iJ, S), np.einsum("qak,qna->qnk", J, C) / det[:, None, None]


def _locate(coords, pts):
    """Lowest element that contains each point to 1e-12 in barycentric coordinates."""
    c = torch.from_numpy(coords)
    T = (c[:, :3] - c[:, 3:]).transpose(1, 2)
    inv = torch.linalg.inv(T)
    out = np.full(len(pts), -1)
    for q, x in enumerate(torch.from_numpy(pts)):
        lam = torch.einsum("eab,eb->ea", inv, x - c[:, 3])
        lam = torch.cat([lam, 1.0 - lam.sum(1, keepdim=True)], 1)
        hit = torch.nonzero(((lam >= -1e-12) & (lam <= 1 + 1e-12)).all(1))
        if len(hit):
            out[q] = int(hit[0])
    return out


def _fields(t, coords, elements, pts, x, om):
    N, C = _basis_at(t, coords, elements, pts)
    xe = x[t.dofs[elements]]
    return np.concatenate([np.einsum("qn,qnk->qk", xe, N),
                           np.einsum("qn,qnk->qk", xe, C) / (1j * om * MU0)], 1)


def _pair(z):
    z = torch.as_tensor(z)
    return torch.view_as_real(z.contiguous())


def _source(t, coords, el, pos, moment, om):
    N, _ = _basis_at(t, coords, np.array([el]), pos[None])
    b = np.zeros(t.ndof, np.complex128)
    b[t.dofs[el]] += 1j * om * MU0 * (N[0] @ moment)
    return b


def exact(case, seed):
    t, coords, sigma, r = _model(case, seed)
    kind = case["kind"]
    om = 2.0 * math.pi * case.get("frequency", 1.0)
    dev = torch.device("cuda")
    if kind == "points":
        el, pos = _source_of(coords, r)
        rx, moment = _line(case["receivers"], r), r.standard_normal(3)
        x, coef = (torch.view_as_complex(_vectors(seed + k, s)).cpu().numpy()
                   for k, s in ((0, (t.ndof, 2)), (1, (case["receivers"], 3, 2))))
        at = _locate(coords, rx)
        N, _ = _basis_at(t, coords, at, rx)
        f = np.zeros(t.ndof, np.complex128)
        np.add.at(f, t.dofs[at], np.einsum("qk,qnk->qn", coef, N))
        return {"elements": None, "b": _pair(_source(t, coords, el, pos, moment, om)),
                "fields": _pair(_fields(t, coords, at, rx, x, om)), "f": _pair(f)}
    if kind == "matrices":
        n = t.dofs.shape[1]
        M = torch.empty((t.n_elems, n, n), dtype=torch.float64, device=dev)
        K = torch.empty_like(M)
        for k, _, m, q in _Exact(t, coords, sigma, dev).parts():
            M[k], K[k] = m, q
        return {"M": M, "K": K}
    X = _Exact(t, coords, sigma, dev)
    if kind == "gradient":
        x = torch.view_as_complex(_vectors(seed, (case["nrhs"], t.ndof, 2), zero=t.boundary_dofs))
        lam = torch.view_as_complex(_vectors(seed + 1, (case["nrhs"], t.ndof, 2),
                                             zero=t.boundary_dofs))
        w = torch.from_numpy(om * np.linspace(1.0, 2.0, case["nrhs"])).to(dev) * MU0
        g = torch.zeros(t.n_elems, dtype=torch.float64, device=dev)
        for k, d, M, _ in X.parts():
            for i in range(case["nrhs"]):
                xe = torch.view_as_real(x[i][d])
                y = torch.view_as_complex((M.unsqueeze(-1) * xe[:, None]).sum(2).contiguous())
                g[k] -= w[i] * (lam[i][d] * y).sum(1).imag
        return {"gradient": g}
    if kind == "apply":
        wide = torch.float64 if case["dtype"] == "complex128" else torch.float32
        x = _vectors(seed, (t.ndof, 2), wide, t.boundary_dofs).double()
        y = torch.zeros_like(x)
        wm = om * MU0
        for _, d, M, K in X.parts():
            xe = x[d]
            ye = (K.unsqueeze(-1) * xe[:, None]).sum(2)
            me = (M.unsqueeze(-1) * xe[:, None]).sum(2)
            ye = ye + wm * torch.stack([me[..., 1], -me[..., 0]], -1)
            y.index_add_(0, d.ravel(), ye.reshape(-1, 2))
        y[torch.from_numpy(t.boundary_dofs).to(dev)] = 0.0  # identity rows, x = 0 there
        return {"y": y}
    row, col, Kv, Mv, bc = X.km()
    if kind == "assemble":
        return {"values": torch.stack([Kv, -om * MU0 * Mv], 1)}
    if kind == "solve":
        el, pos = _source_of(coords, r)
        b = torch.from_numpy(_source(t, coords, el, pos, np.array([1.0, 0, 0]), om)).to(dev)
        b[bc] = 0.0
        rx = _line(case["receivers"], r)
        x = _cocg(row, col, Kv, Mv, [om], b[:, None])[:, 0]
        f = _fields(t, coords, _locate(coords, rx), rx, x.cpu().numpy(), om)
        return {"x": _pair(x), "fields": _pair(f)}
    B = torch.view_as_complex(_batch_rhs(t, coords, case, r, bc))
    w = [2.0 * math.pi * f for f in _frequencies(case)]
    return {"X": _pair(_cocg(row, col, Kv, Mv, w, B))}
