"""Factored element products (K_e x, M_e x without the element matrices) on meshes
whose elements have arbitrary edge and face orientations: node numbers, element
order and each element's vertex order drawn at random."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from petgem_amd import core  # noqa: E402
from petgem_amd.mesh import Topology  # noqa: E402
from petgem_amd.synthetic import kuhn_grid, layered_sigma  # noqa: E402

DEV = "cuda"
EVEN = np.array([(0, 1, 2, 3), (0, 2, 3, 1), (0, 3, 1, 2), (1, 0, 3, 2), (1, 2, 0, 3),
                 (1, 3, 2, 0), (2, 0, 1, 3), (2, 1, 3, 0), (2, 3, 0, 1), (3, 0, 2, 1),
                 (3, 1, 0, 2), (3, 2, 1, 0)])


def _free(n, p, seed=0, keep=None):
    """A Kuhn grid renumbered at random (`keep`: only its first elements), on the device."""
    rng = np.random.default_rng(seed)
    pts, tets = kuhn_grid(n, 10000.0)
    pts = pts + np.where(np.abs(pts).max(1, keepdims=True) < 4999.0,
                         rng.uniform(-300.0 / n, 300.0 / n, pts.shape), 0.0)
    tets = tets[:keep]
    used = np.unique(tets)
    new = np.full(len(pts), -1)
    new[used] = rng.permutation(used.size)
    q = np.empty((used.size, 3))
    q[new[used]] = pts[used]
    tets = new[tets][rng.permutation(len(tets))]
    tets = np.take_along_axis(tets, EVEN[rng.integers(0, 12, len(tets))], axis=1)
    T = Topology(q, tets, p)
    mesh = core.DeviceMesh.from_topology(T, DEV)
    asm = core.Assembler(mesh)
    sigma = layered_sigma(T.coords.mean(1), noise=0.3, seed=seed)
    asm.geometry(sigma)
    return T, mesh, asm, sigma


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("p,n,nrhs", [(1, 3, 64), (1, 5, 256), (2, 2, 64), (2, 3, 192),
                                      (2, 4, 128)])
def test_batch_products_on_arbitrary_orientations(p, n, nrhs, precision):
    """The batched solve with element products against the same batch on the
    assembled CSR, one to sixteen elements per workgroup.  Both reach a true
    residual of 1e-10; the bar between two such solutions is 1e-7."""
    T, mesh, asm, _ = _free(n, p)
    ent_bc, dof_bc = mesh.entity_mask(T.boundary_dofs)
    K, M = core.assemble_km(asm, ent_bc)
    B = torch.randn((T.ndof, nrhs, 2), dtype=torch.float64, device=DEV,
                    generator=torch.Generator(DEV).manual_seed(n))
    B[dof_bc.bool()] = 0.0
    fr = [0.5 + 0.25 * (r % 5) for r in range(nrhs)]
    kw = dict(rtol=1e-10, block_ptr=mesh.block_ptr(), entity_order=mesh.entity_order(),
              precision=precision, pc="bjacobi")
    ref, _ = core.BatchSolver(asm.plan, K, M, fr, **kw).solve(B)
    eop = core.ElementOperator(asm, core.omega_of(1.0), ent_bc, mesh.entity_order())
    X, info = core.BatchSolver(asm.plan, K, M, fr, eop=eop, **kw).solve(B)
    assert (info["status"] == 0).all() and info["relres"].max() <= 1e-10
    err = float((X - ref).abs().max() / ref.abs().max())
    print(f"batch p={p} n={n} R={nrhs} {precision}: {err:.2e}", flush=True)
    assert err <= 1e-7


@pytest.mark.parametrize("p,n,keep", [(1, 2, 1), (1, 3, 65), (2, 2, 31), (2, 2, 33), (2, 3, 64),
                                      (2, 4, 129), (2, 4, None), (1, 28, None), (3, 2, 1),
                                      (3, 2, 33),
                                      (3, 3, None)])
def test_products_on_arbitrary_orientations(p, n, keep):
    """y = A x on the operator against the assembled CSR: element counts around the
    32 elements of a wave, the 64 of a slot group and the 128 of a workgroup, and
    past the 131 072 from which a workgroup takes two groups, in both precisions
    and, for complex128, x at an address that is not a multiple of 32 bytes.
    Bars as for the structured grids: 1e-12 and 1e-5."""
    T, mesh, asm, _ = _free(n, p, seed=n, keep=keep)
    omega = core.omega_of(0.5)
    vals = asm.assemble(omega)
    eop = core.ElementOperator(asm, omega, None, mesh.entity_order())
    g = torch.Generator(DEV).manual_seed(n)
    xb = torch.randn((T.ndof + 1, 2), dtype=torch.float64, device=DEV, generator=g)
    for x in (xb[:-1], xb[1:]):
        ref = core.spmv(asm.plan, vals, x.contiguous())
        err = float((eop.apply(x) - ref).abs().max() / ref.abs().max())
        err32 = float((eop.apply(x.float()).double() - ref).abs().max() / ref.abs().max())
        assert err <= 1e-12 and err32 <= 1e-5, (err, err32)


@pytest.mark.parametrize("p,n,keep,nrhs", [(1, 2, 1, 1), (1, 3, None, 33), (2, 2, 127, 2),
                                           (2, 3, 129, 65), (3, 2, 47, 3)])
@pytest.mark.parametrize("rows", [False, True])
def test_adjoint_gradient_on_arbitrary_orientations(p, n, keep, nrhs, rows):
    """-omega mu0 Im(lam^T M_e x) with the element matrices of pg_element_matrices in
    64 bits, both column layouts, right-hand sides below, at and past the 32 of
    one launch.  n^2 products of 1e-16 each, summed over the columns: 1e-12 of
    the largest entry."""
    import ctypes

    from petgem_amd import _native as nat
    T, mesh, asm, _ = _free(n, p, seed=n, keep=keep)
    gen = torch.Generator(DEV).manual_seed(nrhs)
    x, lam = (torch.randn((nrhs, T.ndof, 2), dtype=torch.float64, device=DEV, generator=gen)
              for _ in range(2))
    omega = np.linspace(1.0, 9.0, nrhs)
    M, _ = asm.element_matrices()
    d = torch.from_numpy(T.dofs).to(DEV)
    xe, le = torch.view_as_complex(x)[:, d], torch.view_as_complex(lam)[:, d]
    y = (M[None] * xe.real[:, :, None]).sum(-1) + 1j * (M[None] * xe.imag[:, :, None]).sum(-1)
    w = torch.from_numpy(omega).to(DEV) * (4e-7 * np.pi)
    ref = -(w[:, None] * (le * y).sum(-1).imag).sum(0)
    if rows:
        x, lam = (v.transpose(0, 1).contiguous() for v in (x, lam))
    g = torch.zeros(T.n_elems, dtype=torch.float64, device=DEV)
    fn = nat.lib().pg_adjoint_gradient_rows if rows else nat.lib().pg_adjoint_gradient
    nat.check(fn(asm.tables.handle, mesh.n_elems, nat.ptr(asm.workspace), nat.ptr(mesh.dofs),
                 nrhs, ctypes.c_int64(T.ndof), nat.ptr(x), nat.ptr(lam), nat.ptr(omega),
                 nat.ptr(g), nat.stream_handle()))
    assert float((g - ref).abs().max()) <= 1e-12 * float(ref.abs().max())


@pytest.mark.parametrize("sizes", [(8, 3, 9), (16, 17, 4), (40,), (5,) * 1700, (5,) * 6000])
def test_p3_sums_of_many_elements(sizes):
    """y = A x at p = 3 over fans of tetrahedra around an edge each: one, two and more
    steps of eight elements, and both sides of the 131 072 entities up to which a thread
    sums one DOF (61 200 and 216 000 here).  Same bounds as above."""
    pts, tets, b = [], [], 0
    for f, m in enumerate(sizes):
        a = 2 * np.pi * np.arange(m) / m
        x = 4.0 * f
        pts += [np.array([(x, 0.0, -1.0), (x, 0.1, 1.0)]),
                np.stack([x + np.cos(a), np.sin(a), 0.1 * np.cos(3 * a)], axis=1)]
        i = np.arange(m)
        tets.append(np.sort(np.stack([0 * i + b, 0 * i + b + 1, b + 2 + i, b + 2 + (i + 1) % m],
                                     axis=1), axis=1))
        b += m + 2
    T = Topology(np.concatenate(pts), np.concatenate(tets), 3)
    mesh = core.DeviceMesh.from_topology(T, DEV)
    asm = core.Assembler(mesh)
    asm.geometry(np.random.default_rng(1).uniform(0.1, 2.0, (T.n_elems, 2)))
    om = core.omega_of(1.0)
    vals = asm.assemble(om)
    eop = core.ElementOperator(asm, om, None, mesh.entity_order())
    x = torch.randn((T.ndof, 2), dtype=torch.float64, device=DEV,
                    generator=torch.Generator(DEV).manual_seed(3))
    ref = core.spmv(asm.plan, vals, x)
    for dt, bar in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
        y = eop.apply(x.to(dt)).double()
        assert float((y - ref).abs().max()) <= bar * float(ref.abs().max())
