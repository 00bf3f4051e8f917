"""Assembly over entities of every size and waves of every length: bitwise the ordered
sum of the element matrices, for A(omega), for K and M and with the PEC fold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from petgem_amd import core  # noqa: E402
from petgem_amd.synthetic import Workload  # noqa: E402
from petgem_amd.mesh import Topology  # noqa: E402
from oracle import fem, topology as otopo  # noqa: E402

DEV = "cuda"


def _ordered_sums(plan, dofs, vals):
    """Per CSR slot, the sum of its element entries (E, n, n) in element order."""
    ndof = plan.h_rowptr.size - 1
    row = torch.repeat_interleave(torch.arange(ndof, device=DEV),
                                  torch.from_numpy(np.diff(plan.h_rowptr)).to(DEV))
    keys = row * ndof + torch.from_numpy(plan.h_cols).to(DEV).long()
    d = torch.from_numpy(dofs).to(DEV).long()
    slot = torch.searchsorted(keys, (d[:, :, None] * ndof + d[:, None, :]).reshape(-1))
    slot, order = torch.sort(slot, stable=True)
    count = torch.bincount(slot, minlength=keys.numel())
    first = torch.cumsum(count, 0) - count
    out = [torch.zeros(keys.numel(), dtype=torch.float64, device=DEV) for _ in vals]
    for k in range(int(count.max())):
        s = torch.nonzero(count > k).reshape(-1)
        for o, v in zip(out, vals):
            o[s] += v.reshape(-1)[order[first[s] + k]]
    return out, row, keys % ndof


def _check(T, sigma, omega):
    mesh = core.DeviceMesh.from_topology(T, DEV)
    asm = core.Assembler(mesh)
    asm.geometry(sigma)
    M, K = asm.element_matrices()
    (k, m, im), row, col = _ordered_sums(asm.plan, T.dofs, (K, M, -(omega * core.MU0 * M)))
    ent_bc, _ = mesh.entity_mask(T.boundary_dofs[::2])
    # the fold eliminates whole entities: the DOFs are numbered edges, faces, volumes
    p, ne, nf = T.p, mesh.n_edges, mesh.n_faces
    size = torch.full((ent_bc.numel(),), p * (p - 1) * (p - 2) // 2, device=DEV)
    size[:ne], size[ne:ne + nf] = p, p * (p - 1)
    bc = torch.repeat_interleave(ent_bc.bool(), size)
    elim, one = bc[row] | bc[col], (bc[row] & (row == col)).double()
    for fold in (False, True):
        a = asm.assemble(omega, ent_bc=ent_bc if fold else None).reshape(-1, 2)
        gk, gm = core.assemble_km(asm, ent_bc if fold else None)
        for got, ref, diag in ((a[:, 0], k, one), (a[:, 1], im, 0 * one), (gk, k, one),
                               (gm, m, 0 * one)):
            assert torch.equal(got.reshape(-1), torch.where(elim, diag, ref) if fold else ref)
    return asm, M, K


def _fans(sizes):
    """Closed fans of tetrahedra, each around an edge of its own."""
    pts, en = [], []
    for f, m in enumerate(sizes):
        b = len(pts)
        pts += [(4.0 * f, 0.0, -1.0), (4.0 * f, 0.1, 1.0)]
        ang = 2 * np.pi * (np.arange(m) + 0.2 * np.sin(np.arange(m))) / m
        pts += [(4.0 * f + np.cos(x), np.sin(x), 0.1 * np.cos(3 * x)) for x in ang]
        en += [sorted((b, b + 1, b + 2 + i, b + 2 + (i + 1) % m)) for i in range(m)]
    return np.array(pts), np.array(en)


# elements around an edge: one batch holds 64 of them at p = 1, 32 at p = 2 and 21 at
# p = 3, 256 pairs are staged at a time
@pytest.mark.parametrize("p,sizes", [(1, (4, 64, 65, 3, 130)), (2, (5, 32, 33, 3, 70)),
                                     (2, (100, 4)), (3, (21, 4, 22, 43)), (3, (70,)),
                                     (3, (21, 4, 22, 43, 70) * 26)])
def test_entities_beyond_a_batch(p, sizes):
    pts, en = _fans(sizes)
    T = Topology(pts, en, p)
    sigma = np.random.default_rng(p).uniform(0.1, 2.0, (T.n_elems, 2))
    asm, M, K = _check(T, sigma, core.omega_of(2.0))
    eo, fo = otopo.orientations(T.elems_nodes, T.elems_edges, T.edges_nodes, T.elem_faces_edges)
    Mr, Kr = fem.all_element_matrices(T.coords, eo, fo, sigma, p)
    for g, r in ((M.cpu().numpy(), Mr), (K.cpu().numpy(), Kr)):
        scale = np.abs(r).max(axis=(1, 2), keepdims=True)
        assert (np.abs(g - r) / scale).max() <= 1e-12


# a wave takes from one entity to four batches with their number, K_e and M_e apart if few;
# p = 3 from 4096 elements on is assembled like p <= 2
@pytest.mark.parametrize("p,n", [(1, 2), (1, 9), (1, 34), (1, 43), (2, 4), (2, 7), (2, 22), (3, 8),
                                 (3, 9), (3, 17)])
def test_waves_of_several_batches(p, n):
    w = Workload(n, p, noise=0.1, seed=n)
    _check(w.topo, w.sigma, core.omega_of(w.frequency))
