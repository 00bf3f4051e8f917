"""Both sides of the size from which element matrices and assembly are formed without
tables, and entities beyond a batch above it at p = 2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from petgem_amd import core  # noqa: E402
from petgem_amd.mesh import Topology  # noqa: E402
from petgem_amd.synthetic import kuhn_grid  # noqa: E402
from oracle import fem, topology as otopo  # noqa: E402
from test_gpu_assembly import _check, _fans  # noqa: E402


def _checked(T, seed):
    """Assembled values bitwise the ordered sums of the element matrices, those within
    1e-12 of the oracle's largest entry of the element."""
    sigma = np.random.default_rng(seed).uniform(0.1, 2.0, (T.n_elems, 2))
    _, M, K = _check(T, sigma, core.omega_of(2.0))
    pick = np.random.default_rng(seed).permutation(T.n_elems)[:300]
    eo, fo = otopo.orientations(T.elems_nodes, T.elems_edges, T.edges_nodes, T.elem_faces_edges)
    Mr, Kr = fem.all_element_matrices(T.coords[pick], eo[pick], fo[pick], sigma[pick], T.p)
    for g, r in ((M.cpu().numpy()[pick], Mr), (K.cpu().numpy()[pick], Kr)):
        scale = np.abs(r).max(axis=(1, 2), keepdims=True)
        assert (np.abs(g - r) / scale).max() <= 1e-12


@pytest.mark.parametrize("p,line", [(2, 2048), (3, 4096)])
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_sizes_around_the_line(p, line, past):
    n = 7 if line == 2048 else 9
    pts, tets = kuhn_grid(n, 1000.0)
    tets = tets[:line + past]
    used, tets = np.unique(tets, return_inverse=True)
    _checked(Topology(pts[used], tets.reshape(-1, 4), p), line + past)


# as in test_entities_beyond_a_batch, often enough to be assembled without tables
@pytest.mark.parametrize("p,sizes", [(2, (5, 32, 33, 3, 70) * 15),
                                     (2, (100, 4) * 20)])
def test_entities_beyond_a_batch_without_tables(p, sizes):
    pts, en = _fans(sizes)
    _checked(Topology(pts, en, p), p)
