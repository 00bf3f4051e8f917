"""Point location of many points in very few elements: the points are taken in slices, as
many as a launch can hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from petgem_amd import core  # noqa: E402
from petgem_amd.mesh import Topology  # noqa: E402
from petgem_amd.synthetic import kuhn_grid  # noqa: E402


@pytest.mark.parametrize("keep,npts", [(1, 524279), (1, 524288), (1, 600001), (6, 700000)])
def test_many_points_in_few_elements(keep, npts):
    pts, tets = kuhn_grid(1, 2.0)
    used, tets = np.unique(tets[:keep], return_inverse=True)
    T = Topology(pts[used], tets.reshape(-1, 4), 1)
    mesh = core.DeviceMesh.from_topology(T, "cuda")
    lo, hi = T.points.min(0), T.points.max(0)
    x = np.random.default_rng(npts).uniform(lo - 0.1, hi + 0.1, (npts, 3))
    got = core.locate_points(mesh, x).cpu().numpy()
    # barycentric coordinates of every point in every element
    c = T.coords
    lam = np.einsum("eij,enj->eni", np.linalg.inv((c[:, 1:] - c[:, :1]).transpose(0, 2, 1)),
                    x[None] - c[:, :1])
    least = np.minimum(lam.min(2), 1.0 - lam.sum(2))  # of the four
    clear = (np.abs(least) > 1e-6).all(0)  # away from every face
    inside = least > 0.0
    ref = np.where(inside.any(0), inside.argmax(0), -1)
    assert clear.mean() > 0.99
    assert np.array_equal(got[clear], ref[clear])
