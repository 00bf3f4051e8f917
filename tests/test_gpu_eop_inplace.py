"""Element products whose result takes the place of x, or overlaps it."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from petgem_amd import _native as nat, core  # noqa: E402
from petgem_amd.synthetic import Workload  # noqa: E402


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("p,n,bc", [(1, 2, True), (1, 16, True), (1, 16, False), (2, 3, True),
                                    (2, 12, True), (2, 12, False), (3, 4, True), (3, 8, False)])
def test_result_in_the_place_of_x(p, n, bc, dtype):
    """From one workgroup to many; bitwise the product into another array.  Without PEC
    entities (whose rows are copied from x) y may begin anywhere in x, too."""
    w = Workload(n, p, noise=0.1, seed=n)
    T, mesh = w.topo, core.DeviceMesh.from_topology(w.topo, "cuda")
    asm = core.Assembler(mesh)
    asm.geometry(w.sigma)
    ent_bc = mesh.entity_mask(T.boundary_dofs)[0] if bc else None
    eop = core.ElementOperator(asm, core.omega_of(1.0), ent_bc, mesh.entity_order())
    x = torch.randn((T.ndof, 2), dtype=dtype, device="cuda",
                    generator=torch.Generator("cuda").manual_seed(p))
    ref = eop.apply(x)
    fn = nat.lib().pg_eop_apply_z if dtype == torch.float64 else nat.lib().pg_eop_apply_c
    for shift in (0,) if bc else (0, 1, T.ndof // 2, T.ndof - 1):
        for ahead in (False, True):
            both = torch.zeros((T.ndof + shift, 2), dtype=dtype, device="cuda")
            lo, hi = both[:T.ndof], both[shift:]
            src, dst = (lo, hi) if ahead else (hi, lo)
            src.copy_(x)
            nat.check(fn(eop.handle, nat.ptr(src), nat.ptr(dst), nat.stream_handle()))
            assert torch.equal(dst, ref), (shift, ahead)
