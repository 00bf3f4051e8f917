"""Stop flag of the COCG iterations (csrc/pg_stop.h): a launch that stores the flag while
its own waves are still reading it must not split them."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "petgem_amd",
                    "csrc")

# a batch of iterations whose launch `stops` stores the flag: every wave of every launch,
# reading it before or after that store, has to do what the others of its launch do
SOURCE = """
#include "pg_stop.h"
#include <cstdio>
#include <vector>
using namespace pg;
int main() {
  const int iterations = 25;
  std::vector<int32_t> launch;
  for (int k = 0; k < iterations; ++k) {
    launch.push_back(stop_direction(k));
    launch.push_back(stop_update(k));
  }
  int wrong = 0;
  for (size_t stops = 0; stops <= launch.size(); ++stops) {
    const bool other = stops == launch.size();  // set by a kernel of its own, before all
    const int32_t set = other ? kStopOther : launch[stops];
    wrong += set == 0;
    for (size_t l = 0; l < launch.size(); ++l) {
      const int32_t before = other || l > stops ? set : 0;
      const int32_t after = other || l >= stops ? set : 0;
      const bool early = stopped_before(before, launch[l]), late = stopped_before(after, launch[l]);
      wrong += early != late;                  // waves of one workgroup part
      wrong += late != (other || l > stops);  // a later launch goes on, an earlier one stops
    }
  }
  std::printf("%d\\n", wrong);
  return 0;
}
"""


def test_no_launch_is_split_by_its_own_stop(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "stop.cpp", tmp_path / "stop"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout.strip() == "0"


@pytest.mark.gpu
@pytest.mark.parametrize("pc,p,element", [("jacobi", 1, False), ("bjacobi", 2, True),
                                          ("bjacobi", 3, True)])
def test_a_stop_at_any_place_of_a_batch_leaves_the_same_solution(pc, p, element):
    """The iteration limit reached by the kernel that forms p (within a batch) and by the
    batch's last kernel: x and the iteration count do not depend on which."""
    torch = pytest.importorskip("torch")
    from petgem_amd import core
    from petgem_amd.synthetic import Workload

    w = Workload(6, p, noise=0.1, seed=p)
    T, mesh = w.topo, core.DeviceMesh.from_topology(w.topo, "cuda")
    asm = core.Assembler(mesh)
    asm.geometry(w.sigma)
    om = core.omega_of(1.0)
    ent_bc, dof_bc = mesh.entity_mask(T.boundary_dofs)
    vals, order = asm.assemble(om, ent_bc=ent_bc), mesh.entity_order()
    eop = core.ElementOperator(asm, om, ent_bc, order) if element else None
    b = torch.randn((T.ndof, 2), dtype=torch.float64, device="cuda",
                    generator=torch.Generator("cuda").manual_seed(p))
    b[dof_bc.bool()] = 0.0
    first = None
    for limit in (1, 2, 5, 12):
        ref = None
        for check in (1, 2, 3, 25):
            S = core.KrylovSolver(asm.plan, vals, pc=pc, rtol=1e-13, maxit=limit,
                                  check_every=check, block_ptr=mesh.block_ptr(),
                                  entity_order=order, eop=eop,
                                  spmv="element" if element else "row", like=first)
            first = first or S  # the same kernels for all
            x, info = S.solve(b)
            assert info["iterations"] == limit, (limit, check, info)
            ref = x if ref is None else ref
            assert torch.equal(x, ref), (limit, check)
