"""Iteration counts of the multigrid solves: PCG corrects a slightly wrong smoothing epilogue,
restriction or prolongation, which shows in the counts and not in the solution."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# counts (both precisions at most, both operators) with the restriction of one thread a coarse
# node, level 0 in separate kernels and the spectral estimates on the host; two more for the
# order of sums
COUNTS = {(6, 4, 2): 34, (16, 8, 8): 55, (36, 20, 12): 68, (10, 22, 18): 130, (48, 24, 40): 67}


# the mixed solve on the Kuhn operator with level 0 fused, and on the general lattice operator
@pytest.mark.parametrize("precision,kuhn", [("fp64", "1"), ("mixed", "1"), ("mixed", "0")])
@pytest.mark.parametrize("dims", list(COUNTS))
def test_gpu_mg_iteration_counts(monkeypatch, dims, precision, kuhn):
    """Coarse levels of 24 to 6825 nodes: 32 restricted nodes a work-group, the last one cut
    short.  The solution is the block-Jacobi one (both stop at 1e-11 of the load, condition
    numbers below 1e5)."""
    from platoanalyze_amd import workloads as wl
    from platoanalyze_amd.elliptic import Problem

    print(f"case: multigrid counts {dims} {precision} kuhn {kuhn}", flush=True)
    monkeypatch.setenv("PA_BOX_MF_KUHN", kuhn)
    w = wl.make("cantilever_64x32x32", tiny=dims)
    m = wl.model(w)
    z = torch.as_tensor(w.z, device="cuda")
    pb = Problem(m, tolerance=1e-11, precision=precision, preconditioner="multigrid", check_every=1)
    u = pb.solution(z)
    assert pb.stats.converged and pb.stats.iterations <= COUNTS[dims] + 2
    ref = Problem(m, tolerance=1e-11, check_every=1).solution(z)
    assert float((u - ref).norm() / ref.norm()) < 1e-6
