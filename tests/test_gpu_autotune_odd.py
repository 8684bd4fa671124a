"""The autotuner on grids with odd sides, whose finest level runs the paired kernels with bilinear
transfers: it re-picks all three chunk heights, and the timing entry point runs those kernels."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density
from tests.test_gpu_bench_kernels import bench
from topomax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(333, 111), (334, 111), (333, 110)])
def test_heights_are_picked_again(nx, ny):
    gp = gpu_problem(CANTILEVER, nx, ny, precision="mixed", rtol=1e-10)
    gp.set_penalization(3)
    rho = torch.as_tensor(smoothed_density(nx, ny, 5, sigma=3.0), device="cuda:0")
    J0, w0, _ = gp.objective_and_gradient(rho)
    # one chunk for the whole height: a wave walks its 110 rows in turn, some 10 times what the
    # heights to choose from take
    for name in ("sweep_pairs_post", "sweep_pair_restrict"):
        gp.set_option(name, 112)
    slow = {(k, p): bench(gp, k, p, reps=20)[:2] for k in (4, 6) for p in ("fp32", "fp64")}
    gp.autotune()
    for (kernel, precision), (rc, us) in slow.items():
        assert rc == _lib.TMX_OK
        rc, tuned, nbytes = bench(gp, kernel, precision, reps=20)
        print(nx, ny, kernel, precision, us, "->", tuned, flush=True)
        assert rc == _lib.TMX_OK and nbytes > 0
        assert tuned < 0.5 * us
    J1, w1, _ = gp.objective_and_gradient(rho)
    # chunk heights only order sums: both solves are within their tolerance of each other
    assert abs(J1 - J0) <= 1e-9 * abs(J0)
    assert float((w1 - w0).norm() / w0.norm()) <= 1e-8


def test_a_single_level_has_no_transfers():
    gp = gpu_problem(CANTILEVER, 3, 2)
    gp.set_penalization(3)
    gp.objective_and_gradient(torch.full((12,), 0.5, dtype=torch.float64, device="cuda:0"))
    gp.autotune()
    for kernel in (4, 6):
        rc, _, _ = bench(gp, kernel, "fp64")
        assert rc == _lib.TMX_ERR_INVALID
