"""The paired sweeps of a finest elasticity level with an odd side (the transfer to the coarse
grid is bilinear): two pre-sweeps + residual + restriction in one launch and prolongation + two
post-sweeps in another, against the V-cycle with a launch for each.

Both compute the same sweeps in the same order; only the weighted sums of the two transfers are
added in another order, so the preconditioner output agrees to round-off: 1e-12 relative in FP64
and 1e-5 in FP32, as for the nested transfers."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density
from tests.test_gpu_sweep_pairs import FIXED, rel, residual_vector

pytestmark = pytest.mark.gpu

# sides: both odd, one odd, narrow grids, and strip edges (56 owned columns of a 64-lane strip)
SHAPES = [(45, 15), (46, 15), (45, 16), (55, 33), (57, 33), (111, 56), (112, 113), (1, 201),
          (201, 1), (3, 700), (699, 5)]


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("fixed", FIXED, ids=["-".join(f) for f in FIXED])
def test_bilinear_pairs_equal_per_sweep(nx, ny, fixed):
    gp = gpu_problem(dict(CANTILEVER, fixed_sides=fixed), nx, ny)
    gp.set_penalization(3)
    xi = torch.as_tensor(smoothed_density(nx, ny, 1, sigma=2.0), device="cuda:0")
    r = residual_vector(nx, ny, 5)
    for cw in (0, 3):  # sweeps form the cell weights from xi, or read them
        gp.set_option("fine_cell_weights", cw)
        for prec, tol in (("fp64", 1e-12), ("fp32", 1e-5)):
            for opt in ("sweep_pairs", "sweep_pairs_post", "sweep_pair_restrict"):
                gp.set_option(opt, 0)
            z_ref = gp.precondition(r, "elasticity", xi, precision=prec)
            for pre, post, rr in ((8, 0, 0), (8, 0, 8), (8, 1, 0), (2, 7, 2), (16, 6, 3),
                                  (4, 64, 64)):
                gp.set_option("sweep_pairs", pre)
                gp.set_option("sweep_pairs_post", post)
                gp.set_option("sweep_pair_restrict", rr)
                z = gp.precondition(r, "elasticity", xi, precision=prec)
                print(nx, ny, fixed, cw, prec, pre, post, rr, rel(z, z_ref), flush=True)
                assert torch.isfinite(z).all()
                assert rel(z, z_ref) < tol
