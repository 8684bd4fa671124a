"""The P2 solve's PCG: grids around its 8 x 8-cell tiles (a single tile, tiles with one cell, odd
counts, every side fixed) against the direct P2 solve, and the MINRES solve behind it."""

import numpy as np
import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, oracle_problem, smoothed_density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,sides", [(4, 4, ["Left"]), (8, 8, ["Left"]), (9, 8, ["Bottom"]),
                                         (17, 9, ["Left", "Right"]), (33, 7, ["Top"]),
                                         (24, 16, ["Left", "Right", "Top", "Bottom"])])
def test_p2_forward(nx, ny, sides, precision):
    case = dict(CANTILEVER, fixed_sides=sides,
                body_force={"center": (1.4, 0.5), "radius": 0.4, "value": (0.3, -1.0)})
    orc = oracle_problem(case, nx, ny, degree=2)
    gp = gpu_problem(case, nx, ny, rtol=1e-9, degree=2, precision=precision)
    orc.set_penalization(3)
    gp.set_penalization(3)
    xi = smoothed_density(nx, ny, seed=nx, sigma=2.0, lo=0.2)
    u = gp.forward(torch.as_tensor(xi, device="cuda:0")).cpu().numpy()
    ref = orc.forward(xi)
    # the residual's bound times the condition number of K, of order n^2 / lo^3
    assert np.linalg.norm(u - ref) <= 1e-6 * np.linalg.norm(ref)
    assert gp.last_stats["rel_residual"] <= 1e-9
    assert gp.last_stats["iterations"] > 0


def test_p2_tolerance_below_the_round_off_floor_is_refused():
    """PCG's restarts and MINRES both end at the floor of the true residual."""
    from topomax_amd._lib import NotConvergedError
    gp = gpu_problem(CANTILEVER, 120, 40, rtol=1e-15, degree=2)
    gp.set_penalization(3)
    xi = torch.as_tensor(smoothed_density(120, 40, seed=1), device="cuda:0")
    with pytest.raises(NotConvergedError):
        gp.forward(xi)
    u = gp.forward(xi, rtol=1e-8)
    assert torch.isfinite(u).all()
