"""Levels on the 512-thread 16 x 12 tiles of the band kernels (one node per thread, rows kept in
registers), 9-point and cell-weight ones, against the launch-per-sweep V-cycle: the same sweeps in the same order, so the
preconditioner output agrees to round-off, 1e-12 relative in FP64 and 1e-5 in FP32.

Level 1 of these grids has from just below to far above the number of 16 x 12 tiles from which
they are used, with tile remainders of one row or column, and sweep counts of which four make
the extended tile too large for one node per thread."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density

pytestmark = pytest.mark.gpu

# level 1 of a x b cells: tiles of 16 x 12 nodes
SHAPES = [(351, 191), (319, 238), (321, 241), (511, 255), (512, 257), (513, 256), (1, 2399),
          (2, 2401), (3201, 3), (450, 151),
          # level 1 with cell weights: 90, 105, 512, 646 and 1066 tiles, and beside them
          (288, 238), (448, 166), (1022, 382), (1200, 400), (1602, 494)]


def rel(a, b):
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("fixed", [["Left"], ["Left", "Right", "Top", "Bottom"]],
                         ids=["left", "all"])
@pytest.mark.parametrize("nu", [1, 3, 4])
def test_mid_tiles_equal_per_sweep(nx, ny, fixed, nu):
    gp = gpu_problem(dict(CANTILEVER, fixed_sides=fixed), nx, ny)
    gp.set_penalization(3)
    gp.set_option("nu_coarse", nu)
    gp.set_option("filter_dct", 0)  # the filter's V-cycle has 9-point levels too
    xi = torch.as_tensor(smoothed_density(nx, ny, 1, sigma=2.0), device="cuda:0")
    g = torch.Generator(device="cpu").manual_seed(7)
    r = torch.randn(2 * (nx + 1) * (ny + 1), generator=g, dtype=torch.float64).cuda()
    rf = torch.randn((nx + 1) * (ny + 1), generator=g, dtype=torch.float64).cuda()
    for prec, tol in (("fp64", 1e-12), ("fp32", 1e-5)):
        gp.set_option("band", 0)
        z_ref = gp.precondition(r, "elasticity", xi, precision=prec)
        f_ref = gp.precondition(rf, "filter", precision=prec)
        gp.set_option("band", 1)
        z = gp.precondition(r, "elasticity", xi, precision=prec)
        f = gp.precondition(rf, "filter", precision=prec)
        print(nx, ny, fixed, nu, prec, rel(z, z_ref), rel(f, f_ref), flush=True)
        assert rel(z, z_ref) < tol
        assert rel(f, f_ref) < tol
