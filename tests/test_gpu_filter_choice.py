"""Which preconditioner a filter solve takes where the DCT solver needs direct stages (2 ny with a
prime factor from 11 up): on narrow grids with large primes, and with eps near the cell size, the
V-cycle, and both give the filtered density."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem

pytestmark = pytest.mark.gpu


def filtered(nx, ny, ratio, precision):
    """The filtered density by default, with the V-cycle, and the problem: square cells, eps of
    `ratio` cells."""
    h = 1.0 / 64
    case = dict(CANTILEVER, width=nx * h, height=ny * h, filter_radius=ratio * h,
                tractions=[{"side": "Right", "center": ny * h / 2, "length": ny * h,
                            "value": (0.0, -1.0)}])
    gp = gpu_problem(case, nx, ny, precision=precision)
    gen = torch.Generator(device="cpu").manual_seed(nx + ny)
    rho = torch.rand((nx + 1) * (ny + 1), generator=gen, dtype=torch.float64).cuda()
    a = gp.filter.apply(rho)
    gp.set_option("filter_dct", 0)
    return a, gp.filter.apply(rho)


# cells, eps/h: primes 349, 347, 337 and 257 of narrow columns; 37 and 53 (two direct stages) of a
# long one; 37 of a wide grid with eps below the cell size
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,ratio", [(4, 349, 1.5), (3, 347, 16.0), (5, 337, 8.0),
                                         (16, 257, 16.0), (2, 1961, 2.0), (333, 111, 0.25)])
def test_slow_direct_stages_leave_the_v_cycle(nx, ny, ratio, precision):
    a, b = filtered(nx, ny, ratio, precision)
    assert torch.equal(a, b)


# the same on the other side of the rule (37, 257, 11 and 13, 347)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,ratio", [(333, 111, 5.0), (256, 257, 50.0), (64, 143, 16.0),
                                         (66, 22, 1.0), (999, 333, 16.0)])
def test_direct_stages_where_they_pay(nx, ny, ratio, precision):
    a, b = filtered(nx, ny, ratio, precision)
    assert not torch.equal(a, b)
    # both to a relative residual of 1e-12, times the condition of mass plus stiffness, of order
    # 1 + 8 ratio^2
    assert float((a - b).norm() / b.norm()) <= 2e-12 * (1.0 + 8.0 * ratio ** 2)
