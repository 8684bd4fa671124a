"""The one-workgroup bottom of the V-cycle against the launch-per-step V-cycle, at the sizes where
its thread and LDS layout changes: one or two nodes per thread on the top level, the largest level
it takes, one-cell-wide grids (whose levels shrink in one direction only), odd and even counts."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density

pytestmark = pytest.mark.gpu

# cells of the finest grid and what the tail's top level is
SHAPES = [
    (45, 15),    # 24 x 9 nodes: one node per thread
    (125, 15),   # 64 x 9 = 576: a second node for some threads
    (61, 61),    # 32 x 32 = 1024: two nodes for every thread
    (63, 61),    # 33 x 32 = 1056: too many, the level below is the top
    (2, 999),    # 2 x 501 = 1002 over 2 x 251
    (2, 1021),   # 2 x 512 = 1024 over 2 x 257 = 514 nodes: too many there
    (999, 2),
    (1, 300),    # never coarsened in x
    (333, 111),
]


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("sweeps", [1, 3, 4])
def test_tail_equals_launch_per_step(nx, ny, sweeps):
    gp = gpu_problem(CANTILEVER, nx, ny)
    gp.set_penalization(3)
    gp.set_option("filter_dct", 0)
    gp.set_option("nu_coarse", sweeps)
    gp.set_option("nu_coarse_filter", sweeps)
    gp.set_option("band", 0)
    xi = torch.as_tensor(smoothed_density(nx, ny, 5, sigma=2.0), device="cuda:0")
    gen = torch.Generator(device="cpu").manual_seed(5)
    nv = (nx + 1) * (ny + 1)
    r = torch.randn(2 * nv, generator=gen, dtype=torch.float64).cuda()
    rf = torch.randn(nv, generator=gen, dtype=torch.float64).cuda()
    # about 100 rounding steps, amplified by no more than the condition of the level operators
    # (of order n^2); FP32 on the square-ish grids only, at the bound of FP32 against FP64
    tol = {"fp64": 100 * 1.2e-16 * max(nx, ny) ** 2, "fp32": 1e-4}
    for precision in ("fp64", "fp32"):
        if precision == "fp32" and max(nx, ny) > 200:
            continue
        out = []
        for tail in (0, 1):
            gp.set_option("tail", tail)
            out.append((gp.precondition(r, "elasticity", xi, precision=precision),
                        gp.precondition(rf, "filter", precision=precision)))
        for a, b in zip(*out):
            assert torch.isfinite(b).all()
            assert float((a - b).norm() / a.norm()) <= tol[precision]


# finest grids whose nested levels end in the tail: its top is an element level with explicit
# rows (25 x 9, 33 x 31 and 31 x 33 nodes), or the level below it is already the coarsest
NESTED = [(48, 16), (64, 60), (60, 64), (32, 8)]


@pytest.mark.parametrize("nx,ny", NESTED)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tail_takes_element_levels(nx, ny, precision):
    gp = gpu_problem(CANTILEVER, nx, ny)
    gp.set_penalization(3)
    xi = torch.as_tensor(smoothed_density(nx, ny, 6, sigma=2.0), device="cuda:0")
    gen = torch.Generator(device="cpu").manual_seed(6)
    r = torch.randn(2 * (nx + 1) * (ny + 1), generator=gen, dtype=torch.float64).cuda()
    out = []
    for tail in (0, 1):  # 0: the element level's own sweeps from its cell weights
        gp.set_option("tail", tail)
        out.append(gp.precondition(r, "elasticity", xi, precision=precision))
    tol = {"fp64": 100 * 1.2e-16 * max(nx, ny) ** 2, "fp32": 1e-4}[precision]
    assert float((out[0] - out[1]).norm() / out[0].norm()) <= tol
