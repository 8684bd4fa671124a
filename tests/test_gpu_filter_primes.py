"""The filter's fast preconditioner as it runs by default: A' = eps^2 K plus the consistent mass
averaged over the two diagonals, and columns whose length has prime factors above 7 (direct stages
of the FFT).  Checked as in test_gpu_filter_dct.py, by applying A' to the result."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem
from tests.test_gpu_filter_dct import a_prime, tolerance

pytestmark = pytest.mark.gpu


def a_averaged(z, nx, ny, hx, hy, eps):
    """eps^2 K z + M' z, M' the mass matrices of the 'right' and the 'left' mesh averaged."""
    stiffness = a_prime(z, nx, ny, hx, hy, eps) - a_prime(z, nx, ny, hx, hy, 0.0)
    Z = z.reshape(ny + 1, nx + 1)
    out = torch.zeros_like(Z)
    c = [Z[:-1, :-1], Z[:-1, 1:], Z[1:, :-1], Z[1:, 1:]]  # the corners of each cell
    o = [out[:-1, :-1], out[:-1, 1:], out[1:, :-1], out[1:, 1:]]
    for tri in ((0, 1, 3), (0, 2, 3), (0, 1, 2), (1, 2, 3)):
        total = sum(c[k] for k in tri)
        for k in tri:
            o[k] += 0.5 * hx * hy / 24.0 * (total + c[k])
    return stiffness + out.reshape(-1)


# 2 ny = 4 * 11, 4 * 13, 2 * 37, 2 * 11 * 11, 2 * 11 * 13 (two direct stages), 2 * 311, 2 * 349
# (the largest prime in FP64), 2 * 27 * 37 (four columns a workgroup in FP32), 16 * 127 (the
# longest column with a direct stage and radix 4), 2 * 6 * 337 near the LDS limit; then radices
# 2 to 5 alone, with the longest row and the longest column
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny", [(66, 22), (150, 26), (100, 37), (90, 121), (61, 143), (40, 311),
                                   (7, 349), (9, 999), (2, 1016), (1, 2022),
                                   (60, 20), (3071, 4), (45, 15), (3, 2048)])
def test_averaged_operator(nx, ny, precision):
    gp = gpu_problem(CANTILEVER, nx, ny)
    gp.set_penalization(3)
    gen = torch.Generator(device="cpu").manual_seed(ny)
    r = torch.randn((nx + 1) * (ny + 1), generator=gen, dtype=torch.float64).cuda()
    z = gp.precondition(r, "filter", precision=precision)
    hx, hy = CANTILEVER["width"] / nx, CANTILEVER["height"] / ny
    back = a_averaged(z, nx, ny, hx, hy, CANTILEVER["filter_radius"])
    assert torch.isfinite(z).all()
    assert float((back - r).norm() / r.norm()) < tolerance(precision, ny)


@pytest.mark.parametrize("precision,nx,ny", [("fp64", 30, 353), ("fp32", 30, 457), ("fp64", 33, 11),
                                             ("fp32", 33, 11)])
def test_larger_primes_and_small_grids_keep_the_v_cycle(precision, nx, ny):
    gp = gpu_problem(CANTILEVER, nx, ny)
    gp.set_penalization(3)
    gen = torch.Generator(device="cpu").manual_seed(3)
    r = torch.randn((nx + 1) * (ny + 1), generator=gen, dtype=torch.float64).cuda()
    a = gp.precondition(r, "filter", precision=precision)
    gp.set_option("filter_dct", 0)
    assert torch.equal(a, gp.precondition(r, "filter", precision=precision))
