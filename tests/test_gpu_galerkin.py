"""The Galerkin operators of the 9-point levels: with a vanishing smoothing step the V-cycle is
P A_c^-1 P' alone, with A_c = P' K P the coarsest operator after one or more products, and is
held to the same product formed with numpy.

Sides: odd and even, ending with a half-width coarse cell or not, one and two cells wide."""

import numpy as np
import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem

pytestmark = pytest.mark.gpu

# one product to the coarsest grid (at most 64 nodes), then two and three
GRIDS = [(9, 7), (13, 9), (14, 9), (9, 14), (1, 40), (41, 1), (2, 33), (3, 31), (45, 15), (63, 23), (29, 21), (41, 33), (33, 65)]


def interpolation(n, nc, finest):
    """Cells are paired from the near and the far side on alternate levels."""
    if n > 1 and n % 2 and ((n - 1).bit_length() - (finest - 1).bit_length()) % 2:
        return interpolation(n, nc, n)[::-1, ::-1]
    p = np.zeros((n + 1, nc + 1))
    for f in range(n + 1):
        if n == nc:
            p[f, f] = 1.0
        elif f % 2 == 0:
            p[f, f // 2] = 1.0
        elif f == n:
            p[f, nc] = 1.0
        else:
            p[f, f // 2] = p[f, f // 2 + 1] = 0.5
    return p


@pytest.mark.parametrize("nx,ny", GRIDS)
@pytest.mark.parametrize("fixed", [["Left"], ["Right", "Bottom"]], ids=["left", "right-bottom"])
def test_galerkin_products(nx, ny, fixed):
    gp = gpu_problem(dict(CANTILEVER, fixed_sides=fixed), nx, ny)
    gp.set_penalization(3)
    gp.set_option("cheb_elast", 0)
    gp.set_option("omega_elast", 1e-14)
    rng = np.random.default_rng(nx * 100 + ny)
    nv = (nx + 1) * (ny + 1)
    xi = torch.as_tensor(rng.uniform(0.7, 1.0, nv), device="cuda:0")
    A = np.zeros((2 * nv, 2 * nv))
    for j in range(2 * nv):
        e = torch.zeros(2 * nv, dtype=torch.float64, device="cuda:0")
        e[j] = 1.0
        A[:, j] = gp.matvec(xi, e).cpu().numpy()

    def free(cx, cy):
        m = np.ones((cy + 1, cx + 1))
        if "Left" in fixed:
            m[:, 0] = 0
        if "Right" in fixed:
            m[:, -1] = 0
        if "Bottom" in fixed:
            m[0] = 0
        return np.repeat(m.ravel(), 2)

    r = rng.standard_normal(2 * nv) * free(nx, ny)
    P = np.diag(free(nx, ny))
    cx, cy = nx, ny
    while (cx + 1) * (cy + 1) > 64:
        mx, my = (cx + 1) // 2, (cy + 1) // 2
        I = np.kron(np.kron(interpolation(cy, my, ny), interpolation(cx, mx, nx)), np.eye(2))
        P = (P @ I) * free(mx, my)
        cx, cy = mx, my
    keep = free(cx, cy) > 0
    P = P[:, keep]
    Ac = P.T @ A @ P
    ref = P @ np.linalg.solve(Ac, P.T @ r)
    z = gp.precondition(torch.as_tensor(r, device="cuda:0"), "elasticity", xi).cpu().numpy()
    err = np.linalg.norm(z - ref) / np.linalg.norm(ref)
    print(nx, ny, fixed, err, flush=True)
    # backward error of the coarsest inverse; the sweeps add 1e-14 times D^-1 r each
    assert err <= 1e-11 + 10 * Ac.shape[0] * 1.2e-16 * np.linalg.cond(Ac)
