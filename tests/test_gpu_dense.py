"""The coarsest grid's inverse: on grids of at most 64 nodes (elasticity) the whole V-cycle is that
inverse, so it is held to a direct solve, at sizes around its 4 x 4 blocks and thread counts."""

import numpy as np
import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, oracle_problem

pytestmark = pytest.mark.gpu

# unknowns: 8, 12, 18, 32, 40, 64, 66, 112, 126, 128 (elasticity)
GRIDS = [(1, 1), (2, 1), (2, 2), (3, 3), (4, 3), (7, 3), (10, 2), (7, 6), (8, 6), (7, 7)]


@pytest.mark.parametrize("nx,ny", GRIDS)
def test_coarsest_inverse(nx, ny):
    gp = gpu_problem(CANTILEVER, nx, ny)
    orc = oracle_problem(CANTILEVER, nx, ny)
    gp.set_penalization(3)
    gp.set_option("filter_dct", 0)
    rng = np.random.default_rng(nx * 100 + ny)
    nv = (nx + 1) * (ny + 1)
    xi = torch.as_tensor(rng.uniform(0.7, 1.0, nv), device="cuda:0")
    # the operator itself, column by column (identity on the fixed rows)
    eye = torch.eye(2 * nv, dtype=torch.float64, device="cuda:0")
    K = torch.stack([gp.matvec(xi, e) for e in eye], dim=1).cpu().numpy()
    free = np.setdiff1d(np.arange(2 * nv), orc.fixed_dofs)
    r = np.zeros(2 * nv)
    r[free] = rng.standard_normal(free.size)
    z = gp.precondition(torch.as_tensor(r, device="cuda:0"), "elasticity", xi).cpu().numpy()
    ref = np.linalg.solve(K, r)
    # backward error of elimination without pivoting on an SPD matrix: n eps cond, with room
    tol = 10 * r.size * 1.2e-16 * np.linalg.cond(K)
    assert np.linalg.norm(z - ref) <= tol * np.linalg.norm(ref)
    rf = rng.standard_normal(nv)
    zf = gp.precondition(torch.as_tensor(rf, device="cuda:0"), "filter").cpu().numpy()
    A = orc.filter_matrix.toarray()
    ref = np.linalg.solve(A, rf)
    assert np.linalg.norm(zf - ref) <= 10 * nv * 1.2e-16 * np.linalg.cond(A) * np.linalg.norm(ref)
