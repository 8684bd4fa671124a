"""The P2 solve's iteration limit and its two solvers: PCG and the MINRES solve behind it share
max_iter, the better iterate is returned, and outer_iterations says whether MINRES ran."""

import ctypes

import numpy as np
import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density
from topomax_amd import _lib
from topomax_amd.elasticity_problem import solve_opts

pytestmark = pytest.mark.gpu


def solve(gp, xi, **opts):
    """tmx_elasticity_solve with these options: code, u, statistics, true relative residual."""
    h = gp._h
    u = torch.full((h.n_dofs,), float("nan"), dtype=torch.float64, device="cuda:0")
    st = _lib.SolveStats()
    h.stream()
    rc = h.lib.tmx_elasticity_solve(h.ptr, ctypes.c_void_p(xi.data_ptr()),
                                    ctypes.c_void_p(u.data_ptr()),
                                    ctypes.byref(solve_opts(**opts)), ctypes.byref(st))
    # b is the load on the free nodes (the operator is the identity on the fixed ones, which
    # returns their entries of a random vector unchanged)
    e = torch.randn_like(u)
    free = (gp.matvec(xi, e) != e).to(torch.float64)
    b = free * gp.load_vector()
    rel = float((b - gp.matvec(xi, u)).norm() / b.norm())
    return rc, u, st.as_dict(), rel


def definite(nx, ny):
    return torch.as_tensor(smoothed_density(nx, ny, seed=5, sigma=2.0, lo=0.1), device="cuda:0")


def indefinite(nx, ny):
    X, Y = np.meshgrid(np.linspace(0, 3, nx + 1), np.linspace(0, 1, ny + 1))
    hole = ((X - 2.0) ** 2 + (Y - 0.5) ** 2 < 0.3 ** 2).ravel()
    xi = np.where(hole, -0.1, 0.3 + 0.7 * smoothed_density(nx, ny, seed=4, sigma=2.0, lo=0.0))
    return torch.as_tensor(xi, device="cuda:0")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_iterations_stay_within_the_limit(precision):
    gp = gpu_problem(CANTILEVER, 30, 10, degree=2, precision=precision)
    gp.set_penalization(3)
    xi = definite(30, 10)
    rc, _, st, rel = solve(gp, xi, rtol=1e-10)
    assert rc == _lib.TMX_OK and st["outer_iterations"] == 1 and rel <= 1.01e-10
    full = st["iterations"]
    assert full > 4
    last = 2.0  # of the zero vector: 1
    for limit in (1, 2, full // 2, full - 1):
        rc, u, st, rel = solve(gp, xi, rtol=1e-10, max_iter=limit)
        assert rc == _lib.TMX_ERR_NOT_CONVERGED
        assert st["iterations"] <= limit and st["outer_iterations"] == 1
        assert torch.isfinite(u).all()
        # the returned iterate is the one that the statistics are of
        assert abs(rel - st["rel_residual"]) <= 1e-3 * rel + 1e-12
        if limit > 2:  # (PCG's residual norm need not fall in its first iterations)
            assert rel < last
        last = rel
    rc, _, st, rel = solve(gp, xi, rtol=1e-10, max_iter=full)
    assert rc == _lib.TMX_OK and st["iterations"] == full


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_minres_takes_over_within_the_limit(precision):
    gp = gpu_problem(CANTILEVER, 30, 10, degree=2, precision=precision)
    gp.set_penalization(3)
    xi = indefinite(30, 10)
    rc, _, st, rel = solve(gp, xi, rtol=1e-9)
    assert rc == _lib.TMX_OK and rel <= 1.01e-9
    assert st["outer_iterations"] == 2
    full = st["iterations"]
    for limit in (1, 3, full // 2):
        rc, u, st, rel = solve(gp, xi, rtol=1e-9, max_iter=limit)
        assert rc == _lib.TMX_ERR_NOT_CONVERGED and st["iterations"] <= limit
        assert torch.isfinite(u).all()
        assert abs(rel - st["rel_residual"]) <= 1e-3 * rel


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_below_the_round_off_floor_the_better_iterate_is_returned(precision):
    gp = gpu_problem(CANTILEVER, 120, 40, degree=2, precision=precision)
    gp.set_penalization(3)
    xi = torch.as_tensor(smoothed_density(120, 40, seed=1), device="cuda:0")
    rc, u, st, rel = solve(gp, xi, rtol=1e-15)
    assert rc == _lib.TMX_ERR_NOT_CONVERGED and st["outer_iterations"] == 2
    # the floor: a few rounding errors of K u against b, so the two evaluations of the residual
    # agree to its size
    assert rel <= 2.0 * st["rel_residual"] and st["rel_residual"] <= 2.0 * rel
    assert torch.isfinite(u).all()
    rc, _, st, _ = solve(gp, xi, rtol=10.0 * rel)
    assert rc == _lib.TMX_OK and st["outer_iterations"] == 1
