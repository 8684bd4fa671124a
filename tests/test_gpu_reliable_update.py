"""The reliable-update solve's replacement period: its FP32 recursion takes about as many iterations
as the mixed scheme's FP64 one, in one round, at sizes where a longer period costs several."""

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,rtol", [(60, 20, 1e-10), (333, 111, 1e-10), (1200, 400, 1e-10),
                                        (1800, 600, 1e-8), (2400, 800, 1e-8)])
def test_iterations_follow_the_mixed_scheme(nx, ny, rtol):
    xi = torch.as_tensor(smoothed_density(nx, ny, 3, sigma=max(2.0, nx / 100)), device="cuda:0")
    gp = gpu_problem(CANTILEVER, nx, ny, precision="mixed", rtol=rtol)
    gp.set_penalization(3)
    gp.forward(xi)
    mixed = gp.last_stats["iterations"]
    gp.forward(xi, precision="mixed-ru")
    st = gp.last_stats
    print(nx, ny, "mixed", mixed, "mixed-ru", st, flush=True)
    # one iteration for the replaced residuals' break in the recursion; a second round would mean
    # that the recursive residual had left the true one behind
    assert st["iterations"] <= mixed + 1 and st["outer_iterations"] == 1
