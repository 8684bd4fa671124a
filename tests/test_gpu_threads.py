"""Solves of different handles on several host threads at once, each on its own stream, against the
same solves one after the other: sizes whose V-cycle tails take 127, 94, 81 and 46 KiB of LDS."""

import threading

import pytest
import torch

from tests.cases import CANTILEVER, gpu_problem, smoothed_density

pytestmark = pytest.mark.gpu

SIZES = [(2, 999), (61, 61), (320, 160), (333, 111)]


def test_handles_on_threads_keep_their_results():
    probs, rhos, alone = [], [], []
    for k, (nx, ny) in enumerate(SIZES):
        case = dict(CANTILEVER, width=3.0, height=3.0 * ny / nx, filter_radius=6.0 / nx,
                    tractions=[{"side": "Right", "center": 1.5 * ny / nx, "length": 3.0 * ny / nx,
                                "value": (0.0, -1.0)}])
        gp = gpu_problem(case, nx, ny, rtol=1e-9)
        gp.set_penalization(3)
        rho = torch.as_tensor(smoothed_density(nx, ny, k, sigma=2.0, lo=0.1), device="cuda:0")
        probs.append(gp)
        rhos.append(rho)
        alone.append(gp.objective_and_gradient(rho)[:2])
    torch.cuda.synchronize()
    failures = []

    def run(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(25):
                    J, w, _ = probs[k].objective_and_gradient(rhos[k])
                    torch.cuda.current_stream().synchronize()
                    if J != alone[k][0] or not torch.equal(w, alone[k][1]):
                        failures.append((SIZES[k], J, alone[k][0]))
        except Exception as e:  # noqa: BLE001 (reported below, with the size)
            failures.append((SIZES[k], repr(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(SIZES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[:4]
