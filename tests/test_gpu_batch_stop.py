"""A batch ends when its last system has stopped, whatever stopped each: the
check of the residual, the start's tolerance rule (AAR.c:76) or a least-squares
solve that does not converge (here on NaN)."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu

CYCLES = 60000


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("p", [1, 6])
def test_every_stop_is_counted(gpu, p, mixed):
    print("batch stops", p, mixed, flush=True)
    a, tol = P.poisson_a(0.5), 1e-3
    shapes = [(16, 17, 18), (13, 13, 13), (20, 14, 15), (16, 16, 16)]
    args = []
    for k, sh in enumerate(shapes):
        b = torch.from_numpy(P.rhs_uniform(sh, 60 + k)).cuda()
        args.append([torch.zeros_like(b), b, sh, a, 0.5])
    args[1][1] *= 1e6                       # tol + 1 <= tol ||b||: no iteration runs
    args[2][0][5] = float("nan")            # the Gram of the first window is NaN
    st = gpu.AAR_batch([tuple(v) for v in args], 0.6, 0.6, 7, p, CYCLES * p, tol, mixed=mixed)
    assert [s["iterations"] for s in st][1] == 0 and not bool(args[1][0].any())
    assert st[0]["converged"] and st[3]["converged"]
    assert st[2]["status"] != 0
    for k in (0, 3):
        x = torch.zeros_like(args[k][1])
        t = (gpu.AAR_mixed if mixed else gpu.AAR)(x, args[k][1], shapes[k], a, 0.6, 0.6, 7, p, CYCLES * p, tol,
                                                  sigma=0.5)
        assert t["iterations"] == st[k]["iterations"]
    # a few cycles of about 0.2 ms; a batch that misses a stop replays all of its 60000
    assert st[0]["solve_ms"] < 300
