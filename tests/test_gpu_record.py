"""The residual record of the sweeps between two checks: cycles shorter than,
equal to and longer than the sets of partials kept, ending on a check or not."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,its", [(1, 5), (2, 9), (6, 24), (63, 64), (64, 130), (65, 131), (66, 70), (150, 149)])
@pytest.mark.parametrize("solver", ["aar", "pgr", "helm"])
def test_record(gpu, oracle, solver, p, its):
    print("record", solver, p, its, flush=True)
    shape, a, m = (13, 15, 14), P.poisson_a(0.5), 3
    n = int(np.prod(shape))
    if solver == "helm":
        b, c = P.rhs_complex_normal(shape, 3), P.helmholtz_coefficient(shape, 7)
        x = torch.zeros(n, dtype=torch.complex128, device="cuda")
        st = gpu.helm_aar(x, torch.from_numpy(b).cuda(), shape, a, torch.from_numpy(c).cuda(), 0.3, 0.5, 0.6, 0.6, m, p,
                          its, 1e-30)
        _, d = oracle.aar_complex(np.zeros_like(b), b, shape, a, c, 0.3, 0.5, 0.6, 0.6, m, p, its, 1e-30)
    else:
        b = np.random.default_rng(9).standard_normal(n)
        x, bd = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.from_numpy(b).cuda()
        if solver == "aar":
            st = gpu.AAR(x, bd, shape, a, 0.6, 0.6, m, p, its, 1e-30, sigma=0.5)
            _, d = oracle.aar(np.zeros(n), b, shape, a, 0.6, 0.6, m, p, its, 1e-30, sigma=0.5)
        else:
            st = gpu.PGR(x, bd, shape, a, 0.6, m, p, its, 1e-30, sigma=0.5)
            _, d = oracle.pgr(np.zeros(n), b, shape, a, 0.6, m, p, its, 1e-30, sigma=0.5)
    h, tr = gpu.history(), d["trace"]
    assert st["iterations"] == d["iterations"] and len(h) == len(tr)
    # a recorded norm may miss by the rounding of a few hundred sweeps against
    # the largest one: 1e3 * 37 eps < 1e-11 of it (three columns: the
    # least-squares step adds nothing of that size)
    assert np.all(np.abs(h - tr) <= 1e-11 * tr.max() + 1e-6 * tr)
