"""The complex sweeps where their forms change: boxes of 2 and of 4 planes at
their edges and remainders, and the march beyond them."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(12, 13, 14), (31, 15, 17), (32, 16, 18), (33, 17, 19), (64, 48, 25), (65, 80, 69),
                                   (96, 81, 66), (97, 82, 67), (128, 128, 153), (70, 200, 180)])
def test_helm_sweeps(gpu, oracle, shape):
    print("helm sweeps", shape, flush=True)
    n = int(np.prod(shape))
    u, b = P.rhs_complex_normal(shape, 5), P.rhs_complex_normal(shape, 6)
    c, a = P.helmholtz_coefficient(shape, 7), P.poisson_a(0.5)
    cd, ud = torch.from_numpy(c).cuda(), torch.from_numpy(u).cuda()
    y = gpu.helm_matvec(ud, shape, a, cd, 0.3, 0.5).cpu().numpy()
    assert np.array_equal(y, oracle.matvec_complex(u, shape, a, c, 0.3, 0.5))
    # four Richardson steps: the true residual of u, then the recurrence.  A
    # step's rounding is below 60 eps of the largest value and the damped
    # Jacobi step does not amplify it: 4 * 60 * 2.2e-16 < 1e-13
    st = gpu.helm_aar(ud, torch.from_numpy(b).cuda(), shape, a, cd, 0.3, 0.5, 0.6, 0.6, 7, 6, 4, 1e-30)
    uo, do = oracle.aar_complex(u.copy(), b, shape, a, c, 0.3, 0.5, 0.6, 0.6, 7, 6, 4, 1e-30)
    assert st["iterations"] == do["iterations"] == 4
    assert np.abs(ud.cpu().numpy() - uo).max() <= 1e-13 * np.abs(uo).max()
