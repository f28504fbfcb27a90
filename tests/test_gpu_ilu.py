"""ILU(0) at the sides where its tiles can go wrong: a last tile of 1, 7 or 8
rows, the sides below 19 where a row's wrapped entries meet its unwrapped ones,
and unequal sides; both triangles, transposed too, real and complex.  Rows are
eliminated and solved in the oracle's order, so the results are its bits."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu

SHAPES = [(13, 13, 13), (14, 16, 13), (15, 13, 17), (16, 16, 16), (17, 17, 17), (18, 18, 18), (18, 19, 24),
          (19, 19, 19), (24, 20, 19), (25, 24, 23), (20, 33, 41), (13, 40, 13), (64, 13, 26)]


@pytest.mark.parametrize("shape", SHAPES)
def test_ilu0_tiles_bitwise(gpu, oracle, shape):
    print("ilu0", shape, flush=True)
    a, c = P.poisson_a(0.5), P.helmholtz_coefficient(shape, 7)
    r = np.random.default_rng(3).standard_normal(int(np.prod(shape)))
    F = oracle.ilu0_factor(shape, a, sigma=0.0, c=c)
    for trans in (False, True):
        z = gpu.ilu0_apply(torch.from_numpy(r).cuda(), shape, a, c=torch.from_numpy(c).cuda(), trans=trans)
        assert np.array_equal(z.cpu().numpy(), oracle.ilu0_apply(shape, F, r, trans=trans)), trans


@pytest.mark.parametrize("shape", SHAPES)
def test_helm_ilu0_tiles_bitwise(gpu, oracle, shape):
    print("helm ilu0", shape, flush=True)
    a, c0, eta = P.poisson_a(0.5), 0.3, 0.5
    c, r = P.helmholtz_coefficient(shape, 7), P.rhs_complex_normal(shape, 1007)
    F = oracle.ilu0_factor_complex(shape, a, c, c0, eta)
    for trans in (0, 1):
        z = gpu.helm_ilu0_apply(torch.from_numpy(r).cuda(), shape, a, c=torch.from_numpy(c).cuda(), c0=c0, eta=eta,
                                trans=trans)
        assert np.array_equal(z.cpu().numpy(), oracle.ilu0_apply_complex(shape, F, r, trans)), trans
