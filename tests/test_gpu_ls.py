"""The device least-squares solve at the sizes where its instantiations end
(8, 16, 32 columns) and below, on Gram matrices like the solvers' own (well
conditioned to numerically singular), bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3, 6, 7, 8, 9, 13, 15, 16, 17, 26, 31, 32])
@pytest.mark.parametrize("decay", [1.0, 0.3, 1e-3])
def test_pinv_bitwise(gpu, oracle, m, decay):
    print("pinv", m, decay, flush=True)
    rng = np.random.default_rng(100 * m)
    F = rng.standard_normal((m, 60)) * decay ** np.arange(m)[:, None]
    A, b = F @ F.T, F @ rng.standard_normal(60)
    x, _, _ = gpu.pinv(A, b)
    xo = oracle.pinv_times_vec(A, b)
    xo = xo[0] if isinstance(xo, tuple) else xo
    assert np.array_equal(x, xo)
