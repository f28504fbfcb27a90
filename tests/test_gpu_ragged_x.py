"""Sweeps on x-sides that are not a multiple of a 16-byte vector: tiles that start
early so that no vector wraps inside (sides from a tile and its halo up), the
tile before the last one where its halo would, and narrower grids, in FP32 vectors
of two parts, else point by point.
Every point is written, and the norms count it once."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P
from test_gpu_sweeps import dev, matvec

pytestmark = pytest.mark.gpu

# around 32 + 6 and 64 + 6 (FP64 boxes and march), 64 + 8 (FP32), and every
# distance of the last tile's end from nx at which the tile before it moves
SIDES = [1, 3, 5, 6, 7, 9, 37, 39, 62, 65, 67, 69, 70, 71, 73, 74, 75, 77, 97, 99, 101, 103, 129, 130, 131, 133, 135, 137, 193, 195, 199]
# boxes of 1, 2 and 4 planes, and the march
FORMS = [((9, 7), None), ((40, 60), None), ((70, 90), None), ((35, 19), (9, 8, 4)), ((18, 19), (5, 4, 4))]


@pytest.mark.parametrize("nx", SIDES)
def test_operator(gpu, nx):
    for (ny, nz), tune in FORMS:
        shape = (nx, ny, nz)
        print("ragged x", shape, tune, flush=True)
        x = np.random.default_rng(nx).standard_normal(nx * ny * nz)
        if tune:
            gpu.set_tuning(*tune)
        try:
            y = gpu.Lap_Vec_mult(dev(x), shape, -4.0, 0.7).cpu().numpy()
            y32 = gpu.Lap_Vec_mult(dev(x, torch.float32), shape, -4.0, 0.7).double().cpu().numpy()
        finally:
            gpu.set_tuning()
        assert np.array_equal(y, matvec(x, shape, -4.0, 0.7))
        # 37 terms of the difference form, each rounded
        yo = matvec(x.astype(np.float32).astype(np.float64), shape, -4.0, 0.7)
        assert np.max(np.abs(y32 - yo)) <= 40 * 2.0 ** -23 * 4.0 * 10.0 * np.max(np.abs(x))


@pytest.mark.parametrize("nx", [5, 7, 37, 66, 69, 73, 74, 75, 99, 130, 133, 135, 199])
@pytest.mark.parametrize("form", range(len(FORMS)))
def test_recurrence_and_norms(gpu, oracle, nx, form):
    """Six iterations with two Anderson steps of AAR, constant coefficient and
    c(x).  FP64 to 1e-12 (rounding, amplified by far less than 1e3); FP32
    corrections of relative rounding 2^-24 each, summed over the six with signs and
    the steps' coefficients of a few: 2e-6.  The recorded norms likewise, with c(x)
    to the hardware reciprocal of its diagonal (2^-24); a column of points lost or
    taken twice moves them by 1/(2 nx)."""
    (ny, nz), tune = FORMS[form]
    shape, a = (nx, ny, nz), -16.0
    print("ragged x solvers", shape, tune, flush=True)
    n = nx * ny * nz
    b = P.rhs_normal(shape, 21)
    c = 1.0 + 0.5 * np.sin(np.arange(n) * 0.01)
    args = (0.6, 0.6, 4, 3, 6, 1e-14)
    xr, dr = oracle.aar(np.zeros(n), b, shape, a, *args, sigma=0.5)
    xv, dv = oracle.aar_vc(np.zeros(n), b, shape, a, c, *args)
    if tune:
        gpu.set_tuning(*tune)
    try:
        for mixed, tol in ((False, 1e-12), (True, 2e-6)):
            for ref, d, rec, go in ((xr, dr, 10 * tol, lambda x: (gpu.AAR_mixed if mixed else gpu.AAR)(x, dev(b), shape, a, *args,
                                                                                             sigma=0.5)),
                               (xv, dv, 10 * tol + 1e-7,
                                lambda x: gpu.AAR_vc(x, dev(b), shape, a, dev(c), *args, mixed=mixed))):
                x = dev(np.zeros(n))
                go(x)
                assert np.linalg.norm(x.cpu().numpy() - ref) <= tol * np.linalg.norm(ref)
                h, t = gpu.history(), d["trace"]
                assert len(h) == len(t) and np.all(np.abs(h - t) <= rec * t[0])
    finally:
        gpu.set_tuning()
