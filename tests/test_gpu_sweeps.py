"""The two forms of the stencil sweep (z-march and one-shot boxes) where their
tiles can go wrong: sides around a vector, a tile and a box, odd x-sides whose
edge tiles wrap inside a vector, the smallest grids; bit
for bit in FP64."""
import numpy as np
import pytest

from aar_hip import problems as P

pytestmark = pytest.mark.gpu

# boxes of 1, 2 and 4 planes; x-sides 1 mod 2, 1..3 mod 4, below a vector
SHAPES = [(1, 1, 1), (2, 3, 1), (3, 5, 2), (5, 4, 3), (7, 9, 13), (13, 8, 5), (63, 9, 7), (64, 8, 4), (65, 17, 9),
          (66, 33, 6), (67, 7, 21), (121, 23, 90), (127, 33, 18), (131, 99, 90), (129, 130, 131)]


def dev(v, dtype=None):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(v)).to("cuda")
    return t if dtype is None else t.to(dtype)


def matvec(x, shape, a, sigma=0.0):
    """system.c:189-205 for sides down to 1 (numpy rounds every operation, in
    that order)."""
    nx, ny, nz = shape
    w = [a * c for c in P.lap_weights(6)]
    u = x.reshape(nz, ny, nx)
    y = (u * 3) * w[0]
    for o in range(1, 7):
        nb = np.roll(u, o, 2) + np.roll(u, -o, 2)
        for axis in (1, 0):
            nb = nb + np.roll(u, o, axis)
            nb = nb + np.roll(u, -o, axis)
        y = y + nb * w[o]
    if sigma != 0.0:
        y = y + sigma * u
    return y.reshape(-1)


def _x(shape, seed=3):
    return np.random.default_rng(seed + sum(shape)).standard_normal(int(np.prod(shape)))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_boxes(gpu, shape):
    import torch
    print("boxes", shape, flush=True)
    x = _x(shape)
    y = gpu.Lap_Vec_mult(dev(x), shape, -4.0, 0.7).cpu().numpy()
    yo = matvec(x, shape, -4.0, 0.7)
    assert np.array_equal(y, yo)
    # off a 16-byte boundary
    buf = torch.zeros(x.size + 1, dtype=torch.float64, device="cuda")
    buf[1:] = dev(x)
    assert np.array_equal(gpu.Lap_Vec_mult(buf[1:], shape, -4.0, 0.7).cpu().numpy(), yo)
    # FP32: 37 terms of the difference form, each rounded: 40 eps32 of the
    # largest weight times the largest value
    x32 = dev(x, torch.float32)
    y32 = gpu.Lap_Vec_mult(x32, shape, -4.0, 0.7).double().cpu().numpy()
    yo = matvec(x32.double().cpu().numpy(), shape, -4.0, 0.7)
    assert np.max(np.abs(y32 - yo)) <= 40 * 2.0 ** -23 * 4.0 * 10.0 * np.max(np.abs(x))


@pytest.mark.parametrize("shape", [(121, 40, 36), (67, 37, 20), (66, 33, 19), (5, 6, 40)], ids=str)
@pytest.mark.parametrize("lz,wy,py", [(16, 8, 4), (5, 4, 8), (7, 8, 2), (20, 4, 4), (3, 4, 2)])
def test_march_edge_tiles(gpu, shape, lz, wy, py):
    import torch
    print("march", shape, lz, wy, py, flush=True)
    x = _x(shape, 5)
    gpu.set_tuning(lz, wy, py)
    try:
        y = gpu.Lap_Vec_mult(dev(x), shape, -16.0).cpu().numpy()
        y32 = gpu.Lap_Vec_mult(dev(x, torch.float32), shape, -16.0).double().cpu().numpy()
    finally:
        gpu.set_tuning()
    assert np.array_equal(y, matvec(x, shape, -16.0))
    yo = matvec(x.astype(np.float32).astype(np.float64), shape, -16.0)
    assert np.max(np.abs(y32 - yo)) <= 40 * 2.0 ** -23 * 16.0 * 10.0 * np.max(np.abs(x))


@pytest.mark.parametrize("shape", [(15, 13, 13), (66, 33, 19), (67, 37, 20), (121, 99, 17)], ids=str)
@pytest.mark.parametrize("march", [False, True])
def test_sweeps_of_the_solvers(gpu, oracle, shape, march):
    """A few iterations of each solver: the norms count every point once (the
    history), and the sweeps' second outputs reach the iterate.  Six steps
    amplify the rounding of the sums by far less than 1e3: 1e-12."""
    print("solvers", shape, march, flush=True)
    n = int(np.prod(shape))
    b = P.rhs_uniform(shape, 77)
    c = 1.0 + 0.5 * np.sin(np.arange(n))
    if march:
        gpu.set_tuning(9, 8, 4)
    try:
        for name, go, ref in (
                ("aar", lambda x: gpu.AAR(x, dev(b), shape, -16.0, 0.6, 0.6, 4, 3, 6, 1e-14),
                 lambda: oracle.aar(np.zeros(n), b, shape, -16.0, 0.6, 0.6, 4, 3, 6, 1e-14)),
                ("pgr", lambda x: gpu.PGR(x, dev(b), shape, -16.0, 0.6, 4, 3, 6, 1e-14),
                 lambda: oracle.pgr(np.zeros(n), b, shape, -16.0, 0.6, 4, 3, 6, 1e-14)),
                ("cg", lambda x: gpu.CG(x, dev(b), shape, -16.0, 6, 1e-14),
                 lambda: oracle.cg(np.zeros(n), b, shape, -16.0, 6, 1e-14)),
                ("pgr_vc", lambda x: gpu.PGR(x, dev(b), shape, -16.0, 0.6, 4, 3, 6, 1e-14, c=dev(c)),
                 lambda: oracle.pgr_vc(np.zeros(n), b, shape, -16.0, c, 0.6, 4, 3, 6, 1e-14)),
                ("cg_vc", lambda x: gpu.CG(x, dev(b), shape, -16.0, 6, 1e-14, c=dev(c)),
                 lambda: oracle.cg_vc(np.zeros(n), b, shape, -16.0, c, 6, 1e-14))):
            x = dev(np.zeros(n))
            go(x)
            h0 = gpu.history()[0]
            xr = ref()[0]
            assert abs(h0 - np.linalg.norm(b)) <= 1e-13 * np.linalg.norm(b), name
            assert np.linalg.norm(x.cpu().numpy() - xr) <= 1e-12 * np.linalg.norm(xr), name
    finally:
        gpu.set_tuning()
