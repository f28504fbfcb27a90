"""The register Gram walks its points in chunks.  Where the right-hand side
sits in one chunk, that chunk carries the coefficients of the first Anderson
step: leaving it out moves the iterate by more than half, walking it twice by more
than 1% (test_a_lost_chunk_shows, on the host).  A step within 1e-3 of the oracle's
has every chunk once, in FP32 history too."""
import numpy as np
import pytest

from aar_hip import problems as P

A, OMEGA, BETA, SIGMA, M, STEP = P.poisson_a(0.5), 0.6, 0.6, 0.5, 7, 6
SHAPES = [(48, 48, 48), (64, 64, 65), (101, 99, 95), (128, 128, 129)]


def chunk_points(n, itemsize):
    """Points of a chunk (gram_blocks): the longest, from 2048 16-byte vectors
    down, with which the fullest of 512 blocks has the least to walk."""
    v = 16 // itemsize
    nq = (n * itemsize + 15) // 16
    best = None
    for ch in (2048, 1024, 512, 256):
        walk = -(-(-(-nq // ch)) // 512) * ch
        if best is None or walk < best[0]:
            best = (walk, ch * v)
    return best[1]


def rhs(shape, where, itemsize=4):
    """A few points in the middle of chunk `where` and noise a million times
    smaller everywhere."""
    n = int(np.prod(shape))
    c = chunk_points(n, itemsize)
    nch = -(-n // c)
    k = {"first": 0, "middle": nch // 2, "last": nch - 1}[where]
    lo, hi = k * c, min(n, (k + 1) * c)
    b = 1e-6 * np.random.default_rng(5).standard_normal(n)
    mid = (lo + hi) // 2
    b[mid - 3:mid + 3] += [1.0, -2.0, 3.0, -1.5, 2.5, 1.0]
    return b, lo, hi


def operator(x, shape):
    nx, ny, nz = shape
    w = [A * c for c in P.lap_weights(6)]
    u = x.reshape(nz, ny, nx)
    y = (3.0 * w[0] + SIGMA) * u
    for o in range(1, 7):
        for axis in range(3):
            y = y + w[o] * (np.roll(u, o, axis) + np.roll(u, -o, axis))
    return y.reshape(-1)


def first_step(b, shape, keep=None):
    """AAR.c up to the first Anderson step, the Gram over the points `keep`."""
    d = 3.0 * A * P.lap_weights(6)[0] + SIGMA
    xs, fs = [np.zeros_like(b)], []
    for k in range(STEP):
        fs.append((b - operator(xs[-1], shape)) / d)
        if k < STEP - 1:
            xs.append(xs[-1] + OMEGA * fs[-1])
    df = np.array([fs[k + 1] - fs[k] for k in range(STEP - 1)])
    dx = np.array([xs[k + 1] - xs[k] for k in range(STEP - 1)])
    s = slice(None) if keep is None else keep
    gamma = np.linalg.lstsq(df[:, s] @ df[:, s].T, df[:, s] @ fs[-1][s], rcond=1e-15)[0]
    return xs[-1] + BETA * fs[-1] - (dx + BETA * df).T @ gamma


@pytest.mark.parametrize("where", ["first", "middle", "last"])
@pytest.mark.parametrize("shape", SHAPES[:2], ids=str)
def test_a_lost_chunk_shows(shape, where):
    for itemsize in (4, 8):
        b, lo, hi = rhs(shape, where, itemsize)
        x = first_step(b, shape)
        keep = np.ones(b.size, bool)
        keep[lo:hi] = False
        assert np.linalg.norm(first_step(b, shape, keep) - x) > 0.5 * np.linalg.norm(x)
        twice = np.concatenate([np.arange(b.size), np.arange(lo, hi)])
        assert np.linalg.norm(first_step(b, shape, twice) - x) > 0.01 * np.linalg.norm(x)


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["first", "middle", "last"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("mixed", [False, True])
def test_gram_with_its_weight_in_one_chunk(gpu, oracle, shape, where, mixed):
    import torch
    print("gram chunk", shape, where, mixed, flush=True)
    b, _, _ = rhs(shape, where, 4 if mixed else 8)
    n = b.size
    x, bd = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.from_numpy(b).cuda()
    (gpu.AAR_mixed if mixed else gpu.AAR)(x, bd, shape, A, OMEGA, BETA, M, STEP, STEP, 1e-30, sigma=SIGMA)
    xo, _ = oracle.aar(np.zeros(n), b, shape, A, OMEGA, BETA, M, STEP, STEP, 1e-30, sigma=SIGMA)
    # FP32 history: columns of relative rounding 2^-24, coefficients conditioned by
    # the five columns (1e4 at most)
    assert np.linalg.norm(x.cpu().numpy() - xo) <= (1e-3 if mixed else 1e-9) * np.linalg.norm(xo)
