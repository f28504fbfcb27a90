"""Planes of more than 2^32 bytes (2^29 points FP64, 2^30 FP32), where 32-bit
byte offsets in a plane would wrap onto its first rows: the sweeps of the
operator, PGR, PL2R, CG with c(x), AAR, mixed AAR and the batch, against the
same arithmetic in plain torch.  The small shapes hold that arithmetic itself to
the sweeps that run elsewhere."""
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu

A = -4.0
WIDE = (23171, 23171, 1)           # 2^29 + 24329 points: a row and more past 4 GiB
WIDE32 = (32769, 32769, 1)         # 2^30 + 65537
SMALL = (37, 29, 1)


@pytest.fixture(autouse=True)
def give_back(gpu):
    yield
    gpu.release()
    torch.cuda.empty_cache()


def field(shape, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(shape[0] * shape[1] * shape[2], dtype=torch.float64, device="cuda", generator=g) - 0.5


def matvec(x, shape, c=None):
    """system.c:189-205, every operation rounded, in that order."""
    nx, ny, nz = shape
    w = [A * v for v in P.lap_weights(6)]
    u = x.view(nz, ny, nx)
    y = (u * 3).mul_(w[0])
    for o in range(1, 7):
        nb = torch.roll(u, o, 2).add_(torch.roll(u, -o, 2))
        for axis in (1, 0):
            nb.add_(torch.roll(u, o, axis))
            nb.add_(torch.roll(u, -o, axis))
        y.add_(nb.mul_(w[o]))
    y = y.view(-1)
    if c is not None:
        y.add_(c * x)
    return y


def diag():
    return A * 3.0 * P.lap_weights(6)[0]


def richardson(b, shape, steps, c=None):
    x = torch.zeros_like(b)
    d = diag() if c is None else diag() + c
    for _ in range(steps):
        x.add_((b - matvec(x, shape, c)).div_(d).mul_(0.6))
    return x


def rel(x, y):
    return float((x - y).norm() / y.norm())


@pytest.mark.parametrize("shape", [SMALL, WIDE], ids=str)
def test_matvec(gpu, shape):
    print("wide matvec", shape, flush=True)
    x = field(shape, 1)
    assert torch.equal(gpu.Lap_Vec_mult(x, shape, A), matvec(x, shape))


@pytest.mark.parametrize("shape", [SMALL, WIDE32], ids=str)
def test_matvec_f32(gpu, shape):
    """37 terms of the difference form, each rounded: 40 eps32 of the largest
    weight times the largest value."""
    print("wide matvec f32", shape, flush=True)
    x = field(shape, 2).float()
    y = gpu.Lap_Vec_mult(x, shape, A).double().sub_(matvec(x.double(), shape))
    assert float(y.abs().max()) <= 40 * 2.0 ** -23 * 4.0 * 10.0 * 0.5


# two Richardson steps (no projection or Anderson step before p): FP64 to the
# rounding of the points, FP32 corrections to theirs
@pytest.mark.parametrize("shape", [SMALL, WIDE], ids=str)
@pytest.mark.parametrize("solver", ["pgr", "pl2r_vc", "aar", "mixed", "batch", "batch_mixed"])
def test_steps(gpu, shape, solver):
    print("wide", solver, shape, flush=True)
    b = field(shape, 3)
    c = 1.0 + field(shape, 4) if solver.endswith("vc") else None
    x = torch.zeros_like(b)
    if solver == "pgr":
        gpu.PGR(x, b, shape, A, 0.6, 1, 6, 2, 1e-30)
    elif solver == "pl2r_vc":
        gpu.PL2R(x, b, shape, A, 0.6, 1, 6, 2, 1e-30, c=c)
    elif solver == "aar":
        gpu.AAR(x, b, shape, A, 0.6, 0.6, 1, 6, 2, 1e-30)
    elif solver == "mixed":
        gpu.AAR_mixed(x, b, shape, A, 0.6, 0.6, 1, 6, 2, 1e-30)
    else:
        b2 = field(SMALL, 5)
        x2 = torch.zeros_like(b2)
        gpu.AAR_batch([(x2, b2, SMALL, A, 0.0), (x, b, shape, A, 0.0)], 0.6, 0.6, 1, 6, 2, 1e-30,
                      mixed=solver.endswith("mixed"))
        assert rel(x2, richardson(b2, SMALL, 2)) <= 1e-6
    assert rel(x, richardson(b, shape, 2, c)) <= (1e-6 if solver.endswith("mixed") else 1e-14)


@pytest.mark.parametrize("shape", [SMALL, WIDE], ids=str)
@pytest.mark.parametrize("vc", [False, True])
def test_cg(gpu, shape, vc):
    print("wide cg", shape, vc, flush=True)
    b, c = field(shape, 6), (1.0 + field(shape, 7) if vc else None)
    x = torch.zeros_like(b)
    gpu.CG(x, b, shape, A, 2, 1e-30, c=c)
    d = diag() if c is None else diag() + c
    xr, r = torch.zeros_like(b), b.clone()
    p = r / d
    rs = float(r @ p)
    for _ in range(2):
        q = matvec(p, shape, c)
        al = rs / float(p @ q)
        xr.add_(p, alpha=al)
        r.sub_(q, alpha=al)
        s = r / d
        rs, old = float(r @ s), rs
        p = s.add_(p, alpha=rs / old)
    assert rel(x, xr) <= 1e-12        # two steps on sums of 2^29 terms in another order
