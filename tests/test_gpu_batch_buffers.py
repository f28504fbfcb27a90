"""The batch's buffers are one allocation of its own: a batch run again after a
larger and a smaller one, and after solves of its own, gives the same bits, and
its memory is the caller's again when it returns."""
import numpy as np
import pytest
import torch

from aar_hip import problems as P

pytestmark = pytest.mark.gpu


def run(gpu, sides, mixed, max_iter=200):
    args = []
    for k, s in enumerate(sides):
        shape = (s, s + 1, s + 2)
        b = torch.from_numpy(P.rhs_uniform(shape, 40 + k)).cuda()
        args.append((torch.zeros_like(b), b, shape, P.poisson_a(0.5), 0.5))
    st = gpu.AAR_batch(args, 0.6, 0.6, 7, 6, max_iter, 1e-8, mixed=mixed)
    return [a[0].cpu().numpy() for a in args], [t["iterations"] for t in st]


@pytest.mark.parametrize("mixed", [False, True])
def test_kept_buffers(gpu, mixed):
    print("batch buffers", mixed, flush=True)
    x0, it0 = run(gpu, [13, 24, 18], mixed)
    run(gpu, [20, 40, 33, 13, 26], not mixed)
    run(gpu, [12], mixed, 0)
    run(gpu, [14], mixed, 4)
    x1, it1 = run(gpu, [13, 24, 18], mixed)
    assert it0 == it1
    assert all(np.array_equal(a, b) for a, b in zip(x0, x1))


def test_buffers_are_given_back(gpu):
    print("batch memory", flush=True)
    run(gpu, [13], False)                       # the library's own context
    torch.cuda.synchronize()
    b = torch.zeros(96 * 97 * 98, dtype=torch.float64, device="cuda")
    args = [(torch.zeros_like(b), b + 1.0, (96, 97, 98), P.poisson_a(0.5), 0.5) for _ in range(4)]
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    gpu.AAR_batch(args, 0.6, 0.6, 7, 6, 12, 1e-8)      # 4 rings of 9 fields: 263 MB
    assert torch.cuda.mem_get_info()[0] >= before - (32 << 20)
