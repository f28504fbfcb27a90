"""The batch's buffers are one allocation, kept up to a bound: a batch run again
after a larger and a smaller one, and after solves of its own, gives the same
bits."""
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


def free_memory():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def batch(gpu, side, count):
    b = torch.ones(side ** 3, dtype=torch.float64, device="cuda")
    args = [(torch.zeros_like(b), b, (side, side, side), P.poisson_a(0.5), 0.5) for _ in range(count)]
    before = free_memory()
    gpu.AAR_batch(args, 0.6, 0.6, 7, 6, 12, 1e-8)
    return before


def test_what_is_kept_and_given_back(gpu):
    """Above 1 GiB nothing is kept; below, the block goes when another allocation
    of the library finds no memory, and with release()."""
    print("batch memory", flush=True)
    run(gpu, [13], False)                       # the library's own context
    gpu.release()
    slack = 32 << 20
    before = batch(gpu, 128, 9)                 # 9 rings of 9 fields and 2 more each: 1.6 GB
    assert free_memory() >= before - slack
    before = batch(gpu, 96, 8)                  # 0.6 GB
    assert before - (1 << 30) <= free_memory() <= before - (400 << 20)
    # a history of 34 fields of 17 GB: more than any card holds, refused by the host
    x = torch.empty(1290 ** 3, dtype=torch.float64, device="cuda")
    b = torch.empty_like(x)
    with pytest.raises(Exception, match="memory"):
        gpu.AAR(x, b, (1290, 1290, 1290), P.poisson_a(0.5), 0.6, 0.6, 32, 6, 12, 1e-8)
    del x, b
    torch.cuda.empty_cache()
    assert free_memory() >= before - slack
    before = batch(gpu, 96, 8)
    gpu.release()
    assert free_memory() >= before - slack
    run(gpu, [14], False)                       # nothing left over from the refusal
