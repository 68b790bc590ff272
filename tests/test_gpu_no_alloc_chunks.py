"""The allocation-free adjoint where the plan's own chunks (32 to 128 nodes) need more
slots than its 64 MiB scratch holds and 256-node chunks do not: it takes those, so its
sums run in another order than the allocating adjoint's.  Against the oracle and the
allocating adjoint (both FP64, 1e-12), a second call with the same bits, and a plan that
fits with its own chunks next to it, bit for bit with the allocating adjoint.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MiB = 1 << 20
# n, m, M, tile extent, nodes per chunk of such a plan
CASES = [([64, 64, 64], 4, 40900, 8, 128), ([1024, 1024], 6, 32000, 32, 32)]


def slot_bytes(n, m, M, tile, chunk):
    cells = (tile + 2 * m + 1) ** len(n)
    return (int(np.prod([v // tile for v in n])) + -(-M // chunk)) * cells * 16


def run(gpu, N, n, m, x, f):
    M, Nt = len(x), int(np.prod(N))
    h = [torch.full((Nt,), complex("nan"), dtype=torch.complex128, device="cuda") for _ in range(3)]
    with gpu.Plan(N, M, n=n, m=m) as p:
        p.set_nodes_dev(x.data_ptr())
        p.adjoint_noalloc_dev(f.data_ptr(), h[0].data_ptr())
        p.adjoint_noalloc_dev(f.data_ptr(), h[1].data_ptr())
        p.adjoint_dev(f.data_ptr(), h[2].data_ptr())
        torch.cuda.synchronize()
    return h


@pytest.mark.parametrize("n,m,M,tile,chunk", CASES)
def test_longest_chunks(gpu, orc, n, m, M, tile, chunk):
    rest = M * (4 * 4 + 2 * 32 + 16)    # keys, descriptors, sorted coefficients
    assert slot_bytes(n, m, M, tile, chunk) + rest > 64 * MiB > slot_bytes(n, m, M, tile, 256) + rest + MiB
    N = [v // 2 for v in n]
    r = np.random.default_rng(M)
    x = r.uniform(-0.5, 0.5, (M, len(n)))
    fv = r.standard_normal(M) + 1j * r.standard_normal(M)
    xd, fd = torch.from_numpy(x).cuda(), torch.from_numpy(fv).cuda()
    a, b, ref = run(gpu, N, n, m, xd, fd)
    assert torch.equal(a, b)
    assert float((a - ref).norm() / ref.norm()) <= 1e-12
    assert orc.rel_l2(orc.nfft_adjoint(N, n, m, x, fv), a.cpu().numpy()) <= 1e-12
    few = M // 4
    a, b, ref = run(gpu, N, n, m, xd[:few].contiguous(), fd[:few].contiguous())
    assert torch.equal(a, b) and torch.equal(a, ref)
