"""1D gridding with 64 and with 256 threads per workgroup: plans on both sides of the rule
(2048 tiles of 256 cells, 256 nodes per tile; 2^19 nodes, 2^15 per tile), tiles of one and of many chunks, and
batches with fewer chunks than the 8192 that change the width, and with 8192.

Plans against the oracle: FP64 1e-12, FP32 1e-5 as the other 1D tests.  A batch's problem
against the oracle, FP32 1e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inputs(r, N, M, single):
    c = r.standard_normal((4, max(N, M)))
    fh, fv = (c[0] + 1j * c[1])[:N], (c[2] + 1j * c[3])[:M]
    if single:
        fh, fv = (v.astype(np.complex64).astype(np.complex128) for v in (fh, fv))
    return fh, fv


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("single", 1e-5)])
@pytest.mark.parametrize("tiles,M", [(1024, 5000), (2048, 5000), (2048, 524288), (2048, 524289),
                                     (4, 20001), (1, 257), (1, 5001), (16, 524288), (16, 524287)])
def test_plan(gpu, orc, tiles, M, precision, tol):
    n, N, m = 256 * tiles, 128 * tiles, 2
    r = np.random.default_rng(tiles + M)
    x = r.uniform(-0.5, 0.5, (M, 1))
    x[:M // 4] = 0.1 + 1e-4 * x[:M // 4]     # a tile of several chunks
    fh, fv = inputs(r, N, M, precision == "single")
    with gpu.Plan([N], M, n=[n], m=m, precision=precision) as p:
        p.x[:], p.f_hat[:] = x, fh
        p.copyDataToDevice()
        p.transform()
        p.copyDataToHost()
        f = p.f.astype(np.complex128).copy()
        p.f[:] = fv
        p.copyDataToDeviceAd()
        p.adjoint()
        p.copyDataToHostAd()
        h = p.f_hat.astype(np.complex128).copy()
    ef = orc.rel_l2(orc.nfft_trafo([N], [n], m, x, fh), f)
    eh = orc.rel_l2(orc.nfft_adjoint([N], [n], m, x, fv), h)
    assert ef <= tol and eh <= tol, (ef, eh)


@pytest.mark.parametrize("short", [1, 0])
def test_batch(gpu, orc, short):
    """32 problems x 64 right-hand sides with nodes in each of 4 tiles: 8192 chunks, and two
    tiles without nodes in one problem: 128 fewer."""
    import torch

    from cunfft_amd.batch import Batch

    P, R, N, n, m = 32, 64, 512, 1024, 3
    r = np.random.default_rng(short)
    M = r.integers(150, 400, P)
    b = Batch([[N]] * P, M, m=m, n_rhs=R, n=[[n]] * P, precision="single")
    xs, fhs, fvs = [], [], []
    for i in range(P):
        x = (np.arange(M[i]) + r.uniform(0, 1, M[i]))[:, None] / M[i] - 0.5   # in every tile
        if short and i == 3:
            x *= 0.2
        fh, fv = inputs(r, N * R, int(M[i]) * R, True)
        xs.append(x), fhs.append(fh.reshape(R, N)), fvs.append(fv.reshape(R, M[i]))
        xd = torch.from_numpy(x).cuda()
        b.set_nodes_dev(i, xd.data_ptr())
        torch.cuda.synchronize()
        fhat_in, _, f_in, _ = b.tensors(i)
        fhat_in.copy_(torch.from_numpy(fhs[i]).to(torch.complex64))
        f_in.copy_(torch.from_numpy(fvs[i]).to(torch.complex64))
    torch.cuda.synchronize()
    b.execute()
    torch.cuda.synchronize()
    for i, k in ((0, 0), (3, 17), (P - 1, R - 1)):
        _, f, _, h = (t[k].cpu().numpy().astype(np.complex128) for t in b.tensors(i))
        ef = orc.rel_l2(orc.nfft_trafo([N], [n], m, xs[i], fhs[i][k]), f)
        eh = orc.rel_l2(orc.nfft_adjoint([N], [n], m, xs[i], fvs[i][k]), h)
        assert ef <= 1e-5 and eh <= 1e-5, (i, ef, eh)
    b.close()
