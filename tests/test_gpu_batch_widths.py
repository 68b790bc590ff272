"""A batch whose problems' FFT lines need workgroups of different widths in one launch (1 to
256 threads: lines of 8 to 4096 points, powers of two and with factors 3, beside a length
that runs the generic pass), in 1D, 2D and 3D, FP32 and FP64, against the oracle: FP64
1e-12, FP32 1e-5.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BATCHES = {
    1: [[256], [512], [4096], [768], [1536], [2304], [256]],
    2: [[32, 64], [4096, 32], [32, 4096], [96, 288], [1024, 96], [64, 32]],
    3: [[8, 8, 8], [64, 16, 8], [8, 24, 192], [16, 256, 8], [48, 8, 16]],
}


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("single", 1e-5)])
@pytest.mark.parametrize("d", [1, 2, 3])
def test_mixed_widths(gpu, orc, d, precision, tol):
    from cunfft_amd.batch import Batch

    n = BATCHES[d]
    N = [[v // 2 for v in row] for row in n]
    P, R, m = len(n), 2, 1
    r = np.random.default_rng(d)
    M = r.integers(100, 400, P)
    ct = torch.complex128 if precision == "double" else torch.complex64
    b = Batch(N, M, m=m, n_rhs=R, n=n, precision=precision)
    data = []
    for i in range(P):
        Nt = int(np.prod(N[i]))
        x = r.uniform(-0.5, 0.5, (M[i], d))
        c = r.standard_normal((2, R, max(Nt, M[i]))).astype(np.float32).astype(np.float64)
        fh, fv = (c[0] + 1j * c[1])[:, :Nt], (c[1] - 1j * c[0])[:, :M[i]]
        xd = torch.from_numpy(x).cuda()
        b.set_nodes_dev(i, xd.data_ptr())
        torch.cuda.synchronize()
        fhat_in, _, f_in, _ = b.tensors(i)
        fhat_in.copy_(torch.from_numpy(fh).to(ct))
        f_in.copy_(torch.from_numpy(fv).to(ct))
        data.append((x, fh, fv))
    torch.cuda.synchronize()
    for _ in range(2):     # the graph's second launch too
        b.execute()
        torch.cuda.synchronize()
    for i, (x, fh, fv) in enumerate(data):
        _, f, _, h = (t.cpu().numpy().astype(np.complex128) for t in b.tensors(i))
        for k in range(R):
            ef = orc.rel_l2(orc.nfft_trafo(N[i], n[i], m, x, fh[k]), f[k])
            eh = orc.rel_l2(orc.nfft_adjoint(N[i], n[i], m, x, fv[k]), h[k])
            assert ef <= tol and eh <= tol, (n[i], k, ef, eh)
    b.close()
