"""FFT passes at every line length with a register-resident kernel, and beside them.

Per line length n: a 2D plan with the axis last (rows) and first (columns), the
other axis 32 points, forward and adjoint against the oracle NFFT.  The crop is
not half the line and the line count is no multiple of a workgroup's, so pruned
slices, partial workgroups and every radix sequence run.  Lengths 18, 36, 108 and
864 have no such kernel (generic pass); 8192 .. 12288 are split axes.

Tolerance: an FFT of n points carries a relative rms error of a few eps log2(n)
(eps 1.1e-16 / 6e-8, log2 <= 18), window weights and sums of as many roundings
again: below 100 eps = 1.2e-14 / 6e-6; the bounds used are 1e-13 and 1e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINES = [16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 48, 72, 96, 144, 192, 288, 384, 576, 768,
         1152, 1536, 18, 36, 108, 864]
SPLIT = [8192, 9216, 12288]


def check(gpu, orc, N, n, precision, M=300, m=2):
    r = np.random.default_rng(sum(n))
    d = len(N)
    x = r.uniform(-0.5, 0.5, (M, d))
    ct = np.complex128 if precision == "double" else np.complex64
    cr = lambda k: (r.standard_normal(k) + 1j * r.standard_normal(k)).astype(ct)   # noqa: E731
    fh, fv = cr(int(np.prod(N))), cr(M)
    with gpu.Plan(N, M, n=n, m=m, precision=precision) as p:
        p.x[:] = x
        p.f_hat[:] = fh
        p.copyDataToDevice()
        p.transform()
        p.copyDataToHost()
        f = p.f.astype(np.complex128)
        p.f[:] = fv
        p.copyDataToDeviceAd()
        p.adjoint()
        p.copyDataToHostAd()
        h = p.f_hat.astype(np.complex128)
    tol = 1e-13 if precision == "double" else 1e-5
    ef = orc.rel_l2(orc.nfft_trafo(N, n, m, x, fh.astype(np.complex128)), f)
    eh = orc.rel_l2(orc.nfft_adjoint(N, n, m, x, fv.astype(np.complex128)), h)
    assert ef <= tol and eh <= tol, (N, n, ef, eh)


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n", LINES)
def test_line_lengths_as_rows_and_columns(gpu, orc, n, precision):
    N = max(2, int(0.45 * n) // 2 * 2)
    check(gpu, orc, [14, N], [32, n], precision)
    check(gpu, orc, [N, 14], [n, 32], precision)


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n", SPLIT)
def test_split_axes(gpu, orc, n, precision):
    N = int(0.45 * n) // 2 * 2
    check(gpu, orc, [N], [n], precision)
    check(gpu, orc, [N, 14], [n, 32], precision)
    check(gpu, orc, [14, N], [32, n], precision)


@pytest.mark.parametrize("precision", ["double", "single"])
def test_batch_of_mixed_line_lengths(gpu, orc, precision):
    """Register-resident (64 .. 512, 288, 384) and generic (864) lines in one batch."""
    import torch

    from cunfft_amd.batch import Batch

    n = np.array([[64, 288], [864, 96], [512, 384], [192, 864]])
    N = (0.45 * n).astype(int) // 2 * 2
    M = [200, 333, 500, 257]
    r = np.random.default_rng(3)
    ct = np.complex128 if precision == "double" else np.complex64
    tol = 1e-13 if precision == "double" else 1e-5
    with Batch(N, M, m=2, n_rhs=2, n=n, precision=precision) as b:
        b.config = gpu.TILE_SHAPES   # node lanes: their 32^2 tiles
        keep = []
        for i in range(4):
            x = r.uniform(-0.5, 0.5, (M[i], 2))
            xt = torch.from_numpy(x).cuda()
            Nt = int(np.prod(N[i]))
            fh = (r.standard_normal((2, Nt)) + 1j * r.standard_normal((2, Nt))).astype(ct)
            fv = (r.standard_normal((2, M[i])) + 1j * r.standard_normal((2, M[i]))).astype(ct)
            b.set_nodes_dev(i, xt.data_ptr())
            fi, _, ai, _ = b.tensors(i)
            fi.copy_(torch.from_numpy(fh).cuda())
            ai.copy_(torch.from_numpy(fv).cuda())
            keep.append((x, xt, fh, fv))
        b.execute()
        torch.cuda.synchronize()
        for i in range(4):
            x, _, fh, fv = keep[i]
            _, fo, _, ho = b.tensors(i)
            for k in range(2):
                args = (N[i].tolist(), n[i].tolist(), 2, x)
                ef = orc.rel_l2(orc.nfft_trafo(*args, fh[k].astype(np.complex128)),
                                fo[k].cpu().numpy().astype(np.complex128))
                eh = orc.rel_l2(orc.nfft_adjoint(*args, fv[k].astype(np.complex128)),
                                ho[k].cpu().numpy().astype(np.complex128))
                assert ef <= tol and eh <= tol, (i, k, ef, eh)
