"""Axes of 4 and 8 grid points (one thread per FFT line) in every place of a grid: first,
middle and last, beside axes of other kinds (power of two, with factors 3, unlisted
length, split), forward, adjoint and node gradient against the oracle.

Tolerances: FP64 1e-12, FP32 1e-5 (as the other sizes'); the FP32 gradient against the
FP64 plan's, 1e-5.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GRIDS = [[4], [8], [8, 8], [4, 48], [36, 8], [8, 16384], [18432, 4], [8, 64, 16], [64, 8, 96],
         [32, 12, 8], [4, 8, 4]]


@pytest.mark.parametrize("n", GRIDS)
def test_short_axes(gpu, orc, n):
    N = [max(2, v // 4 * 2) for v in n]
    m, M, d = 1, 777, len(n)
    r = np.random.default_rng(sum(n))
    x = r.uniform(-0.5, 0.5, (M, d))
    Nt = int(np.prod(N))
    fh = (r.standard_normal((2, Nt)).astype(np.float32) * np.array([[1], [1j]])).sum(0)
    fv = (r.standard_normal((2, M)).astype(np.float32) * np.array([[1], [1j]])).sum(0)
    ref_f, ref_h = orc.nfft_trafo(N, n, m, x, fh), orc.nfft_adjoint(N, n, m, x, fv)
    grads = []
    for precision, ct, rt, tol in (("double", torch.complex128, torch.float64, 1e-12),
                                   ("single", torch.complex64, torch.float32, 1e-5)):
        xd = torch.from_numpy(x).cuda()
        fhd, fvd = (torch.from_numpy(v).to(ct).cuda() for v in (fh, fv))
        f, h = torch.empty_like(fvd), torch.empty_like(fhd)
        gx = torch.empty(M, d, dtype=rt, device="cuda")
        with gpu.Plan(N, M, n=n, m=m, precision=precision) as p:
            p.set_nodes_dev(xd.data_ptr())
            p.transform_dev(fhd.data_ptr(), f.data_ptr())
            p.adjoint_dev(fvd.data_ptr(), h.data_ptr())
            p.grad_x_dev(fhd.data_ptr(), fvd.data_ptr(), gx.data_ptr())
            torch.cuda.synchronize()
        ef, eh = orc.rel_l2(ref_f, f.cpu().numpy()), orc.rel_l2(ref_h, h.cpu().numpy())
        assert ef <= tol and eh <= tol, (precision, ef, eh)
        grads.append(gx.double())
    assert float((grads[0] - grads[1]).norm() / grads[0].norm()) <= 1e-5
