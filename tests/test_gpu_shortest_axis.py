"""Grids whose last axis is a single tile and shorter than the pitch of a staged row
(stage_column in grid_tile.hpp): 8 columns with m = 3 in 3D, 16 with m = 6 and 7 on the
16^2 tiles in 2D, and the axes just above; forward and node gradient (both stage the
tile), adjoint, against the oracle.  FP64 1e-12, FP32 1e-5 (2e-5 for m = 7, whose
roll-off at oversampling 2 lifts the rounding of the band edge).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [([16, 24, 8], 3, 0), ([8, 8, 8], 3, 0), ([16, 16, 16], 3, 0), ([16, 32, 8], 3, 2),
         ([64, 16], 6, 1), ([32, 16], 7, 1), ([32, 32], 7, 1)]


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n,m,config", CASES)
def test_shortest_axis(gpu, orc, n, m, config, precision):
    N = [v // 2 for v in n]
    M, d, Nt = 900, len(n), int(np.prod([v // 2 for v in n]))
    r = np.random.default_rng(sum(n) + m)
    x = r.uniform(-0.5, 0.5, (M, d))
    fh = (r.standard_normal((2, Nt)).astype(np.float32) * np.array([[1], [1j]])).sum(0)
    fv = (r.standard_normal((2, M)).astype(np.float32) * np.array([[1], [1j]])).sum(0)
    ct = torch.complex128 if precision == "double" else torch.complex64
    rt = torch.float64 if precision == "double" else torch.float32
    xd = torch.from_numpy(x).cuda()
    fhd, fvd = (torch.from_numpy(v).to(ct).cuda() for v in (fh, fv))
    f, h = torch.empty_like(fvd), torch.empty_like(fhd)
    g = [torch.empty(M, d, dtype=rt, device="cuda") for _ in range(2)]
    tol = 1e-12 if precision == "double" else 2e-5 if m == 7 else 1e-5
    for k, flags in enumerate((0, gpu.PLAIN_GATHER | gpu.ATOMIC_SCATTER)):
        with gpu.Plan(N, M, n=n, m=m, precision=precision,
                      flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS | flags) as p:
            if k == 0:
                p.config = config
            p.set_nodes_dev(xd.data_ptr())
            p.transform_dev(fhd.data_ptr(), f.data_ptr())
            p.adjoint_dev(fvd.data_ptr(), h.data_ptr())
            p.grad_x_dev(fhd.data_ptr(), fvd.data_ptr(), g[k].data_ptr())
            torch.cuda.synchronize()
        if k == 0:
            ef = orc.rel_l2(orc.nfft_trafo(N, n, m, x, fh), f.cpu().numpy())
            eh = orc.rel_l2(orc.nfft_adjoint(N, n, m, x, fv), h.cpu().numpy())
            assert ef <= tol and eh <= tol, (ef, eh)
    assert float((g[0] - g[1]).norm() / g[1].norm()) <= tol
