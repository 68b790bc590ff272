"""Kaiser-Bessel plans with cut-offs m = 9 .. 16 (the untiled kernels), at oversampling 2,
9/2 and 9, where a weight's sinh(b m) / (pi m) comes close to the end of the FP32 range:
exp(b m) leaves it at m = 16, n/N = 9/2 (b m = 89.4) and m = 15, n/N = 9 (89.0), the
weight does not.  Forward and adjoint against the oracle.

The adjoint's coefficients are 1e-3 in magnitude, so its sums (at most M times the
coefficient times I0(b m)) stay in the range wherever the weights do; a plan whose own
weight sinh(b m) / (pi m) passes the range is not listed for FP32.

Tolerances: FP64 1e-12.  FP32: the weight's argument b sqrt(m^2 - s^2) <= 101 is rounded
twice (6e-8 each), so a weight, and a sum of them in 1D, is off by at most 1.2e-5; the
coefficients times the roll-off 1 / I0 (down to 1e-38) are rounded to steps of 1.4e-45,
below 1e-6 of them: 2e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(128, 256), (128, 576), (64, 576)]
CASES = [(m, N, n, p) for m in range(9, 17) for N, n in GRIDS for p in ("double", "single")
         if p == "double" or np.pi * (2 - N / n) * m < 89.4]


def test_cases_reach_past_the_range_of_exp():
    z = [np.pi * (2 - N / n) * m for m, N, n, p in CASES if p == "single"]
    assert sum(v > np.log(np.finfo(np.float32).max) for v in z) == 2


@pytest.mark.parametrize("m,N,n,precision", CASES)
def test_large_cutoffs(gpu, orc, m, N, n, precision):
    M = 700
    r = np.random.default_rng(100 * m + n)
    x = r.uniform(-0.5, 0.5, (M, 1))
    x[:200] = np.floor(x[:200] * n) / n            # the peak of the window on a grid point
    c = r.standard_normal((2, M))
    fh, fv = (c[0] + 1j * c[1])[:N], 1e-3 * (c[1] + 1j * c[0])
    if precision == "single":
        fh, fv = (v.astype(np.complex64).astype(np.complex128) for v in (fh, fv))
    with orc.window("kaiser_bessel"):
        ref_f, ref_h = orc.nfft_trafo([N], [n], m, x, fh), orc.nfft_adjoint([N], [n], m, x, fv)
    with gpu.Plan([N], M, n=[n], m=m, precision=precision,
                  flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.KAISER_BESSEL) as p:
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
    tol = 1e-12 if precision == "double" else 2e-5
    ef, eh = orc.rel_l2(ref_f, f), orc.rel_l2(ref_h, h)
    assert ef <= tol and eh <= tol, (ef, eh)
