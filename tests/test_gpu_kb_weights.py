"""Kaiser-Bessel weights where their evaluation changes branch: nodes at grid points (a
tap at |s| = m exactly, where the Taylor sum takes over), next to them, and at random,
for every cut-off m = 1 .. 8 and for oversampling 1.5 to 8, against the oracle.

Tolerances: FP64 1e-12 as the other windows' (W^2 <= 324 products and the FFT at
2.2e-16 each, a few hundred eps).  FP32: the weight's argument b sqrt(m^2 - s^2) <= 50
is rounded twice (6e-8 each), so a weight is off by up to 50 x 1.2e-7 = 6e-6 and a
product of two by 1.2e-5; the sum of many is below its worst term: 2e-5.
The window is not normalised, sinh(b m) / (pi m) at its peak: FP32 sums past 3e38 are
infinite, so a case whose two peaks times the node count reach that is left out
(m = 8 at oversampling 4 and 8).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("single", 2e-5)])
@pytest.mark.parametrize("m", range(1, 9))
@pytest.mark.parametrize("N,n", [([32, 32], [64, 64]), ([64, 32], [96, 96]), ([16, 8], [64, 64])])
def test_kb_weights(gpu, orc, m, precision, tol, N, n):
    M = 1500
    peak = np.prod([np.sinh(np.pi * (2 - a / b) * m) / (np.pi * m) for a, b in zip(N, n)])
    if precision == "single" and peak * M > 3e38:
        pytest.skip("the sums leave the FP32 range")
    r = np.random.default_rng(m)
    x = r.uniform(-0.5, 0.5, (M, 2))
    k = np.floor(x[:1000] * n)
    x[:1000] = k / n                                        # s is a whole number on both axes
    x[500:1000] += r.choice([-1, 1], (500, 2)) * 10.0 ** r.uniform(-9, -2, (500, 2)) / n
    x = np.clip(x, -0.5, 0.4999)
    c = r.standard_normal((2, max(M, N[0] * N[1])))
    fh, fv = (c[0] + 1j * c[1])[:N[0] * N[1]], (c[1] + 1j * c[0])[:M]
    if precision == "single":
        fh, fv = (v.astype(np.complex64).astype(np.complex128) for v in (fh, fv))
    with orc.window("kaiser_bessel"):
        ref_f, ref_h = orc.nfft_trafo(N, n, m, x, fh), orc.nfft_adjoint(N, n, m, x, fv)
    with gpu.Plan(N, M, n=n, m=m, precision=precision,
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
    ef, eh = orc.rel_l2(ref_f, f), orc.rel_l2(ref_h, h)
    assert ef <= tol and eh <= tol, (ef, eh)
