"""The 3D matrix-core adjoint on both sides of the rule by which it takes chains of chunks
or single ones (chain_shift in bin.hpp: the chunks against the tiles, and how full they
are), on grids of 4096 tiles and more, and with fewer chunks than workgroups, about as
many, and many more (the persistent kernel's static and dynamic tickets), against the
untiled kernels (PLAIN_GATHER, ATOMIC_SCATTER).  A second call gives the same bits.

Tolerance: both sides sum the same products in another order: 1e-12 (FP64); FP32 1e-5,
with up to 20011 nodes in one tile 2e-5 (the untiled side adds them one after the other).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SETS = {
    "few": 100, "sparse": 700, "eighth": 1500, "uniform": 20011, "patch": 60011, "point": 20011,
    "one": 1,
}


def nodes(kind, r):
    x = r.uniform(-0.5, 0.5, (SETS[kind], 3))
    if kind == "patch":
        x = 0.1 * x + 0.05
    if kind == "point":
        x = 0.1234 + 1e-4 * x
    return x


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 4, 6])
@pytest.mark.parametrize("kind", SETS)
def test_rule(gpu, precision, m, kind):
    import torch

    n = [128, 128, 128] if m != 1 else [128, 192, 96]
    N = [v // 2 for v in n]
    r = np.random.default_rng(m)
    x = torch.from_numpy(nodes(kind, r)).cuda()
    M = len(x)
    dt = torch.float64 if precision == "double" else torch.float32
    f = torch.from_numpy(r.standard_normal((M, 2))).cuda().to(dt)
    out = []
    for flags in (0, gpu.PLAIN_GATHER | gpu.ATOMIC_SCATTER):
        with gpu.Plan(N, M, n=n, m=m, precision=precision,
                      flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS | flags) as p:
            h = [torch.full((int(np.prod(N)), 2), float("nan"), dtype=dt, device="cuda") for _ in range(2)]
            p.set_nodes_dev(x.data_ptr())
            for v in h:
                p.adjoint_dev(f.data_ptr(), v.data_ptr())
            torch.cuda.synchronize()
            out.append(h)
    (a, b), (ref, _) = out
    assert torch.equal(a, b)
    err = float((a - ref).norm() / ref.norm())
    assert err <= (1e-12 if precision == "double" else 2e-5 if kind == "point" else 1e-5), err
