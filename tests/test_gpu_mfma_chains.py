"""The 3D matrix-core adjoint's chains (grid_mfma.hpp) against the untiled kernels
(PLAIN_GATHER, ATOMIC_SCATTER), which use no binning and no slots.

Node sets that end chains at every place: uniform, clustered, one tile with 6000 nodes
(many chunks kept in the accumulators) and a sparse set that leaves gaps in the tile
rows; tile rows of 2 to 16 tiles; every window width of the kernel (W = 4 .. 14, the
last with nodes in both plane sets), FP32 and FP64; and a grid of 16384 tiles, where
FP64 chains are four chunks long.  A second call gives the same bits.

Tolerance: both sides sum the same products in another order, as many per cell as
nodes share it, errors of a few hundred eps: 1e-12 (FP64) and, with 6000 nodes in one
tile in FP32, 1e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def nodes(kind, r):
    M = 300 if kind == "sparse" else 20011
    x = r.uniform(-0.5, 0.5, (M, 3))
    if kind == "cluster":
        x[::2] = np.clip(0.1 * r.standard_normal(x[::2].shape), -0.5, 0.4999)
    if kind == "tile":
        x[:6000] = 0.11 + 1e-3 * r.uniform(0, 1, (6000, 3))
    return x


def check(gpu, precision, n, m, x):
    import torch

    dt = torch.float64 if precision == "double" else torch.float32
    N = [v // 2 for v in n]
    xt = torch.from_numpy(x).cuda()
    fv = torch.from_numpy(np.random.default_rng(m).standard_normal((len(x), 2))).cuda().to(dt)
    out = []
    for flags in (0, gpu.PLAIN_GATHER | gpu.ATOMIC_SCATTER):
        with gpu.Plan(N, len(x), n=n, m=m, precision=precision,
                      flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS | flags) as p:
            h = [torch.full((int(np.prod(N)), 2), float("nan"), dtype=dt, device="cuda") for _ in range(2)]
            p.set_nodes_dev(xt.data_ptr())
            for v in h:
                p.adjoint_dev(fv.data_ptr(), v.data_ptr())
            torch.cuda.synchronize()
            out.append(h)
    (a, b), (ref, _) = out
    assert torch.equal(a, b)
    err = float((a - ref).norm() / ref.norm())
    assert err <= (1e-12 if precision == "double" else 1e-5), err


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", range(1, 7))
@pytest.mark.parametrize("kind", ["uniform", "cluster", "tile", "sparse"])
def test_chains(gpu, precision, m, kind):
    x = nodes(kind, np.random.default_rng(m))
    for n in ([64, 64, 64], [32, 64, 128], [32, 32, 16 if m < 4 else 32]):
        check(gpu, precision, n, m, x)


@pytest.mark.parametrize("kind", ["cluster", "tile"])
def test_chains_of_four(gpu, kind):
    check(gpu, "double", [128, 256, 256], 4, nodes(kind, np.random.default_rng(9)))
