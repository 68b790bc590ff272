"""Node counts and tile counts at the edges of the binning's kernels.

The tiled gridding visits exactly the nodes the binning lists, so a node lost,
doubled or put in a wrong tile shows in the transform.  Each case is compared
with the untiled kernels (PLAIN_GATHER, ATOMIC_SCATTER), which use no binning:
wavefront, workgroup and block edges of the radix pass, both sides of its change
to a separate scan (65536 nodes) and of its block size (2^20), node sets that leave
almost all tiles empty (first, last, one middle tile) and more than 65536 tiles
(the chunk counts in two kernels).

Tolerance (FP64): both sides sum the same <= 10^3 products per node in another
order, and per cell as many as nodes share it: errors of a few hundred eps; 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def nodes(kind, M, d, r):
    if kind == "uniform":
        return r.uniform(-0.5, 0.5, (M, d))
    centre = {"first": 1e-3, "last": -0.07, "middle": -0.5}[kind]
    return np.clip(centre + 1e-4 * r.standard_normal((M, d)), -0.5, 0.4999)


def both(gpu, N, n, m, x, config=None):
    import torch

    M, d = x.shape
    r = np.random.default_rng(M)
    fh = torch.from_numpy(r.standard_normal((int(np.prod(N)), 2))).cuda()
    fv = torch.from_numpy(r.standard_normal((M, 2))).cuda()
    xt = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    out = []
    base = gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS
    for flags in (0, gpu.PLAIN_GATHER | gpu.ATOMIC_SCATTER):
        with gpu.Plan(N, M, n=n, m=m, flags=base | flags) as p:
            if config is not None and not flags:
                p.config = config
            f, h = torch.zeros_like(fv), torch.zeros_like(fh)
            p.set_nodes_dev(xt.data_ptr())
            p.transform_dev(fh.data_ptr(), f.data_ptr())
            p.adjoint_dev(fv.data_ptr(), h.data_ptr())
            torch.cuda.synchronize()
            out.append((f, h))
    (f, h), (f0, h0) = out
    ef, eh = float((f - f0).norm() / f0.norm()), float((h - h0).norm() / h0.norm())
    assert ef <= 1e-12 and eh <= 1e-12, (N, M, ef, eh)


@pytest.mark.parametrize("M", [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 4095, 4097, 65535,
                               65536, 65537, 262145, (1 << 20) - 1, (1 << 20) + 1])
def test_node_counts(gpu, M):
    r = np.random.default_rng(M)
    both(gpu, [60, 64], [128, 128], 2, nodes("uniform", M, 2, r))


@pytest.mark.parametrize("d", [1, 2, 3])
@pytest.mark.parametrize("kind", ["uniform", "first", "last", "middle"])
def test_node_distributions(gpu, d, kind):
    r = np.random.default_rng(d)
    n = {1: [4096], 2: [256, 512], 3: [64, 128, 64]}[d]
    both(gpu, [v // 2 for v in n], n, 3, nodes(kind, 5003, d, r))


@pytest.mark.parametrize("kind", ["uniform", "last"])
def test_many_tiles(gpu, kind):
    r = np.random.default_rng(7)
    both(gpu, [64, 2048], [8192, 4096], 1, nodes(kind, 30011, 2, r), config=1)   # 131072 tiles
