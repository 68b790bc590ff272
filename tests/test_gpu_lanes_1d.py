"""The 1D gridding kernels (one wavefront per chunk; a tile in one chunk stores the cells
that are its alone and adds the others) against the untiled kernels.

Grids of 1, 2 and many 256-cell tiles, every window width, node counts on both sides of
each chunk length, and node sets that leave tiles empty, in one chunk and in many side
by side; the output buffer of the grid holds the last call's cells each time.

Tolerance: the same products in another order, as many per cell as nodes share it:
1e-12 in FP64, 1e-5 in FP32 (up to 3000 nodes in one tile).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(gpu, n, m, x, precision):
    import torch

    dt = torch.float64 if precision == "double" else torch.float32
    r = np.random.default_rng(len(x))
    fh = torch.from_numpy(r.standard_normal((n // 2, 2))).cuda().to(dt)
    fv = torch.from_numpy(r.standard_normal((len(x), 2))).cuda().to(dt)
    xt = torch.from_numpy(x).cuda()
    out = []
    for flags in (0, gpu.PLAIN_GATHER | gpu.ATOMIC_SCATTER):
        with gpu.Plan([n // 2], len(x), n=[n], m=m, precision=precision,
                      flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS | flags) as p:
            f, h = torch.zeros_like(fv), torch.zeros_like(fh)
            p.set_nodes_dev(xt.data_ptr())
            p.transform_dev(fh.data_ptr(), f.data_ptr())   # leaves its values in the grid
            p.adjoint_dev(fv.data_ptr(), h.data_ptr())
            p.adjoint_dev(fv.data_ptr(), h.data_ptr())
            torch.cuda.synchronize()
            out.append((f, h))
    tol = 1e-12 if precision == "double" else 1e-5
    for a, b in zip(*out):
        assert float((a - b).norm() / b.norm()) <= tol, (n, m, len(x))


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", range(1, 9))
@pytest.mark.parametrize("n", [256, 512, 6144])
def test_tiles(gpu, n, m, precision):
    r = np.random.default_rng(m)
    x = r.uniform(-0.5, 0.5, (700, 1))
    dense = np.clip(0.2 + r.uniform(0, 200 / n, (3000, 1)), -0.5, 0.4999)
    for v in (x, x[:1], dense, np.concatenate([x[:40], dense])):
        check(gpu, n, m, np.ascontiguousarray(v), precision)


@pytest.mark.parametrize("M", [63, 64, 65, 32768, 32769, 65536, 65537])
def test_node_counts(gpu, M):
    r = np.random.default_rng(M)
    check(gpu, 65536, 4, r.uniform(-0.5, 0.5, (M, 1)), "double")
