"""cunfft_initDevicePara, cunfft_reinit and cunfft_reinitAd have cleared the
device arrays when they return: what a call on another stream copies in after
them stays.  The grid is large (512^3), so that clearing it takes longer than
the host needs to reach the copy.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["initDevicePara", "reinit", "reinitAd"])
@pytest.mark.parametrize("single", [False, True])
def test_nodes_set_after_a_reset_stay(gpu, call, single):
    torch = pytest.importorskip("torch")
    M = 1000
    x = np.random.default_rng(41).uniform(-0.5, 0.5, (M, 3))
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with gpu.Plan([64] * 3, M, n=[512] * 3, m=4, precision="single" if single else "double",
                  flags=gpu.CUFFT_INIT | gpu.CUFFT_BOTH | gpu.NO_HOST_BUFFERS) as p:
        getattr(p, call)()
        p.set_nodes_dev(xd.data_ptr(), s.cuda_stream)
        torch.cuda.synchronize()
        assert np.array_equal(np.asarray(p.copy_x_toHost()).reshape(M, 3), x)
