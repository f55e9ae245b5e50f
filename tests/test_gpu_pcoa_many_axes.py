"""PCoA of more axes than a launch has rows of blocks (65,535): the leading ones give
the distances back as they do alone, those past the samples are 0."""
import numpy as np
import pytest

from test_gpu_stats_edges import distances

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dims", [(5, 65536), (5, 70001), (3, 1048561)])
def test_pcoa_many_axes(ssu, n, dims):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")
    d = distances(n, n - 1, 7)
    b = -0.5 * d * d
    b = b - b.mean(0) - b.mean(1)[:, None] + b.mean()
    w = np.sort(np.linalg.eigvalsh(b))[::-1]
    print("[gpu-case] pcoa", n, dims, flush=True)
    ssu.lib().ssu_set_random_seed(5)
    e, s, prop = ssu.pcoa(d, dims)
    tol = 1e-11 * 4 * n * (d * d).max()   # (as for few axes)
    assert s.shape == (n, dims) and np.abs(e[:n] - w).max() <= n * tol
    assert np.abs(s[:, :n] @ s[:, :n].T - b).max() <= n * tol
    assert not e[n:].any() and not s[:, n:].any() and not prop[n:].any()
