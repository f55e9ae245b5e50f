"""PERMANOVA of more than 256 groups, whose label rows are shuffled on the host and
turned sample major on the device, 64 x 64 at a time: sample and label row counts
around 64 and labels far apart, against the restated permutations."""
import numpy as np
import pytest

from test_gpu_stats_edges import distances, first_draw, pseudo_f, shuffled

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


@pytest.mark.parametrize("n,groups,spread,perms", [(300, 257, 1, 62), (319, 300, 1, 63), (320, 290, 1, 64),
                                                   (321, 300, 1, 129), (50, 3, 200, 20), (64, 63, 5, 1)])
def test_permanova_host_labels(ssu, n, groups, spread, perms):
    d = distances(n, 6, n)
    rng = np.random.default_rng(groups)
    g = np.concatenate([np.arange(groups), rng.integers(0, groups, n)])[:n] * spread
    rng.shuffle(g)
    assert g.max() > 255
    print("[gpu-case] permanova", n, groups, spread, perms, flush=True)
    ssu.lib().ssu_set_random_seed(n + groups)
    seed = first_draw(n + groups)
    f, p = ssu.permanova(d, g, perms)
    f0 = pseudo_f(d, g)
    assert abs(f - f0) <= 1e-10 * f0
    fs = np.array([pseudo_f(d, shuffled(g, seed, q)) for q in range(1, perms + 1)])
    tie = np.abs(fs - f0) <= 1e-9 * f0
    lo, hi = ((fs >= f0) & ~tie).sum(), ((fs >= f0) | tie).sum()
    got = round(p * (perms + 1)) - 1
    assert abs(p * (perms + 1) - 1 - got) < 1e-3 and lo <= got <= hi
