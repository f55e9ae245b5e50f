"""VAW of FP64 names where some distances are small and the totals many and far apart:
their one-sided sums are taken at every total, not from a series (whose rounding a small
distance does not cancel as it cancels the sums' own).  Bit-equal to the sums at every
total, and within 1e-11 of the FP64 oracle as in the other parity tests."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


@pytest.mark.parametrize("name", ["weighted_normalized_fp64", "weighted_unnormalized_fp64", "unweighted_fp64",
                                  "generalized_fp64"])
@pytest.mark.parametrize("theta", [None, "1"])
@pytest.mark.parametrize("q", [6, 20, 28, 41, 59, 71, 96])
def test_vaw_fp64_small_distances(ssu, synth, O, monkeypatch, name, theta, q):
    if theta:
        monkeypatch.setenv("SSU_VAW_SPLIT", theta)
    rng = np.random.default_rng(q + 900)
    tips, n = int(rng.integers(2, 60)), int(rng.integers(66, 200))
    tree = synth.random_tree(tips, q)
    obs, smp, ip, ix, data = synth.random_table(tips, n, [0.05, 0.3, 0.9][q % 3], q + 1)
    data = np.array(data, float)
    assert np.unique(np.bincount(ix, data, n)).size > 64
    table = (obs, smp, ip, ix, data)

    def matrix():
        p = ssu.Plan(ssu.Inputs(*tree, *table), name, variance_adjust=True, alpha=0.5)
        p.execute()
        m = p.matrix()
        p.close()
        return m

    m = matrix()
    monkeypatch.setenv("SSU_VAW_POINTS", "0")
    assert np.array_equal(m, matrix(), equal_nan=True)
    ref = O.matrix(O.Tree(tree[0].astype(np.uint8), tree[1], tree[2]), O.Table(*table),
                   name.replace("_fp64", ""), variance_adjust=True, alpha=0.5)
    err = rel_err(m, ref)
    print("[gpu-case] VAW small distances", name, theta, tips, n, "max rel err", err, flush=True)
    assert err <= 1e-11
