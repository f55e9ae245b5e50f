"""VAW plans of more than 524,287 nodes, few of them dense: their dense list (built
with the plan, 4 bytes an entry) is smaller than one of all nodes by more than the
2 MiB granularity of device blocks.  Against the FP64 oracle, to 1e-6 as in the
other parity tests of FP32 names."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TIPS, SAMPLES, DENSE_TIPS = 262200, 8, 500


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


@pytest.fixture(scope="module")
def large(synth):
    tree = synth.random_tree(TIPS, 11)
    rng = np.random.default_rng(12)
    first = rng.integers(0, SAMPLES, TIPS)
    indptr, indices = [0], []
    for t in range(TIPS):
        indices += range(SAMPLES) if t < DENSE_TIPS else [first[t]]
        indptr.append(len(indices))
    data = rng.integers(1, 40, len(indices)).astype(float)   # (totals below 2^24)
    return tree, (["t%d" % t for t in range(TIPS)], ["s%d" % s for s in range(SAMPLES)],
                  np.array(indptr, np.uint32), np.array(indices, np.uint32), data)


def test_vaw_list_outlives_the_execution(ssu, O, monkeypatch, large):
    tree, table = large
    name = "weighted_normalized"
    monkeypatch.setenv("SSU_VAW_SPLIT", "0.99")   # dense: held by every sample
    print("[gpu-case] VAW", name, "nodes", 2 * TIPS - 2, flush=True)
    p = ssu.Plan(ssu.Inputs(*tree, *table), name, variance_adjust=True)
    ref = O.matrix(O.Tree(tree[0].astype(np.uint8), tree[1], tree[2]), O.Table(*table), name, variance_adjust=True)
    for _ in range(2):
        p.execute()
        terms = p.kernel_terms()
        assert 0 < terms < 64 * 64 * 100000   # one tile, the dense nodes only
        err = rel_err(p.matrix(), ref)
        print("[gpu-case] dense nodes", terms // 4096, "max rel err", err, flush=True)
        assert err <= 1e-6
    p.close()
