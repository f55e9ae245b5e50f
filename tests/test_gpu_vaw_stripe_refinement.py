"""Unnormalised VAW, FP32: a stripe range refines the near-duplicates among its own
pairs only.  The tiles compute whole blocks, whose pairs outside the range lack their
rare nodes' shares and must not be taken for near-duplicates.  Every pair is in one
stripe (two in the last one of an even number of samples), so over the stripes the
refined pairs add up to those of the whole matrix."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [101, 201])
def test_stripes_refine_their_own_pairs(ssu, synth, O, monkeypatch, n):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")
    monkeypatch.setenv("SSU_VAW_SPLIT", "0.6")   # some nodes dense, the shares of the others large
    tree = synth.random_tree(600, 9)
    rng = np.random.default_rng(10)
    common, rows = rng.choice(600, 40, replace=False), []   # tips held by every sample in about equal numbers
    for t in range(600):
        held = np.arange(n) if t in common else np.nonzero(rng.random(n) < 0.03)[0]
        rows.append((held, rng.integers(98, 103, held.size) if t in common else np.full(held.size, 40)))
    rows = [(("t%d" % t), h, v) for t, (h, v) in enumerate(rows) if h.size]
    obs, smp = [r[0] for r in rows], ["s%d" % s for s in range(n)]
    ip = np.cumsum([0] + [r[1].size for r in rows]).astype(np.uint32)
    ix = np.concatenate([r[1] for r in rows]).astype(np.uint32)
    data = np.concatenate([r[2] for r in rows]).astype(float)
    inp = ssu.Inputs(*tree, obs, smp, ip, ix, data)
    p = ssu.Plan(inp, "weighted_unnormalized", variance_adjust=True)
    assert 0 < p.split_theta() < 1
    got, k = 0, np.arange(n)
    ref = O.matrix(O.Tree(tree[0].astype(np.uint8), tree[1], tree[2]), O.Table(obs, smp, ip, ix, data),
                   "weighted_unnormalized", variance_adjust=True)
    for a in range(0, n // 2, 10):   # (first: nothing has been written to the outputs yet)
        b = min(a + 10, n // 2)
        p.execute_stripes(a, b)
        got += p.refined_pairs()
        want = np.stack([ref[k, (k + s + 1) % n] for s in range(a, b)])
        assert (np.abs(p.stripes(a, b) - want) <= 1e-6 * want).all()
    p.execute_stripes(0, 0)   # every pair
    assert got > 0
    print("[gpu-case] VAW stripes", n, "refined pairs", got, "whole", p.refined_pairs(), flush=True)
    assert got == p.refined_pairs()
    p.close()
