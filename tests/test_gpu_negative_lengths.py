"""Trees with negative branch lengths (neighbour joining gives them): every method
against the FP64 oracle, whose terms carry the sign.  One length in 25 is negative
and a tenth as long.  Tolerances: those of the other parity tests (FP32 1e-6, FP64
1e-11) of the sums of the terms' magnitudes, which bound the rounding errors; here
they are within 5% of the sums themselves (KAPPA)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

KAPPA = 1.05
TOL = {"fp32": 1e-6 * KAPPA ** 2, "fp64": 1e-11 * KAPPA ** 2}   # (numerator and denominator)
METHODS = ["weighted_normalized", "weighted_unnormalized", "generalized", "unweighted", "unweighted_unnormalized"]


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


def negative_case(synth, tips, n, density, seed):
    st, le, nm = synth.random_tree(tips, seed)
    rng = np.random.default_rng(seed + 2)
    pos = np.nonzero(le > 0)[0]
    le = le.copy()
    le[rng.choice(pos, max(1, pos.size // 25), replace=False)] *= -0.1
    return (st, le, nm), synth.random_table(tips, n, density, seed + 1, zipf_s=0.8)


def oracle_matrix(O, tree, table, name, **kw):
    return O.matrix(O.Tree(np.asarray(tree[0], np.uint8), tree[1], tree[2]), O.Table(*table),
                    name.replace("_fp64", ""), **kw)


def check(name, m, ref):
    err = rel_err(m, ref)
    print("[gpu-case] negative lengths", name, m.shape, "max rel err", err, flush=True)
    assert err <= TOL["fp64" if name.endswith("_fp64") else "fp32"]


CASES = [(m + p, kw) for m in METHODS for p in ("", "_fp64")
         for kw in ({}, {"variance_adjust": True}, {"normalize": False})]


@pytest.mark.parametrize("name,kw", CASES, ids=["-".join([m, *k]) for m, k in CASES])
@pytest.mark.parametrize("tips,n", [(60, 20), (700, 131), (2500, 300)])
def test_negative_lengths(ssu, synth, O, name, kw, tips, n):
    tree, table = negative_case(synth, tips, n, 0.25 if tips < 100 else 0.08, tips + n)
    kw = dict(kw, alpha=0.4)
    ref = oracle_matrix(O, tree, table, name, **kw)
    mag = oracle_matrix(O, (tree[0], np.abs(tree[1]), tree[2]), table, "weighted_unnormalized")
    own = oracle_matrix(O, tree, table, "weighted_unnormalized")
    off = ~np.eye(n, dtype=bool)
    assert (mag[off] <= KAPPA * own[off]).all()
    s, m = ssu.matrix_inmem(ssu.Inputs(*tree, *table), name, **kw)
    assert s == ssu.OKAY, ssu.last_error()
    check(name, m, ref)


@pytest.mark.parametrize("name", ["weighted_normalized", "weighted_unnormalized", "weighted_normalized_fp64",
                                  "generalized"])
@pytest.mark.parametrize("block", [None, "128"])
def test_negative_lengths_stripes_and_blocks(ssu, synth, O, monkeypatch, name, block):
    """A stripe range of a plan, and embeddings in column blocks."""
    if block:
        monkeypatch.setenv("SSU_EMBED_BLOCK_SAMPLES", block)
    n = 300
    tree, table = negative_case(synth, 900, n, 0.08, 5)
    ref = oracle_matrix(O, tree, table, name, alpha=0.4)
    p = ssu.Plan(ssu.Inputs(*tree, *table), name, alpha=0.4)
    p.execute()
    check(name, p.matrix(), ref)
    p.execute_stripes(3, 40)
    k = np.arange(n)
    check(name, p.stripes(3, 40), np.stack([ref[k, (k + s + 1) % n] for s in range(3, 40)]))
    p.close()


def test_negative_lengths_rarefied(ssu, synth, O):
    """Replicates of a rarefaction: each against the oracle on its drawn counts."""
    names = ["weighted_normalized", "weighted_unnormalized"]
    tree, table = negative_case(synth, 500, 90, 0.15, 8)
    b = ssu.Rarefaction(ssu.Inputs(*tree, *table), names, 100, 2, seed=3)
    b.execute()
    samples, rows, ip, ix = b.kept()
    for rep in range(2):
        counts = b.counts(rep)
        ids, ptr, held = [], [0], counts > 0   # entries and rows without counts dropped
        for i in range(len(rows)):
            if held[ip[i]:ip[i + 1]].any():
                ids.append(table[0][rows[i]])
                ptr.append(ptr[-1] + int(held[ip[i]:ip[i + 1]].sum()))
        drawn = (ids, [table[1][s] for s in samples], np.array(ptr, np.uint32), ix[held], counts[held])
        for k, name in enumerate(names):
            check(name, b.matrix(k, rep), oracle_matrix(O, tree, drawn, name))
    b.close()


@pytest.mark.parametrize("theta", ["0", "0.3", "1"])
@pytest.mark.parametrize("name", ["weighted_normalized", "weighted_unnormalized", "generalized",
                                  "weighted_normalized_fp64", "weighted_unnormalized_fp64", "generalized_fp64"])
def test_negative_lengths_split(ssu, synth, O, monkeypatch, theta, name):
    """Nodes of negative length stay on the tiles at any threshold of the split."""
    monkeypatch.setenv("SSU_SPARSE_SPLIT", theta)
    tree, table = negative_case(synth, 900, 200, 0.08, 6)
    p = ssu.Plan(ssu.Inputs(*tree, *table), name, alpha=0.4)
    p.execute()
    check(name, p.matrix(), oracle_matrix(O, tree, table, name, alpha=0.4))
    assert (p.sparse_terms() > 0) == (theta != "0")
    p.close()


@pytest.mark.parametrize("name,tol", [("weighted_unnormalized", 1e-6), ("weighted_unnormalized_fp64", 1e-11)])
def test_negative_length_larger_than_the_rest(ssu, synth, O, monkeypatch, name, tol):
    """A tip that holds half of every sample, with a negative length that takes away
    most of the samples' sums (which then bound no sum of the other nodes) and
    leaves the distances alone.  Rounding errors against the terms' magnitudes."""
    monkeypatch.setenv("SSU_SPARSE_SPLIT", "1")   # every other node on the posting lists
    (st, le, nm), (obs, smp, ip, ix, data) = synth.random_tree(400, 3), synth.random_table(400, 90, 0.1, 4)
    tot = np.bincount(ix, data, 90)
    one = oracle_matrix(O, (st, le, nm), (obs, smp, ip, ix, data), "weighted_unnormalized")
    with np.errstate(invalid="ignore"):
        pair = one / oracle_matrix(O, (st, le, nm), (obs, smp, ip, ix, data), "weighted_normalized")   # S_i + S_j
    i, j, k = (np.arange(90) + s for s in range(3))
    sums = (pair[i % 90, j % 90] + pair[i % 90, k % 90] - pair[j % 90, k % 90]) / 2
    st = np.concatenate([[True], st, [True, False, False]])
    le = np.concatenate([[0.0], le, [-0.95 * sums.min(), 0.0, 0.0]])
    nm = [""] + list(nm) + ["half", "", ""]
    table = (list(obs) + ["half"], smp, np.concatenate([ip, [ip[-1] + 90]]), np.concatenate([ix, np.arange(90)]),
             np.concatenate([data, tot]))
    ref = oracle_matrix(O, (st, le, nm), table, "weighted_unnormalized")
    assert np.abs(ref - one / 2).max() < 1e-12
    p = ssu.Plan(ssu.Inputs(st, le, nm, *table), name)
    p.execute()
    err = np.abs(p.matrix() - ref).max() / one.max()
    print("[gpu-case] negative tip", name, "max err of the magnitudes", err, flush=True)
    assert err <= tol
    p.close()
