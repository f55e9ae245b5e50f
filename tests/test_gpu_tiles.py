"""The pair tiles over the dense nodes: sample counts at the edges of a tile
(128 x 128 pairs) and of the round of resident tiles, node counts at the edges
of an LDS stage (16 nodes) and of a part (64 nodes), every node dense, a split
that leaves few dense nodes, and embeddings in column blocks.  Against the FP64
oracle, to the tolerances of the other parity tests (FP32 1e-6, FP64 1e-11)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-6, "fp64": 1e-11}
OPS = [("weighted_normalized", {}), ("weighted_unnormalized", {}), ("weighted_normalized_fp64", {}),
       ("weighted_unnormalized_fp64", {}), ("generalized", {"alpha": 0.5}), ("generalized", {"alpha": 1.0}),
       ("generalized", {"alpha": 0.3}), ("generalized", {"alpha": 0.0}), ("generalized_fp64", {"alpha": 0.5}),
       ("generalized_fp64", {"alpha": 1.0}), ("generalized_fp64", {"alpha": 0.3})]
VAW = {"variance_adjust": True}
OPS += [(m + p, dict(VAW, **k)) for p in ("", "_fp64")
        for m, k in (("weighted_normalized", {}), ("weighted_unnormalized", {}), ("unweighted", {}),
                     ("generalized", {"alpha": 0.5}), ("generalized", {"alpha": 1.0}), ("generalized", {"alpha": 0.3}))]


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


def case(ssu, synth, O, tips, n, density, seed):
    st, le, nm = synth.random_tree(tips, seed)
    table = synth.random_table(tips, n, density, seed + 1, zipf_s=0.8)
    return ssu.Inputs(st, le, nm, *table), O.Tree(st.astype(np.uint8), le, nm), O.Table(*table)


def check(ssu, O, inp, otree, otab, name, kw):
    prec = "fp64" if name.endswith("_fp64") else "fp32"
    p = ssu.Plan(inp, name, **kw)
    p.execute()
    err = rel_err(p.matrix(), O.matrix(otree, otab, name.replace("_fp64", ""), **kw))
    print("[gpu-case]", name, kw, inp.n_samples, len(inp.obs_ids), "max rel err", err, flush=True)
    assert err <= TOL[prec]
    p.close()


@pytest.mark.parametrize("name,kw", OPS, ids=[f"{m}{'-vaw' if 'variance_adjust' in k else ''}{k.get('alpha', '')}"
                                               for m, k in OPS])
@pytest.mark.parametrize("theta", [None, "0", "0.3"])
@pytest.mark.parametrize("tips,n", [(9, 2), (12, 127), (40, 128), (41, 129), (300, 257), (700, 520), (1500, 90)])
def test_tile_edges(ssu, synth, O, monkeypatch, name, kw, theta, tips, n):
    if theta is not None:
        for v in ("SSU_SPARSE_SPLIT", "SSU_VAW_SPLIT"):
            monkeypatch.setenv(v, theta)
    check(ssu, O, *case(ssu, synth, O, tips, n, 0.25 if tips < 100 else 0.08, 17 * tips + n), name, kw)


@pytest.mark.parametrize("name,kw", [o for o in OPS if not o[0].endswith("_fp64")],
                         ids=[f"{m}{'-vaw' if 'variance_adjust' in k else ''}{k.get('alpha', '')}"
                              for m, k in OPS if not m.endswith("_fp64")])
def test_tiles_blocked_embedding(ssu, synth, O, monkeypatch, name, kw):
    # (the postings then take their values from the operand rows, which must not be scaled)
    monkeypatch.setenv("SSU_EMBED_BLOCK_SAMPLES", "128")
    check(ssu, O, *case(ssu, synth, O, 400, 300, 0.06, 5), name, kw)


@pytest.mark.parametrize("name", ["weighted_normalized", "unweighted", "weighted_normalized_fp64", "unweighted_fp64",
                                  "generalized_fp64"])
@pytest.mark.parametrize("totals", ["few", "narrow", "wide", "beyond", "with_zero"])
def test_vaw_one_sided_points(ssu, synth, O, monkeypatch, name, totals):
    """One-sided VAW sums at the distinct totals themselves (at most 64), from a
    series over totals within a factor of 2 and of 10,000, summed at every total
    beyond that, and with an empty sample's zero total: against the oracle, and
    against the sums at every total."""
    monkeypatch.setenv("SSU_VAW_SPLIT", "1")   # every node on the posting lists
    n, rng = 150, np.random.default_rng(3)
    tree = synth.random_tree(200, 21)
    obs, smp, ip, ix, data = synth.random_table(200, n, 0.15, 22)
    data = rng.integers(1, 99, data.size).astype(float)
    ix = np.asarray(ix)
    if totals == "few":
        data[:] = 1.0
    elif totals in ("wide", "beyond"):   # one sample scaled up (the FP32 names then compute in FP64 past 2^24)
        data[ix == 7] *= 3000 if totals == "wide" else 40000
    table = [obs, smp, ip, ix, data]
    if totals == "with_zero":
        data[ix == 11] = 0.0
    inp = ssu.Inputs(*tree, *table)
    tot = np.bincount(ix, data, n)
    kw = {"variance_adjust": True, "alpha": 0.4}
    p = ssu.Plan(inp, name, **kw)
    p.execute()
    m = p.matrix()
    monkeypatch.setenv("SSU_VAW_POINTS", "0")
    q = ssu.Plan(inp, name, **kw)
    q.execute()
    ref = O.matrix(O.Tree(tree[0].astype(np.uint8), *tree[1:]), O.Table(*table), name.replace("_fp64", ""), **kw)
    tol = TOL["fp64" if name.endswith("fp64") else "fp32"]
    pos = tot[tot > 0]
    assert (np.unique(tot).size <= 64) == (totals == "few")
    print("[gpu-case]", name, totals, "distinct", np.unique(tot).size, "range", pos.max() / pos.min(), "err",
          rel_err(m, ref), "against every total", rel_err(m, q.matrix()), flush=True)
    assert rel_err(m, ref) <= tol and rel_err(m, q.matrix()) <= tol
