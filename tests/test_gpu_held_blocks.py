"""The embedding by blocks of 16 samples that hold something below a node: every
distance the same bits as with every block written and read, at sample counts around
a block (16), a word of blocks (512) and a wave (128), with the embedding in column
blocks that do not start at a word, with explicit zeros, nodes of one and of several
children, and with other values left in the buffers by a plan before."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OPS = [("weighted_normalized", {}), ("weighted_unnormalized_fp64", {}), ("generalized", {"alpha": 0.5}),
       ("generalized_fp64", {"alpha": 0.3}), ("weighted_normalized", {"variance_adjust": True}),
       ("unweighted_fp64", {"variance_adjust": True})]


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


def tree(synth, tips, seed):
    """A random tree with every seventh closing bracket's node merged into its parent
    (three or more children) and every fifth tip below a node of its own (one child)."""
    st, le, nm = synth.random_tree(tips, seed)
    st, le, nm = list(map(bool, st)), list(le), list(nm)
    stack, match = [], {}
    for i, b in enumerate(st):
        if b:
            stack.append(i)
        else:
            match[stack.pop()] = i
    inner = [i for i in match if match[i] != i + 1 and i > 0]
    drop = {j for i in inner[::7] for j in (i, match[i])}
    out = ([], [], [])
    for i, b in enumerate(st):
        if i in drop:
            continue
        tip = b and match[i] == i + 1
        if tip and i % 5 == 0:   # (x) -> ((x))
            out[0].extend([True, True]), out[1].extend([0.25, le[i]]), out[2].extend(["", nm[i]])
        elif not b and st[i - 1] and (i - 1) % 5 == 0:
            out[0].extend([False, False]), out[1].extend([0.0, 0.0]), out[2].extend(["", ""])
        else:
            out[0].append(b), out[1].append(le[i]), out[2].append(nm[i])
    return np.array(out[0]), np.array(out[1]), out[2]


@pytest.mark.parametrize("name,kw", OPS, ids=[m + "".join(k) for m, k in OPS])
@pytest.mark.parametrize("n,block", [(15, None), (16, None), (17, None), (129, None), (512, None), (530, None),
                                     (530, "64"), (530, "448")])
def test_held_blocks(ssu, synth, monkeypatch, name, kw, n, block):
    if block:
        monkeypatch.setenv("SSU_EMBED_BLOCK_SAMPLES", block)
    for v in ("SSU_SPARSE_SPLIT", "SSU_VAW_SPLIT"):
        monkeypatch.setenv(v, "0.2")
    st, le, nm = tree(synth, 400, n)
    table = list(synth.random_table(400, n, 0.03, n + 1))
    table[4] = np.asarray(table[4], dtype=np.float64).copy()
    table[4][::11] = 0.0
    other = list(synth.random_table(400, n, 0.9, n + 2))
    dirty, inp = ssu.Inputs(st, le, nm, *other), ssu.Inputs(st, le, nm, *table)
    print("[gpu-case]", name, kw, n, block, flush=True)
    got = []
    for held in ("0", "1"):
        monkeypatch.setenv("SSU_HELD_BLOCKS", held)
        p = ssu.Plan(dirty, name, **kw)
        p.execute()
        p.close()
        p = ssu.Plan(inp, name, **kw)
        for _ in range(2):
            p.execute()
        got.append(p.matrix())
        p.close()
    assert np.array_equal(got[0], got[1], equal_nan=True)
