"""The int8 Gram of unweighted UniFrac at the edges of its tiles (128 samples) and
stages (128 columns; a launch keeps three in flight), with few tiles and many columns
(split over several workgroups a tile), with lengths in one exponent
chunk and over many.  Against the FP64 oracle at the tolerances of the other parity
tests (FP32 1e-6, FP64 1e-11; the digits are exact), and, where lengths span 40
octaves, to the rounding of the totals: a distance is T_i + T_j - 2 G_ij (over
T_i + T_j - G_ij), each of T and G an FP64 sum of at most 32 chunks, so it is off by
at most (4 * 32 + 4) 2^-53 = 1.5e-14 of T_i + T_j (of 2, normalized), and a pair that
differs in short branches alone has no more digits than that."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


@pytest.mark.parametrize("tips,n", [(4, 2), (20, 127), (64, 128), (66, 129), (130, 40), (200, 300), (330, 257),
                                    (2600, 130), (260, 3), (4000, 20), (1500, 700)])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("name", ["unweighted", "unweighted_fp64", "unweighted_unnormalized_fp64"])
def test_gram_edges(ssu, synth, O, monkeypatch, tips, n, wide, name):
    monkeypatch.setenv("SSU_GRAM_SPLIT", "0")   # every node a Gram column
    st, le, nm = synth.random_tree(tips, tips + n)
    if wide:   # exponents over 40 octaves, and zero lengths
        rng = np.random.default_rng(tips)
        le = np.asarray(le) * 2.0 ** rng.integers(-30, 10, len(le)) * (rng.random(len(le)) > 0.05)
    table = synth.random_table(tips, n, 0.3 if tips < 100 else 0.08, tips)
    inp = ssu.Inputs(st, le, nm, *table)
    p = ssu.Plan(inp, name)
    p.execute()
    want = O.matrix(O.Tree(st.astype(np.uint8), le, nm), O.Table(*table), name.replace("_fp64", ""))
    got = p.matrix().astype(np.float64)
    rel = 1e-11 if name.endswith("_fp64") else 1e-6
    scale = 2.0 * np.sum(le) if "unnormalized" in name else 2.0
    floor = 1.5e-14 * scale if wide else 0.0
    print("[gpu-case]", name, tips, n, wide, "max rel err", rel_err(got, want), "abs", np.abs(got - want).max(), flush=True)
    assert np.all(np.abs(got - want) <= rel * np.abs(want) + floor)
    p.close()


@pytest.mark.parametrize("name", ["unweighted", "unweighted_fp64"])
def test_gram_parts_of_a_stripe_range(ssu, synth, name):
    """Columns split over workgroups: a stripe range's tiles hold the same bits as
    the full matrix's (the split follows the matrix, not the tiles of a launch)."""
    n = 513
    st, le, nm = synth.random_tree(2500, 5)
    inp = ssu.Inputs(st, le, nm, *synth.random_table(2500, n, 0.05, 6))
    p = ssu.Plan(inp, name)
    p.execute()
    full = p.matrix()
    print("[gpu-case] stripes", name, flush=True)
    p.execute_stripes(100, 110)
    part = p.matrix()
    k = np.arange(n)
    for s in range(100, 110):
        assert np.array_equal(part[k, (k + s + 1) % n], full[k, (k + s + 1) % n])
    p.close()
