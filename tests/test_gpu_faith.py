"""Faith PD from presence bits: bit-equal to the oracle, whose FP64 sums run over
every node in postorder, at sample counts around a wave (64) and node counts
around a round of 256 nodes and around a group of four, with samples that hold
nothing and, for tables with negative values, through the FP64 embedding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("tips", [2, 3, 65, 128, 129, 130, 500])
@pytest.mark.parametrize("kind", ["counts", "low", "negative"])
def test_faith_bits(ssu, synth, O, n, tips, kind):
    st, le, nm = synth.random_tree(tips, 7 * tips + n)
    obs, smp, ip, ix, data = synth.random_table(tips, n, max(0.05, 2 / tips), tips + n)
    data = np.asarray(data)
    if kind == "low":          # totals below 1 are dropped, explicit zeros hold nothing
        data = data.copy()
        data[np.asarray(ix) % 5 == 3] = 0.0
        data[np.asarray(ix) == n - 1] = 1.0
    if kind == "negative":
        data = data.copy()
        data[::7] *= -0.001
    inp = ssu.Inputs(st, le, nm, obs, smp, ip, ix, data)
    tot = np.bincount(np.asarray(ix), data, n)
    keep = np.nonzero(tot >= 1)[0]
    status, vals, ids = ssu.faith_pd_inmem(inp)
    assert status == ssu.OKAY and ids == [smp[i] for i in keep]
    # the oracle on the kept samples and rows
    ind, col, dat, rows = [0], [], [], []
    new = {s: k for k, s in enumerate(keep)}
    for i in range(len(obs)):
        e = [(new[s], v) for s, v in zip(ix[ip[i]:ip[i + 1]], data[ip[i]:ip[i + 1]]) if s in new]
        if e:
            rows.append(obs[i])
            col += [s for s, _ in e]
            dat += [v for _, v in e]
            ind.append(len(col))
    ref = O.faith_pd(O.Tree(st.astype(np.uint8), le, nm),
                     O.Table(rows, [smp[i] for i in keep], np.array(ind, np.uint32), np.array(col, np.uint32),
                             np.array(dat)))
    assert np.array_equal(vals, ref)
