"""In-memory Faith PD of tables that its filter changes: samples with a total below
1, rows without entries, rows held by dropped samples only, alone and together.
Bit-equal to the oracle on the kept samples and rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


def kept_table(obs, smp, ip, ix, data):
    tot = np.bincount(ix, data, len(smp))
    keep = np.nonzero(tot >= 1)[0]
    new = {s: k for k, s in enumerate(keep)}
    ind, col, dat, rows = [0], [], [], []
    for i in range(len(obs)):
        e = [(new[s], v) for s, v in zip(ix[ip[i]:ip[i + 1]], data[ip[i]:ip[i + 1]]) if s in new]
        if e:
            rows.append(obs[i])
            col += [s for s, _ in e]
            dat += [v for _, v in e]
            ind.append(len(col))
    return rows, [smp[i] for i in keep], np.array(ind, np.uint32), np.array(col, np.uint32), np.array(dat)


@pytest.mark.parametrize("low", [[], [0], [3, 70, 71, 199], list(range(1, 200))], ids=["none", "first", "four", "all but one"])
@pytest.mark.parametrize("rows", ["held", "empty", "lost", "both"])
@pytest.mark.parametrize("zeros", [False, True])
def test_faith_filtered(ssu, synth, O, low, rows, zeros):
    n, tips = 200, 400
    st, le, nm = synth.random_tree(tips, 41)
    obs, smp, ip, ix, data = synth.random_table(tips, n, 0.06, 42)
    ip, ix, data = np.asarray(ip), np.asarray(ix), np.array(data)
    if zeros:
        data[::9] = 0.0
    data[np.isin(ix, low)] = 0.0 if zeros else 0.001
    if rows in ("lost", "both") and low:      # the second row: only in the first dropped sample
        ix = np.concatenate([ix[:ip[1]], [low[0]], ix[ip[2]:]])
        data = np.concatenate([data[:ip[1]], [0.002], data[ip[2]:]])
        ip = np.concatenate([ip[:2], ip[2:] - (ip[2] - ip[1] - 1)])
    if rows in ("empty", "both"):             # the first and the last row empty
        drop = ip[1]
        ix, data = ix[drop:ip[-2]], data[drop:ip[-2]]
        ip = np.clip(ip - drop, 0, ix.size)
    assert ip[-1] == ix.size and len(obs) + 1 == ip.size
    table = (obs, smp, ip.astype(np.uint32), ix.astype(np.uint32), data)
    keep = kept_table(*table)
    status, vals, ids = ssu.faith_pd_inmem(ssu.Inputs(st, le, nm, *table))
    assert status == ssu.OKAY and ids == keep[1]
    assert np.array_equal(vals, O.faith_pd(O.Tree(st.astype(np.uint8), le, nm), O.Table(*keep)))


def test_faith_nothing_left(ssu, synth):
    st, le, nm = synth.random_tree(50, 1)
    obs, smp, ip, ix, data = synth.random_table(50, 20, 0.2, 2)
    status, vals, ids = ssu.faith_pd_inmem(ssu.Inputs(st, le, nm, obs, smp, ip, ix, np.full(len(data), 1e-3)))
    assert status == ssu.OKAY and ids == list(smp) and not vals.any()


@pytest.mark.parametrize("values", [(5e-324, 1e8), (1e-310, 1e20), (1e308, 1.7e308)], ids=["least", "subnormal", "overflow"])
def test_faith_of_proportions_that_vanish(ssu, synth, O, values):
    """A value whose proportion underflows to 0, or of a total that overflows, does not
    count as present: a node held only through it adds nothing."""
    st, le, nm = synth.random_tree(60, 5)
    obs, smp, ip, ix, data = synth.random_table(60, 30, 0.2, 6)
    ip, ix, data = np.asarray(ip), np.asarray(ix), np.array(data, float)
    own = np.nonzero(ix == ix[0])[0]
    data[own] = 2.0
    data[own[::2]], data[own[1::2]] = values
    table = (obs, smp, ip, ix, data)
    status, vals, _ = ssu.faith_pd_inmem(ssu.Inputs(st, le, nm, *table))
    ref = O.faith_pd(O.Tree(st.astype(np.uint8), le, nm), O.Table(*table))
    assert status == ssu.OKAY and np.array_equal(vals, ref)
    full = O.faith_pd(O.Tree(st.astype(np.uint8), le, nm), O.Table(obs, smp, ip, ix, np.ones(data.size)))
    assert ref[ix[0]] < full[ix[0]]
