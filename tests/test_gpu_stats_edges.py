"""PCoA and PERMANOVA at the edges of their kernels' blocks: sample counts around
16 (a product's row tile), 64 (a permutation tile) and 256 (its column chunk), probe
counts around 16 columns, label rows around 64, and groups past 256, whose labels
do not fit bytes.  The permutations are restated here, so the p-value is held
exactly but for permuted statistics that tie with the observed one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


@pytest.fixture(scope="module", autouse=True)
def _need_device(ssu):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")


def mix64(z):
    z = (z + 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def first_draw(seed):
    """The first output of std::mt19937_64 (Nishimura & Matsumoto), the library's stream."""
    mt = [seed & M64]
    for i in range(1, 157):
        mt.append((6364136223846793005 * (mt[-1] ^ (mt[-1] >> 62)) + i) & M64)
    x = (mt[0] & ~0x7FFFFFFF) | (mt[1] & 0x7FFFFFFF)
    x = mt[156] ^ (x >> 1) ^ (0xB5026F5AA96619E9 if x & 1 else 0)
    x ^= (x >> 29) & 0x5555555555555555
    x ^= (x << 17) & 0x71D67FFFEDA60000
    x ^= (x << 37) & 0xFFF7EEE000000000
    return x ^ (x >> 43)


def shuffled(g, seed, p):
    g = list(g)
    key = mix64(seed ^ mix64(p))
    for i in range(len(g) - 1, 0, -1):
        j = mix64((key + i) & M64) % (i + 1)
        g[i], g[j] = g[j], g[i]
    return np.array(g)


def distances(n, rank, seed):
    x = np.random.default_rng(seed).normal(size=(n, rank)) / np.arange(1, rank + 1)
    d = np.sqrt(((x[:, None, :] - x[None, :, :]) ** 2).sum(-1))
    np.fill_diagonal(d, 0.0)
    return d


def pseudo_f(d, g):
    n, ids = len(g), np.unique(g)
    d2 = np.triu(d * d, 1)
    st = d2.sum() / n
    sw = sum(d2[np.ix_(g == i, g == i)].sum() / (g == i).sum() for i in ids)
    return ((st - sw) / (len(ids) - 1)) / (sw / (n - len(ids)))


@pytest.mark.parametrize("n,groups,perms", [(3, 2, 1), (63, 2, 62), (64, 3, 63), (65, 64, 64), (129, 5, 65),
                                            (256, 256, 20), (300, 257, 20), (321, 4, 130), (1300, 7, 10)])
@pytest.mark.parametrize("fp32", [False, True])
def test_permanova_blocks(ssu, n, groups, perms, fp32):
    d = distances(n, 6, n)
    if fp32:
        d = d.astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(groups)
    g = np.concatenate([np.arange(groups), rng.integers(0, groups, n)])[:n]
    if n == groups:
        g[0] = 1
    rng.shuffle(g)
    print("[gpu-case] permanova", n, groups, perms, fp32, flush=True)
    ssu.lib().ssu_set_random_seed(n + groups)
    seed = first_draw(n + groups)
    f, p = ssu.permanova(d, g, perms, fp32=fp32)
    f0 = pseudo_f(d, g)
    assert abs(f - f0) <= (1e-6 if fp32 else 1e-10) * f0   # sums of FP64; the result is rounded to FP32
    fs = np.array([pseudo_f(d, shuffled(g, seed, q)) for q in range(1, perms + 1)])
    tie = np.abs(fs - f0) <= 1e-9 * f0
    lo, hi = ((fs >= f0) & ~tie).sum(), ((fs >= f0) | tie).sum()
    got = round(p * (perms + 1)) - 1
    assert abs(p * (perms + 1) - 1 - got) < 1e-3 and lo <= got <= hi


@pytest.mark.parametrize("n", [2, 15, 16, 17, 65, 130, 1025])
@pytest.mark.parametrize("dims", [1, 3, 14, 15, 30])
@pytest.mark.parametrize("fp32", [False, True])
def test_pcoa_blocks(ssu, n, dims, fp32):
    """Points of rank <= dims: the probes span the whole range, so the coordinates
    give the distances back (the QR and the SVD are backward stable; the centred
    matrix is rounded to FP32 where the input is)."""
    rank = min(dims, n - 1)
    d = distances(n, rank, 100 * n + dims)
    print("[gpu-case] pcoa", n, dims, fp32, flush=True)
    ssu.lib().ssu_set_random_seed(5)
    e, s, prop = ssu.pcoa(d, dims, fp32=fp32)
    e, s = e.astype(np.float64), s.astype(np.float64)
    # FP32: n x n rounding errors of up to 2^-24 of the largest entry each
    tol = (n * 6e-8 if fp32 else 1e-11) * 4 * (d * d).max()
    b = -0.5 * d * d
    b = b - b.mean(0) - b.mean(1)[:, None] + b.mean()
    w = np.sort(np.linalg.eigvalsh(b))[::-1][:rank]
    assert np.abs(e[:rank] - w).max() <= n * tol
    if not fp32:
        assert np.abs(s @ s.T - b).max() <= n * tol
        assert abs(prop.sum() - 1.0) <= 1e-9
    else:
        # the leading coordinate, away from the noise of the small ones
        assert abs((s[:, 0] ** 2).sum() - e[0]) <= n * tol
