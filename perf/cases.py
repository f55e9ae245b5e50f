"""Timed cases: the calls that a program using this library makes.

Sizes are those of the benchmark workloads and tests of this repository (256
samples on 1,000 tips up to 16,384 samples on 100,000 tips) and ragged ones
between them.  Tables are drawn like the benchmark's: Zipf(1.1) tip
popularity, lognormal counts, a different richness in every sample; the tip
order of the table is not that of the tree.

Kinds of cases:
  matrix  one call of one_off_matrix_inmem_v3 / _fp32_v3: host table and tree
          to the host matrix (the drop-in call)
  plan    a resident plan (ssu_plan_create_inmem) that the program keeps:
          ssu_plan_execute, then ssu_plan_copy_matrix into its own buffer
  rarefy  a rarefaction batch the program keeps: every replicate of every
          method drawn, computed and copied out
  faith   ssu_faith_pd_inmem
  stats   PCoA, then PERMANOVA, on one distance matrix
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "unifrac-binaries_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "unifrac-binaries_amd"))
import ssu  # noqa: E402


def listed():
    return [
        # the smallest calls: a study of a few hundred samples, where latency counts
        dict(name="unweighted_256", kind="matrix", method="unweighted", samples=256, tips=1000, richness=50),
        dict(name="weighted_fp64_131", kind="matrix", method="weighted_normalized_fp64", samples=131, tips=2011,
             richness=90),
        # ordinary calls: a few thousand samples, every metric family, host to host
        dict(name="unweighted_2001", kind="matrix", method="unweighted", samples=2001, tips=20000, richness=400),
        dict(name="weighted_3000", kind="matrix", method="weighted_normalized", samples=3000, tips=20000,
             richness=400),
        dict(name="generalized_1777", kind="matrix", method="generalized", alpha=0.5, samples=1777, tips=20000,
             richness=400),
        # resident plans: variance adjusted, and double precision
        dict(name="vaw_1500_plan", kind="plan", method="weighted_normalized", vaw=True, samples=1500, tips=15000,
             richness=300),
        dict(name="weighted_fp64_3001_plan", kind="plan", method="weighted_normalized_fp64", samples=3001, tips=20000,
             richness=400),
        # the largest: the benchmark's workload, weighted in a plan and unweighted in one call
        dict(name="weighted_16384_plan", kind="plan", method="weighted_normalized", samples=16384, tips=100000,
             richness=1000),
        dict(name="unweighted_16384", kind="matrix", method="unweighted", samples=16384, tips=100000, richness=1000),
        # rarefaction: replicates of one table at depth 1,000, two methods
        dict(name="rarefy_1024x4", kind="rarefy", method="unweighted,weighted_normalized", samples=1024, tips=20000,
             richness=400, depth=1000, reps=4),
        # alpha diversity of a whole study
        dict(name="faith_4000", kind="faith", samples=4000, tips=20000, richness=400),
        # ordination and test of one matrix: 10 axes, 999 permutations, 6 groups
        dict(name="pcoa_permanova_2500", kind="stats", samples=2500, dims=10, perms=999, groups=6),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matrix"] * 4 + ["plan"] * 3 + ["rarefy", "faith", "stats"])
    if kind == "stats":
        return dict(kind=kind, samples=_log_int(rng, 100, 6000), dims=rng.choice([3, 5, 10]),
                    perms=rng.choice([199, 499, 999]), groups=rng.randint(2, 12))
    tips = _log_int(rng, 1000, 100000)
    case = dict(kind=kind, tips=tips, richness=max(20, int(tips * rng.uniform(0.008, 0.05) * (1000 / tips) ** 0.2)))
    if kind == "faith":
        return dict(case, samples=_log_int(rng, 100, 8000))
    if kind == "rarefy":
        methods = rng.choice(["unweighted,weighted_normalized", "weighted_unnormalized", "generalized",
                              "unweighted_fp64"])
        case["tips"] = min(tips, 30000)
        case["richness"] = min(max(case["richness"], 200), 600)   # (every sample reaches the depth)
        return dict(case, method=methods, alpha=rng.choice([0.5, 0.3]), samples=_log_int(rng, 100, 2000),
                    depth=rng.choice([500, 1000]), reps=rng.randint(2, 5))
    method = rng.choice(["unweighted", "unweighted_unnormalized", "weighted_normalized", "weighted_normalized",
                         "weighted_unnormalized", "generalized"])
    fp64 = rng.random() < 0.3
    vaw = rng.random() < 0.15
    if method == "generalized":
        case["alpha"] = rng.choice([0.5, 0.5, 1.0, 0.25, 0.7])
    # the dearer terms on smaller matrices, so that no drawn case costs more than the largest listed one
    most = 12000 if method.startswith("unweighted") and not vaw else 9000 if not (fp64 or vaw) else 4500
    if method == "generalized":
        most = 1200 if fp64 else 3000 if vaw else 5000
    return dict(case, method=method + ("_fp64" if fp64 else ""), vaw=vaw, samples=_log_int(rng, 64, most))


# ------------------------------------------------------------------ inputs


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _tree(tips, rng):
    """A random (Yule) binary tree: parentheses arrays, the tips' positions in tree order, every node's tip range."""
    size = 2 * (2 * tips - 1)
    structure = np.zeros(size, bool)
    lengths = np.zeros(size)
    tip_pos = np.zeros(tips, np.int64)
    pos, k, first = np.zeros(1, np.int64), np.full(1, tips, np.int64), np.zeros(1, np.int64)
    nodes = []
    while pos.size:
        structure[pos] = True
        lengths[pos] = rng.exponential(0.1, pos.size).astype(np.float32)
        nodes.append((pos, first, first + k))
        leaf = k == 1
        tip_pos[first[leaf]] = pos[leaf]
        pos, k, first = pos[~leaf], k[~leaf], first[~leaf]
        left = 1 + np.floor(rng.random(pos.size) * (k - 1)).astype(np.int64)
        pos, k, first = (np.concatenate([pos + 1, pos + 1 + 2 * (2 * left - 1)]), np.concatenate([left, k - left]),
                         np.concatenate([first, first + left]))
    lengths[0] = 0.0
    ranges = np.concatenate([np.stack(n, 1) for n in nodes[1:]])   # without the root: position, first tip, last + 1
    return structure, lengths, tip_pos, ranges


def _table(tips, samples, richness, seed):
    """Tip-major entries: indptr over every tip, sample indices and counts (host arrays)."""
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    w = (torch.randperm(tips, generator=g, device=dev) + 1).double() ** -1.1
    want = (richness * torch.exp(0.4 * torch.randn(samples, generator=g, device=dev).double() - 0.08)).clamp(
        richness / 2, tips / 3)
    # tip t is in sample s with probability 1 - exp(-rate_s w_t); rate_s gives the wanted richness
    grid = torch.logspace(-4, 9, 400, dtype=torch.float64, device=dev)
    got = torch.stack([(-torch.expm1(-r * w)).sum() for r in grid])
    rate = grid[torch.searchsorted(got, want).clamp(max=399)].float()
    wf = w.float()
    step = max(1, (1 << 27) // samples)
    counts, index = [], []
    for t0 in range(0, tips, step):
        p = -torch.expm1(-wf[t0:t0 + step, None] * rate[None, :])
        hit = torch.rand(p.shape, generator=g, device=dev) < p
        counts.append(hit.sum(1))
        index.append(hit.nonzero()[:, 1].to(torch.int32))
    index = torch.cat(index)
    data = torch.exp(3.0 + 1.5 * torch.randn(index.numel(), generator=g, device=dev)).ceil().double()
    indptr = np.zeros(tips + 1, np.int64)
    np.cumsum(torch.cat(counts).cpu().numpy(), out=indptr[1:])
    return indptr, index.cpu().numpy().view(np.uint32), data.cpu().numpy()


def _inputs(case, seed):
    """The program's table and tree, and what exact() needs of them."""
    rng = np.random.default_rng(seed)
    tips, samples = case["tips"], case["samples"]
    structure, lengths, tip_pos, ranges = _tree(tips, rng)
    indptr, index, data = _table(tips, samples, case["richness"], seed)
    place = rng.permutation(tips)          # tip i of the table is tip place[i] of the tree
    names = [""] * structure.size
    for i, p in enumerate(tip_pos[place]):
        names[p] = "t%d" % i
    seen = np.nonzero(np.diff(indptr))[0]  # only observed tips become rows
    rows = np.concatenate([[0], indptr[seen + 1]])
    inp = ssu.Inputs(structure, lengths, names, ["t%d" % i for i in seen], ["s%d" % i for i in range(samples)], rows,
                     index, data)
    return inp, dict(ranges=ranges, lengths=lengths, place=place, indptr=indptr, index=index, data=data)


def _distances(case, seed):
    """A distance matrix with group structure, as FP32 UniFrac gives one, and the grouping."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    group = rng.integers(0, case["groups"], n).astype(np.uint32)
    group[:case["groups"]] = np.arange(case["groups"])
    scale = 0.8 ** np.arange(40)
    x = torch.from_numpy((rng.normal(size=(n, 40)) + 0.8 * rng.normal(size=(case["groups"], 40))[group]) * scale)
    x = x.to(_device())
    d = torch.cdist(x, x, compute_mode="donot_use_mm_for_euclid_dist")
    noise = torch.from_numpy(rng.random(n)).to(d.device)
    d = d / d.max() * (0.97 + 0.03 * (noise[:, None] + noise[None, :]) / 2)
    d.fill_diagonal_(0.0)
    return d.float().cpu().numpy(), group


# ------------------------------------------------------------------ the calls


class _OneOff:
    """A one-off call's inputs."""

    def __init__(self, case, inp):
        self.inp, self.case, self.fp64 = inp, case, case["method"].endswith("_fp64")

    def run(self):
        L, c = ssu.lib(), self.case
        res = C.POINTER(ssu.MatFullFP64 if self.fp64 else ssu.MatFullFP32)()
        call = L.one_off_matrix_inmem_v3 if self.fp64 else L.one_off_matrix_inmem_fp32_v3
        status = call(C.byref(self.inp.table), C.byref(self.inp.tree), c["method"].encode(),
                      C.c_bool(c.get("vaw", False)), C.c_double(c.get("alpha", 1.0)), C.c_bool(False), C.c_bool(True),
                      C.c_uint(1), C.c_uint(0), C.c_bool(True), None, C.byref(res))
        if status != ssu.OKAY:
            raise RuntimeError("status %d: %s" % (status, ssu.last_error()))
        n, where = res.contents.n_samples, C.cast(res.contents.matrix, C.c_void_p).value

        class Matrix((C.c_double if self.fp64 else C.c_float) * (n * n)):   # the library's matrix, destroyed with it
            def __del__(self):
                (L.destroy_mat_full_fp64 if self._type_ is C.c_double else L.destroy_mat_full_fp32)(C.byref(res))

        return np.frombuffer(Matrix.from_address(where), C.c_double if self.fp64 else C.c_float).reshape(n, n)


class _Plan:
    def __init__(self, case, inp):
        self.plan = ssu.Plan(inp, case["method"], variance_adjust=case.get("vaw", False), alpha=case.get("alpha", 1.0))
        wide = ssu.lib().ssu_plan_result_bytes(self.plan.h) == 8
        self.out = np.zeros((case["samples"], case["samples"]), np.float64 if wide else np.float32)

    def run(self):
        self.plan.execute()
        if ssu.lib().ssu_plan_copy_matrix(self.plan.h, self.out.ctypes.data_as(C.c_void_p)) != ssu.OKAY:
            raise RuntimeError(ssu.last_error())
        return self.out


class _Rarefy:
    def __init__(self, case, inp):
        methods = case["method"].split(",")
        self.batch = ssu.Rarefaction(inp, methods, case["depth"], case["reps"], seed=7, alpha=case.get("alpha", 1.0))
        n = self.batch.n
        self.out = [[np.zeros((n, n), np.float64 if m.endswith("_fp64") else np.float32) for _ in range(case["reps"])]
                    for m in methods]

    def run(self):
        L = ssu.lib()
        self.batch.execute()
        for k, reps in enumerate(self.out):
            for r, m in enumerate(reps):
                if L.ssu_rarefy_copy_matrix(self.batch.h, C.c_int(k), C.c_uint(r),
                                            m.ctypes.data_as(C.c_void_p)) != ssu.OKAY:
                    raise RuntimeError(ssu.last_error())
        return self.out


class _Faith:
    def __init__(self, inp):
        self.inp = inp

    def run(self):
        status, values, _ = ssu.faith_pd_inmem(self.inp)
        if status != ssu.OKAY:
            raise RuntimeError("status %d: %s" % (status, ssu.last_error()))
        return values


class _Stats:
    def __init__(self, case, seed):
        self.case, (self.d, self.group) = case, _distances(case, seed)

    def run(self):
        ssu.lib().ssu_set_random_seed(C.c_uint(11))
        eig, coords, share = ssu.pcoa(self.d, self.case["dims"], fp32=True)
        f, p = ssu.permanova(self.d, self.group, self.case["perms"], fp32=True)
        return dict(eigenvalues=eig, coordinates=coords, proportion=share, f=np.float32(f), p=np.float32(p))


def prepare(case, seed):
    if case["kind"] == "stats":
        return _Stats(case, seed)
    inp, _ = _inputs(case, seed)
    if case["kind"] == "matrix":
        return _OneOff(case, inp)
    if case["kind"] == "plan":
        return _Plan(case, inp)
    return _Rarefy(case, inp) if case["kind"] == "rarefy" else _Faith(inp)


def run(state):
    return state.run()


# ------------------------------------------------------------------ floors and exact values


def _tip_counts(x, dtype, n0, n1):
    """Counts summed over the tips of the tree, in tree order: row t holds those of tips below t (samples n0 .. n1)."""
    dev = _device()
    tips = x["place"].size
    tip = torch.from_numpy(np.repeat(x["place"], np.diff(x["indptr"]))).to(dev)
    smp = torch.from_numpy(x["index"].view(np.int32)).to(dev).long()
    val = torch.from_numpy(x["data"]).to(dev).to(dtype)
    keep = (smp >= n0) & (smp < n1)
    m = torch.zeros((tips + 1, n1 - n0), dtype=dtype, device=dev)
    m[tip[keep] + 1, smp[keep] - n0] = val[keep]
    return torch.cumsum(m, 0, dtype=dtype, out=m)


def work(case):
    """Bytes: the table and the tree read, the results written.  Operations: those of the metric's terms over the
    (pair, node) combinations whose node both samples hold (what one sample holds alone is a sum per sample)."""
    if case["kind"] == "stats":
        n, k = case["samples"], case["dims"] + 2
        return dict(bytes=2 * 4 * n * n, flops=2.0 * n * n * k * 8 + n * n / 2 * case["perms"])
    inp, x = _inputs(case, 1)
    n, nnz = case["samples"], x["index"].size
    read = 12 * nnz + 9 * x["lengths"].size
    if case["kind"] == "faith":
        return dict(bytes=read + 8 * n, flops=float(nnz))
    held = torch.zeros(x["ranges"].shape[0], dtype=torch.int64, device=_device())
    a, b = (torch.from_numpy(x["ranges"][:, q].copy()).to(held.device) for q in (1, 2))
    for n0 in range(0, n, 2048):
        c = _tip_counts(x, torch.int32, n0, min(n, n0 + 2048))
        for k0 in range(0, a.numel(), 16384):
            held[k0:k0 + 16384] += (c[b[k0:k0 + 16384]] > c[a[k0:k0 + 16384]]).sum(1)
    both = float((held.double() * (held.double() - 1) / 2).sum())
    methods = case["method"].split(",")
    ops = sum(2 if m.startswith("unweighted") else 3 if m.startswith("weighted") else 8 for m in methods)
    size = sum(8 if m.endswith("_fp64") else 4 for m in methods)
    reps = case.get("reps", 1)
    return dict(bytes=read + size * n * n * reps, flops=both * reps * (ops + (6 if case.get("vaw") else 0)))


def _exact_matrix(case, x):
    n, method = case["samples"], case["method"]
    K = x["ranges"].shape[0]
    vaw, unweighted = case.get("vaw", False), method.startswith("unweighted")
    cost = float(n) * n * K * (0.002 if unweighted and not vaw else 1 if method.startswith("weighted") and not vaw
                               else 8 if vaw else 5)
    if cost > 1.0e12:   # (about 20 seconds)
        return None
    dev = _device()
    ell = torch.from_numpy(x["lengths"][x["ranges"][:, 0]]).to(dev)
    a, b = (torch.from_numpy(x["ranges"][:, q].copy()).to(dev) for q in (1, 2))
    c = _tip_counts(x, torch.int32 if unweighted and not vaw else torch.float64, 0, n)   # (whole counts: exact sums)
    total = c[-1].double()
    num = torch.zeros((n, n), dtype=torch.float64, device=dev)
    den = torch.zeros((n, n), dtype=torch.float64, device=dev)
    alpha = case.get("alpha", 1.0)
    for k0 in range(0, K, 4096):
        e = c[b[k0:k0 + 4096]] - c[a[k0:k0 + 4096]]
        lk = ell[k0:k0 + 4096, None]
        if unweighted and not vaw:
            p = (e > 0).double()
            num += (p * lk).T @ p          # shared length; turned into distances below
            continue
        u = e / total
        if method.startswith("weighted") and not vaw:
            y = (u * lk).T.contiguous()
            for i in range(0, n, 1024):
                num[i:i + 1024] += torch.cdist(y[i:i + 1024], y, p=1.0)
            s = y.sum(1)
            den += s[:, None] + s[None, :]
            continue
        for i in range(n):
            v, w = (u[:, i:], u[:, i:i + 1]) if not unweighted else ((u[:, i:] > 0).double(), (u[:, i:i + 1] > 0).double())
            s, d = v + w, (v - w).abs()
            if unweighted:
                s = torch.maximum(v, w)
            if vaw:
                mi = e[:, i:] + e[:, i:i + 1]
                q = (mi * (total[i:] + total[i] - mi)).sqrt()
                q = torch.where(q > 0, 1.0 / q, torch.zeros_like(q))
                s, d = s * q, d * q
            if method.startswith("generalized"):
                ss = s ** alpha
                d = torch.where(s > 0, ss * d / s, torch.zeros_like(s))
                s = torch.where(s > 0, ss, torch.zeros_like(s))
            num[i, i:] += (lk * d).sum(0)
            den[i, i:] += (lk * s).sum(0)
    if unweighted and not vaw:
        t = num.diagonal().clone()
        both = t[:, None] + t[None, :]
        num, den = both - 2 * num, both - num
    elif not (method.startswith("weighted") and not vaw):
        num, den = (torch.triu(m) + torch.triu(m, 1).T for m in (num, den))
    out = num if "unnormalized" in method else num / den
    return out.fill_diagonal_(0.0).cpu().numpy()


def exact(case, seed):
    if case["kind"] == "rarefy":   # (the draws are the library's own)
        return None
    if case["kind"] == "stats":
        d, group = _distances(case, seed)
        d = torch.from_numpy(d).double()
        n = d.shape[0]
        if n > 4000:
            return None
        a = -0.5 * d * d
        r = a.mean(1)
        bm = a - r[:, None] - r[None, :] + r.mean()
        e = torch.linalg.eigvalsh(bm).flip(0)[:case["dims"]].clamp(min=0)
        g = torch.from_numpy(group.astype(np.int64))
        size = torch.bincount(g).double()
        d2 = torch.triu(d * d, 1)
        within = float((torch.where(g[:, None] == g[None, :], d2, torch.zeros_like(d2)) / size[g][:, None]).sum())
        total, k = float(d2.sum()) / n, int((size > 0).sum())
        f = ((total - within) / (k - 1)) / (within / (n - k))
        return dict(eigenvalues=e.numpy(), coordinates=None, proportion=(e / bm.trace()).numpy(), f=np.float64(f),
                    p=None)
    inp, x = _inputs(case, seed)
    if case["kind"] != "faith":
        return _exact_matrix(case, x)
    c = _tip_counts(x, torch.int32, 0, case["samples"])
    ell = torch.from_numpy(x["lengths"][x["ranges"][:, 0]]).to(c.device)
    a, b = (torch.from_numpy(x["ranges"][:, q].copy()).to(c.device) for q in (1, 2))
    pd = torch.zeros(case["samples"], dtype=torch.float64, device=c.device)
    for k0 in range(0, ell.numel(), 16384):
        pd += ell[k0:k0 + 16384] @ (c[b[k0:k0 + 16384]] > c[a[k0:k0 + 16384]]).double()
    return pd.cpu().numpy()
