"""Timed cases of the library: what a t-SNE run asks of it, through its Python binding.

Kinds (a case's "kind"):
  run         a whole short FP32 run: new context, P and Y uploaded, iterations, KL, embedding back
  steps       iterations of a resident context (FP32 form or FP64 plain), then the embedding
  batch       iterations of several independent 2D embeddings stepped together
  mirror      one gradient through the host-array entry point (FP64)
  affinities  the sparse P of a data set: exact neighbours, perplexity calibration, symmetrisation
  knn         exact neighbours of a large data set (the FP32-candidate search)
  exact       iterations and KL with the dense P (theta = 0)
  bh          Barnes-Hut iterations

Inputs are Gaussian mixtures: P joins random neighbours of one cluster with rows that sum to one before
symmetrisation, Y holds one blob per cluster.  FP32 contexts hold the embedding in 32 bits, so their
outputs are returned in 32 bits.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fit-sne_amd"))

import fitsne_gpu as fg  # noqa: E402

FLT_MIN = float(np.finfo(np.float32).tiny)
DBL_MIN = float(np.finfo(np.float64).tiny)
DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64


def listed():
    return [
        # a small embedding from start to finish, with early exaggeration: latency, launches and set-up
        dict(name="run_2k", kind="run", N=2000, D=2, df=1.0, per=30, span=35.0, steps=20, exag=12.0),
        # a mid-size embedding with the heavier-tailed kernel and late exaggeration
        dict(name="steps_2d_df_70k", kind="steps", prec="fp32", N=70001, D=2, df=0.7, per=45, span=40.0, steps=10,
             exag=4.0),
        # a million points in 2D, about 90 neighbours each: the headline size
        dict(name="steps_2d_1m", kind="steps", prec="fp32", N=1000000, D=2, df=1.0, per=45, span=70.0, steps=10,
             exag=1.0),
        # 1D embedding, heavy tails, late exaggeration
        dict(name="steps_1d_1m", kind="steps", prec="fp32", N=1000003, D=1, df=0.5, per=30, span=280.0, steps=10,
             exag=4.0),
        # a sweep: independent embeddings of 2,000 to 60,000 points stepped together
        dict(name="batch_24", kind="batch", count=24, nmin=2000, nmax=60000, D=2, df=1.0, per=30, span=35.0, steps=10,
             exag=1.0),
        # the double-precision path, resident
        dict(name="steps_fp64_200k", kind="steps", prec="fp64", N=200003, D=2, df=1.0, per=45, span=50.0, steps=4,
             exag=1.0),
        # one gradient on the caller's host arrays, as a program that keeps its own loop calls it
        dict(name="mirror_10k", kind="mirror", N=10000, D=2, df=1.0, per=45, span=35.0),
        # P of a usual data set (50 principal components, perplexity 30)
        dict(name="affinities_10k", kind="affinities", N=10000, D=50, clusters=10, perplexity=30),
        # P of a larger one, odd sizes, perplexity 50
        dict(name="affinities_40k", kind="affinities", N=40009, D=37, clusters=40, perplexity=50),
        # neighbours of a large data set
        dict(name="knn_300k", kind="knn", N=300000, D=100, clusters=200, K=90),
        # theta = 0 with its dense P
        dict(name="exact_8k", kind="exact", N=8001, D=2, df=1.0, data_dim=50, perplexity=30, steps=3, exag=1.0),
        # Barnes-Hut
        dict(name="bh_100k", kind="bh", N=100000, D=2, theta=0.5, per=30, span=50.0, steps=3, exag=1.0),
    ]


def draw(rng):
    def size(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["run", "steps", "steps", "steps64", "batch", "mirror", "affinities", "knn", "exact", "bh"])
    exag = rng.choice([1.0, 1.0, 4.0, 12.0])
    if kind == "run":
        return dict(kind=kind, N=size(2000, 20000), D=2, df=rng.choice([1.0, 1.0, 0.6]), per=rng.randint(15, 45),
                    span=round(rng.uniform(25, 40), 2), steps=rng.randint(10, 30), exag=exag)
    if kind == "steps":
        D = rng.choice([1, 2, 2])
        N = size(20000, 900000)
        return dict(kind=kind, prec="fp32", N=N, D=D, df=rng.choice([1.0, 1.0, 0.5, 0.8]), per=rng.randint(15, 40),
                    span=round(rng.uniform(30, 70) if D == 2 else rng.uniform(50, 280), 2), steps=rng.randint(5, 10),
                    exag=exag)
    if kind == "steps64":
        D = rng.choice([1, 2, 2])
        return dict(kind="steps", prec="fp64", N=size(5000, 200000), D=D, df=rng.choice([1.0, 1.0, 0.7]),
                    per=rng.randint(15, 45), span=round(rng.uniform(30, 60), 2), steps=rng.randint(2, 4), exag=exag)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(4, 16), nmin=2000, nmax=size(6000, 50000), D=2, df=1.0,
                    per=rng.randint(15, 40), span=round(rng.uniform(25, 40), 2), steps=rng.randint(5, 10), exag=exag)
    if kind == "mirror":
        return dict(kind=kind, N=size(2000, 60000), D=rng.choice([1, 2, 2]), df=rng.choice([1.0, 0.6]),
                    per=rng.randint(15, 45), span=round(rng.uniform(20, 50), 2))
    if kind == "affinities":
        return dict(kind=kind, N=size(2000, 40000), D=rng.choice([20, 50, 50, rng.randint(4, 120)]),
                    clusters=rng.randint(5, 60), perplexity=rng.choice([10, 30, 30, 50]))
    if kind == "knn":
        return dict(kind=kind, N=size(50000, 250000), D=rng.choice([50, 100, rng.randint(20, 128)]),
                    clusters=rng.randint(50, 200), K=rng.choice([30, 90, 90, 150]))
    if kind == "exact":
        return dict(kind=kind, N=size(1000, 8000), D=rng.choice([1, 2, 2, 3]), df=rng.choice([1.0, 1.0, 0.7]),
                    data_dim=rng.choice([20, 50]), perplexity=rng.choice([10, 30]), steps=rng.randint(2, 4), exag=exag)
    return dict(kind="bh", N=size(5000, 90000), D=rng.choice([2, 2, 3]), theta=rng.choice([0.5, 0.5, 0.8]),
                per=rng.randint(15, 30), span=round(rng.uniform(25, 50), 2), steps=rng.randint(2, 3), exag=exag)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _labels(N, k, g):
    """Cluster of every point: k clusters of unequal weight, none of them empty."""
    w = torch.rand(k, generator=g, device=DEV, dtype=F64) + 0.1
    lab = torch.multinomial(w, N, replacement=True, generator=g)
    lab[:k] = torch.arange(k, device=DEV)
    return lab


def _blobs(lab, k, D, span, g):
    """One blob per cluster, centres uniform in [-span, span]^D; zero mean."""
    cen = (torch.rand(k, D, generator=g, device=DEV, dtype=F64) * 2 - 1) * span
    Y = cen[lab] + torch.randn(lab.numel(), D, generator=g, device=DEV, dtype=F64) * (span / 23.0)
    return Y - Y.mean(0, keepdim=True)


def _sparse_p(lab, k, per, g):
    """Symmetric normalised P (CSR: row, col, val): `per` random neighbours of the point's own cluster each, weights
    falling with a squared distance of relative spread 0.2, rows normalised, then (P + P^T) / sum."""
    N = lab.numel()
    order = torch.argsort(lab, stable=True)
    cnt = torch.bincount(lab, minlength=k)
    start = torch.cumsum(cnt, 0) - cnt
    pick = (torch.rand(N, per, generator=g, device=DEV, dtype=torch.float32) * cnt[lab][:, None]).long()
    pick = torch.minimum(pick, cnt[lab][:, None] - 1)
    nbr = order[start[lab][:, None] + pick]
    w = torch.exp(-(1 + 0.2 * torch.randn(N, per, generator=g, device=DEV, dtype=torch.float32))).to(F64)
    own = torch.arange(N, device=DEV)[:, None]
    w = torch.where(nbr == own, torch.zeros_like(w), w)
    w /= w.sum(1, keepdim=True).clamp_min(1e-30)
    i, j, w = own.expand(N, per).reshape(-1), nbr.reshape(-1), w.reshape(-1)
    keep = w > 0
    i, j, w = i[keep], j[keep], w[keep]
    key = torch.cat([i * N + j, j * N + i])
    key, at = torch.sort(key)
    w = torch.cat([w, w])[at]
    del at, i, j, keep, nbr, pick
    first = torch.ones_like(key, dtype=torch.bool)
    first[1:] = key[1:] != key[:-1]
    at = torch.nonzero(first)[:, 0]
    val = w[at]
    for r in range(1, 8):  # a pair drawn again is the next entry: its weights add up
        nxt = (at + r).clamp_max(key.numel() - 1)
        val += torch.where((key[nxt] == key[at]) & (nxt == at + r), w[nxt], 0.0)
    key = key[at]
    del first, at, w
    val /= val.sum()
    row = torch.zeros(N + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.cumsum(torch.bincount(key // N, minlength=N), 0)
    return row, key % N, val


def _sizes(case):
    """Sizes of a batch's problems, spread over the logarithm of their range."""
    n = case["count"]
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [int(round(math.exp(lo + (hi - lo) * i / max(1, n - 1)))) + i % 2 for i in range(n)]


def _embedding(case, N, seed):
    """(P, Y0) of one embedding problem, on the device."""
    g = _gen(seed)
    k = 50 if N >= 20000 else 10
    lab = _labels(N, k, g)
    Y = _blobs(lab, k, case["D"], case["span"], g)
    return _sparse_p(lab, k, case["per"], g), Y


def _host_p(P):
    row, col, val = P
    return (row.to(torch.int32).cpu().numpy().view(np.uint32), col.to(torch.int32).cpu().numpy().view(np.uint32),
            val.cpu().numpy())


def _data(case, D, seed):
    """Centred mixture scaled by its largest absolute value, as a run prepares its data."""
    g = _gen(seed)
    N, k = case["N"], case.get("clusters", 10)
    lab = _labels(N, k, g)
    X = (torch.randn(k, D, generator=g, device=DEV, dtype=F64) * 4)[lab] + torch.randn(
        N, D, generator=g, device=DEV, dtype=F64)
    X -= X.mean(0, keepdim=True)
    return X / X.abs().max()


def _lr(N):
    return max(200.0, N / 12.0)


def _context(case, N, P, Y):
    prec = {"fp32": fg.FP32, "fp64": fg.FP64_PLAIN, "bh": fg.FP64_BH}[case.get("prec", "fp32")]
    ctx = fg.Context(no_dims=case["D"], precision=prec, df=case.get("df", 1.0))
    ctx.set_P(*P)
    ctx.set_exaggeration(case["exag"])
    ctx.set_Y(Y)
    return ctx


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind in ("run", "steps", "mirror"):
        P, Y = _embedding(case, case["N"], seed)
        s["P"], s["Y"] = _host_p(P), Y.cpu().numpy()
        if kind == "steps":
            s["ctx"] = _context(case, case["N"], s.pop("P"), s.pop("Y"))
    elif kind == "batch":
        s["ctx"] = []
        for i, N in enumerate(_sizes(case)):
            P, Y = _embedding(case, N, seed * 101 + i)
            s["ctx"].append(_context(case, N, _host_p(P), Y.cpu().numpy()))
        s["batch"] = fg.Batch(s["ctx"])
    elif kind in ("affinities", "knn"):
        s["X"] = _data(case, case["D"], seed).cpu().numpy()
        if kind == "affinities":  # the caller's arrays of the symmetric P, as long as it can become
            N, K = case["N"], 3 * case["perplexity"]
            s["sym"] = (np.zeros(N + 1, dtype=np.uint32), np.zeros(2 * N * K, dtype=np.uint32), np.zeros(2 * N * K))
    elif kind == "exact":
        X, Y = _data(case, case["data_dim"], seed), _start(case, seed)
        s["ctx"] = fg.Context(no_dims=case["D"], precision=fg.FP64_EXACT, df=case["df"])
        s["ctx"].exact_affinities(X.cpu().numpy(), perplexity=case["perplexity"], download=False)
        s["ctx"].set_exaggeration(case["exag"])
        s["ctx"].set_Y(Y.cpu().numpy())
    else:
        P, Y = _embedding(case, case["N"], seed)
        s["ctx"] = _context(dict(case, prec="bh"), case["N"], _host_p(P), Y.cpu().numpy())
        s["ctx"].set_theta(case["theta"])
    return s


def _start(case, seed):
    g = _gen(seed + 5)
    return torch.randn(case["N"], case["D"], generator=g, device=DEV, dtype=F64) * 8


# ---------------------------------------------------------------- one pass

def _f32(v):
    return np.asarray(v, dtype=np.float32)


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "mirror":
        dC, Z = fg.compute_fft_gradient(s["P"], s["Y"], df=case["df"])
        return {"dC": dC, "Z": Z}
    if kind == "affinities":
        K = 3 * case["perplexity"]
        idx, dist = fg.knn_exact(s["X"], K)
        P, beta, iters = fg.distances2similarities(dist, float(case["perplexity"]), squared=True)
        row = np.arange(case["N"] + 1, dtype=np.uint32) * np.uint32(K)
        srow, scol, sval = s["sym"]
        fg.check(fg.lib().fitsne_symmetrize(row, idx.reshape(-1).view(np.uint32), P.reshape(-1), case["N"], srow, scol,
                                            sval, None))
        return {"idx": idx, "dist": dist, "beta": beta, "iters": iters, "row": srow.view(np.int32),
                "col": scol.view(np.int32), "val": sval}
    if kind == "knn":
        idx, dist, _ = fg.knn_mfma(s["X"], case["K"])
        return {"idx": idx, "dist": dist}
    if kind == "batch":
        prm = [(0.8, _lr(c.N), 5.0) for c in s["ctx"]]
        for _ in range(case["steps"]):
            s["batch"].step(prm)
        return [_f32(c.get_Y()) for c in s["ctx"]]
    if kind == "run":
        ctx = _context(case, case["N"], s["P"], s["Y"])
        for _ in range(case["steps"]):
            ctx.step(0.8, _lr(case["N"]))
        out = {"kl": _f32(ctx.kl()), "Y": _f32(ctx.get_Y())}
        ctx.close()
        return out
    ctx = s["ctx"]
    for _ in range(case["steps"]):
        ctx.step(0.8, _lr(case["N"]))
    if kind == "exact":
        return {"kl": ctx.kl(), "Y": ctx.get_Y()}
    Y = ctx.get_Y()
    return {"Y": _f32(Y) if case.get("prec") == "fp32" else Y}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "affinities":
        # input, distances, P and the symmetric P out; a subtraction, product and sum per coordinate and pair
        N, D, K = case["N"], case["D"], 3 * case["perplexity"]
        return {"bytes": 8.0 * N * D + N * K * (4 + 8 + 8) + 1.5 * N * K * 12, "flops": 3.0 * N * N * D}
    if kind == "knn":
        N, D, K = case["N"], case["D"], case["K"]
        return {"bytes": 8.0 * N * D + 12.0 * N * K, "flops": 3.0 * N * N * D}
    if kind == "exact":
        N, D = case["N"], case["D"]
        return {"bytes": case["steps"] * (8.0 * N * N + 72.0 * N * D) + 8.0 * N * N,
                "flops": (case["steps"] + 1) * N * N * (8.0 + 7 * D)}
    if kind == "batch":
        return {k: sum(work(dict(case, kind="steps", prec="fp32", N=N))[k] for N in _sizes(case))
                for k in ("bytes", "flops")}
    N, D, per = case["N"], case["D"], case["per"]
    nnz = 2.0 * N * per
    if kind == "bh":
        # P, Y and the state; a tree walk opens a few cells per level for each point
        return {"bytes": case["steps"] * (12.0 * nnz + 72.0 * N * D),
                "flops": case["steps"] * (nnz * (5 + 4 * D) + N * 40 * math.log2(N) * (4 + 3 * D))}
    wide = 2 if kind == "mirror" or case.get("prec") == "fp64" else 1
    nb = max(50, 2.2 * case["span"])
    m = 2 * 3 * nb
    grid = m ** D
    flops = nnz * (5 + 4 * D) + N * (3 ** D) * 16 + 8 * 2.5 * grid * math.log2(grid)
    step = nnz * (4 + 4 * wide) + 28.0 * wide * N * D
    if kind == "mirror":
        return {"bytes": 12.0 * nnz + 16.0 * N * D, "flops": flops}
    once = 12.0 * nnz + 16.0 * N * D if kind == "run" else 8.0 * N * D
    return {"bytes": case["steps"] * step + once, "flops": case["steps"] * flops}


# ---------------------------------------------------------------- the same in 64 bits, plain torch

def _rows_of(row):
    return torch.repeat_interleave(torch.arange(row.numel() - 1, device=row.device), row[1:] - row[:-1])


def _edges(P, chunk=1 << 24):
    row, col, val = P
    own = _rows_of(row)
    for a in range(0, col.numel(), chunk):
        yield own[a:a + chunk], col[a:a + chunk], val[a:a + chunk]


def _attraction(P, Y, df, exag):
    pos = torch.zeros_like(Y)
    for i, j, v in _edges(P):
        diff = Y[i] - Y[j]
        q = 1 / (1 + (diff * diff).sum(1) / df)
        pos.index_add_(0, i, (exag * v * q)[:, None] * diff)
    return pos


_BOXES = (25, 36, 50, 55, 60, 65, 70, 75, 80, 85, 90, 96, 100, 110, 120, 130, 140, 150, 175, 200)


def _grid(Y, p=3, ipi=1.0, mni=50):
    D = Y.shape[1]
    flat = Y.reshape(-1)
    mx = flat.max().item()
    mn = (flat[1:] if D == 2 else flat).min().item()  # in 2D the first coordinate opens the search unread
    nb = int(max(float(mni), (mx - mn) / ipi))
    if D == 2 and nb < 200:
        nb = next(b for b in _BOXES if b >= nb)
    bw = (mx - mn) / nb
    box = ((Y - mn) / bw).long().clamp(0, nb - 1)
    t = (Y - (box.to(F64) * bw + mn)) / bw
    node = (torch.arange(p, device=Y.device, dtype=F64) + 0.5) / p
    L = []
    for a in range(p):
        v = torch.ones_like(t)
        for b in range(p):
            if b != a:
                v = v * (t - node[b]) / (node[a] - node[b])
        L.append(v)
    return nb * p, bw / p, box * p, torch.stack(L, -1)  # nodes a side, spacing, first node [N, D], weights [N, D, p]


def _potentials(Y, charges, kernel, grid):
    """sum_j kernel(|y_i - y_j|^2) charges_j by interpolation on the grid's nodes and a circulant convolution."""
    n, h, first, L = grid
    N, D = Y.shape
    p = L.shape[2]
    r = torch.arange(2 * n, device=Y.device, dtype=F64)
    r = torch.minimum(r, 2 * n - r) * h
    if D == 1:
        node = first + torch.arange(p, device=Y.device)
        w = L[:, 0, :]
        kt = torch.fft.rfft(kernel(r * r))
    else:
        a = first[:, 0, None] + torch.arange(p, device=Y.device)
        b = first[:, 1, None] + torch.arange(p, device=Y.device)
        node = (a[:, :, None] * n + b[:, None, :]).reshape(N, p * p)
        w = (L[:, 0, :, None] * L[:, 1, None, :]).reshape(N, p * p)
        kt = torch.fft.rfft2(kernel(r[:, None] ** 2 + r[None, :] ** 2))
    out = []
    for c in charges:
        g = torch.zeros(n ** D, device=Y.device, dtype=F64)
        g.index_add_(0, node.reshape(-1), (w * c[:, None]).reshape(-1))
        if D == 1:
            v = torch.fft.irfft(torch.fft.rfft(g, 2 * n) * kt, 2 * n)[:n]
        else:
            v = torch.fft.irfft2(torch.fft.rfft2(g.view(n, n), (2 * n, 2 * n)) * kt, (2 * n, 2 * n))[:n, :n]
        out.append((w * v.reshape(-1)[node]).sum(1))
    return out


def _fft_gradient(P, Y, df, exag):
    N, D = Y.shape
    grid = _grid(Y)
    one = torch.ones(N, device=Y.device, dtype=F64)
    phi = _potentials(Y, [one] + [Y[:, d] for d in range(D)], lambda r2: (1 + r2 / df) ** -(df + 1), grid)
    if df == 1.0:
        sq = (Y * Y).sum(1)
        extra, = _potentials(Y, [sq], lambda r2: (1 + r2) ** -2.0, grid)
        Z = ((1 + sq) * phi[0] - 2 * sum(Y[:, d] * phi[1 + d] for d in range(D)) + extra).sum() - N
    else:
        Z = _potentials(Y, [one], lambda r2: (1 + r2 / df) ** -df, grid)[0].sum() - N
    neg = torch.stack([Y[:, d] * phi[0] - phi[1 + d] for d in range(D)], 1)
    return _attraction(P, Y, df, exag) - neg / Z, Z


def _exact_gradient(P, Y, df, exag):
    N, D = Y.shape
    att, rep, Z = torch.zeros_like(Y), torch.zeros_like(Y), 0.0
    for a in range(0, N, 1024):
        d2 = torch.zeros(min(1024, N - a), N, device=Y.device, dtype=F64)
        for d in range(D):
            d2 += (Y[a:a + 1024, d, None] - Y[None, :, d]) ** 2
        q = 1 / (1 + d2 / df)
        qd = q if df == 1.0 else q ** df
        own = torch.arange(a, min(a + 1024, N), device=Y.device)
        qd = qd.clone()
        qd[own - a, own] = 0
        Z = Z + qd.sum()
        for w, out in ((exag * P[a:a + 1024] * q, att), (qd * q, rep)):
            w[own - a, own] = 0
            out[a:a + 1024] = Y[a:a + 1024] * w.sum(1, keepdim=True) - w @ Y
    return att - rep / Z, Z


def _bh_forces(Y, theta):
    """Barnes-Hut repulsion and Z: cells level by level, then every point's open cells level by level."""
    N, D = Y.shape
    dev = Y.device
    mean = Y.mean(0)
    hw = torch.maximum(Y.max(0).values - mean, mean - Y.min(0).values) + 1e-5
    cen, cell, live = mean[None, :], torch.zeros(N, dtype=torch.int64, device=dev), torch.arange(N, device=dev)
    pt, at = torch.arange(N, device=dev), torch.zeros(N, dtype=torch.int64, device=dev)
    neg, Q = torch.zeros_like(Y), torch.zeros(N, dtype=F64, device=dev)
    while pt.numel():
        C = cen.shape[0]
        cum = torch.bincount(cell, minlength=C)
        com = torch.zeros(C, D, dtype=F64, device=dev).index_add_(0, cell, Y[live]) / cum[:, None]
        leaf = cum == 1
        one = torch.full((C,), -1, dtype=torch.int64, device=dev)
        one[cell[leaf[cell]]] = live[leaf[cell]]
        # children of the cells that hold several points: upper half of a dimension first
        inner = ~leaf[cell]
        live, parent = live[inner], cell[inner]
        up = Y[live] >= cen[parent]
        code = sum((~up[:, d]).long() << d for d in range(D))
        key, nxt = torch.unique(parent * (1 << D) + code, return_inverse=True)
        child = torch.full((C, 1 << D), -1, dtype=torch.int64, device=dev)
        child.view(-1)[key] = torch.arange(key.numel(), device=dev)
        # the points' open cells of this level
        keep = one[at] != pt
        pt, at = pt[keep], at[keep]
        diff = Y[pt] - com[at]
        d2 = (diff * diff).sum(1)
        take = leaf[at] | (hw.max() / d2.sqrt() < theta)
        q = 1 / (1 + d2[take])
        m = cum[at[take]] * q
        Q.index_add_(0, pt[take], m)
        neg.index_add_(0, pt[take], (m * q)[:, None] * diff[take])
        pt, at = pt[~take], at[~take]
        sub = child[at]
        pt = pt[:, None].expand_as(sub)[sub >= 0]
        at = sub[sub >= 0]
        down = torch.stack([((key >> d) & 1).to(F64) for d in range(D)], 1)
        cen = cen[key >> D] + (1 - 2 * down) * 0.5 * hw
        hw, cell = 0.5 * hw, nxt
    return neg, Q.sum()


def _iterate(Y, steps, lr, gradient):
    u, gains, Z = torch.zeros_like(Y), torch.ones_like(Y), None
    for _ in range(steps):
        dY, Z = gradient(Y)
        gains = torch.where(torch.sign(dY) != torch.sign(u), gains + 0.2, gains * 0.8).clamp_min(0.01)
        u = 0.8 * u - lr * gains * dY
        norm = (u * u).sum(1, keepdim=True).sqrt()
        u = torch.where(norm > 5.0, u * (5.0 / norm), u)
        Y = Y + u
        Y = Y - Y.mean(0, keepdim=True)
    return Y, Z


def _neighbours(X, K):
    N = X.shape[0]
    sq = (X * X).sum(1)
    step = max(64, min(4096, (1 << 28) // N))
    out = []
    for a in range(0, N, step):
        d2 = sq[a:a + step, None] + sq[None, :] - 2 * (X[a:a + step] @ X.T)
        own = torch.arange(a, min(a + step, N), device=X.device)
        d2[own - a, own] = math.inf
        near = torch.topk(d2, min(K + 8, N - 1), dim=1, largest=False).indices
        diff = X[a:a + step, None, :] - X[near]
        d = (diff * diff).sum(2).sqrt()
        d, at = torch.sort(d, dim=1)
        out.append((d[:, :K], torch.gather(near, 1, at)[:, :K]))
    return torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out])


def _calibrate(d2, perplexity, skip=None):
    """Rows of exp(-beta d2) / sum with entropy log(perplexity) within 1e-5: doubling and halving from 1, then bisection."""
    n = d2.shape[0]
    beta = torch.ones(n, 1, device=d2.device, dtype=F64)
    lo, hi = torch.full_like(beta, -math.inf), torch.full_like(beta, math.inf)
    out_beta, at = torch.ones(n, device=d2.device, dtype=F64), torch.arange(n, device=d2.device)
    P = torch.empty_like(d2)
    for _ in range(200):
        v = torch.exp(-beta * d2[at])
        if skip is not None:
            v[torch.arange(at.numel(), device=d2.device), skip[at]] = DBL_MIN
        s = v.sum(1, keepdim=True) + DBL_MIN
        H = beta * (d2[at] * v).sum(1, keepdim=True) / s + torch.log(s)
        off = H - math.log(perplexity)
        done = (off.abs() < 1e-5)[:, 0]
        P[at[done]] = (v / s)[done]
        out_beta[at[done]] = beta[done, 0]
        lo, hi = torch.where(off > 0, beta, lo), torch.where(off > 0, hi, beta)
        beta = torch.where(off > 0, torch.where(torch.isinf(hi), beta * 2, (beta + hi) / 2),
                           torch.where(torch.isinf(lo), beta / 2, (beta + lo) / 2))
        lo, hi, beta, at = lo[~done], hi[~done], beta[~done], at[~done]
        if not at.numel():
            return P, out_beta
    return None


def _symmetric_values(idx, P):
    """Values of (P + P^T) / 2 row by row, each row's in the order of the directed entries that make it."""
    N, K = idx.shape
    n = torch.arange(N, device=idx.device)[:, None].expand(N, K).reshape(-1)
    c, v = idx.reshape(-1), P.reshape(-1)
    key, at = torch.sort(n * N + c)
    where = torch.searchsorted(key, c * N + n).clamp_max(key.numel() - 1)
    has = key[where] == c * N + n
    v2 = torch.where(has, v + v[at[where]], v) / 2
    e = torch.nonzero(~has | (n <= c))[:, 0]
    rows, both = torch.cat([n[e], c[e]]), torch.cat([e, e])
    val = v2[both][torch.argsort(rows * key.numel() + both)]
    return torch.cat([val, torch.zeros(2 * N * K - val.numel(), device=val.device, dtype=F64)])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("affinities", "knn"):
        X = _data(case, case["D"], seed)
        if kind == "knn":
            return {"idx": None, "dist": _neighbours(X, case["K"])[0]}
        dist, idx = _neighbours(X, 3 * case["perplexity"])
        got = _calibrate(dist, float(case["perplexity"]))
        if got is None:
            return None
        return {"idx": None, "dist": dist, "beta": got[1], "iters": None, "row": None, "col": None,
                "val": _symmetric_values(idx, got[0])}
    if kind == "exact":
        X, Y, N = _data(case, case["data_dim"], seed), _start(case, seed), case["N"]
        d2 = torch.zeros(N, N, device=DEV, dtype=F64)
        for d in range(X.shape[1]):
            d2 += (X[:, d, None] - X[None, :, d]) ** 2
        got = _calibrate(d2, float(case["perplexity"]), torch.arange(N, device=DEV))
        if got is None:
            return None
        P = got[0] + got[0].T
        P.fill_diagonal_(DBL_MIN)
        P /= P.sum()
        Y, _ = _iterate(Y, case["steps"], _lr(N), lambda y: _exact_gradient(P, y, case["df"], case["exag"]))
        _, Z = _exact_gradient(P, Y, case["df"], case["exag"])
        kl = 0.0
        for a in range(0, N, 1024):
            r2 = torch.zeros(min(1024, N - a), N, device=DEV, dtype=F64)
            for d in range(case["D"]):
                r2 += (Y[a:a + 1024, d, None] - Y[None, :, d]) ** 2
            Q = (1 / (1 + r2 / case["df"])) ** case["df"]
            own = torch.arange(a, min(a + 1024, N), device=DEV)
            Q[own - a, own] = DBL_MIN
            p = case["exag"] * P[a:a + 1024]
            kl = kl + (p * torch.log((p + FLT_MIN) / (Q / Z + FLT_MIN))).sum()
        return {"kl": float(kl), "Y": Y}
    if kind == "batch":
        out = []
        for i, N in enumerate(_sizes(case)):
            P, Y = _embedding(case, N, seed * 101 + i)
            out.append(_iterate(Y, case["steps"], _lr(N), lambda y: _fft_gradient(P, y, case["df"], case["exag"]))[0])
        return out
    P, Y = _embedding(case, case["N"], seed)
    if kind == "mirror":
        dC, Z = _fft_gradient(P, Y, case["df"], 1.0)
        return {"dC": dC, "Z": float(Z)}
    if kind == "bh":
        def gradient(y):
            neg, Z = _bh_forces(y, case["theta"])
            return _attraction(P, y, 1.0, case["exag"]) - neg / Z, Z
    else:
        def gradient(y):
            return _fft_gradient(P, y, case["df"], case["exag"])
    Y, Z = _iterate(Y, case["steps"], _lr(case["N"]), gradient)
    if kind != "run":
        return {"Y": Y}
    kl = 0.0
    for i, j, v in _edges(P):
        r2 = ((Y[i] - Y[j]) ** 2).sum(1)
        p = case["exag"] * v
        kl = kl + (p * torch.log((p + FLT_MIN) / ((1 / (1 + r2 / case["df"])) ** case["df"] / Z + FLT_MIN))).sum()
    return {"kl": float(kl), "Y": Y}
