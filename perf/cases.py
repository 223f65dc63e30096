"""The work that programs have this package do on one MI355X, as cases to time.

Five kinds of pass, each through the entry points that a program calls:

=======  ==============================================================================
kind     one pass
=======  ==============================================================================
fit      the whole ``HipKMeans.fit`` on host data: tolerance, upload, k-means++, Lloyd
         to convergence, final E-step, results back on the host
lloyd    a fit from given centres on an X that is resident in HBM (``LloydHandle``:
         set_centers, run, centers, labels), as a program with several runs makes it
seed     k-means++ seeding of a resident X with given draws
parinit  skmetal's k-means|| seeding (``kmeans_parallel_init``) of a resident X
apply    predict and transform of host rows against given centres
=======  ==============================================================================

Data: Gaussian blobs of unit width ("blobs"; ``spread`` is the standard deviation of
the blobs' centres per feature, so a small spread makes them overlap as real clusters
do), the same with Zipf(1.2) blob sizes ("zipf"), unit vectors around random directions
("unit", the law of text and image embeddings), and colours in [0, 1] ("colours").
All data are fp32, the one type that the package takes.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from skmetal_amd import _bridge
from skmetal_amd.estimators.cluster import HipKMeans, kmeans_parallel_init

MAX_FLOPS = 1.9e12  # 2nkd over the steps of a drawn case (the largest listed one: 2.2e12)
MAX_VALUES = 1.3e8  # n * d of a drawn case (the largest listed one: 1.28e8)


def listed():
    return [
        # a small table through the estimator: host work, launches and latency
        dict(name="fit_2k_16_k8", kind="fit", n=2_000, d=16, k=8, law="blobs", spread=2.0, iters=300),
        # the README's headline size through the estimator, from host rows to labels
        dict(name="fit_500k_100_k50", kind="fit", n=500_000, d=100, k=50, law="blobs", spread=5.0, iters=300),
        # the small resident fit: short kernels, where launches count
        dict(name="lloyd_100k_32_k8", kind="lloyd", n=100_000, d=32, k=8, law="blobs", spread=0.6, iters=20),
        # the headline size, resident
        dict(name="lloyd_500k_100_k50", kind="lloyd", n=500_000, d=100, k=50, law="blobs", spread=0.45, iters=20),
        # hundreds of clusters: distance work bound by the matrix cores
        dict(name="lloyd_1m_128_k256", kind="lloyd", n=1_000_000, d=128, k=256, law="blobs", spread=0.4, iters=10),
        # a codebook of a thousand centres on skewed clusters
        dict(name="lloyd_2m_64_k1024", kind="lloyd", n=2_000_000, d=64, k=1024, law="zipf", spread=0.9, iters=5),
        # embedding vectors: long rows, thousands of centres
        dict(name="lloyd_100k_768_k2048", kind="lloyd", n=100_000, d=768, k=2048, law="unit", spread=0.15, iters=6),
        # colour quantisation of a picture of a million pixels
        dict(name="lloyd_1m_3_k64", kind="lloyd", n=1_000_000, d=3, k=64, law="colours", spread=0.1, iters=10),
        # no size a multiple of anything
        dict(name="lloyd_250007_37_k101", kind="lloyd", n=250_007, d=37, k=101, law="blobs", spread=0.6, iters=10),
        # seeding alone, many centres
        dict(name="seed_300k_60_k200", kind="seed", n=300_000, d=60, k=200, law="blobs", spread=0.5, iters=1),
        # skmetal's own seeding at the headline size
        dict(name="parinit_500k_100_k50", kind="parinit", n=500_000, d=100, k=50, law="blobs", spread=0.5, iters=1),
        # new rows against a fitted model: labels and distances
        dict(name="apply_200k_100_k50", kind="apply", n=200_000, d=100, k=50, law="blobs", spread=0.5, iters=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["fit", "lloyd", "lloyd", "lloyd", "lloyd", "seed", "parinit", "apply"])
        n, d = _log(rng, 1_000, 2_000_000), _log(rng, 2, 768)
        k = _log(rng, 2, 2048 if kind == "lloyd" else 256)
        iters = rng.randint(3, 20) if kind == "lloyd" else 300 if kind == "fit" else 1
        if kind == "lloyd":
            law = rng.choice(["blobs", "zipf", "unit" if d >= 64 else "blobs", "colours" if d <= 4 else "blobs"])
        else:
            law = "blobs"
        # overlapping blobs for a given number of steps, separate ones where a fit runs to convergence
        spread = {"unit": 0.15, "colours": 0.1}.get(law) or (5.0 if kind == "fit" else round(rng.uniform(4, 6) / math.sqrt(d), 3))
        steps = {"lloyd": iters, "fit": 10, "seed": 2 + int(math.log(k)), "parinit": 2 + int(math.log(k)), "apply": 2}[kind]
        if 8 * k <= n and n * d <= MAX_VALUES and 2.0 * n * d * k * steps <= MAX_FLOPS and n * k <= 1e9:
            if kind != "apply" or n * k <= 2e7:
                return dict(kind=kind, n=n, d=d, k=k, law=law, spread=spread, iters=iters)


class KMeans:
    """An estimator's parameters under scikit-learn's names, and what a fit sets on it."""

    def __init__(self, n_clusters, init, max_iter, random_state):
        self.n_clusters = n_clusters
        self.init = init
        self.n_init = 1
        self.max_iter = max_iter
        self.tol = 1e-4
        self.random_state = random_state


def _data(case, seed):
    """X [n x d] and k starting centres, on the device, from the seed.  The centres are the
    means of the blobs' rows in a sample of X, as a fit of that sample gives them: from
    random rows instead, fits of many clusters split blobs at random, and the steps then
    amplify the last bit of every sum until no two correct programs agree."""
    n, d, k, law, spread = case["n"], case["d"], case["k"], case["law"], case["spread"]
    g = torch.Generator(device="cuda").manual_seed(1_000_003 * (seed % 1_000_000) + 17)
    cen = torch.randn(k, d, device="cuda", generator=g)
    if law == "zipf":
        w = torch.arange(1, k + 1, device="cuda", dtype=torch.float64) ** -1.2
        edge = torch.cumsum(w, 0) / w.sum()
        lab = torch.searchsorted(edge, torch.rand(n, device="cuda", generator=g, dtype=torch.float64)).clamp_(max=k - 1)
    else:
        lab = torch.randint(0, k, (n,), device="cuda", generator=g)
    X = torch.randn(n, d, device="cuda", generator=g)
    if law == "unit":
        X.mul_(spread).add_(torch.nn.functional.normalize(cen, dim=1)[lab])
        X = torch.nn.functional.normalize(X, dim=1)
    elif law == "colours":
        X.mul_(spread).add_((0.5 + 0.2 * cen)[lab]).abs_()
        X = torch.where(X > 1.0, 2.0 - X, X).clamp_(min=0.0)
    else:
        X.add_((cen * spread)[lab])
    m = min(n // 2, 64 * k) if law in ("zipf", "unit") else min(n, 16 * k)
    C = torch.zeros(k, d, device="cuda", dtype=torch.float64).index_add_(0, lab[:m], X[:m].double())
    size = torch.bincount(lab[:m], minlength=k)
    C = torch.where(size[:, None] > 0, C / size.clamp(min=1)[:, None], X[n - k:].double()).float()
    return X, C


def prepare(case, seed):
    n, d, k, kind = case["n"], case["d"], case["k"], case["kind"]
    X, C = _data(case, seed)
    X, C = X.cpu().numpy(), C.cpu().numpy()
    state = dict(case=case, seed=seed % (1 << 31))
    if kind in ("fit", "parinit", "apply"):
        state["X"] = X
    if kind in ("lloyd", "seed", "parinit"):
        state["h"] = _bridge.LloydHandle(n, d, k)
        state["h"].load(X, center=kind != "parinit")
    if kind in ("lloyd", "apply"):
        state["C"] = C
    if kind == "seed":
        state["draws"] = _bridge.plusplus_draws(np.random.RandomState(state["seed"]), n, k)
    return state


def run(state):
    case = state["case"]
    n, d, k, kind = case["n"], case["d"], case["k"], case["kind"]
    if kind == "fit":
        est = KMeans(k, "k-means++", case["iters"], state["seed"])
        HipKMeans(est).fit(state["X"])
        return dict(centers=est.cluster_centers_, labels=est.labels_, inertia=est.inertia_)
    if kind == "lloyd":
        h = state["h"]
        h.set_centers(state["C"])
        _, inertia = h.run(case["iters"], 0.0, strict=False)
        return dict(centers=h.centers(), labels=h.labels(), inertia=inertia)
    if kind == "seed":
        rows = state["h"].plusplus_with(*state["draws"])
        return dict(rows=rows, centers=state["h"].centers())
    if kind == "parinit":
        return dict(centers=kmeans_parallel_init(state["X"], k, np.random.RandomState(state["seed"]), state["h"]))
    labels = np.empty(n, np.int32)
    _bridge.kmeans_assign(state["X"], state["C"], labels, n, d, k)
    return dict(labels=labels, distances=_bridge.kmeans_transform(state["X"], state["C"]))


def work(case):
    n, d, k, kind = case["n"], case["d"], case["k"], case["kind"]
    X, trials = 4.0 * n * d, 2 + int(math.log(k))
    if kind == "lloyd":  # every step needs every row; the labels come out once
        return dict(bytes=(case["iters"] + 1) * X + 4.0 * n, flops=(case["iters"] + 1) * 2.0 * n * k * d)
    if kind == "seed":  # every centre is drawn by the distances to the one before
        return dict(bytes=k * (X + 8.0 * n), flops=((k - 1) * trials + 1) * 2.0 * n * d)
    if kind == "parinit":  # a round's rows are drawn by the distances to the round before
        return dict(bytes=trials * (X + 8.0 * n), flops=((trials - 1) * k + 1) * 2.0 * n * d)
    if kind == "apply":
        return dict(bytes=X + 4.0 * n + 4.0 * n * k, flops=2 * 2.0 * n * k * d)
    # fit: the column variances, the seeding, two steps and the final E-step at least
    return dict(bytes=2 * X + k * (X + 8.0 * n) + 3 * X + 4.0 * n, flops=((k - 1) * trials + 1 + 3 * k) * 2.0 * n * d)


def tolerance(case):
    """fp32 results.  Rows that lie within the rounding of the distances of two centres
    may take either label, and a centre then moves by that row's share of it."""
    kind = case["kind"]
    if kind == "lloyd":  # ten rows a centre in the smallest clusters of unit vectors
        return dict(rel=1e-2 if case["law"] == "unit" else 5e-4, max=3e-1, differ=1e-3)
    if kind == "fit":
        return dict(rel=2e-3, max=3e-1, differ=2e-3)
    if kind == "seed":
        return dict(rel=1e-6, max=1e-5, differ=0.0)
    if kind == "parinit":
        return dict(rel=1e-5, max=1e-3, differ=0.0)
    return dict(rel=1e-6, max=1e-3, differ=1e-4)


# ---- the same results in 64 bits ----


def _sq(A, B):
    """Squared distances of A's rows to B's, [a x b], fp64."""
    return (A.square().sum(1)[:, None] - 2.0 * (A @ B.T) + B.square().sum(1)[None, :]).clamp_(min=0.0)


def _blocks(n, width):
    step = max(1, (1 << 26) // max(1, width))
    return [(s, min(n, s + step)) for s in range(0, n, step)]


def _assign(X, C):
    lab = torch.empty(len(X), dtype=torch.int64, device=X.device)
    low = torch.empty(len(X), dtype=torch.float64, device=X.device)
    for a, b in _blocks(len(X), max(X.shape[1], len(C))):
        low[a:b], lab[a:b] = _sq(X[a:b].double(), C).min(1)
    return lab, low


def _lloyd(X, C, max_iter, tol, strict):
    """scikit-learn's Lloyd loop: centres, labels, inertia.  X fp32 on the device, C fp64."""
    k, old = len(C), None
    converged = False
    for _ in range(max_iter):
        lab, low = _assign(X, C)
        S = torch.zeros_like(C)
        for a, b in _blocks(len(X), X.shape[1]):
            S.index_add_(0, lab[a:b], X[a:b].double())
        cnt = torch.bincount(lab, minlength=k).double()
        empty = torch.nonzero(cnt == 0).flatten().tolist()
        if empty and float(low.max()) > 0:  # the farthest rows move to the empty clusters
            for j, r in zip(empty, torch.argsort(low, descending=True, stable=True)[: len(empty)].tolist()):
                o, x = int(lab[r]), X[r].double()
                S[o] -= x
                cnt[o] -= 1
                S[j], cnt[j] = x, 1
        new = S / cnt.clamp(min=1)[:, None]
        new[cnt == 0] = new[int(cnt.argmax())].clone()
        shift = float((new - C).square().sum())
        C = new
        if strict and old is not None and torch.equal(old, lab):
            converged = True
            break
        if shift <= tol:
            break
        old = lab
    if not converged:
        lab, _ = _assign(X, C)
    inertia = sum(float((X[a:b].double() - C[lab[a:b]]).square().sum()) for a, b in _blocks(len(X), X.shape[1]))
    return C, lab, inertia


def _nearest(X, C, low):
    """low, lowered by the fp32 squared distances to C's rows: [len(C) x n] fp32."""
    D = torch.empty(len(C), len(X), dtype=torch.float32, device=X.device)
    for a, b in _blocks(len(X), X.shape[1]):
        D[:, a:b] = _sq(X[a:b].double(), C).T.float()
    return torch.minimum(D, low[None, :])


def _plusplus(X, trials, first, u):
    """k-means++ from given draws: the rows taken."""
    rows = [first]
    low = _nearest(X, X[[first]].double(), torch.full((len(X),), math.inf, device=X.device))[0]
    for r in u:
        sums = torch.cumsum(low.double(), 0)
        pot = float(sums[-1].float())
        at = torch.searchsorted(sums, torch.from_numpy(r * pot).to(X.device)).clamp_(max=len(X) - 1)
        D = _nearest(X, X[at].double(), low)
        best = int(D.double().sum(1).argmin())
        rows.append(int(at[best]))
        low = D[best]
    return rows


def _parallel(X, k, rng):
    """skmetal's k-means|| seeding: k centres."""
    n = len(X)
    rows = [int(rng.randint(n))]
    taken, new = {0}, rows[:]
    low = torch.full((n,), math.inf, device=X.device)
    for _ in range(max(1, int(2 + np.log(k)))):
        for a in range(0, len(new), 32):
            low = _nearest(X, X[new[a:a + 32]].double(), low).min(0).values
        w = np.maximum(low.cpu().numpy(), np.float32(1e-30))
        new = []
        for i in rng.choice(n, min(k, n), replace=False, p=w / w.sum()).tolist():
            if i not in taken:
                taken.add(i)
                new.append(i)
        rows += new
    cand = X[rows]
    if len(rows) <= k:
        return cand[[i % len(rows) if i >= len(rows) else i for i in range(k)]].double()
    mean = cand.double().mean(0).float()
    C, _, _ = _lloyd(cand - mean, (cand[:k] - mean).double(), 1, 0.0, True)
    return C + mean.double()


def exact(case, seed):
    k, kind = case["k"], case["kind"]
    X, C = _data(case, seed)
    if kind == "apply":
        lab, dist = [], []
        for a, b in _blocks(len(X), max(X.shape[1], k)):
            D = _sq(X[a:b].double(), C.double())
            lab.append(D.argmin(1))
            dist.append(D.sqrt())
        return dict(labels=torch.cat(lab), distances=torch.cat(dist))
    seed %= 1 << 31
    if kind == "parinit":
        return dict(centers=_parallel(X, k, np.random.RandomState(seed)))
    mean = X.double().mean(0).float()
    Xc = X - mean  # fp32, as scikit-learn centres its data
    if kind == "lloyd":
        C, lab, inertia = _lloyd(Xc, (C - mean).double(), case["iters"], 0.0, False)
        return dict(centers=C + mean.double(), labels=lab, inertia=inertia)
    rows = _plusplus(Xc, *_bridge.plusplus_draws(np.random.RandomState(seed), len(X), k))
    if kind == "seed":
        return dict(rows=torch.tensor(rows), centers=X[rows].double())
    tol = 1e-4 * float(X.double().var(0, unbiased=False).mean())
    C, lab, inertia = _lloyd(Xc, Xc[rows].double(), case["iters"], tol, True)
    return dict(centers=C + mean.double(), labels=lab, inertia=inertia)
