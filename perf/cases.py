"""The calls by which this package's speed is measured.

Every case is one call that a user of the package makes with the data at hand:
a merge tree (`linkage`), a fitted estimator (`AgglomerativeClustering`,
`HDBSCAN`) or a distance matrix (`pairwise_distances`). The listed sizes are
those of the package's own benchmark and tests, and general ones beside them;
`draw` gives others of the same ranges.

A case's keys:
  path      "pairwise", "linkage", "agglomerative" or "hdbscan"
  n, d      points and features (m: rows of the second matrix of a pairwise call)
  metric    the distance
  method    the linkage, where there is one
  k         HDBSCAN's min_cluster_size (and min_samples)
  clusters  flat clusters an AgglomerativeClustering is asked for
  data      "normal" (i.i.d. N(0, 1)), "unit" (N(0, 1) rows of norm 1) or
            "blobs" (20 Gaussian blobs, every tenth point uniform noise)
  held      where the program holds its points: "device" (a float32 tensor in
            GPU memory), "host" (a float32 array) or "host64" (a float64 array)
"""

import math

import numpy as np
import torch

import cuhc_amd as cuhc

# Above these sizes the 64-bit results take too long in plain torch.
PRIM_MOST = 60_000
CHAIN_MOST = 6_000


def listed():
    return [
        # A distance matrix between two sets of embeddings, ragged on both sides.
        dict(name="pairwise_12k_7k_d50", path="pairwise", n=12_345, m=6_789, d=50,
             metric="euclidean", data="normal", held="device"),
        # An interactive call on a small table: latency and launches.
        dict(name="single_500_d2", path="linkage", n=500, d=2, metric="euclidean",
             method="single", data="blobs", held="host64"),
        # The ordinary single-linkage tree (the benchmark's small workload).
        dict(name="single_20k_d32", path="linkage", n=20_000, d=32, metric="euclidean",
             method="single", data="normal", held="device"),
        # Another metric, with the points in host memory and few features: FP32 passes.
        dict(name="single_manhattan_50k_d10", path="linkage", n=50_021, d=10, metric="manhattan",
             method="single", data="normal", held="host"),
        # The headline tree of a million points.
        dict(name="single_1M_d32", path="linkage", n=1_000_000, d=32, metric="euclidean",
             method="single", data="normal", held="device"),
        # A notebook's HDBSCAN: a few thousand rows of a table in float64.
        dict(name="hdbscan_2k_d5", path="hdbscan", n=2_003, d=5, metric="euclidean", k=5,
             data="blobs", held="host64"),
        # HDBSCAN of an ordinary data set.
        dict(name="hdbscan_100k_d8", path="hdbscan", n=100_000, d=8, metric="euclidean", k=25,
             data="blobs", held="host"),
        # HDBSCAN of a million points already on the GPU.
        dict(name="hdbscan_1M_d8", path="hdbscan", n=1_000_000, d=8, metric="euclidean", k=25,
             data="blobs", held="device"),
        # The estimator's default (ward) on a table of a few thousand rows.
        dict(name="ward_3k_d13", path="agglomerative", n=3_001, d=13, metric="euclidean",
             method="ward", clusters=8, data="blobs", held="host64"),
        # The large Ward tree.
        dict(name="ward_100k_d32", path="linkage", n=100_000, d=32, metric="euclidean",
             method="ward", data="normal", held="device"),
        # A stored distance matrix, ordinary size.
        dict(name="complete_5k_d20", path="linkage", n=5_003, d=20, metric="euclidean",
             method="complete", data="normal", held="host"),
        # The largest stored matrix (20 GB): average linkage of embeddings by cosine.
        dict(name="average_cosine_100k_d64", path="linkage", n=100_000, d=64, metric="cosine",
             method="average", data="unit", held="device"),
    ]


def _size(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["pairwise", "linkage", "linkage", "agglomerative", "hdbscan", "dense"])
    held = rng.choice(["device", "host", "host64"])
    if path == "pairwise":
        return dict(path=path, n=_size(rng, 300, 20_000), m=_size(rng, 300, 10_000),
                    d=_size(rng, 2, 256), data="normal", held="device",
                    metric=rng.choice(["euclidean", "sqeuclidean", "manhattan", "cosine"]))
    if path == "hdbscan":
        return dict(path=path, n=_size(rng, 1_000, 500_000), d=rng.randint(2, 10),
                    metric=rng.choice(["euclidean", "euclidean", "manhattan"]),
                    k=_size(rng, 5, 50), data="blobs", held=held)
    if path == "agglomerative":
        return dict(path=path, n=_size(rng, 500, 60_000), d=_size(rng, 4, 64),
                    metric="euclidean", method="ward", clusters=rng.randint(2, 30),
                    data=rng.choice(["normal", "blobs"]), held=held)
    if path == "dense":
        metric = rng.choice(["euclidean", "cosine"])
        return dict(path="linkage", n=_size(rng, 500, 40_000), d=_size(rng, 8, 128),
                    metric=metric, method=rng.choice(["complete", "average"]),
                    data="unit" if metric == "cosine" else "normal", held=held)
    if rng.random() < 0.5:  # features enough for the matrix cores
        return dict(path="linkage", n=_size(rng, 500, 800_000), d=rng.randint(16, 64),
                    metric=rng.choice(["euclidean", "sqeuclidean"]), method="single",
                    data="normal", held=held)
    return dict(path="linkage", n=_size(rng, 500, 100_000), d=_size(rng, 2, 100),
                metric=rng.choice(["euclidean", "manhattan", "chebyshev", "cosine"]),
                method="single", data=rng.choice(["normal", "blobs"]), held=held)


def _points(case, seed, n):
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = case["d"]
    X = torch.randn(n, d, generator=g, device="cuda")
    if case["data"] == "unit":
        X /= X.norm(dim=1, keepdim=True)
    elif case["data"] == "blobs":
        centres = torch.rand(20, d, generator=g, device="cuda") * 20 - 10
        X += centres[torch.arange(n, device="cuda") % 20]
        low, high = X.min(0).values, X.max(0).values
        noise = torch.rand(n, d, generator=g, device="cuda") * (high - low) + low
        every_tenth = (torch.arange(n, device="cuda") // 20 % 10 == 9).unsqueeze(1)
        X = torch.where(every_tenth, noise, X)
    return X.contiguous()


def _held(X, where):
    if where == "device":
        return X
    X = X.cpu().numpy()
    return X.astype(np.float64) if where == "host64" else X


def prepare(case, seed):
    X = _points(case, 2 * seed, case["n"])
    state = dict(case, X=_held(X, case["held"]))
    if case["path"] == "pairwise":
        state["Y"] = _held(_points(case, 2 * seed + 1, case["m"]), case["held"])
    return state


def _tree(Z):
    """A scipy-format tree as its columns (views): whole numbers and heights apart."""
    return {"merged": Z[:, :2], "heights": Z[:, 2], "sizes": Z[:, 3]}


def run(state):
    path = state["path"]
    if path == "pairwise":
        out = cuhc.pairwise_distances(state["X"], state["Y"], metric=state["metric"])
        return {"distances": torch.as_tensor(out, device="cuda")}
    if path == "linkage":
        return _tree(cuhc.linkage(state["X"], method=state["method"], metric=state["metric"]))
    if path == "agglomerative":
        fit = cuhc.AgglomerativeClustering(n_clusters=state["clusters"], metric=state["metric"],
                                           linkage=state["method"], compute_distances=True)
        fit.fit(state["X"])
        return {"labels": fit.labels_, "children": fit.children_, "distances": fit.distances_}
    fit = cuhc.HDBSCAN(min_cluster_size=state["k"], metric=state["metric"]).fit(state["X"])
    return {"labels": fit.labels_, "probabilities": fit.probabilities_,
            "core_distances": fit.core_distances_, "tree": _tree(fit._single_linkage_tree_)}


def work(case):
    n, d, path = case["n"], case["d"], case["path"]
    points, tree = 4.0 * n * d, 32.0 * (n - 1)
    if path == "pairwise":
        m = case["m"]
        return {"bytes": 4.0 * d * (n + m) + 4.0 * n * m, "flops": 2.0 * n * m * d}
    if path == "hdbscan":
        # k neighbours of every point and the tree's edges: pruning may skip the rest.
        return {"bytes": points + tree + 20.0 * n, "flops": 2.0 * d * n * (case["k"] + 1)}
    pairs = 0.5 * n * (n - 1)
    if case["method"] in ("complete", "average"):
        # Every distance once, and one update for each cluster left at each merge.
        return {"bytes": points + tree, "flops": pairs * (2.0 * d + 3.0)}
    return {"bytes": points + tree, "flops": pairs * 2.0 * d}


# ---- The results in 64 bits -------------------------------------------------


def _row_distances(X, i, metric):
    """Distances of point i to every point."""
    diff = X - X[i]
    if metric == "manhattan":
        return diff.abs().sum(1)
    if metric == "chebyshev":
        return diff.abs().amax(1)
    if metric == "cosine":  # rows of norm 1
        return 1.0 - (X * X[i]).sum(1)
    sq = diff.square().sum(1)
    return sq if metric == "sqeuclidean" else sq.sqrt()


def _matrix(X, Y, metric):
    if metric == "cosine":
        return 1.0 - X @ Y.T.contiguous()
    D = torch.zeros(len(X), len(Y), dtype=X.dtype, device=X.device)
    for f in range(X.shape[1]):
        diff = X[:, f].unsqueeze(1) - Y[:, f].unsqueeze(0)
        if metric == "manhattan":
            D += diff.abs()
        elif metric == "chebyshev":
            D = torch.maximum(D, diff.abs())
        else:
            D += diff.square()
    return D.sqrt() if metric == "euclidean" else D


def _prim_heights(X, metric, core=None):
    """Sorted edge weights of the minimum spanning tree."""
    n = len(X)
    best = torch.full((n,), math.inf, dtype=X.dtype, device=X.device)
    left = torch.zeros_like(best)  # infinite once a point is in the tree
    weights = torch.empty(n - 1, dtype=X.dtype, device=X.device)
    i = torch.zeros(1, dtype=torch.int64, device=X.device)
    for e in range(n - 1):
        left.index_fill_(0, i, math.inf)
        w = _row_distances(X, i, metric)
        if core is not None:
            w = torch.maximum(torch.maximum(w, core), core[i])
        best = torch.minimum(best, w)
        value, i = (best + left).min(0, keepdim=True)
        weights[e:e + 1] = value
    return weights.sort().values


def _chain_heights(D, method):
    """Sorted merge heights of a reducible linkage from its distance matrix
    (nearest-neighbour chain with Lance-Williams updates; ward on squares)."""
    n = len(D)
    D = D.square() if method == "ward" else D.clone()
    D.fill_diagonal_(math.inf)
    size = torch.ones(n, dtype=D.dtype, device=D.device)
    alive = np.ones(n, dtype=bool)
    heights, chain, first = [], [], 0
    while len(heights) < n - 1:
        if not chain:
            while not alive[first]:
                first += 1
            chain.append(first)
        a = chain[-1]
        low, at = D[a].min(0)
        low, b = torch.stack([low, at.to(low.dtype)]).tolist()
        b = int(b)
        if len(chain) > 1 and float(D[a, chain[-2]]) <= low:
            b = chain[-2]
        if len(chain) < 2 or b != chain[-2]:
            chain.append(b)
            continue
        heights.append(low)
        del chain[-2:]
        if method == "complete":
            row = torch.maximum(D[a], D[b])
        elif method == "average":
            row = (size[a] * D[a] + size[b] * D[b]) / (size[a] + size[b])
        else:
            row = ((size[a] + size) * D[a] + (size[b] + size) * D[b] - size * low) / (
                size[a] + size[b] + size)
        size[a] += size[b]
        row[a] = row[b] = math.inf
        row = torch.where(torch.isfinite(D[a]) & torch.isfinite(D[b]), row, math.inf)
        D[a], D[:, a] = row, row
        D[b], D[:, b] = math.inf, math.inf
        alive[b] = False
    out = torch.tensor(heights, dtype=torch.float64).sort().values
    return out.sqrt() if method == "ward" else out


def _core(X, k, metric):
    """The k-th smallest distance of each point (itself counted)."""
    step = max(1, 200_000_000 // len(X))
    return torch.cat([_matrix(X[a:a + step], X, metric).kthvalue(k, dim=1).values
                      for a in range(0, len(X), step)])


def exact(case, seed):
    path, metric, n = case["path"], case["metric"], case["n"]
    most = CHAIN_MOST if case.get("method") in ("ward", "complete", "average") else PRIM_MOST
    if path != "pairwise" and n > most:
        return None
    X = _points(case, 2 * seed, n).double()
    if metric == "cosine":
        X /= X.norm(dim=1, keepdim=True)
    if path == "pairwise":
        Y = _points(case, 2 * seed + 1, case["m"]).double()
        if metric == "cosine":
            Y /= Y.norm(dim=1, keepdim=True)
        return {"distances": _matrix(X, Y, metric)}
    if path == "hdbscan":
        core = _core(X, case["k"], metric)
        return {"labels": None, "probabilities": None, "core_distances": core,
                "tree": {"merged": None, "heights": _prim_heights(X, metric, core),
                         "sizes": None}}
    if case["method"] == "single":
        return {"merged": None, "heights": _prim_heights(X, metric), "sizes": None}
    heights = _chain_heights(_matrix(X, X, metric), case["method"])
    if path == "agglomerative":
        return {"labels": None, "children": None, "distances": heights}
    return {"merged": None, "heights": heights, "sizes": None}
