"""
The measured cases of this package: what its users call, from the smallest calls to the largest.

``listed()`` names the cases, ``draw(rng)`` makes further ones over the same ranges, ``prepare`` builds what a
user's program holds before the call (data on the GPU as DNDarrays, initial centroids, a fitted estimator) and
``run`` is one pass through the public entry points of ``heat_amd``.

Data: Gaussian blobs with centres uniform in a box, uneven cluster sizes (a Dirichlet draw) and optionally a share
of uniform background noise, rows in random order -- what clusterings, neighbour searches and distance matrices
are run on.  Everything is drawn on the GPU from the seed.
"""

from __future__ import annotations

import math
import warnings

import torch

import heat_amd as ht

_CHUNK_VALUES = 1 << 26  # values generated at a time


def listed():
    return [
        # the reference's continuous benchmark: 20 000 points in space in four balls, k-means++ initialisation,
        # default stop rule -- a few hundred small launches and looks from the host
        {"name": "fit_plusplus_small", "path": "fit_plusplus", "n": 20000, "d": 3, "k": 4, "max_iter": 300,
         "tol": 1e-4, "box": 8.0, "sigma": 0.5},
        # k-means++ on a data set that fills the card: the initialiser reads the rows once per round
        {"name": "fit_plusplus_1m", "path": "fit_plusplus", "n": 1000000, "d": 32, "k": 256, "max_iter": 10,
         "tol": 0.0, "box": 5.0, "sigma": 0.5},
        # a fit small enough that launches and hand-overs count
        {"name": "fit_100k_d8_k16", "path": "fit", "n": 100000, "d": 8, "k": 16, "max_iter": 20, "box": 10.0,
         "sigma": 1.0},
        # an ordinary table: row count and width that are multiples of nothing
        {"name": "fit_odd_d50_k100", "path": "fit", "n": 999983, "d": 50, "k": 100, "max_iter": 10, "box": 5.0,
         "sigma": 1.0},
        # the headline configuration of the benchmark
        {"name": "fit_10m_d32_k256", "path": "fit", "n": 10000000, "d": 32, "k": 256, "max_iter": 10, "box": 5.0,
         "sigma": 0.5},
        # embeddings: wide rows, many clusters
        {"name": "fit_2m_d512_k1024", "path": "fit", "n": 2000000, "d": 512, "k": 1024, "max_iter": 5, "box": 3.5,
         "sigma": 1.0},
        # a point cloud: narrow rows, few clusters, some background noise
        {"name": "fit_200m_d3_k8", "path": "fit", "n": 200000000, "d": 3, "k": 8, "max_iter": 10, "box": 100.0,
         "sigma": 5.0, "noise": 0.05},
        # tables read with numpy arrive in float64 and stay there
        {"name": "fit_f64_1m_d18_k16", "path": "fit", "n": 1000000, "d": 18, "k": 16, "max_iter": 10, "box": 5.0,
         "sigma": 1.0, "dtype": "float64"},
        # labelling new rows with a finished clustering (distance + argmin, the benchmark's second configuration);
        # i.i.d. normal rows: no cluster is near
        {"name": "predict_1m_d64_k1024", "path": "predict", "n": 1048576, "d": 64, "k": 1024, "box": 0.0,
         "sigma": 1.0},
        # the reference's distance-matrix benchmark: 40 000 rows of 18 features against themselves, default form
        {"name": "cdist_40k_d18", "path": "cdist", "n": 40000, "m": 0, "d": 18, "box": 2.0, "sigma": 1.0,
         "expand": False},
        # classification of a test set by its nearest training rows
        {"name": "knn_32k_d64", "path": "knn", "n": 32768, "m": 32768, "d": 64, "k": 5, "box": 2.0, "sigma": 1.0},
        # the robust sibling estimator
        {"name": "kmedians_1m_d32_k64", "path": "kmedians", "n": 1000000, "d": 32, "k": 64, "max_iter": 10,
         "box": 5.0, "sigma": 1.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        path = rng.choice(["fit", "fit", "fit", "fit", "fit", "fit64", "fit_plusplus", "predict", "cdist", "knn",
                           "kmedians"])
        d = _log_int(rng, 2, 512)
        if path in ("fit", "fit64"):
            c = {"path": "fit", "n": _log_int(rng, 20000, 100000000), "d": d, "k": _log_int(rng, 2, 1024),
                 "max_iter": rng.choice([5, 10, 20]), "box": rng.choice([3.5, 5.0, 10.0]),
                 "sigma": rng.choice([0.5, 1.0, 2.0])}
            if d > 128:
                c["max_iter"] = 5  # wide rows are stopped early: see tolerance()
            if rng.random() < 0.3:
                c["noise"] = 0.05
            if path == "fit64":
                c.update(n=_log_int(rng, 20000, 4000000), d=_log_int(rng, 2, 64), k=_log_int(rng, 2, 128),
                         dtype="float64")
        elif path == "fit_plusplus":
            c = {"path": path, "n": _log_int(rng, 20000, 4000000), "d": _log_int(rng, 2, 64),
                 "k": _log_int(rng, 4, 256), "max_iter": 10, "tol": 0.0, "box": 5.0, "sigma": 0.5}
        elif path == "predict":
            c = {"path": path, "n": _log_int(rng, 1000, 10000000), "d": d, "k": _log_int(rng, 4, 2048),
                 "box": rng.choice([0.0, 3.0]), "sigma": 1.0}
        elif path == "cdist":
            c = {"path": path, "n": _log_int(rng, 1000, 40000), "m": rng.choice([0, _log_int(rng, 1000, 40000)]),
                 "d": _log_int(rng, 2, 256), "box": 2.0, "sigma": 1.0, "expand": rng.random() < 0.5}
        elif path == "knn":
            c = {"path": path, "n": _log_int(rng, 1000, 300000), "m": _log_int(rng, 1000, 100000),
                 "d": _log_int(rng, 2, 128), "k": rng.choice([1, 3, 5, 10]), "box": 2.0, "sigma": 1.0}
        else:
            c = {"path": path, "n": _log_int(rng, 20000, 4000000), "d": _log_int(rng, 2, 64),
                 "k": _log_int(rng, 2, 256), "max_iter": rng.choice([5, 10]), "box": 5.0, "sigma": 1.0}
        w = work(c)
        rows = (c["n"] + c.get("m", 0)) * c["d"] * (8 if c.get("dtype") == "float64" else 4)
        # vector-ALU paths reach a fraction of the matrix cores' rate
        slow = 8 if path in ("fit64", "kmedians", "cdist") else 1
        if c["n"] >= 4 * c.get("k", 1) and rows <= 4.2e9 and w["flops"] * slow <= 8e12 and w["bytes"] <= 24e9:
            return c


def _iters(case):
    """Passes over the rows that a run makes: the set number of iterations, or about what the default stop rule
    and the initialiser's rounds come to."""
    if case["path"] in ("fit", "kmedians"):
        return case["max_iter"]
    if case["path"] == "fit_plusplus":
        return 15 + min(case["max_iter"], 10)
    return 1


def work(case):
    """Bytes: the rows once per pass over them (once in all where they fit the last-level cache) and every output
    once.  Flops: one multiply-add per row, centroid (training row, column) and feature."""
    size = 8 if case.get("dtype") == "float64" else 4
    n, d, path = case["n"], case["d"], case["path"]
    if path == "cdist":
        m = case["m"] or n
        return {"bytes": 4 * (n * d + (m * d if case["m"] else 0) + n * m), "flops": 2 * n * m * d}
    if path == "knn":
        return {"bytes": 4 * (n + case["m"]) * d + 8 * case["m"] * (case["k"] + 1), "flops": 2 * n * case["m"] * d}
    passes = _iters(case)
    reads = passes if size * n * d > 256e6 else 1
    return {"bytes": size * n * d * reads + 8 * n + size * case["k"] * d, "flops": 2 * n * case["k"] * d * passes}


def tolerance(case):
    """Of two correct implementations at the same precision: about four times what the same rows give when they are
    scaled by a number near 1 (every rounding another one) or taken in float64.  Labels and neighbours differ where
    two distances agree to the rounding of the expansion |x|^2 + |c|^2 - 2 x.c, a row that changes sides moves its
    two centroids by 1 / (their rows), and the iterations after that amplify it: most for wide rows, where several
    initial centroids share a blob at nearly equal distances."""
    path = case["path"]
    if path == "cdist":
        # expanded: a row against itself gives the square root of the rounding error in place of 0
        return {"rel": 2e-5, "max": 4e-3} if case["expand"] else {"rel": 2e-6, "max": 1e-5}
    if path == "knn":
        return {"differ": 2e-4}
    if path == "predict":
        return {"rel": 1e-6, "differ": 1e-5}
    if case.get("dtype") == "float64":
        return {"rel": 1e-9, "max": 1e-8, "differ": 1e-6}
    if case["d"] > 64:
        return {"rel": 8e-3, "max": 0.5, "differ": 1e-2}
    return {"rel": 2e-3, "max": 2e-2, "differ": 5e-3}


def _blobs(gen, n, d, blobs, box, sigma, noise, dtype):
    """n rows in random order around ``blobs`` centres."""
    dev = torch.device("cuda")
    centres = (torch.rand((blobs, d), generator=gen, device=dev) * 2.0 - 1.0) * box
    share = torch.rand((blobs,), generator=gen, device=dev, dtype=torch.float64).clamp_min(1e-12).log().neg() + 0.05
    edges = torch.cumsum(share / share.sum(), 0).float()
    x = torch.empty((n, d), dtype=dtype, device=dev)
    step = max(1, _CHUNK_VALUES // d)
    for s in range(0, n, step):
        e = min(n, s + step)
        u = torch.rand((e - s,), generator=gen, device=dev)
        lab = torch.searchsorted(edges, u).clamp_max_(blobs - 1)
        rows = torch.randn((e - s, d), generator=gen, device=dev, dtype=dtype).mul_(sigma).add_(centres[lab])
        if noise:
            far = torch.rand((e - s,), generator=gen, device=dev) < noise
            back = (torch.rand((int(far.sum()), d), generator=gen, device=dev) * 2.0 - 1.0) * (box + 3 * sigma)
            rows[far] = back.to(dtype)
        x[s:e] = rows
    return x


def _some_rows(gen, x, k):
    """k distinct rows, one from each of k equal stretches."""
    n = x.shape[0]
    at = (torch.arange(k, device=x.device) + torch.rand((k,), generator=gen, device=x.device, dtype=torch.float64)) * (n / k)
    return x[at.long().clamp_max_(n - 1)].clone()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    path, n, d = case["path"], case["n"], case["d"]
    dtype = torch.float64 if case.get("dtype") == "float64" else torch.float32
    blobs = case["k"] if path in ("fit", "fit_plusplus", "kmedians", "predict") else 10
    x = _blobs(gen, n, d, blobs, case["box"], case["sigma"], case.get("noise", 0.0), dtype)
    state = {"case": case, "x": ht.array(x, split=0)}
    if path in ("fit", "kmedians"):
        state["init"] = ht.array(_some_rows(gen, x, case["k"]))
    elif path == "predict":
        # a finished clustering: centroids from one iteration on some of the rows
        few = x[: 16 * case["k"]]
        km = ht.cluster.KMeans(n_clusters=case["k"], init=ht.array(_some_rows(gen, few, case["k"])), max_iter=1)
        state["model"] = km.fit(ht.array(few, split=0))
    elif path == "cdist":
        if case["m"]:
            state["y"] = ht.array(_blobs(gen, case["m"], d, blobs, case["box"], case["sigma"], 0.0, dtype))
    elif path == "knn":
        both = _blobs(gen, n + case["m"], d, blobs, case["box"], case["sigma"], 0.0, dtype)
        side = torch.randn((d, blobs), generator=gen, device=x.device)
        labels = torch.argmax(both[:n] @ side, dim=1)
        model = ht.classification.KNeighborsClassifier(n_neighbors=case["k"])
        model.fit(ht.array(both[:n].clone(), split=0), ht.array(labels, split=0))
        state["model"] = model
        state["x"] = ht.array(both[n:].clone(), split=0)
    return state


def run(state):
    case = state["case"]
    path, x = case["path"], state["x"]
    if path == "cdist":
        return ht.spatial.cdist(x, state.get("y"), quadratic_expansion=case["expand"]).larray
    if path == "knn":
        model = state["model"]
        classes = model.predict(x)
        return {"classes": classes.larray, "neighbours": model.kneighbors_.larray}
    if path == "predict":
        model = state["model"]
        labels = model.predict(x)
        return {"labels": labels.larray, "functional_value": model.functional_value_.larray}
    if path == "fit_plusplus":
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")  # the default oversampling is raised for many clusters
            model = ht.cluster.KMeans(n_clusters=case["k"], init="kmeans++", max_iter=case["max_iter"],
                                      tol=case["tol"], random_state=1).fit(x)
        return {"labels": model.labels_.larray, "centers": model.cluster_centers_.larray}
    estimator = ht.cluster.KMedians if path == "kmedians" else ht.cluster.KMeans
    keys = {"random_state": 1} if path == "kmedians" else {}
    model = estimator(n_clusters=case["k"], init=state["init"], max_iter=case["max_iter"], tol=0.0, **keys).fit(x)
    return {"labels": model.labels_.larray, "centers": model.cluster_centers_.larray}
