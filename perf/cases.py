"""The work whose time is followed on an MI355X: one case per way a program uses this library.

    find           LinearKNNSearch::find for a handful of rows: an interactive lookup.  The
                   smallest call; launches, copies and latency are what it costs.
    classify       KNNClassifier.fit + predict from host arrays (the 10,000 x 32 f64 mixture
                   of the classifier configuration; default parameters but for k).
    knn_f64        batched search of f64 host queries in the default (FP64) form.
    knn_f32        the same for f32 rows with queries and outputs on the device, at a row
                   width that is not a multiple of the padding.
    knn_mixed      the mixed (BF16 MFMA + FP64 rescoring) search, device-resident: the
                   4,000,000 x 128 configuration.
    knn_manhattan  the mixed Manhattan search, device-resident.
    serve          one burst of uneven requests to the serving loop (2,000,000 x 96 rows,
                   k = 20, one request in five Manhattan): submitted together, all awaited.
    radius         LinearKNNSearch::find_radius for a batch of host queries, with distances.
    dbscan         DBSCAN.fit over resident rows (200,000 x 8 f64).
    lloyd          the Lloyd loop on resident f32 rows, mixed form (1,000,000 x 64, k = 64,
                   100 iterations).
    kmeans_fit     KMeans.fit (k-means++ seeding and the Lloyd loop, default FP64 form) and
                   predict on the same host rows: what an estimator user calls.
    kmeans_batch   many small fits in one call: the uneven batch's distribution of problems,
                   fewer of them.

`draw` takes one of these at random and spreads its sizes over the range the kind is used at.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from smartcore_amd import _capi as S

DEV = "cuda:0"


def listed():
    return [
        {"name": "find", "kind": "find", "n": 10_000, "d": 32, "q": 1, "k": 5},
        {"name": "classify", "kind": "classify", "n": 10_000, "d": 32, "q": 2_000, "k": 5},
        {"name": "knn_f64", "kind": "knn_f64", "n": 200_000, "d": 64, "q": 4_096, "k": 10},
        {"name": "knn_f32", "kind": "knn_f32", "n": 750_000, "d": 100, "q": 3_001, "k": 5},
        {"name": "knn_mixed", "kind": "knn_mixed", "n": 4_000_000, "d": 128, "q": 65_536, "k": 10},
        {"name": "knn_manhattan", "kind": "knn_manhattan", "n": 1_000_000, "d": 96, "q": 1_024,
         "k": 20},
        {"name": "serve", "kind": "serve", "n": 2_000_000, "d": 96, "k": 20, "requests": 16,
         "rows_max": 4_096},
        {"name": "radius", "kind": "radius", "n": 100_000, "d": 16, "q": 5_000, "hits": 40},
        {"name": "dbscan", "kind": "dbscan", "n": 200_000, "d": 8, "eps": 1.5, "min_samples": 10},
        {"name": "lloyd", "kind": "lloyd", "n": 1_000_000, "d": 64, "k": 64, "iters": 100},
        {"name": "kmeans_fit", "kind": "kmeans_fit", "n": 100_000, "d": 16, "k": 10, "iters": 100},
        {"name": "kmeans_batch", "kind": "kmeans_batch", "problems": 64, "n_lo": 1_000,
         "n_hi": 200_000, "iters": 20},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice([c["kind"] for c in listed()])
    k = rng.randint(1, 32)
    if kind == "find":
        return {"kind": kind, "n": _log_int(rng, 1_000, 100_000), "d": rng.randint(4, 128),
                "q": rng.randint(1, 8), "k": k}
    if kind == "classify":
        return {"kind": kind, "n": _log_int(rng, 2_000, 40_000), "d": rng.randint(4, 64),
                "q": _log_int(rng, 100, 4_000), "k": rng.randint(2, 16)}
    if kind in ("knn_f64", "knn_f32"):
        n, d = _log_int(rng, 20_000, 1_000_000), rng.randint(6, 130)
        q = min(_log_int(rng, 100, 10_000), 2 * 10**11 // (n * d))
        return {"kind": kind, "n": n, "d": d, "q": q, "k": k}
    if kind == "knn_mixed":
        n, d = _log_int(rng, 100_000, 4_000_000), rng.randint(16, 128)
        return {"kind": kind, "n": n, "d": d, "q": _log_int(rng, 200, 65_536), "k": k}
    if kind == "knn_manhattan":
        n, d = _log_int(rng, 100_000, 2_000_000), rng.randint(16, 128)
        q = min(_log_int(rng, 100, 8_192), 4 * 10**11 // (n * d))
        return {"kind": kind, "n": n, "d": d, "q": q, "k": k}
    if kind == "serve":
        return {"kind": kind, "n": _log_int(rng, 200_000, 2_000_000), "d": rng.randint(32, 128),
                "k": k, "requests": rng.randint(4, 20), "rows_max": rng.randint(64, 4_096)}
    if kind == "radius":
        return {"kind": kind, "n": _log_int(rng, 10_000, 400_000), "d": rng.randint(2, 48),
                "q": _log_int(rng, 100, 20_000), "hits": rng.randint(1, 80)}
    if kind == "dbscan":
        return {"kind": kind, "n": _log_int(rng, 10_000, 200_000), "d": 8,
                "eps": rng.uniform(1.2, 1.6), "min_samples": rng.randint(4, 12)}
    if kind == "lloyd":
        return {"kind": kind, "n": _log_int(rng, 20_000, 1_000_000), "d": rng.randint(4, 64),
                "k": rng.randint(4, 64), "iters": rng.randint(20, 100)}
    if kind == "kmeans_fit":
        return {"kind": kind, "n": _log_int(rng, 5_000, 200_000), "d": rng.randint(4, 40),
                "k": rng.randint(2, 32), "iters": rng.randint(20, 100)}
    return {"kind": kind, "problems": rng.randint(8, 64), "n_lo": 1_000, "n_hi": 200_000,
            "iters": 20}


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, n, d, dtype=torch.float32):
    return torch.randn((n, d), generator=g, device=DEV, dtype=dtype)


def _mixture(g, n, q, d, dtype, classes=10):
    """Rows and queries of one Gaussian mixture (centres ~ N(0, 16 I), unit noise), and labels."""
    centres = 4.0 * _normal(g, classes, d, dtype)
    lab = torch.randint(0, classes, (n + q,), generator=g, device=DEV)
    x = centres[lab] + _normal(g, n + q, d, dtype)
    return x[:n].contiguous(), x[n:].contiguous(), lab[:n].to(torch.int32)


def _lognormal(g, n, d):
    """Rows ~ N(0, I) scaled by per-row norms ~ LogNormal(0, 0.5), f32."""
    x = torch.empty((n, d), device=DEV)
    for s in range(0, n, 1 << 20):
        e = min(n, s + (1 << 20))
        x[s:e] = _normal(g, e - s, d) * torch.exp(0.5 * _normal(g, e - s, 1))
    return x


def _blobs(g, n, d, k, dtype=torch.float32):
    """k Gaussian blobs (centres ~ U(-10, 10), standard deviations ~ U(0.5, 2), uneven sizes)."""
    def uni(*shape):
        return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)
    centres = (20.0 * uni(k, d) - 10.0).to(dtype)
    std = (0.5 + 1.5 * uni(k, 1)).to(dtype)
    weight = -torch.log(uni(k))
    lab = torch.multinomial(weight, n, replacement=True, generator=g)
    return centres[lab] + std[lab] * _normal(g, n, d, dtype)


def _index(rows):
    np_dtype = np.float64 if rows.dtype == torch.float64 else np.float32
    torch.cuda.synchronize()
    return S.Index(device_ptr=rows.data_ptr(), n=rows.shape[0], d=rows.shape[1], dtype=np_dtype)


def _device_search(rows, queries, k, metric, mode):
    q = queries.shape[0]
    return {"index": _index(rows), "queries": queries, "k": k, "metric": metric, "mode": mode,
            "idx": torch.empty((q, k), dtype=torch.int64, device=DEV),
            "dist": torch.empty((q, k), dtype=torch.float64, device=DEV),
            "count": torch.empty((q,), dtype=torch.int32, device=DEV)}


def _request_rows(case):
    """Rows of each request of a burst: log-spaced sizes, not in order of size."""
    m = case["requests"]
    sizes = [int(round(case["rows_max"] ** (i / max(m - 1, 1)))) for i in range(m)]
    return [sizes[(7 * i + 3) % m] if math.gcd(7, m) == 1 else sizes[i] for i in range(m)]


def _radius_of(case):
    """A radius at which N(0, I) rows of this width give about `hits` neighbours per query:
    ||x - y||^2 / 2 has a chi-square distribution of d degrees."""
    p = min(0.4, case["hits"] / case["n"])
    shape = torch.tensor(0.5 * case["d"], dtype=torch.float64)
    lo, hi = 0.0, 10.0 * case["d"]
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        if float(torch.special.gammainc(shape, torch.tensor(0.5 * mid, dtype=torch.float64))) < p:
            lo = mid
        else:
            hi = mid
    return math.sqrt(2.0 * hi)


def _capacity(case):
    """Entries of a caller's result buffers: the expected neighbours with room to spare."""
    return 2 * case["q"] * case["hits"] + 64 * case["hits"] + 4_096


def _inputs(case, seed):
    """The inputs of a case as device tensors, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("find", "classify", "knn_f64", "knn_f32"):
        dtype = torch.float32 if kind == "knn_f32" else torch.float64
        rows, queries, labels = _mixture(g, case["n"], case["q"], case["d"], dtype)
        return {"rows": rows, "queries": queries, "labels": labels}
    if kind == "knn_mixed":
        return {"rows": _lognormal(g, case["n"], case["d"]),
                "queries": _lognormal(g, case["q"], case["d"])}
    if kind == "knn_manhattan":
        return {"rows": _normal(g, case["n"], case["d"]), "queries": _normal(g, case["q"], case["d"])}
    if kind == "serve":
        return {"rows": _normal(g, case["n"], case["d"]),
                "requests": [_normal(g, r, case["d"]) for r in _request_rows(case)]}
    if kind == "radius":
        return {"rows": _normal(g, case["n"], case["d"]), "queries": _normal(g, case["q"], case["d"])}
    if kind == "dbscan":
        return {"rows": _mixture(g, case["n"], 0, case["d"], torch.float64)[0]}
    if kind in ("lloyd", "kmeans_fit"):
        dtype = torch.float32 if kind == "lloyd" else torch.float64
        rows = _blobs(g, case["n"], case["d"], case["k"], dtype)
        pick = torch.randperm(case["n"], generator=g, device=DEV)[:case["k"]].sort().values
        return {"rows": rows, "centroids": rows[pick].double()}
    problems = []
    r = np.random.default_rng(1234)  # the shapes of a batch are its case's, the values the seed's
    for _ in range(case["problems"]):
        n = int(round(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        d, k = int(r.choice((8, 16, 32, 64))), int(r.integers(4, 129))
        centres = 4.0 * _normal(g, k, d)
        x = centres[torch.randint(0, k, (n,), generator=g, device=DEV)] + _normal(g, n, d)
        problems.append((x, x[torch.randperm(n, generator=g, device=DEV)[:k].sort().values].double()))
    return {"problems": problems}


def prepare(case, seed):
    kind = case["kind"]
    v = _inputs(case, seed)
    if kind in ("find", "knn_f64"):
        return {"kind": kind, "index": _index(v["rows"]), "queries": v["queries"].cpu().numpy(),
                "k": case["k"]}
    if kind == "classify":
        from smartcore_amd import smartcore as sm
        params = sm.KNNClassifierParameters().with_k(case["k"])
        return {"kind": kind, "fit": sm.KNNClassifier.fit, "params": params,
                "x": v["rows"].cpu().numpy(), "y": v["labels"].cpu().numpy(),
                "queries": v["queries"].cpu().numpy()}
    if kind == "knn_f32":
        return {"kind": kind, **_device_search(v["rows"], v["queries"], case["k"], S.SC_EUCLIDIAN,
                                               S.SC_PLAIN_FP64)}
    if kind == "knn_mixed":
        return {"kind": kind, **_device_search(v["rows"], v["queries"], case["k"], S.SC_EUCLIDIAN,
                                               S.SC_MIXED)}
    if kind == "knn_manhattan":
        return {"kind": kind, **_device_search(v["rows"], v["queries"], case["k"], S.SC_MANHATTAN,
                                               S.SC_MIXED)}
    if kind == "serve":
        index = _index(v["rows"])
        return {"kind": kind, "server": S.Server(index), "k": case["k"],
                "requests": [x.cpu().numpy() for x in v["requests"]],
                "metrics": [S.SC_MANHATTAN if i % 5 == 2 else S.SC_EUCLIDIAN
                            for i in range(case["requests"])]}
    if kind == "radius":
        return {"kind": kind, "index": _index(v["rows"]), "queries": v["queries"].cpu().numpy(),
                "radius": _radius_of(case), "offsets": np.zeros(case["q"] + 1, np.uint64),
                "idx": np.zeros(_capacity(case), np.int64), "dist": np.zeros(_capacity(case))}
    if kind == "dbscan":
        return {"kind": kind, "index": _index(v["rows"]), "eps": case["eps"],
                "min_samples": case["min_samples"]}
    if kind == "lloyd":
        return {"kind": kind, "index": _index(v["rows"]), "iters": case["iters"],
                "centroids": v["centroids"].cpu().numpy()}
    if kind == "kmeans_fit":
        from smartcore_amd import smartcore as sm
        params = sm.KMeansParameters().with_k(case["k"]).with_max_iter(case["iters"])
        return {"kind": kind, "fit": sm.KMeans.fit, "params": params, "x": v["rows"].cpu().numpy()}
    return {"kind": kind, "iters": case["iters"],
            "problems": [(x.cpu().numpy(), c.cpu().numpy()) for x, c in v["problems"]]}


# ---------------------------------------------------------------- one pass


def _radius_search(state):
    """sc_radius_search as a C caller uses it: the CSR offsets, rows and distances go to buffers
    that the program keeps."""
    lib, queries = S.lib(), state["queries"]
    handle = ctypes.c_void_p()
    S.check(lib.sc_radius_search(state["index"].handle, queries.ctypes.data, queries.shape[0],
                                 state["radius"], S.SC_EUCLIDIAN, 2, ctypes.byref(handle)))
    try:
        total = lib.sc_radius_result_total(handle)
        offsets, idx, dist = state["offsets"], state["idx"], state["dist"]
        if total > idx.size:
            raise RuntimeError(f"{total} neighbours do not fit the caller's buffers")
        S.check(lib.sc_radius_result_copy(handle, offsets.ctypes.data, idx.ctypes.data,
                                          dist.ctypes.data))
    finally:
        lib.sc_radius_result_free(handle)
    return {"offsets": offsets, "idx": idx, "dist": dist}


def run(state):
    kind = state["kind"]
    if kind in ("find", "knn_f64"):
        idx, dist, count = state["index"].knn(state["queries"], state["k"])
        return {"idx": idx, "dist": dist, "count": count}
    if kind == "classify":
        model = state["fit"](state["x"], state["y"], state["params"])
        return {"labels": model.predict(state["queries"])}
    if kind in ("knn_f32", "knn_mixed", "knn_manhattan"):
        queries = state["queries"]
        state["index"].knn_device(queries.data_ptr(), queries.shape[0], state["k"],
                                  state["idx"].data_ptr(), state["dist"].data_ptr(),
                                  state["count"].data_ptr(), state["metric"], 2, state["mode"],
                                  torch.cuda.current_stream().cuda_stream)
        return {"idx": state["idx"], "dist": state["dist"], "count": state["count"]}
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(x, state["k"], m, 2, S.SC_MIXED)
                   for x, m in zip(state["requests"], state["metrics"])]
        answers = [server.wait(t) for t in tickets]
        return [{"idx": a[0], "dist": a[1], "count": a[2]} for a in answers]
    if kind == "radius":
        return _radius_search(state)
    if kind == "dbscan":
        labels, clusters = state["index"].dbscan_fit(state["eps"], state["min_samples"])
        return {"labels": labels, "clusters": clusters}
    if kind == "lloyd":
        centroids, labels, size, distortion, iters = state["index"].kmeans_run(
            state["centroids"], state["iters"], S.SC_MIXED)
        return {"centroids": centroids, "labels": labels, "size": size, "distortion": distortion,
                "iters": iters}
    if kind == "kmeans_fit":
        model = state["fit"](state["x"], state["params"])
        return {"centroids": model.centroids, "labels": model.labels, "size": model.size,
                "distortion": model.distortion, "iters": model.iterations,
                "predicted": model.predict(state["x"])}
    out = S.kmeans_batch_run(state["problems"], state["iters"], S.SC_MIXED)
    # every problem's arrays are views of these three
    return {"centroids": out[0][0].base, "labels": out[0][1].base, "sizes": out[0][2].base,
            "distortion": np.array([o[3] for o in out]), "iters": np.array([o[4] for o in out])}


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind in ("find", "classify", "knn_f64", "knn_f32", "knn_mixed", "knn_manhattan", "serve"):
        n, d, k = case["n"], case["d"], case["k"]
        q = sum(_request_rows(case)) if kind == "serve" else case["q"]
        es = 8 if kind in ("find", "classify", "knn_f64") else 4
        out = 4 * q if kind == "classify" else q * (16 * k + 4)
        return {"bytes": (n + q) * d * es + out, "flops": 2.0 * n * q * d}
    if kind == "radius":
        n, d, q = case["n"], case["d"], case["q"]
        return {"bytes": (n + q) * d * 4 + 16 * q * case["hits"], "flops": 2.0 * n * q * d}
    if kind == "dbscan":
        n, d = case["n"], case["d"]
        return {"bytes": n * d * 8 + 4 * n, "flops": 1.0 * n * n * d}
    if kind in ("lloyd", "kmeans_fit"):
        # a Lloyd iteration reads every row; the seeding makes k passes more and predict one
        n, d, k, it = case["n"], case["d"], case["k"], case["iters"]
        es, passes = (4, it) if kind == "lloyd" else (8, it + k + 1)
        seed = 0.0 if kind == "lloyd" else 3.0 * n * k * d + 2.0 * n * k * d
        return {"bytes": passes * n * d * es + 4 * n, "flops": it * 2.0 * n * k * d + seed}
    r = np.random.default_rng(1234)
    total = {"bytes": 0.0, "flops": 0.0}
    for _ in range(case["problems"]):
        n = int(round(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        d, k = int(r.choice((8, 16, 32, 64))), int(r.integers(4, 129))
        total["bytes"] += case["iters"] * n * d * 4 + 4 * n
        total["flops"] += case["iters"] * 2.0 * n * d * k
    return total


# ---------------------------------------------------------------- the same results in 64 bits


def _pairwise(rows, queries, metric):
    """Distances of every query to every row, f64: the widened values' differences, one
    dimension after another, in pieces that stay in cache."""
    out = torch.empty((queries.shape[0], rows.shape[0]), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 23) // rows.shape[0])
    columns = rows.T.contiguous()
    for s in range(0, queries.shape[0], step):
        part = out[s:s + step].zero_()
        for x, r in zip(queries[s:s + step].T, columns):
            diff = x[:, None] - r
            if metric == S.SC_MANHATTAN:
                part += diff.abs_()
            else:
                part.addcmul_(diff, diff)
        if metric != S.SC_MANHATTAN:
            part.sqrt_()
    return out


def _heap_order(dist, k):
    """Distances in the order LinearKNNSearch::find leaves them: a k-entry max-heap whose root is
    replaced by every row that beats it, in row order; one heap per query, side by side."""
    q, n = dist.shape
    rows, cols = [], []
    edge, kth = 0, torch.full((q, 1), math.inf, dtype=torch.float64, device=dist.device)
    while edge < n:
        end = min(n, max(64, 2 * edge))
        hit = (dist[:, edge:end] < kth).nonzero()
        rows.append(hit[:, 0])
        cols.append(hit[:, 1] + edge)
        if end >= k:
            kth = torch.topk(dist[:, :end], k, dim=1, largest=False).values[:, -1:]
        edge = end
    rows, cols = torch.cat(rows), torch.cat(cols)
    order = torch.argsort(rows * n + cols)
    value = dist[rows[order], cols[order]].cpu().numpy()
    count = torch.bincount(rows, minlength=q).cpu().numpy()
    first = np.concatenate([[0], np.cumsum(count)[:-1]])
    heap, who = np.full((q, k), np.inf), np.arange(q)
    for j in range(int(count.max())):
        v = np.where(j < count, value[np.minimum(first + j, value.size - 1)], np.inf)
        enter = v < heap[:, 0]
        heap[enter, 0] = v[enter]
        at, live = np.zeros(q, np.int64), enter
        while True:
            child = 2 * at
            live = live & (child <= k - 1)
            if not live.any():
                break
            child = np.where(live, child, 0)
            nxt = np.minimum(child + 1, k - 1)
            child = np.where(live & (child < k - 1) & (heap[who, child] < heap[who, nxt]), nxt, child)
            live = live & (heap[who, at] < heap[who, child])
            a, c, w = at[live], child[live], who[live]
            heap[w, a], heap[w, c] = heap[w, c].copy(), heap[w, a].copy()
            at = np.where(live, child, at)
            if not live.any():
                break
    return heap


def _exact_search(rows, queries, k, metric):
    return _heap_order(_pairwise(rows.double(), queries.double(), metric), k)


def _lloyd(x, centroids, iters):
    """KMeans::fit's loop in f64: centroids, sizes and the distortion it stops with."""
    x, c = x.double(), centroids.clone().double()
    k, best = c.shape[0], math.inf
    size = None
    for _ in range(iters):
        label = torch.empty(x.shape[0], dtype=torch.int64, device=DEV)
        cost = 0.0
        for s in range(0, x.shape[0], 1 << 17):
            part = x[s:s + (1 << 17)]
            near = (c.square().sum(dim=1) - 2.0 * part @ c.T).argmin(dim=1)
            label[s:s + (1 << 17)] = near
            cost += float((part - c[near]).square().sum())
        size = torch.bincount(label, minlength=k)
        sums = torch.zeros_like(c).index_add_(0, label, x)
        c = torch.where(size[:, None] > 0, sums / size.clamp(min=1)[:, None], c)
        if best <= cost:
            break
        best = cost
    return c.cpu().numpy(), best


def _too_long(case, q):
    return case["n"] * q > 4e9 or case["n"] * q * case["d"] > 4e11


def exact(case, seed):
    kind = case["kind"]
    if kind in ("classify", "dbscan", "kmeans_fit"):
        return None  # labels; or a seeding drawn from a random stream of the library's own
    if kind == "serve":
        sizes = _request_rows(case)
        if _too_long(case, sum(sizes)):
            return None
        v = _inputs(case, seed)
        return [{"dist": _exact_search(v["rows"], x, case["k"],
                                       S.SC_MANHATTAN if i % 5 == 2 else S.SC_EUCLIDIAN)}
                for i, x in enumerate(v["requests"])]
    if kind in ("find", "knn_f64", "knn_f32", "knn_mixed", "knn_manhattan"):
        if _too_long(case, case["q"]):
            return None
        v = _inputs(case, seed)
        metric = S.SC_MANHATTAN if kind == "knn_manhattan" else S.SC_EUCLIDIAN
        return {"dist": _exact_search(v["rows"], v["queries"], case["k"], metric)}
    if kind == "radius":
        if _too_long(case, case["q"]):
            return None
        v = _inputs(case, seed)
        full = _pairwise(v["rows"].double(), v["queries"].double(), S.SC_EUCLIDIAN)
        near = full[full <= _radius_of(case)].cpu().numpy()
        dist = np.zeros(_capacity(case))
        dist[:near.size] = near
        return {"dist": dist}
    if kind == "lloyd":
        v = _inputs(case, seed)
        c, cost = _lloyd(v["rows"], v["centroids"], case["iters"])
        return {"centroids": c, "distortion": cost}
    v = _inputs(case, seed)
    fits = [_lloyd(x, c, case["iters"]) for x, c in v["problems"]]
    return {"centroids": np.concatenate([c.ravel() for c, _ in fits]),
            "distortion": np.array([cost for _, cost in fits])}
