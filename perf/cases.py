"""The work that users of this package have it do, as measurable cases.

A case is a dict of plain values whose "kind" names an entry point:

* "fit"       kmeans_lloyd_driver / kmeans_lloyd_driver_ex: a whole Lloyd fit
              from given centroids on feature-major data;
* "step"      one iteration of a caller's own Lloyd loop over the single-step
              entry points (half norms, fused step, reduction, division);
* "batch"     kmeans_lloyd_batched: many independent fits of uneven sizes;
* "estimator" KMeans.fit: sample-major data, k-means++ seeding, a fit;
* "predict"   KMeans.predict with a fitted model;
* "transform" KMeans.transform with a fitted model.

Data are Gaussian blobs, one row of each first (per-blob standard deviation 0.5 to 2, centres
uniform in [-20, 20]^d), the distribution of this repository's benchmark.
"""
import math

import numpy as np
import torch

import kmeans_dpcpp_amd as kd

_DTYPES = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # one small request: launch count and host time decide
        {"name": "fit_small", "kind": "fit", "n": 1000, "d": 16, "k": 8, "dtype": "f32",
         "precision": "fp32", "max_iter": 100, "tol": 1e-4},
        # an ordinary table of 50,000 rows, fitted until it converges
        {"name": "fit_ordinary", "kind": "fit", "n": 50_000, "d": 14, "k": 127,
         "dtype": "f32", "precision": "fp32", "max_iter": 100, "tol": 1e-4},
        # the largest single fit of the benchmark, in float32
        {"name": "fit_large", "kind": "fit", "n": 10_000_000, "d": 32, "k": 256,
         "dtype": "f32", "precision": "fp32", "max_iter": 10, "tol": 0.0},
        # wide rows and many clusters in float32 (the large request of a
        # served stream, a quarter of its rows)
        {"name": "fit_wide", "kind": "fit", "n": 500_000, "d": 96, "k": 512,
         "dtype": "f32", "precision": "fp32", "max_iter": 10, "tol": 0.0},
        # the mixed-precision option at the size it is meant for
        {"name": "fit_bf16", "kind": "fit", "n": 2_000_000, "d": 128, "k": 1024,
         "dtype": "f32", "precision": "bf16", "max_iter": 6, "tol": 0.0},
        # float64 data, an odd number of rows
        {"name": "fit_f64", "kind": "fit", "n": 1_000_003, "d": 32, "k": 256,
         "dtype": "f64", "precision": "fp32", "max_iter": 6, "tol": 0.0},
        # embedding-like rows beyond 128 features, odd sizes, given one sample
        # of each blob as a caller's own k-means++ would give
        {"name": "fit_embedding", "kind": "fit", "n": 200_003, "d": 300, "k": 100,
         "dtype": "f32", "precision": "fp32", "max_iter": 8, "tol": 0.0},
        # a caller's own loop over few clusters: bound by reading the samples
        {"name": "step_few_clusters", "kind": "step", "n": 9_999_999, "d": 32, "k": 8},
        # many uneven fits at once
        {"name": "batch", "kind": "batch", "fits": 128, "sizes_seed": 1, "n_min": 1000,
         "n_max": 200_000, "precision": "fp32"},
        # the estimator's whole fit, seeding included
        {"name": "estimator_fit", "kind": "estimator", "n": 1_000_000, "d": 32, "k": 64},
        # labels of new rows
        {"name": "predict", "kind": "predict", "n": 3_000_001, "d": 48, "k": 200},
        # distances of new rows to every centre
        {"name": "transform", "kind": "transform", "n": 1_000_000, "d": 32, "k": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "fit", "fit", "fit", "fit", "step", "batch",
                       "estimator", "predict", "transform"])
    if kind == "batch":
        return {"kind": kind, "fits": _log_int(rng, 2, 128),
                "sizes_seed": rng.randrange(1 << 20), "n_min": 1000,
                "n_max": _log_int(rng, 5000, 200_000),
                "precision": rng.choice(["fp32", "bf16"])}
    while True:
        n = _log_int(rng, 500, 10_000_000)
        if kind == "fit":
            d, k = _log_int(rng, 2, 512), _log_int(rng, 2, 1024)
            dtype = rng.choice(["f32", "f32", "f32", "f64"])
            cap = 10 * 10_000_000 * 32 * 256 // (1 if dtype == "f32" else 8)
            # a fit until convergence on small and middle sizes, a fixed
            # number of iterations on the others
            to_end = dtype == "f32" and d <= 128 and n * d <= 4_000_000
            iters = 25 if to_end else rng.randint(2, 10)
            precision = rng.choice(["fp32", "fp32", "bf16"]) if dtype == "f32" else "fp32"
            if k * 10 > n or n * d > 300_000_000 or n * d * k * iters > cap:
                continue
            # without matrix-core kernels a wide or a float64 fit is slow
            if (d > 128 or dtype == "f64") and n * d * k > 4_000_000_000:
                continue
            return {"kind": kind, "n": n, "d": d, "k": k, "dtype": dtype,
                    "precision": precision, "max_iter": 100 if to_end else iters,
                    "tol": 1e-4 if to_end else 0.0}
        d, k = _log_int(rng, 2, 128), _log_int(rng, 2, 512)
        if k * 10 > n or n * d > 320_000_000 or n * k > 400_000_000:
            continue
        if kind == "estimator" and n * d > 40_000_000:
            continue
        if kind == "transform" and n * k > 100_000_000:
            continue
        return {"kind": kind, "n": n, "d": d, "k": k}


def _blobs(n, d, k, gen, dtype, by_sample):
    """Blob samples, (d, n) or by_sample (n, d)."""
    dev = gen.device
    centres = torch.rand((k, d), generator=gen, device=dev, dtype=dtype) * 40.0 - 20.0
    std = torch.rand((k,), generator=gen, device=dev, dtype=dtype) * 1.5 + 0.5
    blob = torch.randint(0, k, (n,), generator=gen, device=dev)
    blob[:k] = torch.arange(k, device=dev)
    X = torch.empty((n, d) if by_sample else (d, n), dtype=dtype, device=dev)
    for s in range(0, n, 1 << 21):
        b = blob[s:s + (1 << 21)]
        z = torch.randn((b.numel(), d), generator=gen, device=dev, dtype=dtype)
        rows = z.mul_(std[b, None]).add_(centres[b])
        if by_sample:
            X[s:s + b.numel()] = rows
        else:
            X[:, s:s + b.numel()] = rows.T
    return X


def _sample_init(X_t, k, gen):
    """k distinct samples as initial centroids (d, k).  Beyond 128 features
    sample j is of blob j: there two centroids in one blob split it by the last
    bits of their coordinates, and no two runs would agree."""
    n = X_t.shape[1]
    if X_t.shape[0] > 128:
        return X_t[:, :k].contiguous()
    idx = torch.randperm(n, generator=gen, device=gen.device)[:k]
    return X_t[:, idx].contiguous()


def _batch_sizes(case):
    rng = np.random.default_rng(case["sizes_seed"])
    sizes = []
    for _ in range(case["fits"]):
        n = int(np.exp(rng.uniform(np.log(case["n_min"]), np.log(case["n_max"]))))
        d = int(rng.choice([16, 32, 64]))
        k = int(rng.choice([8, 32, 64, 128, 256]))
        while k >= n / 10:
            k = int(rng.choice([8, 32, 64, 128, 256]))
        sizes.append((n, d, k))
    return sizes


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "batch":
        sizes = _batch_sizes(case)
        # results of all fits live in two buffers, each fit's part aligned
        pad = 64
        lab = torch.zeros(sum(-(-n // pad) * pad for n, _, _ in sizes), dtype=torch.int32,
                          device=dev)
        cen = torch.zeros(sum(-(-d * k // pad) * pad for _, d, k in sizes), device=dev)
        fits, at, ac = [], 0, 0
        for n, d, k in sizes:
            X_t = _blobs(n, d, k, gen, torch.float32, False)
            fits.append((X_t, torch.ones(n, device=dev), _sample_init(X_t, k, gen),
                         lab[at:at + n], cen[ac:ac + d * k].view(d, k)))
            at += -(-n // pad) * pad
            ac += -(-d * k // pad) * pad
        return {"case": case, "fits": fits, "labels": lab, "centroids": cen}
    n, d, k = case["n"], case["d"], case["k"]
    dtype = _DTYPES[case.get("dtype", "f32")]
    if kind in ("estimator", "predict", "transform"):
        X = _blobs(n, d, k, gen, dtype, True)
        if kind == "estimator":
            return {"case": case, "X": X, "seed": seed}
        # a fitted model: its centres are a few Lloyd steps from samples
        m = min(n, 16 * k + 1000)
        model = kd.KMeans(k, init=X[:k].contiguous(), n_init=1, max_iter=2, tol=0.0)
        model.fit(X[:m])
        return {"case": case, "X": X, "model": model}
    X_t = _blobs(n, d, k, gen, dtype, False)
    init = _sample_init(X_t, k, gen)
    state = {"case": case, "X_t": X_t, "w": torch.ones(n, dtype=dtype, device=dev),
             "init": init, "labels": torch.zeros(n, dtype=torch.int32, device=dev)}
    if kind == "fit":
        state["res"] = torch.zeros_like(init)
        return state
    copies = kd.compute_number_of_private_copies(X_t, n, d, k, 0.7, 128)
    state["copies"] = torch.empty((copies, d, k), dtype=dtype, device=dev)
    state["size_copies"] = torch.empty((copies, k), dtype=dtype, device=dev)
    state["half_norm"] = torch.empty(k, dtype=dtype, device=dev)
    state["sizes"] = torch.empty(k, dtype=dtype, device=dev)
    state["next"] = torch.empty_like(init)
    state["empty"] = torch.empty(k, dtype=torch.int32, device=dev)
    state["n_empty"] = torch.empty(1, dtype=torch.int32, device=dev)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    q = torch.cuda.current_stream()
    if kind == "fit":
        init = state["init"].clone()   # the fit overwrites its initial centroids
        if case["precision"] == "fp32":
            n_iter, inertia = kd.kmeans_lloyd_driver(
                state["X_t"], state["w"], init, state["labels"], state["res"],
                case["tol"], False, case["max_iter"], 8, 128, 0.7, q)
        else:
            n_iter, inertia, _ = kd.kmeans_lloyd_driver_ex(
                state["X_t"], state["w"], init, state["labels"], state["res"],
                case["tol"], False, case["max_iter"], case["precision"], q)
        return {"labels": state["labels"], "centroids": state["res"],
                "n_iter": int(n_iter), "inertia": float(np.asarray(inertia).reshape(-1)[0])}
    if kind == "batch":
        fits = [(X_t, w, init.clone(), lab, res, 1e-4, 100)
                for X_t, w, init, lab, res in state["fits"]]
        results, _ = kd.kmeans_lloyd_batched(fits, case["precision"], q)
        return {"labels": state["labels"], "centroids": state["centroids"],
                "n_iter": np.array([r[0] for r in results], dtype=np.int64),
                "inertia": np.array([r[1] for r in results], dtype=np.float64)}
    if kind == "step":
        s = state
        s["copies"].zero_()
        s["size_copies"].zero_()
        s["n_empty"].zero_()
        kd.half_l2_norm_squared(s["init"], s["half_norm"], 128, q)
        kd.fused_lloyd_single_step(s["X_t"], s["w"], s["init"], s["half_norm"], s["labels"],
                                   s["copies"], s["size_copies"], 8, 128, q)
        kd.reduce_centroids_data(s["size_copies"], s["copies"], s["sizes"], s["next"],
                                 s["empty"], s["n_empty"], 128, q)
        kd.broadcast_divide(s["next"], s["sizes"], 128, q)
        return {"labels": s["labels"], "sizes": s["sizes"], "centroids": s["next"]}
    if kind == "estimator":
        model = kd.KMeans(case["k"], random_state=state["seed"] % 1_000_003)
        model.fit(state["X"])
        return {"labels": model.labels_, "centres": model.cluster_centers_,
                "inertia": model.inertia_}
    if kind == "predict":
        return state["model"].predict(state["X"])
    return state["model"].transform(state["X"])


#: Iterations that a fit until convergence takes on these data, about.
_USUAL_ITERS = 16


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = f = 0
        for n, d, k in _batch_sizes(case):
            b += 4 * (n * d + 2 * n + 2 * d * k)
            f += 2 * n * d * k * (_USUAL_ITERS + 1) + 2 * n * d * _USUAL_ITERS
        return {"bytes": b, "flops": f}
    n, d, k = case["n"], case["d"], case["k"]
    s = 8 if case.get("dtype") == "f64" else 4
    if kind == "transform":
        return {"bytes": s * (n * d + d * k + n * k), "flops": 3 * n * d * k}
    if kind == "predict":
        return {"bytes": s * (n * d + d * k) + 4 * n, "flops": 2 * n * d * k}
    if kind == "step":
        return {"bytes": s * (n * d + n + 2 * d * k) + 4 * n, "flops": 2 * n * d * (k + 1)}
    iters = _USUAL_ITERS
    if kind == "fit" and case["tol"] == 0.0:
        iters = case["max_iter"]
    flops = 2 * n * d * k * (iters + 1) + 2 * n * d * iters
    if kind == "estimator":   # seeding: every sample against each new centre's trials
        flops += 2 * n * d * k * (2 + int(math.log(k)))
    return {"bytes": s * (n * d + n + 2 * d * k) + 4 * n, "flops": flops}


def tolerance(case):
    # Labels may differ where two centroids are equally near within rounding.
    kind = case["kind"]
    if kind == "predict":
        return {"rel": 0.0, "differ": 1e-4}
    if kind == "transform":
        return {"rel": 2e-7, "max": 2e-6}
    if kind in ("step", "estimator"):
        return {"rel": 3e-6, "max": 1e-4, "differ": 1e-4}
    if kind == "fit" and case["d"] > 128:
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-5}
    # From sampled centroids two of them may come to lie almost on one another
    # in one blob; their split then carries rounding errors on, enlarged some
    # ten thousand times (9e-4 measured in float32 against float64).
    if case.get("dtype") == "f64":
        return {"rel": 1e-10, "max": 1e-8, "differ": 1e-4}
    return {"rel": 4e-3, "max": 0.2, "differ": 1e-2}


def _lloyd64(X, w, C, max_iter, tol):
    """Lloyd in float64 with the driver's rules, X (n, d) and C (k, d): the
    j-th empty cluster takes the j-th farthest sample, on the undivided sums."""
    k = C.shape[0]
    dev = X.device
    chunk = max(1, (1 << 27) // max(k, X.shape[1]))
    labels = torch.empty(X.shape[0], dtype=torch.int64, device=dev)
    far = torch.empty(X.shape[0], dtype=torch.float64, device=dev)

    def assign(s):
        """Rows from s on with their labels and squared distances (noted)."""
        x = X[s:s + chunk].double()
        lab = torch.argmin((C * C).sum(1)[None, :] / 2 - x @ C.T, dim=1)
        labels[s:s + chunk] = lab
        far[s:s + chunk] = ((x - C[lab]) ** 2).sum(1)
        return x, lab

    it, shift = 0, math.inf
    while it < max_iter and shift > tol:
        S = torch.zeros_like(C)
        N = torch.zeros(k, dtype=C.dtype, device=dev)
        for s in range(0, X.shape[0], chunk):
            x, lab = assign(s)
            hot = torch.zeros((x.shape[0], k), dtype=C.dtype, device=dev)
            hot.scatter_(1, lab[:, None], w[s:s + chunk, None].double())
            S += hot.T.contiguous() @ x
            N += hot.sum(0)
        empty = torch.nonzero(N == 0).flatten().tolist()
        if empty:
            for e, i in zip(empty, torch.topk(far, len(empty)).indices.tolist()):
                wi = w[i].double()
                S[labels[i]] -= wi * X[i].double()
                N[labels[i]] -= wi
                S[e] = wi * X[i].double()
                N[e] = wi
        new = S / N[:, None]
        shift = float(((new - C) ** 2).sum())
        C = new
        it += 1
    for s in range(0, X.shape[0], chunk):
        assign(s)
    return C, float((far * w).sum())


def _seeds64(X, k, seed):
    """Greedy k-means++ on (n, d) float64 data with RandomState(seed)."""
    rs = np.random.RandomState(seed)
    trials = 2 + int(np.log(k))
    n = X.shape[0]
    draws = torch.arange(1, n + 1, dtype=X.dtype, device=X.device) / n
    first = int(torch.searchsorted(draws, rs.random_sample(), right=True))
    ids = [min(first, n - 1)]
    near = ((X - X[ids[0]]) ** 2).sum(1)
    for _ in range(1, k):
        u = torch.as_tensor(rs.uniform(size=trials), device=X.device)
        cand = torch.searchsorted(torch.cumsum(near, 0), u * near.sum()).clamp_(max=n - 1)
        trial = torch.stack([torch.minimum(near, ((X - X[c]) ** 2).sum(1)) for c in cand])
        best = int(torch.argmin(trial.sum(1)))
        near = trial[best]
        ids.append(int(cand[best]))
    return X[torch.tensor(ids, device=X.device)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        return None
    state = prepare(case, seed)
    if kind == "transform":
        X = state["X"].double()
        out = torch.empty((X.shape[0], case["k"]), dtype=X.dtype, device=X.device)
        for c, centre in enumerate(state["model"].cluster_centers_.double()):
            out[:, c] = ((X - centre) ** 2).sum(1).sqrt()
        return out
    if kind == "estimator":
        X = state["X"].double()
        mean = X.mean(0)
        X -= mean
        tol = float(X.var(0, unbiased=False).mean()) * 1e-4
        got = _lloyd64(X, torch.ones(X.shape[0], dtype=X.dtype, device=X.device),
                       _seeds64(X, case["k"], seed % 1_000_003), 300, tol)
        return {"labels": None, "centres": got[0] + mean, "inertia": got[1]}
    if kind == "batch":
        centroids = torch.zeros_like(state["centroids"], dtype=torch.float64)
        inertia, at = [], 0
        for X_t, w, init, _, _ in state["fits"]:
            got = _lloyd64(X_t.T.double(), w, init.T.double(), 100, 1e-4)
            m = init.numel()
            centroids[at:at + m] = got[0].T.reshape(-1)
            at += -(-m // 64) * 64
            inertia.append(got[1])
        return {"labels": None, "centroids": centroids, "n_iter": None,
                "inertia": np.array(inertia)}
    X = state["X_t"].T.contiguous()
    steps = 1 if kind == "step" else case["max_iter"]
    tol = 0.0 if kind == "step" else case["tol"]
    got = _lloyd64(X, state["w"], state["init"].T.double(), steps, tol)
    if kind == "step":
        return {"labels": None, "sizes": None, "centroids": got[0].T.contiguous()}
    return {"labels": None, "centroids": got[0].T.contiguous(), "n_iter": None,
            "inertia": got[1]}
