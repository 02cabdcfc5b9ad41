"""The work that a user of this KMeans engine has it do, as cases to time.

A case is one call of a public entry point on data of one shape:

  fit        `KMeans(...).fit(X)`: validation, centring, seeding, the Lloyd loop, labels and inertia
  lloyd      `drivers.lloyd`: one Lloyd run from given centroids on the transposed array, the call that
             the engine makes once per initialisation
  seed       `drivers.kmeans_plusplus`: the seeding alone
  predict    `KMeans.predict(X)` with fitted centres
  score      `drivers.get_labels_inertia`: the labels and the inertia that `KMeans.score` is taken from
  transform  `KMeans.transform(X)`: the distances to every centre

Data are Gaussian blobs, as the benchmark configurations of `sklearn_numba_dpex_amd.datasets` have them,
drawn on the GPU.  `spread` is the half width of the box that the blob centres lie in (standard deviations
are 0.5 to 2): with a small one the blobs overlap, labels keep moving and a run uses all its iterations.
"""

import math
import warnings

import numpy as np
import torch

from sklearn_numba_dpex_amd.kmeans import drivers
from sklearn_numba_dpex_amd.kmeans.estimator import KMeans

_DTYPES = {"f32": torch.float32, "f64": torch.float64}
_SIZE = {"f32": 4, "f64": 8}


def _case(name, op, n, d, k, dtype, iters=0, weights="unit", spread=10.0, source="device", far=0):
    case = dict(op=op, n=n, d=d, k=k, dtype=dtype, iters=iters, weights=weights, spread=spread, source=source,
                far=far)
    return dict(case, name=name) if name else case


def listed():
    return [
        # serving: labels for a handful of rows, latency only
        _case("predict_small", "predict", 256, 14, 127, "f32"),
        # a table of classroom size with scikit-learn's default type and the default seeding
        _case("fit_small_f64", "fit", 1_500, 20, 8, "f64", iters=10, spread=2.0),
        # the usual call of a scikit-learn program: numpy array in, fp64
        _case("fit_numpy_f64", "fit", 100_000, 30, 20, "f64", iters=10, spread=2.0, source="host"),
        # the first benchmark configuration: 14 features, 127 clusters, few samples (launches count)
        _case("lloyd_100k_d14_k127", "lloyd", 100_000, 14, 127, "f32", iters=20),
        # the headline configuration: many samples, few features, weights
        _case("lloyd_5m_d14_k127", "lloyd", 5_000_000, 14, 127, "f32", iters=20, weights="random"),
        # the contraction-bound configuration
        _case("lloyd_1m_d256_k1024", "lloyd", 1_000_000, 256, 1_024, "f32", iters=5, spread=3.5),
        # the fp64 configuration, with centroids that empty on the first iteration and are relocated
        _case("lloyd_2m_d32_k64_f64", "lloyd", 2_000_000, 32, 64, "f64", iters=12, far=16),
        # few clusters of wide samples (images as rows), seeding included
        _case("fit_70k_d784_k10", "fit", 70_000, 784, 10, "f32", iters=10, spread=1.0),
        # fp64, more features than the narrow kernels take, odd number of samples
        _case("lloyd_1m_d100_k100_f64", "lloyd", 1_000_003, 100, 100, "f64", iters=4, weights="random", spread=2.0),
        # the seeding configuration
        _case("seed_1m_d64_k256", "seed", 1_000_000, 64, 256, "f32", spread=5.0),
        # evaluation of a fitted model on held-out rows, odd sizes
        _case("score_1m_d50_k100_f64", "score", 1_000_003, 50, 100, "f64", weights="random", spread=4.0),
        # distances as features for another model
        _case("transform_300k_d100_k64", "transform", 300_007, 100, 64, "f32", spread=4.0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        op = rng.choice(["fit", "fit", "lloyd", "lloyd", "lloyd", "seed", "predict", "score", "transform"])
        dtype = rng.choice(["f32", "f64"])
        n = _log_uniform(rng, 250, 5_000_000)
        d = _log_uniform(rng, 2, 800)
        k = _log_uniform(rng, 2, 1_024)
        iters = rng.choice([4, 10, 20]) if op in ("fit", "lloyd") else 0
        spread = rng.choice([2.0, 4.0, 10.0])
        weights = rng.choice(["unit", "random"])
        source = "host" if op in ("fit", "predict") and n * d * _SIZE[dtype] <= 64 << 20 and rng.random() < 0.25 else "device"
        passes = max(1, iters)
        products = 2.0 * n * d * k * passes
        # at least sixteen samples a cluster, and no more work than the largest of the listed cases
        if n < 16 * k or n * d * _SIZE[dtype] > 800 << 20 or products > (1e12 if dtype == "f32" else 2.5e11):
            continue
        if op in ("seed", "fit") and (k * n * d * _SIZE[dtype] > 40e9 or k > 300):
            continue
        if n * d * _SIZE[dtype] * passes > 6 << 30 or op == "transform" and n * k * _SIZE[dtype] > 1 << 30:
            continue
        return _case(None, op, n, d, k, dtype, iters, weights, spread, source)


def _blobs(case, gen):
    n, d, k, dtype = case["n"], case["d"], case["k"], _DTYPES[case["dtype"]]
    blobs = k - case["far"] * 3 // 4 if case["far"] else k
    dev = gen.device
    centres = (torch.rand(blobs, d, generator=gen, device=dev) * 2 - 1) * case["spread"]
    std = 0.5 + 1.5 * torch.rand(blobs, generator=gen, device=dev)
    X = torch.empty(n, d, dtype=dtype, device=dev)
    step = max(1, (1 << 26) // d)
    for lo in range(0, n, step):
        hi = min(n, lo + step)
        which = torch.randint(0, blobs, (hi - lo,), generator=gen, device=dev)
        noise = torch.randn(hi - lo, d, generator=gen, device=dev, dtype=dtype)
        X[lo:hi] = centres[which].to(dtype).addcmul_(std[which].to(dtype)[:, None], noise)
    return X


def _centres(case, X, gen):
    """`k` rows of X, the last `far` of them replaced by points far away from every sample."""
    rows = torch.randperm(case["n"], generator=gen, device=X.device)[: case["k"]]
    centres = X[rows].clone()
    for j in range(case["far"]):
        centres[case["k"] - 1 - j] = 1e3 * (1 + j * 1e-3)
    return centres


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op, n, k = case["op"], case["n"], case["k"]
    X = _blobs(case, gen)
    w = None
    if case["weights"] == "random":
        w = 0.5 + torch.rand(n, generator=gen, device="cuda", dtype=X.dtype)
    state = dict(case=dict(case), seed=seed)
    if op in ("lloyd", "seed", "score"):
        X -= X.mean(0)  # what the engine hands on is centred
        state["w"] = torch.ones(n, dtype=X.dtype, device="cuda") if w is None else w
        state["X_t"] = X.T.contiguous()
        if op != "seed":
            state["centres_t"] = _centres(case, X, gen).T.contiguous()
        return state
    if op in ("predict", "transform"):
        model = KMeans(n_clusters=k, init=_centres(case, X, gen).cpu().numpy(), n_init=1, max_iter=1, tol=0.0)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            model.fit(X[: min(n, 64 * k)])
        state["model"] = model
    host = case["source"] == "host"
    state["X"] = X.cpu().numpy() if host else X
    state["w"] = w.cpu().numpy() if host and w is not None else w
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "fit":
        model = KMeans(n_clusters=case["k"], init="k-means++", n_init=1, max_iter=case["iters"], tol=0.0,
                       random_state=state["seed"] % (1 << 31))
        model.fit(state["X"], sample_weight=state["w"])
        return dict(centres=model.cluster_centers_, labels=model.labels_, inertia=model.inertia_, n_iter=model.n_iter_)
    if op == "lloyd":
        labels, inertia, centres_t, n_iter = drivers.lloyd(
            state["X_t"], state["w"], state["centres_t"], case["weights"] == "unit", case["iters"], False, 0.0)
        return dict(centres=centres_t, labels=labels, inertia=inertia, n_iter=n_iter)
    if op == "seed":
        centres_t, indices = drivers.kmeans_plusplus(
            state["X_t"], state["w"], case["k"], np.random.RandomState(state["seed"] % (1 << 31)))
        return dict(centres=centres_t, indices=indices)
    if op == "predict":
        return state["model"].predict(state["X"])
    if op == "score":
        labels, inertia = drivers.get_labels_inertia(state["X_t"], state["centres_t"], state["w"], True)
        return dict(labels=labels, inertia=inertia)
    return state["model"].transform(state["X"])


def work(case):
    """X is read once per Lloyd iteration and once for the final labels; seeding reads it once per centre
    (each centre is drawn from the distances to those before it)."""
    n, d, k, s, op, iters = case["n"], case["d"], case["k"], _SIZE[case["dtype"]], case["op"], case["iters"]
    X, centres, labels = n * d * s, k * d * s, 4 * n
    trials = 2 + int(math.log(k))
    seeding = dict(bytes=k * X, flops=3 * n * d * (1 + trials * (k - 1)))
    loop = dict(bytes=(iters + 1) * (X + n * s + labels + 2 * centres), flops=(iters + 1) * 2 * n * d * k + iters * 2 * n * d)
    if op == "seed":
        return dict(bytes=seeding["bytes"] + centres, flops=seeding["flops"])
    if op == "lloyd":
        return loop
    if op == "fit":
        return {u: seeding[u] + loop[u] for u in loop}
    if op == "transform":
        return dict(bytes=X + centres + n * k * s, flops=3 * n * d * k)
    return dict(bytes=X + centres + labels + (n * s if op == "score" else 0), flops=2 * n * d * k)


def tolerance(case):
    """About four times what a run in fp64 shows against one in fp32 (fp64: samples in another order), over the
    listed cases and two dozen drawn ones.  Within one Lloyd run of fp32 a sample midway between two centres
    may go either way, and the iterations after it carry the difference on: centres then differ by up to
    1e-3 in norm and 5e-2 in a coordinate of a small cluster, labels by up to 2 in 1000.  fp64 shows 4e-16
    for another order of the samples; sums in 64-bit fixed point, which some kernels use, are good to 1e-14.
    Seeding is all or nothing: one other pick changes all that follow."""
    op, f32 = case["op"], case["dtype"] == "f32"
    if op == "seed":
        return "exact"
    if op in ("fit", "lloyd"):
        return dict(rel=4e-3, max=0.2, differ=8e-3) if f32 else dict(rel=1e-13, max=1e-12, differ=0.0)
    # one labelling or one set of distances (fp32 seen: 8e-8 in norm, 5e-7 at most)
    return dict(rel=4e-7, max=4e-6, differ=1e-5) if f32 else dict(rel=1e-13, max=1e-12, differ=0.0)
