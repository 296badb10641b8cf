"""What a user of this package has it do, as measurable cases.

Every case is one call (or the two or three calls that belong together) through
the public entry points: a fit of a point set over the range of sizes,
dimensions and precision forms that the package takes, a parameter scan, a
batch of small data sets, a re-fit of a resident graph, the prediction of new
points and a fit from a distance matrix.  Outputs are labels: whole numbers.

Data are drawn as the package meets them: molecular-dynamics projections
(d = 2, 3: anisotropic basins visited in dwell times of some hundred frames,
plus noise), descriptors (d = 8) and learned features (d >= 16: unit Gaussians
around separated centres, in random order).  The radius is a low percentile
``q`` (in percent) of the pair distances, so a point has about q/100 * n
neighbours.
"""

import math

import numpy as np
import torch

from commonnnclustering_amd import Clustering, engine

DEVICE = "cuda"


def listed():
    return [
        # The reference's tutorial: one small 2-d set from a host array through the
        # user class; latency of the whole call.
        {"name": "tutorial_2d_2k", "kind": "clustering", "n": 2000, "d": 2, "dtype": "f64", "precision": "f64",
         "q": 2.0, "c": 5, "k": 4},
        # A short trajectory projected on three coordinates, default (plain FP64) form.
        {"name": "fit_3d_30k_f64", "kind": "fit", "n": 30011, "d": 3, "dtype": "f64", "precision": "f64",
         "q": 0.5, "c": 10, "k": 8},
        # A long trajectory: the largest low-dimensional fit, banded form.
        {"name": "fit_3d_1m_band", "kind": "fit", "n": 1000000, "d": 3, "dtype": "f32", "precision": "f32_band",
         "q": 0.15, "c": 10, "k": 8},
        # Descriptors at the largest dimension of the spatial order, ragged size.
        {"name": "fit_8d_80k_band", "kind": "fit", "n": 80021, "d": 8, "dtype": "f32", "precision": "f32_band",
         "q": 0.5, "c": 10, "k": 10},
        # A served request of middling size in 16 dimensions.
        {"name": "fit_16d_100k_band", "kind": "fit", "n": 100003, "d": 16, "dtype": "f32", "precision": "f32_band",
         "q": 1.0, "c": 20, "k": 16},
        # Learned features: the largest high-dimensional fit, banded form.
        {"name": "fit_64d_200k_band", "kind": "fit", "n": 200000, "d": 64, "dtype": "f32", "precision": "f32_band",
         "q": 1.0, "c": 20, "k": 20},
        # The same kind of features with the default (plain FP64) form.
        {"name": "fit_64d_50k_f64", "kind": "fit", "n": 50001, "d": 64, "dtype": "f32", "precision": "f64",
         "q": 1.0, "c": 20, "k": 20},
        # A parameter scan: 8 radii times 8 similarity cutoffs on one 2-d set.
        {"name": "scan_2d_50k", "kind": "scan", "n": 50000, "d": 2, "dtype": "f32", "precision": "f32_band",
         "q": 2.0, "c": 1, "k": 6},
        # Many small data sets in one call (sizes 500 to 20000).
        {"name": "batch_3d_256", "kind": "batch", "n": 256, "d": 3, "dtype": "f32", "precision": "f32_band",
         "q": 2.0, "c": 5, "k": 6},
        # A resident graph fitted again at a smaller radius and another cutoff.
        {"name": "refit_3d_300k", "kind": "refit", "n": 299993, "d": 3, "dtype": "f32", "precision": "f32_band",
         "q": 0.3, "c": 10, "k": 8},
        # New frames labelled from a clustered trajectory.
        {"name": "predict_3d_100k", "kind": "predict", "n": 100000, "d": 3, "dtype": "f32", "precision": "f32_band",
         "q": 0.3, "c": 10, "k": 8},
        # A precomputed distance matrix: lists by threshold, labels, sort by size.
        {"name": "distances_8k", "kind": "distances", "n": 8001, "d": 3, "dtype": "f64", "precision": "f64",
         "q": 1.0, "c": 5, "k": 6},
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["clustering", "fit", "fit", "fit", "fit", "scan", "batch", "refit", "predict", "distances"])
    case = {"kind": kind, "n": 0, "d": 3, "dtype": rng.choice(["f32", "f32", "f64"]),
            "precision": rng.choice(["f32_band", "f32_band", "f64"]), "q": 1.0, "c": rng.choice([2, 5, 10, 20, 50]),
            "k": rng.randint(3, 24)}
    if kind == "clustering":
        case.update(n=_between(rng, 500, 20000), d=rng.choice([2, 3, 8, 16]), q=rng.uniform(0.5, 2.0))
    elif kind == "fit":
        d = rng.choice([1, 2, 3, 3, 3, 5, 8, 11, 16, 24, 32, 64, 64, 100])
        top = 1000000 if d <= 3 else 200000 if d <= 8 else 150000 if d <= 64 else 60000
        if case["precision"] == "f64" or 8 < d < 16:
            top = min(top, 500000 if d <= 3 else 50000)
        n = _between(rng, 1000, top)
        # about 30 to 1500 neighbours a point, at most two percent of the points
        case.update(n=n, d=d, q=min(2.0, 100.0 * _between(rng, 30, 1500) / n))
    elif kind == "scan":
        case.update(n=_between(rng, 2000, 50000), d=rng.choice([2, 3]), q=rng.uniform(0.5, 2.0), c=rng.choice([1, 2]))
    elif kind == "batch":
        case.update(n=_between(rng, 8, 256), d=rng.choice([2, 3, 5, 8]), q=rng.uniform(1.0, 2.0), c=5)
    elif kind == "refit":
        n = _between(rng, 2000, 300000)
        case.update(n=n, d=rng.choice([2, 3, 3, 8, 16]), q=min(2.0, 100.0 * _between(rng, 50, 1000) / n))
        if case["d"] > 3:
            case["n"] = min(n, 60000)
    elif kind == "predict":
        n = _between(rng, 2000, 100000)
        case.update(n=n, d=rng.choice([2, 3, 3, 8, 16]), q=min(2.0, 100.0 * _between(rng, 50, 500) / n))
        if case["d"] > 3:
            case["n"] = min(n, 40000)
    else:
        case.update(n=_between(rng, 500, 8000), d=rng.choice([2, 3, 8]), q=rng.uniform(0.3, 2.0))
    return case


def _dtype(case):
    return np.float64 if case["dtype"] == "f64" else np.float32


def _centres(rng, d, k):
    if d <= 8:
        return rng.uniform(-5.0, 5.0, size=(k, d)), rng.uniform(0.2, 0.8, size=(k, d))
    return 2.0 * rng.normal(size=(k, d)), np.ones((k, d))


def _points(rng, n, d, k, model=None):
    """(n, d) float64: basins in dwell-time order with 5 % noise (d <= 8), or unit
    Gaussians in random order (d > 8).  ``model``: the centres and widths to draw from."""
    centres, widths = _centres(rng, d, k) if model is None else model
    k = len(centres)
    if d <= 8:
        of = rng.integers(0, k, size=n // 400 + 2).repeat(400)[:n]
    else:
        of = rng.choice(k, size=n, p=rng.dirichlet(np.full(k, 5.0)))
    x = rng.standard_normal((n, d))
    x *= widths[of]
    x += centres[of]
    if d <= 8:
        noise = rng.random(n) < 0.05
        x[noise] = rng.uniform(-6.0, 6.0, size=(int(noise.sum()), d))
    return x


def _radius(rng, x, q):
    """The q-th percentile of the distances of 400,000 random pairs."""
    n = len(x)
    i = rng.integers(0, n, size=400_000)
    j = (i + 1 + rng.integers(0, n - 1, size=400_000)) % n
    s = np.zeros(len(i))
    for a in range(x.shape[1]):
        c = np.ascontiguousarray(x[:, a])
        s += (c[i] - c[j]) ** 2
    return float(np.sqrt(np.percentile(s, q)))


def _device(x, case):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=_dtype(case))).to(DEVICE)


def _batch_sizes(n):
    """n sizes spread over the logarithm of 500..20000."""
    return np.round(500.0 * 40.0 ** ((np.arange(n) + 0.5) / n)).astype(np.int64)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, n, d, k, c = case["kind"], case["n"], case["d"], case["k"], case["c"]
    state = {"case": case, "c": c}
    if kind == "batch":
        sizes = rng.permutation(_batch_sizes(n))
        sets = [_points(rng, int(m), d, k) for m in sizes]
        state["r2"] = np.array([_radius(rng, x[:2000], case["q"]) ** 2 for x in sets])
        state["offsets"] = np.concatenate([[0], np.cumsum(sizes)])
        state["X"] = _device(np.concatenate(sets), case)
        return state
    model = _centres(rng, d, k)
    x = _points(rng, n, d, k, model)
    r = state["r"] = _radius(rng, x, case["q"])
    if kind == "clustering":
        state["X"] = np.ascontiguousarray(x, dtype=_dtype(case))
        state["recipe"] = "coordinates" if case["precision"] == "f64" else "coordinates_f32"
    elif kind == "scan":
        state["X"] = _device(x, case)
        state["radii"] = np.geomspace(r / 8.0, r, 8)
        state["cutoffs"] = [c * m for m in (1, 2, 5, 10, 20, 40, 80, 160)]
    elif kind == "refit":
        state["graph"] = engine.build_graph(_device(x, case), r * r, precision=case["precision"])
        state["r2_small"] = (0.8 * r) ** 2
    elif kind == "predict":
        X = state["X"] = _device(x, case)
        labels = engine.fit(X, r * r, c + 2, c + 1, precision=case["precision"], member_cutoff=10)[0]
        state["labels"] = labels
        state["clusters"] = list(range(1, int(labels.max()) + 1))
        state["Y"] = _device(_points(rng, n // 5 + 1, d, k, model), case)
    elif kind == "distances":
        X = torch.from_numpy(x).to(DEVICE)
        D = torch.zeros((n, n), dtype=torch.float64, device=DEVICE)
        for a in range(d):
            D += (X[:, a, None] - X[None, :, a]) ** 2
        state["D"] = D.sqrt_().to(torch.float64 if case["dtype"] == "f64" else torch.float32)
    else:
        state["X"] = _device(x, case)
    return state


def run(state):
    case, c = state["case"], state["c"]
    kind, precision = case["kind"], case["precision"]
    if kind == "clustering":
        clustering = Clustering(state["X"], recipe=state["recipe"])
        clustering.fit(state["r"], c, member_cutoff=10, v=False)
        return clustering.labels
    if kind == "scan":
        return engine.fit_scan(state["X"], state["radii"], state["cutoffs"], precision=precision, member_cutoff=10)[0]
    if kind == "batch":
        return engine.fit_batch(state["X"], state["offsets"], state["r2"], c + 2, c + 1, precision=precision)[0]
    if kind == "refit":
        graph = state["graph"].rethreshold(state["r2_small"])
        labels = graph.fit(2 * c + 2, 2 * c + 1, member_cutoff=10)[0]
        graph.release()
        return labels
    if kind == "predict":
        labels, consider, _ = engine.predict(state["X"], state["labels"], state["Y"], state["r"] ** 2, c + 2, c + 1,
                                             state["clusters"], precision=precision)
        return labels, consider
    if kind == "distances":
        # the lists themselves have no fixed length: their offsets stand for them
        row_ptr, col, _ = engine.precomputed_csr(state["D"], state["r"])
        labels = engine.labels_from_csr(row_ptr, col, c + 2, c + 1)[0]
        engine.sort_by_size(labels, member_cutoff=10)
        return labels, row_ptr
    return engine.fit(state["X"], state["r"] ** 2, c + 2, c + 1, precision=precision, member_cutoff=10)[0]


def work(case):
    """Each input read once and each label written once; 3 d operations for every pair
    within the radius (the neighbour relation itself: a pair is decided once)."""
    kind, n, d = case["kind"], case["n"], case["d"]
    size = 8 if case["dtype"] == "f64" else 4
    share = case["q"] / 100.0
    if kind == "batch":
        sizes = _batch_sizes(n).astype(np.float64)
        return {"bytes": float(sizes.sum()) * (d * size + 8), "flops": 1.5 * d * share * float((sizes ** 2).sum())}
    pairs = 0.5 * share * n * n
    if kind == "scan":
        return {"bytes": n * (d * size + 64 * 8), "flops": 3.0 * d * pairs}
    if kind == "predict":
        m = n // 5 + 1
        return {"bytes": (n + m) * (d * size + 8) + 2 * m, "flops": 3.0 * d * (pairs + share * n * m)}
    if kind == "distances":
        return {"bytes": n * n * size + 16.0 * n, "flops": float(n) * n}
    return {"bytes": n * (d * size + 8), "flops": 3.0 * d * pairs}
