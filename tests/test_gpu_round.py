"""The label pass on tile-pair words at the places where its kernels can go
wrong: tests that fail over many columns (batches of several columns a row, the
queue of tile pairs, also when it is full), tiles with more common candidate tiles
than one chunk of the match holds, ragged tiles, a cutoff of zero, mixed
components per tile.
Labels are whole numbers: equal to the oracle's."""

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import _lib, engine

pytestmark = pytest.mark.gpu


def _blobs(n, d, sep, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n, d))
    x[: n // 2, 0] += sep
    x[-n // 20:] = rng.uniform(-4.0, 4.0 + sep, size=(len(x[-n // 20:]), d))
    return x[rng.permutation(n)]


# (n, d, separation, radius, cutoffs): the degrees run from a few to thousands,
# the cutoffs from passing everywhere to failing for most edges
CASES = [
    (65, 2, 3.0, 1.0, (0, 3, 20)),
    (129, 3, 3.0, 0.8, (0, 2, 8)),
    (5003, 3, 2.0, 0.3, (2, 6, 12, 25)),
    (20011, 2, 3.0, 1.2, (50, 900, 1800, 2600)),
    (4111, 16, 6.0, 4.6, (5, 60, 200)),
]


@pytest.mark.parametrize("n,d,sep,r,cuts", CASES)
def test_round_matches_oracle(cuda, n, d, sep, r, cuts):
    x = _blobs(n, d, sep, n)
    X = torch.from_numpy(x).cuda()
    for c in cuts:
        want = C.fit(x, r, c, member_cutoff=2)
        lab, _, _, ls = engine.fit(X, r * r, c + 2, c + 1, precision="f64", member_cutoff=2)
        assert (lab.cpu().numpy() == want).all(), f"c={c}"
        if c == 0:  # c_sim = 0: every edge between core points passes
            lab = engine.fit(X, r * r, 0, 1, precision="f64", member_cutoff=1)[0].cpu().numpy()
            full = C.fit(x, r, 0, member_cutoff=1)
            assert ((lab > 0) >= (full > 0)).all()


@pytest.mark.parametrize("kind,n,d,deg,words", [
    ("heavy", 20000, 5, 40, False), ("heavy", 20000, 5, 2000, True), ("uniform", 9000, 24, 30, False),
    ("uniform", 9000, 24, 1500, True), ("basins", 20000, 3, 30, True),
])
@pytest.mark.parametrize("precision", ["f64", "f32_band"])
def test_form_by_candidates_and_fill(cuda, kind, n, d, deg, words, precision):
    """A fit tests similarities on its tile words or, where they are sparse over many
    candidate tiles, on its lists; labels and predictions are the same."""
    rng = np.random.default_rng(n + deg)
    if kind == "heavy":
        x = rng.standard_t(1.5, size=(n, d))
    elif kind == "uniform":
        x = rng.uniform(size=(n, d))
    else:
        x = _blobs(n, d, 4.0, n)
    i, j = rng.integers(0, n, (2, 400_000))
    r = float(np.sqrt(np.quantile(((x[i] - x[j]) ** 2).sum(1), deg / n)))
    c = max(1, deg // 20)
    want = C.fit(x, r, c, member_cutoff=3, use_grid=False)
    X = torch.from_numpy(x).cuda()
    lab, _, gs, ls = engine.fit(X, r * r, c + 2, c + 1, precision=precision, member_cutoff=3)
    assert (lab.cpu().numpy() == want).all()
    assert (ls["sim_form"] == _lib.CNN_SIM_FORM_TILE_WORDS) == words
    # new points, against the lists of both sets together
    y = x[rng.permutation(n)[:100]] + 0.1 * r / np.sqrt(d) * rng.normal(size=(100, d))
    ids = list(range(1, min(int(want.max()), 5) + 1))
    got = engine.predict(X, lab, torch.from_numpy(y).cuda(), r * r, c + 2, c + 1, ids, precision=precision)[0]
    rp, col = C.neighbours_csr(np.concatenate([x, y]), r, use_grid=False)
    refs = [col[rp[q]:rp[q + 1]][col[rp[q]:rp[q + 1]] < n] for q in range(n, n + 100)]
    ref = np.zeros(100, np.int64)
    for q, mine in enumerate(refs):
        for m in mine if len(mine) > c + 1 else ():
            other = col[rp[m]:rp[m + 1]]
            other = other[other < n]
            if want[m] in ids and len(other) > c + 1 and len(np.intersect1d(mine, other, True)) >= c + 2:
                ref[q] = want[m]
                break
    assert (got.cpu().numpy() == ref).all()


@pytest.mark.parametrize("capacity", ["1", "70"])
@pytest.mark.parametrize("n,d,sep,r,cuts", CASES[2:])
def test_full_queue_matches_oracle(cuda, monkeypatch, n, d, sep, r, cuts, capacity):
    """Tile pairs beyond the round's queue are tested where they were found: fits,
    every cutoff of a scan in one launch, and a batch."""
    monkeypatch.setenv("CNN_HIP_ROUND_QUEUE", capacity)
    x = _blobs(n, d, sep, n)
    X = torch.from_numpy(x).cuda()
    want = [C.fit(x, r, c, member_cutoff=2) for c in cuts]
    for c, w in zip(cuts, want):
        lab = engine.fit(X, r * r, c + 2, c + 1, precision="f64", member_cutoff=2)[0].cpu().numpy()
        assert (lab == w).all(), f"c={c}"
    if d > 3:
        return
    lab = engine.fit_scan(X, [r], list(cuts), precision="f64", member_cutoff=2)[0].cpu().numpy()
    for ci, w in enumerate(want):
        assert (lab[0, ci] == w).all(), f"scan c={cuts[ci]}"
    both, offsets = torch.cat([X, X]), np.array([0, n, 2 * n])
    lab = engine.fit_batch(both, offsets, np.full(2, r * r), cuts[-1] + 2, cuts[-1] + 1, precision="f64",
                           member_cutoff=2)[0].cpu().numpy()
    assert (lab[:n] == want[-1]).all() and (lab[n:] == want[-1]).all()


@pytest.mark.parametrize("n,d,sep,r,cuts", [c for c in CASES if c[1] <= 3 and c[0] > 128])
def test_scan_rounds_match_oracle(cuda, n, d, sep, r, cuts):
    """Every cutoff of a radius in one launch, twice over the same graph."""
    x = _blobs(n, d, sep, n)
    radii = [r, 0.7 * r]
    lab, _, _ = engine.fit_scan(torch.from_numpy(x).cuda(), radii, list(cuts), precision="f64", member_cutoff=2)
    lab = lab.cpu().numpy()
    for ri, rad in enumerate(radii):
        for ci, c in enumerate(cuts):
            assert (lab[ri, ci] == C.fit(x, rad, c, member_cutoff=2)).all(), (rad, c)
