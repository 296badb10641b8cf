"""The split FP16 Gram form (banded precision, 16 <= d <= 128): neighbour lists
equal the oracle's FP64 ones at every number of MFMA steps and its remainders,
ragged tiles, the ordered and the plain layout, tiles of very different scales,
subnormal FP16 parts, non-finite and huge points, padding next to far points, and
with the record list full."""

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import engine

pytestmark = pytest.mark.gpu


def _check(x, r):
    want_rp, want_col = C.neighbours_csr(x, r, use_grid=False)
    X = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    rp, col, st = engine.radius_csr(X, float(r) ** 2, "f32_band")
    assert (rp.cpu().numpy() == want_rp).all()
    assert (col.cpu().numpy() == want_col).all()
    return st


def _quantile_radius(x, q):
    y = x[np.random.default_rng(0).permutation(len(x))[:300]].astype(np.float64)
    d2 = ((y[:, None] - y[None]) ** 2).sum(-1)
    return float(np.sqrt(np.quantile(d2[np.triu_indices(len(y), 1)], q)))


@pytest.mark.parametrize("d", [16, 17, 31, 32, 33, 48, 49, 64, 65, 79, 80, 81, 96, 100, 112, 113, 127, 128, 129])
@pytest.mark.parametrize("n,dtype", [(130, np.float32), (2113, np.float64)])
def test_every_step_count(cuda, d, n, dtype):
    rng = np.random.default_rng(d * n)
    x = (2.0 * rng.normal(size=(5, d)))[rng.integers(0, 5, n)] + rng.normal(size=(n, d))
    _check(x.astype(dtype), _quantile_radius(x, 0.1))


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1.0, 1e6, 1e15])
@pytest.mark.parametrize("d", [16, 40])
def test_scales(cuda, d, scale):
    rng = np.random.default_rng(3)
    x = rng.normal(size=(700, d))
    x[::7] *= 1e-4          # small next to large in one tile
    x[64:128] *= 1e-6       # whole tiles small
    x[130] = 0.0
    x = (x * scale).astype(np.float32)
    for q in (0.02, 0.3):
        _check(x, _quantile_radius(x, q))
    _check(x, 1e-7 * scale)  # far below the coordinates: zero and duplicate distances only
    _check(x, 1e3 * scale)   # far above them: all pairs


def test_offset_and_boundary(cuda):
    rng = np.random.default_rng(4)
    x = (rng.integers(-3, 4, size=(900, 24)) + 100.0).astype(np.float32)  # many pairs at exactly r
    st = _check(x, np.sqrt(150.0))
    assert st["band_hits"] > 0
    x = (rng.normal(size=(900, 20)) + 1e4).astype(np.float32)  # far from the origin: most pairs in the band
    _check(x, _quantile_radius(x, 0.1))


def test_nonfinite_and_huge(cuda):
    rng = np.random.default_rng(5)
    x = rng.normal(size=(400, 18)).astype(np.float32)
    x[3, 2], x[70, 0], x[140, 17], x[200], x[399, 1] = np.nan, np.inf, -np.inf, 3e37, 2e18
    _check(x, 4.0)


@pytest.mark.parametrize("records", [None, "1"])
@pytest.mark.parametrize("budget", [None, "512"])
@pytest.mark.parametrize("n,d", [(69, 64), (69, 16), (130, 128)])
def test_padding_next_to_a_far_tile(cuda, monkeypatch, n, d, budget, records):
    """A tile with a coordinate near 1e18 and the origin next to a ragged tile of
    tiny scale: padding values fall inside the pair's band, in one batch and in
    several, with room in the record list and without."""
    for name, value in (("CNN_HIP_MASK_BUDGET", budget), ("CNN_HIP_BAND_RECORDS", records)):
        if value is not None:
            monkeypatch.setenv(name, value)
    rng = np.random.default_rng(n)
    for small in (1e-3, 1e-5):
        x = (rng.uniform(-1.0, 1.0, size=(n, d)) * small).astype(np.float32)
        x[0] = 0.0
        x[1, 0] = 9e17
        _check(x, small)
        _check(x, 0.3 * small * np.sqrt(d))


@pytest.mark.parametrize("records", ["1", "9"])
@pytest.mark.parametrize("d", [16, 64, 100])
def test_full_record_list(cuda, monkeypatch, records, d):
    """Pairs beyond the record list recompute their values and settle them."""
    monkeypatch.setenv("CNN_HIP_BAND_RECORDS", records)
    rng = np.random.default_rng(d)
    x = (rng.integers(-2, 3, size=(1500, d)) + 10.0).astype(np.float32)
    st = _check(x, np.sqrt(4.0 * d))
    assert st["band_hits"] > 0


def _split_d2(x, r2):
    """The split form's FP32 values of d2 for all pairs: scaled parts, products of
    eight dimensions summed and rounded into FP32, the small products' sum last."""
    f32, f64 = np.float32, np.float64
    x = x.astype(f32)
    n, d = x.shape
    tile = np.arange(n) // 64
    m = np.array([max(np.abs(x[tile == t]).max(), np.sqrt(r2)) for t in range(tile[-1] + 1)])
    s = (2.0 ** (13 - np.floor(np.log2(m)))).astype(f32)[tile]
    xs = x * s[:, None]
    h = xs.astype(np.float16)
    low = (xs - h.astype(f32)).astype(np.float16).astype(f64)
    h = h.astype(f64)
    c = (0.25 * r2 - 0.5 * (x.astype(f64) ** 2).sum(1)).astype(f32)
    big = (c * s)[:, None] * s[None] + (c * s)[None] * s[:, None]
    small = np.zeros((n, n), f32)
    for k0 in range(0, d, 8):
        hh, lh, hl = np.zeros((n, n)), np.zeros((n, n)), np.zeros((n, n))
        for k in range(k0, min(k0 + 8, d)):
            hh += h[:, None, k] * h[None, :, k]
            lh += low[:, None, k] * h[None, :, k]
            hl += h[:, None, k] * low[None, :, k]
        small = (small + lh).astype(f32)
        small = (small + hl).astype(f32)
        big = (big + hh).astype(f32)
    return r2 - 2.0 * ((big + small).astype(f64) / (s[:, None].astype(f64) * s[None].astype(f64)))


def _far_case(n, d, far):
    """(x, r): the rows of `far` 1000 from the form's origin (the median of nine
    rows, here all zero), the others at it."""
    x = (np.random.default_rng(n).normal(size=(n, d)) + 1000.0).astype(np.float32)
    far[np.arange(9) * (n - 1) // 8] = False
    x[~far] = 0.0
    return x, np.sqrt(2.0 * d)


def _exact_d2(x):
    y = x.astype(np.float64)
    exact = np.zeros((len(x), len(x)))
    for k in range(x.shape[1]):
        exact += (y[:, None, k] - y[None, :, k]) ** 2
    return exact


@pytest.mark.parametrize("n,d", [(200, 16), (257, 33), (190, 64), (130, 128)])
def test_band_statistics(cuda, n, d):
    """Every pair of the far points (at most 11 a tile) lies inside the band: the
    reported flips and largest error are those of the split form's values."""
    far = np.arange(n) % 64 < 11
    x, r = _far_case(n, d, far)
    st = _check(x, r)
    value, exact = _split_d2(x, r * r), _exact_d2(x)
    tile = np.arange(n) // 64
    pairs = (tile[:, None] <= tile[None]) & far[:, None] & far[None]  # a tile pair is evaluated once
    assert st["band_hits"] == pairs.sum()
    assert st["max_abs_err_band"] == pytest.approx(np.abs(value - exact)[pairs].max(), rel=1e-9)
    assert st["band_flips"] == ((value <= r * r) != (exact <= r * r))[pairs].sum()


@pytest.mark.parametrize("records", [None, "1"])
@pytest.mark.parametrize("n,d", [(200, 16), (257, 33), (190, 64), (130, 128)])
def test_dense_band(cuda, monkeypatch, n, d, records):
    """Nearly every pair inside the band: whole pairs are recomputed, and the values
    of the matrix units lie within the margin (its accumulation, split and rounding
    terms times |x|^2, twice for T = (r2 - d2) / 2) of the FP64 ones."""
    if records is not None:
        monkeypatch.setenv("CNN_HIP_BAND_RECORDS", records)
    far = np.ones(n, bool)
    x, r = _far_case(n, d, far)
    st = _check(x, r)
    tile = np.arange(n) // 64
    pairs = (tile[:, None] <= tile[None]) & far[:, None] & far[None]
    assert st["band_hits"] == pairs.sum()
    w = (x.astype(np.float64) ** 2).sum(1).max()
    units = 21 * ((d + 15) // 16) + 6 + 9
    assert 0.0 < st["max_abs_err_band"] <= 2.0 * units * 2.0 ** -24 * (2.0 * w + 0.5 * r * r)
    exact = _exact_d2(x)[pairs]
    near = np.abs(exact - r * r) <= st["max_abs_err_band"]
    assert st["band_flips"] <= near.sum()


@pytest.mark.parametrize("dtype,shift", [(np.float32, 1024.0), (np.float64, 2.0 ** 30)])
@pytest.mark.parametrize("n,d", [(1, 16), (700, 16), (2000, 40), (300, 128)])
def test_translation_changes_nothing(cuda, n, d, dtype, shift):
    """The form works from a median of the points, so a translation that the input
    holds exactly leaves lists and band statistics the same (in the caller's order,
    n < 2048: beyond it the working order depends on the origin)."""
    rng = np.random.default_rng(n)
    x = np.rint(rng.normal(size=(n, d)) * 256.0) / 256.0
    r = _quantile_radius(x, 0.05) if n > 1 else 1.0
    base = _check(x.astype(dtype), r)
    moved = (x + shift).astype(dtype)
    assert (moved.astype(np.float64) == x + shift).all()
    st = _check(moved, r)
    for name in ("band_hits", "band_flips", "max_abs_err_band"):
        assert st[name] == base[name], name


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["column", "sampled rows", "no finite sample", "far samples"])
def test_origin_of_the_coordinates(cuda, kind, dtype):
    """One far column, and sampled rows that are not finite or far from the others."""
    for n, d in ((70, 64), (2113, 17)):
        rng = np.random.default_rng(n + d)
        x = rng.normal(size=(n, d))
        r = _quantile_radius(x, 0.2)
        sampled = np.arange(9) * (n - 1) // 8
        if kind == "column":
            x[:, -1] = 1e5 + np.sort(rng.uniform(0.0, 2.0 * r, n))
        elif kind == "sampled rows":
            x[sampled[::2], :3] = np.nan
            x[sampled[1], 4:] = -np.inf
        elif kind == "no finite sample":
            x[sampled, 1] = np.inf
        else:
            x[sampled] += 1e14
        _check(x.astype(dtype), r)


def test_row_tile_batches(cuda, monkeypatch):
    """Several row-tile batches: every pair evaluated from both sides."""
    monkeypatch.setenv("CNN_HIP_MASK_BUDGET", str(512 * 200))
    rng = np.random.default_rng(8)
    for n in (1500, 2500):
        x = rng.normal(size=(n, 33)).astype(np.float32)
        _check(x, _quantile_radius(x, 0.05))
