"""The plain FP64 form on the FP64 matrix units (dense layout, 8 < d <= 120):
neighbour lists equal the oracle's at every remainder of the steps and around
the form's limits, ragged tiles, pairs exactly at r, non-finite and huge points,
several row-tile batches."""

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import engine

pytestmark = pytest.mark.gpu


def _check(x, r):
    want_rp, want_col = C.neighbours_csr(x, r, use_grid=False)
    rp, col, _ = engine.radius_csr(torch.from_numpy(np.ascontiguousarray(x)).cuda(), float(r) ** 2, "f64")
    assert (rp.cpu().numpy() == want_rp).all()
    assert (col.cpu().numpy() == want_col).all()


def _quantile_radius(x, q):
    y = x[np.random.default_rng(0).permutation(len(x))[:300]].astype(np.float64)
    d2 = ((y[:, None] - y[None]) ** 2).sum(-1)
    return float(np.sqrt(np.quantile(d2[np.triu_indices(len(y), 1)], q)))


@pytest.mark.parametrize("d", [9, 12, 15, 16, 17, 23, 24, 63, 64, 65, 88, 112, 119, 120, 121])
@pytest.mark.parametrize("n,dtype", [(1, np.float64), (65, np.float64), (130, np.float32), (2113, np.float64)])
def test_every_step_count(cuda, d, n, dtype):
    rng = np.random.default_rng(d * n)
    x = (2.0 * rng.normal(size=(5, d)))[rng.integers(0, 5, n)] + rng.normal(size=(n, d))
    _check(x.astype(dtype), _quantile_radius(x, 0.1) if n > 1 else 1.0)


@pytest.mark.parametrize("offset", [0.0, 1e8])
def test_pairs_at_the_radius(cuda, offset):
    """Integer coordinates: a large share of the pairs lies exactly at r."""
    rng = np.random.default_rng(4)
    x = rng.integers(-3, 4, size=(900, 24)) + offset
    _check(x, np.sqrt(150.0))
    _check(x / 10.0, np.sqrt(1.5))


def test_nonfinite_huge_and_tiny(cuda):
    rng = np.random.default_rng(5)
    x = rng.normal(size=(400, 18))
    x[3, 2], x[70, 0], x[140, 17], x[200], x[399, 1] = np.nan, np.inf, -np.inf, 1e200, 1e151
    _check(x, 4.0)
    _check(rng.normal(size=(300, 10)) * 1e-160, 3e-160)
    _check(rng.normal(size=(300, 10)), np.inf)


@pytest.mark.parametrize("n,d", [(2, 9), (70, 64), (2113, 17)])
@pytest.mark.parametrize("kind", ["offset", "column", "sampled rows", "no finite sample", "far samples"])
def test_origin_of_the_coordinates(cuda, n, d, kind):
    """The form works from a median of nine rows: points far from zero, one far
    column, and sampled rows that are not finite or far from all others."""
    rng = np.random.default_rng(n + d)
    x = rng.normal(size=(n, d))
    r = _quantile_radius(x, 0.2) if n > 2 else 4.0
    sampled = np.arange(9) * (n - 1) // 8
    if kind == "offset":
        for offset in (1e3, 1e8, -1e15):
            _check(x + offset, r)
        return
    if kind == "column":
        x[:, -1] = 1.7e9 + np.sort(rng.uniform(0.0, 2.0 * r, n))
    elif kind == "sampled rows":
        x[sampled[::2], :3] = np.nan
        x[sampled[1], 4:] = -np.inf
    elif kind == "no finite sample":
        x[sampled, 1] = np.inf
    else:
        x[sampled] += 1e14
    _check(x, r)


@pytest.mark.parametrize("r", [1e150, 2.1e150, 1e151, 1.3e154])
@pytest.mark.parametrize("n,d", [(1, 9), (65, 9), (130, 64), (2113, 17)])
def test_radius_beyond_the_padding_term(cuda, monkeypatch, n, d, r):
    """r^2 up to the largest double: padding rows and columns of the ragged tile are
    never neighbours, in one batch and in several."""
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, d))
    x[::5] *= 1e149
    _check(x, r)
    lab = engine.fit(torch.from_numpy(x).cuda(), r * r, 3, 2, precision="f64", member_cutoff=1)[0].cpu().numpy()
    assert (lab == C.fit(x, r, 1, member_cutoff=1)).all()
    monkeypatch.setenv("CNN_HIP_MASK_BUDGET", "512")
    _check(x, r)


def test_row_tile_batches(cuda, monkeypatch):
    monkeypatch.setenv("CNN_HIP_MASK_BUDGET", str(512 * 200))
    rng = np.random.default_rng(8)
    for n in (1500, 2500):
        x = rng.normal(size=(n, 33))
        _check(x, _quantile_radius(x, 0.05))
