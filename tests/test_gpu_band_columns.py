"""The direct FP32 form (d < 16) reads a pair's test from the sign of its sum less
the band's lower end: points that are not finite in FP32, radii for which that end
is not positive, radii that are not finite, and ragged tiles of a packed batch,
against the oracle."""

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import engine

pytestmark = pytest.mark.gpu


# every decision is exact: lists are compared bit for bit
def _same_lists(x, r2):
    g = engine.build_graph(torch.from_numpy(x).cuda(), r2, precision="f32_band")
    row_ptr, col = g.to_csr()
    want_ptr, want_col = C.neighbours_bf(x, r2=r2)
    assert (row_ptr.cpu().numpy() == want_ptr).all()
    assert (col.cpu().numpy() == want_col).all()
    g.release()


# 65: dense layout; 129: the smallest ordered size, one point in the last tile
@pytest.mark.parametrize("n", [65, 129, 500])
@pytest.mark.parametrize("d", [1, 2, 3, 8, 9, 15])
def test_points_not_finite_in_fp32(cuda, n, d):
    x = np.random.default_rng(n * d).normal(size=(n, d))
    x[3] = np.nan
    x[[5, 60]] = 1e200  # equal points beyond FP32
    x[11, 0] = np.inf
    x[12, d - 1] = -np.inf
    _same_lists(x, 0.3 * d)


# integers far from the origin: distances exactly at the radius, and a band wider
# than the small radii (lower end <= 0)
@pytest.mark.parametrize("d", [2, 3, 8])
@pytest.mark.parametrize("r2", [1e-12, 0.0, 4.0, np.inf])
def test_band_ends(cuda, d, r2):
    _same_lists(np.random.default_rng(d).integers(0, 5, size=(700, d)) + 4000.0, r2)


def test_packed_ragged_tiles(cuda):
    rng = np.random.default_rng(2)
    sizes = [64, 1, 65, 127, 200]
    sets = [rng.normal(size=(n, 3)).astype(np.float32) for n in sizes]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    k = np.full(len(sizes), 2)
    lab = engine.fit_batch(torch.from_numpy(np.concatenate(sets)).cuda(), off, np.full(len(sizes), 0.7 * 0.7), k + 2, k + 1,
                           precision="f32_band", member_cutoff=2)[0].cpu().numpy()
    for b, x in enumerate(sets):
        assert (lab[off[b]:off[b + 1]] == C.fit(x, 0.7, 2, member_cutoff=2)).all()


# squares below the smallest normal FP32 number, and below the smallest of all
@pytest.mark.parametrize("n", [65, 500])
@pytest.mark.parametrize("d", [1, 3, 8, 9, 15])
@pytest.mark.parametrize("scale", [1e-18, 1e-20, 1e-22, 1e-24])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_squares_below_fp32(cuda, n, d, scale, dtype):
    x = (np.random.default_rng(n * d).normal(size=(n, d)) * scale).astype(dtype)
    for q in (0.3, 1.0, 4.0):
        _same_lists(x, q * d * float(scale) ** 2)
