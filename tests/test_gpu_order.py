"""The spatial working order (d <= 8) follows a Hilbert curve: tiles of 64
consecutive points are compact, so a build keeps clearly fewer candidate tile
pairs than bit interleaving (Morton order) of the same points would."""

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import engine

pytestmark = pytest.mark.gpu


def _morton_tile_pairs(x, r, bits=8):
    q = np.floor((x - x.min(0)) / (x.max(0) - x.min(0)) * (2 ** bits - 1)).astype(np.int64)
    key = np.zeros(len(x), dtype=np.int64)
    for b in range(bits):
        for k in range(x.shape[1]):
            key |= ((q[:, k] >> b) & 1) << (b * x.shape[1] + k)
    x = x[np.argsort(key, kind="stable")]
    tiles = [x[t:t + 64] for t in range(0, len(x), 64)]
    lo, hi = np.array([t.min(0) for t in tiles]), np.array([t.max(0) for t in tiles])
    gap = np.maximum(0.0, np.maximum(lo[:, None] - hi[None], lo[None] - hi[:, None]))
    return int(((gap ** 2).sum(-1) <= r * r).sum())


# bound: a CPU count over uniform points gives 0.64 to 0.71 of Morton's pairs for d = 2, 3
@pytest.mark.parametrize("d,r", [(2, 0.02), (3, 0.05)])
def test_order_keeps_tiles_compact(cuda, d, r):
    x = np.random.default_rng(5).random((20011, d))
    g = engine.build_graph(torch.from_numpy(x).cuda(), r * r)
    assert g.stats["tile_pairs"] < 0.85 * _morton_tile_pairs(x, r)
    g.release()


# the smallest ordered size, ragged last tiles, one to three curve dimensions,
# constant and equal coordinates
@pytest.mark.parametrize("n", [129, 191, 1025])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 8])
def test_order_edges(cuda, n, d):
    rng = np.random.default_rng(n + d)
    x = rng.normal(size=(n, d))
    x[: n // 3, 0] = 0.25
    x[n // 2:, d - 1] = x[n // 2, d - 1]
    x[-5:] = x[0]
    want = C.fit(x, 0.6 * d, 2, member_cutoff=2)
    for precision in ("f64", "f32_band"):
        got = engine.fit(torch.from_numpy(x).cuda(), (0.6 * d) ** 2, 4, 3, precision=precision)[0]
        assert (got.cpu().numpy() == want).all()
