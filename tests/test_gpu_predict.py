"""Label prediction (Clustering.predict / PredictorFirstmatch.predict) on the
GPU equals the oracle's first-match restatement."""

import numpy as np
import pytest
import torch

from oracle import cnn_oracle as O
from commonnnclustering_amd import Clustering, engine
from commonnnclustering_amd.cluster import Bundle
from kat_data import equalise_labels

pytestmark = pytest.mark.gpu


def _split(n_x, n_y, d, seed):
    """Reference and predictand points drawn from one distribution."""
    Z = _blobs(n_x + n_y, d, seed)
    return Z[:n_x], Z[n_x:]


def _blobs(n, d, seed, k=4, noise=0.15):
    rng = np.random.default_rng(seed)
    centres = rng.uniform(-6, 6, size=(k, d))
    m = n - int(noise * n)
    X = np.concatenate([centres[rng.integers(0, k, size=m)] + rng.normal(0, 0.7, size=(m, d)),
                        rng.uniform(-8, 8, size=(n - m, d))])
    return X[rng.permutation(n)]


@pytest.mark.parametrize("precision", ["f64", "f32_band"])
@pytest.mark.parametrize("d,seed", [(2, 1), (3, 2), (16, 3), (2, 4)])
def test_predict_matches_oracle(cuda, precision, d, seed):
    X, Y = _split(1500, 900, d, seed)
    r = {2: 0.6, 3: 0.9, 16: 3.6}[d]
    c = 4
    labels_x, _ = O.fit(X, r, c, member_cutoff=5)
    want_l, want_c = O.predict_firstmatch(X, labels_x, Y, r, c)
    dtype = np.float32 if precision == "f32_band" else np.float64
    Xd = torch.from_numpy(X.astype(dtype)).cuda()
    Yd = torch.from_numpy(Y.astype(dtype)).cuda()
    lx = torch.from_numpy(labels_x).cuda()
    if dtype == np.float32:  # the oracle sees the exact float64 upcast of the float32 data
        labels_x32, _ = O.fit(X.astype(np.float32), r, c, member_cutoff=5)
        want_l, want_c = O.predict_firstmatch(X.astype(np.float32), labels_x32, Y.astype(np.float32), r, c)
        lx = torch.from_numpy(labels_x32).cuda()
    clusters = set(int(v) for v in lx.cpu().numpy()) - {0}
    lab, con, tests = engine.predict(Xd, lx, Yd, r * r, c + 2, c + 1, clusters, precision=precision)
    assert (lab.cpu().numpy() == want_l).all()
    assert (con.cpu().numpy() == want_c).all()
    assert tests > 0


def test_predict_cluster_subset_and_consider(cuda):
    X, Y = _split(1200, 700, 2, 11)
    r, c = 0.6, 3
    labels_x, _ = O.fit(X, r, c, member_cutoff=5)
    rng = np.random.default_rng(0)
    prior = rng.integers(0, 4, size=len(Y)).astype(np.int64)
    consider = (rng.uniform(size=len(Y)) > 0.3).astype(np.uint8)
    allowed = {1, 3}
    want_l, want_c = O.predict_firstmatch(X, labels_x, Y, r, c, clusters=allowed, labels_y=prior,
                                          consider_y=consider)
    lab, con, _ = engine.predict(torch.from_numpy(X).cuda(), torch.from_numpy(labels_x).cuda(),
                                 torch.from_numpy(Y).cuda(), r * r, c + 2, c + 1, allowed,
                                 labels_y=torch.from_numpy(prior).cuda(),
                                 consider_y=torch.from_numpy(consider).cuda())
    assert (lab.cpu().numpy() == want_l).all()
    assert (con.cpu().numpy() == want_c).all()


def test_predict_mixed_dtypes_and_empty(cuda):
    X, Y = _split(600, 300, 3, 21)
    Y = Y.astype(np.float32)
    r, c = 0.8, 2
    labels_x, _ = O.fit(X, r, c)
    want_l, _ = O.predict_firstmatch(X, labels_x, Y, r, c)
    lab, _, _ = engine.predict(torch.from_numpy(X).cuda(), torch.from_numpy(labels_x).cuda(),
                               torch.from_numpy(Y).cuda(), r * r, c + 2, c + 1, set(labels_x.tolist()) - {0})
    assert (lab.cpu().numpy() == want_l).all()
    # empty Y and empty reference set: nothing changes
    lab, con, tests = engine.predict(torch.from_numpy(X).cuda(), torch.from_numpy(labels_x).cuda(),
                                     torch.zeros((0, 3), dtype=torch.float64).cuda(), r * r, 4, 3, {1})
    assert lab.numel() == 0 and tests == 0
    lab, con, tests = engine.predict(torch.zeros((0, 3), dtype=torch.float32).cuda(),
                                     torch.zeros(0, dtype=torch.int64).cuda(), torch.from_numpy(Y).cuda(),
                                     r * r, 4, 3, {1})
    assert (lab.cpu().numpy() == 0).all() and (con.cpu().numpy() == 1).all()


def test_clustering_predict_moons_reference_case(cuda):
    """test_procedures.py:246-277 through the Clustering API."""
    from sklearn import datasets
    from sklearn.preprocessing import StandardScaler

    X, truth = datasets.make_moons(n_samples=1500, random_state=3)
    X = StandardScaler().fit_transform(X)
    truth = truth + 1
    ref = Clustering(np.ascontiguousarray(X[::2]))
    ref.labels = truth[::2]
    other = Clustering(X)
    ref.predict(other._bundle, 0.2, 2)
    assert (equalise_labels(other.labels) == equalise_labels(truth)).all()
    assert other._bundle._labels.meta["origin"] == "predict"
    assert other._bundle._labels.meta["frozen"] is True


def test_clustering_predict_frozen_labels_accumulate(cuda):
    X, Y = _split(1000, 800, 2, 31)
    ref = Clustering(X)
    ref.fit(0.6, 3, member_cutoff=5, v=False)
    other = Clustering(Y)
    labels = ref.labels
    # first only cluster 1, then (frozen labels kept) the rest
    ref.predict(other, 0.6, 3, clusters={1})
    first = other.labels.copy()
    ref.predict(other, 0.6, 3)
    want1, con1 = O.predict_firstmatch(X, labels, Y, 0.6, 3, clusters={1})
    want2, _ = O.predict_firstmatch(X, labels, Y, 0.6, 3, labels_y=want1, consider_y=con1)
    assert (first == want1).all()
    assert (other.labels == want2).all()
    # purge starts again from zeros
    ref.predict(other, 0.6, 3, clusters={2}, purge=True)
    want3, _ = O.predict_firstmatch(X, labels, Y, 0.6, 3, clusters={2})
    assert (other.labels == want3).all()


# n = 129 and 2048 are where the graphs start to hold words in d = 2 and 16
@pytest.mark.parametrize("d,n_x,n_y", [(2, 100, 20), (2, 128, 1), (2, 300, 65), (3, 63, 1000), (16, 2000, 47),
                                       (16, 2000, 48), (16, 2100, 63)])
def test_predict_on_words_and_lists(cuda, d, n_x, n_y):
    X, Y = _split(n_x, n_y, d, n_x + n_y)
    r, c = {2: 0.9, 3: 1.4, 16: 3.8}[d], 2
    labels_x, _ = O.fit(X, r, c, member_cutoff=3)
    want_l, want_c = O.predict_firstmatch(X, labels_x, Y, r, c)
    lx = torch.from_numpy(labels_x).cuda()
    lab, con, _ = engine.predict(torch.from_numpy(X).cuda(), lx, torch.from_numpy(Y).cuda(), r * r, c + 2, c + 1,
                                 set(labels_x.tolist()) - {0})
    assert (lab.cpu().numpy() == want_l).all()
    assert (con.cpu().numpy() == want_c).all()
