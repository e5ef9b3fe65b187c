"""``hz_knn`` at the edges of its tiles, parts and lists, on data whose FP32
distances are exact (small integers, or one non-zero entry per row): indices
and distances must then equal the (distance, index) order of all pairs, ties
included, whatever the split of the candidates."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing import _neighbors as nb

pytestmark = pytest.mark.gpu
FLT_MAX = float(np.finfo(np.float32).max)


def _expected(full, k):
    order = np.argsort(full, axis=1, kind="stable")[:, :k]
    return order, np.take_along_axis(full, order, axis=1)


@pytest.mark.parametrize("n,d,k", [
    (1, 1, 1), (2, 3, 2), (63, 4, 16), (64, 16, 17), (65, 17, 32), (127, 32, 1), (129, 33, 31),
    (1000, 52, 15), (1025, 53, 32), (2500, 64, 16), (2049, 65, 30), (1300, 100, 16),
    (1300, 101, 32), (700, 128, 8), (5003, 50, 15),
])
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean"])
def test_integer_rows_are_exact(device, metric, n, d, k):
    X = np.random.default_rng(n + d + k).integers(-2, 3, size=(n, d)).astype(np.float32)
    sq = (X.astype(np.int64) ** 2).sum(axis=1)
    full = sq[:, None] + sq[None, :] - 2 * (X @ X.T).astype(np.int64)
    ri, rd = _expected(full, k)
    idx, dist = nb.knn(torch.as_tensor(X, device=device), k, metric)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    rd = np.sqrt(rd.astype(np.float32)) if metric == "euclidean" else rd.astype(np.float32)
    # the device's square root is correctly rounded to 1 ulp
    np.testing.assert_allclose(dist.cpu().numpy(), rd, rtol=1.2e-7, atol=0)


@pytest.mark.parametrize("n,d,k", [(64, 5, 15), (1025, 30, 30), (3001, 100, 16), (300, 128, 32)])
def test_one_entry_rows_cosine(device, n, d, k):
    rng = np.random.default_rng(n + d + k)
    X = np.zeros((n, d), np.float32)
    X[np.arange(n), rng.integers(0, d, n)] = rng.choice([-4.0, 0.5, 1.0, 2.0], n)
    X[n // 2] = 0.0  # no direction: distance 1 to every row
    unit = np.sign(X)
    ri, rd = _expected(1.0 - unit @ unit.T, k)
    idx, dist = nb.knn(torch.as_tensor(X, device=device), k, "cosine")
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(dist.cpu().numpy(), rd.astype(np.float32))


@pytest.mark.parametrize("n,k", [(40, 32), (900, 15)])
def test_rows_without_neighbours(device, n, k):
    """A NaN row is nobody's cosine neighbour and has none itself; a list that
    cannot be filled ends in (-1, FLT_MAX)."""
    d = 8
    X = np.eye(d, dtype=np.float32)[np.random.default_rng(n).integers(0, d, n)]
    X[3:n:2] = np.nan
    good = np.flatnonzero(~np.isnan(X[:, 0]))
    full = 1.0 - X[good] @ X[good].T
    kk = min(k, len(good))
    ri, rd = _expected(full, kk)
    idx, dist = (t.cpu().numpy() for t in nb.knn(torch.as_tensor(X, device=device), k, "cosine"))
    np.testing.assert_array_equal(idx[good][:, :kk], good[ri])
    np.testing.assert_array_equal(dist[good][:, :kk], rd)
    bad = np.setdiff1d(np.arange(n), good)
    assert (idx[bad] == -1).all() and (dist[bad] == np.float32(FLT_MAX)).all()
    assert (idx[good][:, kk:] == -1).all() and (dist[good][:, kk:] == np.float32(FLT_MAX)).all()
