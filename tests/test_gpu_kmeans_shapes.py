"""k-means at the edges of its tiles (rows, clusters, columns) against the
oracle's Lloyd step, on sorted cells, so that neighbours share clusters."""

import numpy as np
import pytest
import torch

from oracle import harmony_oracle as ho
from rapids_singlecell_amd.preprocessing._harmony import kmeans_centroids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-6), (np.float64, 1e-9)])
@pytest.mark.parametrize("n,d,k", [
    (2, 1, 2), (15, 3, 4), (16, 16, 2), (17, 17, 16), (130, 32, 17), (129, 53, 64), (1000, 52, 65),
    (3001, 64, 112), (2000, 33, 113), (4100, 20, 128), (2500, 100, 40), (900, 127, 20),
    (1500, 10, 129), (40000, 7, 30),
])
def test_kmeans(device, dtype, tol, n, d, k):
    rng = np.random.default_rng(n + d + k)
    Z = ho.l2_normalize(rng.normal(size=(n, d)))
    Z = Z[np.argsort(Z[:, 0])].astype(dtype)
    got = kmeans_centroids(torch.as_tensor(Z, device=device), k, 77, max_iter=1).cpu().numpy()
    ref = ho.kmeans_centroids(Z.astype(np.float64), k, 77, max_iter=1)
    # a cluster's mean: float32 rounds the result, the fixed-point sums each
    # value to 2^-33; two scores of random unit rows are equal to a rounding
    # about once in 10^6 cells
    assert np.abs(got - ref).max() <= tol
