"""FP64 centroid pass: column tile counts, groups of cluster tiles and row parts
at their edges, through whole Harmony iterations against the oracle (within the
FP64 path's 1e-8 of Z_corr)."""

import numpy as np
import pytest
import torch

from oracle import harmony_oracle as ho
from rapids_singlecell_amd.datasets import synthetic_pcs
from rapids_singlecell_amd.preprocessing._harmony import harmonize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,B,K", [
    (45, 6, 2, 3), (63, 80, 2, 10), (257, 65, 2, 33), (1030, 96, 3, 64), (1501, 97, 2, 65),
    (1300, 112, 2, 32), (1200, 113, 2, 48), (1100, 127, 2, 60), (9001, 40, 3, 70),
    (33000, 24, 4, 30),
])
def test_whole_iterations(device, n, d, B, K):
    X, obs = synthetic_pcs(n, d, 5, B, seed=n + d)
    X = X.astype(np.float64)
    Y0 = ho.l2_normalize(X)[np.random.default_rng(n).choice(n, K, replace=False)]
    kw = dict(n_clusters=K, init_centroids=Y0, max_iter_harmony=2, max_iter_clustering=3,
              tol_harmony=float("-inf"), tol_clustering=float("-inf"), random_state=3)
    Z = harmonize(torch.as_tensor(X, device=device), obs, "batch", **kw).cpu().numpy()
    codes, cats, _ = ho.batch_codes(obs, "batch")
    kw["Y0"] = kw.pop("init_centroids")
    ref = ho.harmonize(X, codes, len(cats), **kw)
    assert np.linalg.norm(Z - ref) < 1e-8 * np.linalg.norm(ref)
