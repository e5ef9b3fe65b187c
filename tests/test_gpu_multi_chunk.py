"""Several covariates: the rule for the rows per chunk, on both sides of its
lines, against chunks of 64 rows and against the cells' own sums."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd import _native
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu


def _run(X, Y0, cats, levels, pairs, n_levels, counts, precision, chunk):
    _native.set_tuning(row_chunk=chunk)
    try:
        job = HarmonyJob(X, cats, len(pairs), n_clusters=len(Y0),
                         theta_np=np.full(n_levels, 2.0, np.float32), N_b_np=counts,
                         max_iter_clustering=2, tol_clustering=float("-inf"), random_state=1,
                         precision=precision, group_levels=pairs, n_levels0=levels)
        job.init(Y0)
        job.clustering(0)
    finally:
        _native.set_tuning(row_chunk=0)
    return job


# a block of n / 20 rows in chunks of 16 or 32 and its groups' partial chunks
# against 2048 waves: 16 rows, 16 (last), 32, 32 (last), 64
@pytest.mark.parametrize("n,B,D", [
    (3_001, 2, 3), (650_000, 4, 8), (665_003, 4, 8), (1_290_000, 4, 8), (700_000, 40, 50),
])
@pytest.mark.parametrize("precision", [0, 1])
def test_chunk_rule(device, precision, n, B, D):
    K, d = 12, 8
    g = torch.Generator(device=device).manual_seed(n)
    rng = np.random.default_rng(n)
    X = torch.randn(n, d, device=device, generator=g)
    b, dn = rng.integers(0, B, n), rng.integers(0, D, n)
    present, cats = np.unique(b * D + dn, return_inverse=True)
    pairs = np.stack([present // D, B + present % D], axis=1)
    counts = np.concatenate([np.bincount(b, minlength=B), np.bincount(dn, minlength=D)])
    Y0 = X[:K] / X[:K].norm(dim=1, keepdim=True)
    args = (X, Y0.contiguous(), cats.astype(np.int32), B, pairs, B + D, counts.astype(np.float32),
            precision)
    job, wide = _run(*args, 0), _run(*args, 64)
    # chunks are summed in float32 (6e-8 each); a clustering iteration
    # multiplies what O differs by with theta and 2 / sigma = 20
    assert float((job.R - wide.R).norm() / wide.R.norm()) < 1e-5
    hot = torch.zeros(B, K, device=device, dtype=torch.float64)
    hot.index_add_(0, torch.as_tensor(b, device=device), job.R.double())
    assert float((job.O[:B].double() - hot).abs().max()) <= 1e-5 * float(hot.max())
