"""Block sweep at the edges of its stores and of its grid rule (GPU).

R rows leave the sweep in 16-byte quads; a cluster count that is not a
multiple of 4 leaves a quad that straddles the end of a row, stored element by
element.  Every remainder, and counts at the edges of the 16-column tiles, are
checked against the FP64 oracle with the bound of the other FP32 runs (1e-4 of
Z_corr at fixed iteration counts), and R's rows (including the row after each,
which a store past a row's end would damage) must sum to 1.

The number of workgroups follows the block's chunks; the block sums are fixed
point, so every grid must give the same bits.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import harmony_oracle as ho
from rapids_singlecell_amd import _native
from rapids_singlecell_amd.datasets import synthetic_pcs
from rapids_singlecell_amd.preprocessing._harmony import harmonize

pytestmark = pytest.mark.gpu

FIXED = dict(max_iter_harmony=2, max_iter_clustering=4, tol_harmony=float("-inf"),
             tol_clustering=float("-inf"), random_state=3)


def _problem(n, d, B, K, seed):
    X, obs = synthetic_pcs(n, d, 6, B, seed=seed)
    Z = ho.l2_normalize(X.astype(np.float64))
    return X, obs, Z[np.random.default_rng(seed).choice(n, K, replace=False)]


@pytest.mark.parametrize("precision", ["native", "split_bf16"])
@pytest.mark.parametrize("K", [2, 3, 5, 15, 18, 63, 65, 77, 111, 113])
def test_rows_at_every_cluster_remainder(device, precision, K):
    n, d, B = 2511, 19, 3
    X, obs, Y0 = _problem(n, d, B, K, K)
    codes, cats, _ = ho.batch_codes(obs, "batch")
    ref = ho.harmonize(X.astype(np.float64), codes, len(cats), Y0=Y0, n_clusters=K, **FIXED)
    rec = {}
    got = harmonize(torch.as_tensor(X, device=device), obs, "batch", n_clusters=K,
                    init_centroids=Y0.astype(np.float32), precision=precision, record=rec, **FIXED)
    err = np.linalg.norm(got.cpu().numpy() - ref) / np.linalg.norm(ref)
    assert err < (1e-4 if precision == "native" else 1e-3), err
    sums = rec["R"].double().sum(dim=1).cpu().numpy()
    # K values of FP32 rounding each, and the reciprocal's 1 ulp
    assert np.abs(sums - 1).max() < (K + 2) * 2.0**-23


@pytest.mark.parametrize("n,K,B", [(1000, 33, 3), (6000, 100, 2), (25_000, 60, 32), (70_003, 100, 5)])
def test_grid_rule_changes_no_bit(device, n, K, B):
    X, obs, Y0 = _problem(n, 30, B, K, n)
    kw = dict(n_clusters=K, init_centroids=Y0.astype(np.float32), **FIXED)
    X = torch.as_tensor(X, device=device)
    auto = harmonize(X, obs, "batch", **kw).cpu().numpy()
    try:
        for wgs in (7, 256):
            _native.set_tuning(sweep_wg=wgs)
            assert np.array_equal(harmonize(X, obs, "batch", **kw).cpu().numpy(), auto), wgs
    finally:
        _native.set_tuning(sweep_wg=0)
