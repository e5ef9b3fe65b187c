"""FP64 block sweep whose wait for the other workgroups' block sums runs out
(GPU): the call goes on with one launch per block from the iteration that failed.

The waits are cut short from the host (``spin_limit`` polls, with ``spin_retry``
set); every kernel exits normally.  One poll fails in the first iteration of a
call, some tens of polls in any iteration or in none: whichever it is, R, O, E,
the objectives, the iteration counts and Z_corr are those of the path that was
never interrupted, within the bound between the FP64 sweep and one launch per
block (1e-10), and Z_corr within the FP64 path's bound of the oracle (1e-8).
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


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _run(device, X, obs, kw, **tuning):
    _native.set_tuning(**tuning)
    try:
        rec = {}
        Z = harmonize(torch.as_tensor(X, device=device), obs, "batch", record=rec, **kw)
        return [Z.cpu().numpy(), *(rec[k].cpu().numpy() for k in "ROE")], rec
    finally:
        _native.set_tuning(**{k: 0 for k in tuning})


# more clustering iterations than one set of block orders holds (16), and a run
# that stops by its own convergence test
@pytest.mark.parametrize("polls", [1, 12, 40, 200])
@pytest.mark.parametrize("n,d,B,K,kw", [
    (30_000, 20, 4, 40, dict(max_iter_harmony=2, max_iter_clustering=18,
                             tol_harmony=float("-inf"), tol_clustering=float("-inf"))),
    (9_001, 33, 20, 90, dict(max_iter_harmony=2, max_iter_clustering=30,
                             tol_harmony=float("-inf"), tol_clustering=1e-3)),
])
def test_call_goes_on(device, n, d, B, K, kw, polls):
    X, obs = synthetic_pcs(n, d, 6, B, seed=n + polls)
    X = X.astype(np.float64)
    Y0 = ho.l2_normalize(X)[np.random.default_rng(n).choice(n, K, replace=False)]
    kw = dict(kw, n_clusters=K, init_centroids=Y0, random_state=5)
    want, rec_w = _run(device, X, obs, kw)
    got, rec_g = _run(device, X, obs, kw, spin_limit=polls, spin_retry=1)
    assert rec_g["clustering_iters"] == rec_w["clustering_iters"]
    for a, b in zip(got, want):
        assert _rel(a, b) < 1e-10
    np.testing.assert_allclose(rec_g["objectives"], rec_w["objectives"], rtol=1e-11)
    codes, cats, _ = ho.batch_codes(obs, "batch")
    ref = ho.harmonize(X, codes, len(cats), Y0=Y0, **{k: v for k, v in kw.items()
                                                      if k != "init_centroids"})
    assert _rel(got[0], ref) < 1e-8
    # and the next call sweeps again
    again, _ = _run(device, X, obs, kw)
    for a, b in zip(again, want):
        assert np.array_equal(a, b)
