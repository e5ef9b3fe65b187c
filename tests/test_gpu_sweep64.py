"""FP64 block sweep (one launch per clustering iteration) at the edges of its
tiles and of its dispatch rule (GPU).

Every shape runs twice: by the rule (the sweep where it applies) and with the
sweep switched off (one launch per block).  Both stay within the FP64 path's
bound of the NumPy oracle (1e-8 of Z_corr) and within 1e-10 of each other:
both hold the block sums to 2^-40 of a cell or finer and everything else to
FP64 rounding, which 2 / sigma = 20 amplifies per clustering iteration.
Objectives agree to 1e-11 (the sweep forms the entropy's logarithm from the
exponent and the row sums).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import harmony_oracle as ho
from rapids_singlecell_amd import _native
from rapids_singlecell_amd.datasets import synthetic_pcs
from rapids_singlecell_amd.preprocessing._harmony import harmonize
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu

FIXED = dict(max_iter_harmony=2, max_iter_clustering=4, tol_harmony=float("-inf"),
             tol_clustering=float("-inf"), random_state=5)


def _problem(n, d, B, K, seed, dirichlet=False):
    X, obs = synthetic_pcs(n, d, 6, B, seed=seed, dirichlet_batches=dirichlet)
    X = X.astype(np.float64)
    Z = ho.l2_normalize(X)
    return X, obs, Z[np.random.default_rng(seed).choice(n, K, replace=False)]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _both(device, X, obs, **kw):
    out = []
    for no_sweep in (0, 1):
        _native.set_tuning(no_sweep=no_sweep)
        try:
            rec = {}
            Z = harmonize(torch.as_tensor(X, device=device), obs, "batch", record=rec, **kw)
            out.append((Z.cpu().numpy(), rec["R"].cpu().numpy(), rec["objectives"]))
        finally:
            _native.set_tuning(no_sweep=0)
    return out


# K: tile classes of 4, 7 and 8 columns and their edges, above 128 the
# per-block path; d: k-step classes, odd, above 100 the per-block path;
# B: batches beyond one thread's share (K = 128: 32) take the per-block path
@pytest.mark.parametrize("n,d,B,K", [
    (1501, 4, 2, 2), (1501, 5, 3, 15), (1700, 16, 2, 16), (1700, 17, 4, 17),
    (2049, 33, 3, 64), (2049, 32, 5, 65), (2111, 52, 2, 100), (2111, 53, 3, 112),
    (1999, 99, 3, 100), (1700, 101, 2, 20), (1700, 10, 2, 129),
    (3000, 3, 2, 10), (4001, 12, 32, 128), (4001, 12, 33, 128), (2600, 64, 20, 7),
])
def test_shapes(device, n, d, B, K):
    X, obs, Y0 = _problem(n, d, B, K, n + d + K)
    kw = dict(n_clusters=K, init_centroids=Y0, **FIXED)
    (Za, Ra, oa), (Zb, Rb, ob) = _both(device, X, obs, **kw)
    codes, cats, _ = ho.batch_codes(obs, "batch")
    ref = ho.harmonize(X, codes, len(cats), Y0=Y0, n_clusters=K, **FIXED)
    assert _rel(Za, ref) < 1e-8 and _rel(Zb, ref) < 1e-8
    assert _rel(Za, Zb) < 1e-10 and _rel(Ra, Rb) < 1e-10
    np.testing.assert_allclose(oa, ob, rtol=1e-11)


# shapes whose correction is refused (its FP64 apply step needs more LDS than a
# workgroup has): the clustering step alone
@pytest.mark.parametrize("n,d,B,K", [(1999, 99, 3, 113), (1999, 100, 4, 128)])
def test_clustering_of_the_widest(device, n, d, B, K):
    X, obs, Y0 = _problem(n, d, B, K, n + d + K)
    codes, cats, counts = ho.batch_codes(obs, "batch")
    state = []
    for no_sweep in (0, 1):
        _native.set_tuning(no_sweep=no_sweep)
        try:
            job = HarmonyJob(torch.as_tensor(X, device=device), codes, B, n_clusters=K,
                             theta_np=np.full(B, 2.0), N_b_np=counts.astype(np.float64),
                             max_iter_clustering=4, tol_clustering=float("-inf"), random_state=5)
            job.init(torch.as_tensor(Y0, device=device))
            assert job.clustering(0) == 4
            state.append([t.cpu().numpy() for t in (job.R, job.O, job.E, job.last_obj)])
        finally:
            _native.set_tuning(no_sweep=0)
    for a, b in zip(*state):
        assert _rel(a, b) < 1e-10


# rounds: one to several per wave, the staged rounds and past them, uneven
# batches (empty and full chunk ranges), few workgroups and one block
@pytest.mark.parametrize("n,B,prop,wgs", [
    (40_001, 3, 0.05, 0), (40_001, 9, 0.3, 4), (30_000, 2, 0.5, 1), (20_011, 30, 1.0, 3),
    (900, 5, 0.02, 0),
])
def test_rounds(device, n, B, prop, wgs):
    X, obs, Y0 = _problem(n, 11, B, 24, n + B, dirichlet=True)
    kw = dict(n_clusters=24, init_centroids=Y0, block_proportion=prop, **FIXED)
    _native.set_tuning(sweep_wg=wgs)
    try:
        (Za, Ra, oa), (Zb, Rb, ob) = _both(device, X, obs, **kw)
    finally:
        _native.set_tuning(sweep_wg=0)
    assert _rel(Za, Zb) < 1e-10 and _rel(Ra, Rb) < 1e-10
    np.testing.assert_allclose(oa, ob, rtol=1e-11)


def test_repeats_bitwise_and_reports_a_wait_that_runs_out(device):
    X, obs, Y0 = _problem(30_000, 20, 4, 40, 1)
    kw = dict(n_clusters=40, init_centroids=Y0, **FIXED)
    run = lambda: harmonize(torch.as_tensor(X, device=device), obs, "batch", **kw).cpu().numpy()  # noqa: E731
    first = run()
    _native.set_tuning(spin_limit=1)
    try:
        with pytest.raises(_native.HarmonyNativeError, match="timed out"):
            run()
    finally:
        _native.set_tuning(spin_limit=0)
    assert np.array_equal(run(), first)
