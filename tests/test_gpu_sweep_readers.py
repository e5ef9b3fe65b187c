"""FP32 and split-BF16 block sweeps with workgroups that take no rows (GPU): the
automatic grid has eight of them where a thread's share of a block's old-row sums
does not fit its registers (more than 8 x max(1, 256 / clusters) batches).  The
block sums are fixed point, so R, O, E and the objective equal those of fixed
grids, which have none, bit for bit; one clustering step is checked against one
launch per block at that path's bound (1e-3 after three iterations)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from rapids_singlecell_amd import _native
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu


def _state(device, n, d, B, K, precision, **tuning):
    _native.set_tuning(**tuning)
    try:
        g = torch.Generator(device=device).manual_seed(n + B)
        X = torch.randn(n, d, device=device, generator=g)
        cats = np.random.default_rng(n + B).integers(0, B, n).astype(np.int32)
        job = HarmonyJob(X, cats, B, n_clusters=K, theta_np=np.full(B, 2.0, np.float32),
                         N_b_np=np.bincount(cats, minlength=B).astype(np.float32),
                         max_iter_clustering=3, tol_clustering=float("-inf"), random_state=3,
                         precision=precision)
        job.init((X[:K] / X[:K].norm(dim=1, keepdim=True)).contiguous())
        assert job.clustering(0) == 3
        return [t.clone() for t in (job.R, job.O, job.E, job.last_obj)]
    finally:
        _native.set_tuning(**{k: 0 for k in tuning})


# both sides of the line, several rounds per wave, every CU with rows already
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,d,B,K", [
    (3_001, 20, 16, 100), (3_001, 20, 17, 100), (9_000, 50, 32, 100), (40_003, 30, 24, 77),
    (20_000, 10, 9, 250), (20_000, 10, 8, 250), (5_000, 50, 40, 64), (400_000, 20, 24, 100),
])
def test_same_as_fixed_grids(device, n, d, B, K, precision):
    auto = _state(device, n, d, B, K, precision)
    for wgs in (3, 64, 256):
        if wgs == 3 and n > 100_000:
            continue
        for a, b in zip(auto, _state(device, n, d, B, K, precision, sweep_wg=wgs)):
            assert torch.equal(a, b)
    for a, b in zip(auto, _state(device, n, d, B, K, precision, no_sweep=1)):
        assert float((a - b).norm() / b.norm()) < 1e-3
