"""Jobs on both sides of the line between joint launches and a launch per job
and kernel: every job of a batched step equals the same job alone, bit for bit."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing._harmony._batch import clustering_step
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu


def _job(device, n, B, K, seed):
    g = torch.Generator(device=device).manual_seed(seed)
    X = torch.randn(n, 20, device=device, generator=g)
    cats = np.random.default_rng(seed).integers(0, B, n).astype(np.int32)
    job = HarmonyJob(X, cats, B, n_clusters=K, theta_np=np.full(B, 2.0, np.float32),
                     N_b_np=np.bincount(cats, minlength=B).astype(np.float32),
                     max_iter_clustering=3, tol_clustering=float("-inf"), random_state=seed)
    job.init((X[:K] / X[:K].norm(dim=1, keepdim=True)).contiguous())
    return job


# average cells: 300000 (joint), 300001 (a launch per job)
@pytest.mark.parametrize("sizes", [(599_000, 1_000), (599_002, 1_000)])
def test_same_as_alone(device, sizes):
    shapes = [(n, 2 + i, 65 + 20 * i) for i, n in enumerate(sizes)]
    together = [_job(device, *s, seed=i) for i, s in enumerate(shapes)]
    assert clustering_step(together, 0) == [3, 3]
    for i, (s, job) in enumerate(zip(shapes, together)):
        alone = _job(device, *s, seed=i)
        assert alone.clustering(0) == 3
        for name in ("R", "O", "E", "last_obj"):
            assert torch.equal(getattr(job, name), getattr(alone, name)), (i, name)
