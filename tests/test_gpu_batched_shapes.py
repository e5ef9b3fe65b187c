"""Batched clustering of jobs that share a sweep shape but not the shapes of the
joint centroid pass and old-row sums (GPU): one joint launch per number of column
tiles (its workgroup ranges are empty for the other jobs, at the start, in the
middle and at the end), and one for the sums with the lanes of the widest job.
Every job equals the same job alone, bit for bit."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing._harmony._batch import clustering_step, sweep_class
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu


def _job(device, n, d, B, K, seed, precision):
    g = torch.Generator(device=device).manual_seed(seed)
    X = torch.randn(n, d, device=device, generator=g)
    cats = np.random.default_rng(seed).integers(0, B, n).astype(np.int32)
    job = HarmonyJob(X, cats, B, n_clusters=K, theta_np=np.full(B, 2.0, np.float32),
                     N_b_np=np.bincount(cats, minlength=B).astype(np.float32),
                     max_iter_clustering=3, tol_clustering=float("-inf"), random_state=seed,
                     precision=precision)
    job.init((X[:K] / X[:K].norm(dim=1, keepdim=True)).contiguous())
    return job


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shapes", [
    # (cells, PCs, clusters): 3 and 4 column tiles in turn
    [(5_001, 36, 40), (9_000, 50, 33), (2_777, 40, 64), (7_003, 52, 50)],
    [(6_000, 52, 20), (3_001, 36, 60), (4_500, 50, 45)],
    # 150 and 250 clusters: 3 and 4 lanes' worth of columns
    [(8_000, 20, 150), (11_003, 20, 250), (6_001, 24, 129)],
])
def test_same_as_alone(device, shapes, precision):
    specs = [(n, d, 2 + i, K) for i, (n, d, K) in enumerate(shapes)]
    together = [_job(device, *s, seed=i, precision=precision) for i, s in enumerate(specs)]
    classes = {sweep_class(job) for job in together}
    assert len(classes) == 1 and None not in classes  # one call for all of them
    assert clustering_step(together, 0) == [3] * len(specs)
    for i, (s, job) in enumerate(zip(specs, together)):
        alone = _job(device, *s, seed=i, precision=precision)
        assert alone.clustering(0) == 3
        for name in ("R", "O", "E", "last_obj"):
            assert torch.equal(getattr(job, name), getattr(alone, name)), (i, name)
