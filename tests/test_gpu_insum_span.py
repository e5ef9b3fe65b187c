"""Old-row sums at every span of positions per wave: after some clustering
iterations O still equals the column sums of R over each batch, which fails by
whole rows if a span loses or repeats a position."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,B", [(40, 2), (257, 3), (32767, 5), (34817, 7), (70001, 2)])
def test_level_sums_follow_the_rows(device, dtype, n, B):
    K, d, iters = 20, 10, 3
    g = torch.Generator(device=device).manual_seed(n)
    X = torch.randn(n, d, device=device, dtype=dtype, generator=g)
    cats = (np.arange(n) * 7919 % n % B).astype(np.int32)
    counts = np.bincount(cats, minlength=B)
    np_dtype = np.float32 if dtype == torch.float32 else np.float64
    job = HarmonyJob(X, cats, B, n_clusters=K, theta_np=np.full(B, 2.0, np_dtype),
                     N_b_np=counts.astype(np_dtype), max_iter_clustering=iters,
                     tol_clustering=float("-inf"), random_state=n)
    Y0 = X[:K] / X[:K].norm(dim=1, keepdim=True)
    job.init(Y0.contiguous())
    job.clustering(0)
    hot = torch.zeros(B, n, device=device, dtype=torch.float64)
    hot[torch.as_tensor(cats, device=device).long(), torch.arange(n, device=device)] = 1.0
    O = hot @ job.R.double()
    # two roundings of O per block and iteration, and each block's sums added
    # in the rows' type
    eps = torch.finfo(dtype).eps
    tol = (2 * iters * 21 + 16) * eps * float(O.max()) + 1e-6
    assert float((job.O.double() - O).abs().max()) <= tol
