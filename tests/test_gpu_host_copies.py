"""The drop-in call's copies: chunked results equal the plain copy, and a
float32 input widened on the device gives the bits of one widened on the host,
whatever its layout."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd import pp
from rapids_singlecell_amd.datasets import SimpleAnnData, synthetic_pcs
from rapids_singlecell_amd.preprocessing import _harmony_integrate as hi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("chunks", [0.3, 2, 2.5, 5])
def test_chunks(device, dtype, chunks):
    per = hi._CHUNK_BYTES // torch.empty(0, dtype=dtype).element_size()
    t = torch.randn(int(per * chunks) // 3 + 1, 3, device=device, dtype=dtype)
    got = hi._to_host(t)
    np.testing.assert_array_equal(got, t.cpu().numpy())
    assert got.flags.owndata or got.base is not None
    np.testing.assert_array_equal(hi._to_host(t.T), t.cpu().numpy().T)


@pytest.mark.parametrize("layout", ["C", "F", "step", "readonly"])
def test_widened_input(device, layout):
    X, obs = synthetic_pcs(600, 10, 4, 2, seed=2)
    X32 = X.astype(np.float32)
    arr = {"C": X32, "F": np.asfortranarray(X32), "step": np.repeat(X32, 2, axis=1)[:, ::2],
           "readonly": X32.copy()}[layout]
    if layout == "readonly":
        arr.flags.writeable = False
    out = []
    for a in (arr, X32.astype(np.float64)):
        adata = SimpleAnnData(obs, {"X_pca": a})
        pp.harmony_integrate(adata, "batch", max_iter_harmony=2)
        out.append(adata.obsm["X_pca_harmony"])
    assert out[0].dtype == np.float64
    np.testing.assert_array_equal(out[0], out[1])
