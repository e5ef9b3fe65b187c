"""``hz_pca_covariance`` at the edges of its tiles, stages and row slices, with
rows that can and cannot be read 16 bytes at a time, against float64."""

import ctypes

import numpy as np
import pytest
import torch

from rapids_singlecell_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,g", [
    (2, 1), (2, 4), (31, 3), (33, 127), (64, 128), (65, 129), (100, 132), (4097, 256), (5001, 257),
    (20011, 300), (3000, 515),
])
@pytest.mark.parametrize("shift", [0, 1])
def test_covariance(device, n, g, shift):
    rng = np.random.default_rng(n + g)
    X = (rng.normal(size=(n, g)) * rng.uniform(0.5, 2.0, g) + rng.uniform(0, 2, g)).astype(np.float32)
    buf = torch.empty(n * g + 4, dtype=torch.float32, device=device)
    Xd = buf[shift:shift + n * g].view(n, g)  # shift 1: rows off the 16-byte grid
    Xd.copy_(torch.as_tensor(X))
    lib = _native.load()
    nb = lib.hz_pca_workspace_bytes(n, g)
    ws = torch.empty(nb, dtype=torch.uint8, device=device)
    mean = torch.empty(g, dtype=torch.float64, device=device)
    cov = torch.empty((g, g), dtype=torch.float64, device=device)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _native.check(lib.hz_pca_covariance(p(Xd), n, g, p(mean), p(cov), p(ws), nb, s), "cov")
    X64 = X.astype(np.float64)
    np.testing.assert_allclose(mean.cpu().numpy(), X64.mean(axis=0), rtol=1e-12, atol=1e-12)
    ref = np.cov(X64.T).reshape(g, g)
    got = cov.cpu().numpy()
    np.testing.assert_array_equal(got, got.T)
    # float32 products of centred values (the rounding of the centring counts
    # with the means, at most twice the smallest spread of 0.5)
    sd = np.sqrt(np.maximum(np.diag(ref), 1e-2))
    assert (np.abs(got - ref) <= 1e-5 * np.outer(sd, sd)).all()
