"""Leading eigenpairs on the device (``hz_sym_tridiag``, ``hz_tridiag_top``,
``hz_sym_back`` and the host's inverse iteration) against LAPACK's full
eigensolver in float64, at the edges of the kernels' tiles and on matrices whose
reduction degenerates."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing import _pca

pytestmark = pytest.mark.gpu


def _check(device, C, m, must_run=True):
    ref = np.linalg.eigvalsh(C)[::-1][:m]
    scale = max(float(np.abs(np.linalg.eigvalsh(C)).max()), 1e-300)
    found = _pca._device_eigenpairs(torch.as_tensor(C, device=device), m)
    if found is None:
        assert not must_run
        w, v, total = _pca._eigenpairs(torch.as_tensor(C, device=device), m)
        ref = ref.clip(min=0.0)
    else:
        w, v, total = found
    # backward stable: a few rows' worth of roundings of the norm
    tol = 4e-16 * len(C) * scale + 1e-300
    assert np.abs(w - ref).max() <= tol
    assert np.abs(C @ v - v * w).max() <= tol
    assert np.abs(v.T @ v - np.eye(m)).max() <= 1e-11
    assert abs(total - np.trace(C)) <= tol * len(C)


@pytest.mark.parametrize("g,m", [
    (4, 1), (7, 1), (8, 2), (9, 2), (65, 16), (130, 30), (511, 50), (512, 50), (513, 20),
    (1023, 50), (1024, 10), (1025, 50), (2041, 50), (2048, 64),
])
def test_random_covariance(device, monkeypatch, g, m):
    monkeypatch.setattr(_pca, "_MIN_DEVICE_VARS", 3)
    rng = np.random.default_rng(g)
    A = rng.normal(size=(g + 5, g)) * (1 + 3 * 0.97 ** np.arange(g))
    _check(device, A.T @ A / g, m)


@pytest.mark.parametrize("kind", ["diagonal", "identity", "zero", "rank1", "blocks", "tiny", "huge"])
def test_degenerate(device, monkeypatch, kind):
    monkeypatch.setattr(_pca, "_MIN_DEVICE_VARS", 3)
    g, m = 200, 20
    rng = np.random.default_rng(7)
    A = rng.normal(size=(300, g))
    C = A.T @ A
    if kind == "diagonal":
        C = np.diag(rng.permutation(g) + 1.0)
    elif kind == "identity":
        C = np.eye(g)
    elif kind == "zero":
        C = np.zeros((g, g))
    elif kind == "rank1":
        C = np.outer(A[0], A[0])
    elif kind == "blocks":
        C[:100, 100:] = C[100:, :100] = 0.0
        C[100:, 100:] = C[:100, :100]  # every eigenvalue twice
    elif kind == "tiny":
        C = C * 1e-60
    elif kind == "huge":
        C = C * 1e60
    _check(device, C, m, must_run=False)


def test_nan_goes_to_the_host(device):
    C = np.eye(300)
    C[3, 4] = C[4, 3] = np.nan
    assert _pca._device_eigenpairs(torch.as_tensor(C, device=device), 10) is None
