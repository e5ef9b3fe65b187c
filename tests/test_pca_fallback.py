"""PCA eigenpairs where the device reduction cannot run (host side, no GPU):
the host's full eigensolver takes over when the library says that the reduction
is not supported or its workspace does not fit, and any other error is raised."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing import _pca


class _Library:
    """The entry points of the reduction; hz_sym_tridiag returns ``rc``."""

    def __init__(self, rc):
        self.rc = rc
        self.asked = 0

    def hz_sym_eig_workspace_bytes(self, n):
        return 1 << 12

    def hz_sym_tridiag(self, *args):
        self.asked += 1
        return self.rc

    def hz_last_error(self):
        return b"stub"


class _Stream:
    cuda_stream = 0


def _stub(monkeypatch, rc):
    lib = _Library(rc)
    monkeypatch.setattr(_pca._native, "load", lambda: lib)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: _Stream())
    return lib


def _cov(g):
    A = np.random.default_rng(g).normal(size=(2 * g, g))
    return A.T @ A / (2 * g - 1)


def _check(C, m):
    w, v, total = _pca._eigenpairs(torch.as_tensor(C), m)
    ref_w, ref_v = np.linalg.eigh(C)
    np.testing.assert_array_equal(w, ref_w[::-1][:m])
    np.testing.assert_array_equal(v, ref_v[:, ::-1][:, :m])
    assert total == ref_w[::-1].sum()


def test_refused_launch_takes_the_host_solver(monkeypatch):
    lib = _stub(monkeypatch, -4)  # HZ_ERR_UNSUPPORTED
    _check(_cov(240), 20)
    assert lib.asked == 1


def test_no_memory_for_the_workspace_takes_the_host_solver(monkeypatch):
    lib = _stub(monkeypatch, 0)
    real = torch.empty

    def empty(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.cuda.OutOfMemoryError("no memory")
        return real(*size, **kw)

    monkeypatch.setattr(_pca.torch, "empty", empty)
    _check(_cov(240), 20)
    assert lib.asked == 0


@pytest.mark.parametrize("rc", [-1, -2, -3, -5])
def test_other_errors_are_raised(monkeypatch, rc):
    _stub(monkeypatch, rc)
    with pytest.raises(_pca._native.HarmonyNativeError, match=f"status {rc}"):
        _pca._eigenpairs(torch.as_tensor(_cov(240)), 20)
