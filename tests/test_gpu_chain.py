"""Kernels whose workgroups wait for each other, from several threads and streams
at once (GPU): FP64 block sweeps beside each other, beside an FP32 sweep and
beside the Householder reduction.  The library orders such launches on a device
one after the other; every result equals the one obtained alone, bit for bit."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from oracle import harmony_oracle as ho
from rapids_singlecell_amd import _native
from rapids_singlecell_amd.datasets import synthetic_pcs
from rapids_singlecell_amd.preprocessing import _pca
from rapids_singlecell_amd.preprocessing._harmony import harmonize

pytestmark = pytest.mark.gpu

FIXED = dict(max_iter_harmony=2, max_iter_clustering=6, tol_harmony=float("-inf"),
             tol_clustering=float("-inf"))


def _harmony(n, d, B, K, seed, dtype):
    X, obs = synthetic_pcs(n, d, 8, B, seed=seed)
    X = X.astype(dtype)
    Y0 = ho.l2_normalize(X.astype(np.float64))
    Y0 = Y0[np.random.default_rng(seed).choice(n, K, replace=False)].astype(dtype)

    def run(device):
        Z = harmonize(torch.as_tensor(X, device=device), obs, "batch", n_clusters=K,
                      init_centroids=Y0, random_state=seed, **FIXED)
        return [Z.cpu().numpy()]

    return run


def _eigen(g, m, seed):
    A = np.random.default_rng(seed).normal(size=(g + 5, g)) * (1 + 3 * 0.97 ** np.arange(g))
    C = A.T @ A / g

    def run(device):
        w, v, total = _pca._device_eigenpairs(torch.as_tensor(C, device=device), m)
        return [w, v, np.float64(total)]

    return run


@pytest.mark.parametrize("kinds", ["two_f64", "f64_f32_eigen"])
def test_together_as_alone(device, kinds):
    jobs = [_harmony(60_000, 50, 8, 100, 11, np.float64)]
    if kinds == "two_f64":
        jobs.append(_harmony(9_000, 30, 20, 60, 12, np.float64))
    else:
        jobs += [_harmony(40_000, 30, 5, 60, 13, np.float32), _eigen(600, 50, 3)]
    alone = [run(device) for run in jobs]
    results = [None] * len(jobs)
    errors = []

    def worker(i):
        try:
            s = torch.cuda.Stream(device=device)
            with torch.cuda.stream(s):
                results[i] = [jobs[i](device) for _ in range(3)]
            s.synchronize()
        except Exception as e:  # noqa: BLE001 - re-raised below
            errors.append(e)
        finally:
            _native.release_thread()

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors, errors
    for want, got in zip(alone, results):
        for run in got:
            for a, b in zip(want, run):
                np.testing.assert_array_equal(a, b)
