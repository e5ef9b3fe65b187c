"""Workspace of FP64 jobs that run the block sweep (GPU: the layout follows the
device's CU count).  Beside what a job takes with the sweep switched off there
are only every workgroup's copy of O and E (2 x batches x clusters values, one
workgroup per CU), the tables of 16 block orders for 16-row instead of 64-row
chunks (three 4-byte values per chunk) and the centroid partials of another
number of workgroups."""

from __future__ import annotations

import ctypes

import pytest
import torch

from rapids_singlecell_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,K,B", [
    (2_700, 50, 90, 2), (900, 4, 2, 2), (20_000, 50, 100, 8), (36_863, 100, 100, 32),
    (200_000, 50, 100, 8), (5_000, 30, 128, 32),
])
def test_extra_bytes(device, n, d, K, B):
    lib = _native.load()
    bs = int(n * 0.05)
    dims = _native.dims(n, d, K, B, bs, 8, 0)
    need = lib.hz_workspace_bytes(ctypes.byref(dims))
    _native.set_tuning(no_sweep=1)
    try:
        without = lib.hz_workspace_bytes(ctypes.byref(dims))
    finally:
        _native.set_tuning(no_sweep=0)
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    blocks = -(-n // bs)

    def chunks(rows):
        return -(-n // rows) + blocks * B

    def partials(rows):  # of the centroid pass: at most 512, evenly shared chunks
        per = -(-chunks(rows) // min(512, chunks(rows)))
        return -(-chunks(rows) // per)

    extra = (cus * 2 * B * K * 8 + 16 * 3 * 4 * (chunks(16) - chunks(64))
             + (partials(16) - partials(64)) * K * d * 8)
    print(f"\n{n} x {d}, K {K}, B {B}: {need} bytes, {without} without the sweep", flush=True)
    assert without > 0
    assert abs(need - without - extra) <= 64 * 256  # buffers are aligned to 256 bytes
