"""Workspace of the neighbour search (host-only queries): the rows packed in
tiles of 64 with padded dimensions and a line of norms, and lists of k 8-byte
keys per row and part (at most 16 parts) that stay within 128 MiB whatever the
number of rows."""

from __future__ import annotations

import pytest

from rapids_singlecell_amd import _native

# padded dimensions of the kernel's classes
PADDED = {10: 16, 30: 32, 50: 52, 100: 100, 128: 128}


@pytest.mark.parametrize("d", sorted(PADDED))
@pytest.mark.parametrize("n", [1, 64, 5_000, 20_000, 150_001, 265_000, 400_000, 600_000,
                               868_000, 1_458_000, 5_000_000])
def test_lists_are_bounded(n, d):
    lib = _native.load()
    packed = -(-n // 64) * 64 * (PADDED[d] + 1) * 4
    any_k = lib.hz_knn_workspace_bytes(n, d, 0)
    assert packed <= any_k <= packed + (128 << 20) + 2 * 256
    for k in (1, 5, 15, 16, 17, 30, 32):
        got = lib.hz_knn_workspace_bytes_k(n, d, 0, k)
        lists = min(128 << 20, n * 16 * k * 8)
        assert packed <= got <= packed + lists + 2 * 256
        assert got <= any_k


def test_refused_numbers_of_neighbours():
    lib = _native.load()
    assert lib.hz_knn_workspace_bytes_k(100, 10, 0, 0) == 0
    assert lib.hz_knn_workspace_bytes_k(100, 10, 0, 33) == 0
    assert lib.hz_knn_workspace_bytes_k(0, 10, 0, 5) == 0
