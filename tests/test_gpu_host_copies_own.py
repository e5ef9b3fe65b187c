"""A result copied to the host through the pinned buffers owns its memory: a
second copy of the same size leaves the first as it was."""

import numpy as np
import pytest
import torch

from rapids_singlecell_amd.preprocessing import _harmony_integrate as hi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [0.5, 2, 3.5])
def test_results_are_independent(device, chunks):
    n = int(hi._CHUNK_BYTES // 8 * chunks)
    a, b = (torch.randn(n, device=device, dtype=torch.float64) for _ in range(2))
    first = hi._to_host(a)
    second = hi._to_host(b)
    assert not np.shares_memory(first, second)
    np.testing.assert_array_equal(first, a.cpu().numpy())
    np.testing.assert_array_equal(second, b.cpu().numpy())
    first[:] = 0.0  # writable, and the tensor is another memory
    assert bool((a != 0).any())
