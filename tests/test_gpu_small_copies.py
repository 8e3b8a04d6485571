"""Host copies through pinned buffers (csrc/pool.hip): around one bounce buffer, around the words
kernel's limit, odd lengths, and on either side of the size from which pieces go over several threads."""

import numpy as np
import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [1, 4, 16384, 16388, 16390, 1 << 20, (1 << 21) + 4, (3 << 20) + 1, (4 << 20) - 1, 4 << 20, (4 << 20) + 8, (37 << 20) + 5])
def test_small_copies(nbytes):
    a = np.random.default_rng(nbytes).integers(0, 255, nbytes, dtype=np.uint8)
    x = d.DeviceArray.from_numpy(a, dtype=np.uint8)
    assert np.array_equal(x.numpy(), a)
