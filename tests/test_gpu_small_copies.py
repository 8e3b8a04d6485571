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


@pytest.mark.parametrize("sizes", [[4], [20, 4, 16], [240_000, 240_004, 8], [1 << 20, 1 << 20, 1 << 20], [3, 0, (1 << 21) - 16, 40],
                                   [(1 << 21) - 12, 5 << 20, 12, 7]])
def test_several_arrays_come_down_at_once(sizes):
    """Aligned and odd sizes, more than a bounce buffer holds, empty and large ones: all bytes, in their places."""
    rng = np.random.default_rng(len(sizes))
    src = [rng.integers(0, 256, s, dtype=np.uint8) for s in sizes]
    dev = [d.DeviceArray.from_numpy(a, dtype=np.uint8) for a in src]
    got = d.binding._scratch_numpy(*((x, a.shape, np.uint8) for x, a in zip(dev, src)))
    for a, b in zip(got, src):
        assert np.array_equal(a, b)
