"""Freed device blocks that the library keeps: not where the device is nearly full."""

import ctypes as C

import numpy as np
import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu


def _device_free():
    """Free memory as the runtime sees it (device_memory() would give the kept blocks back first)."""
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_nothing_large_is_kept_on_a_full_device():
    d.release_cached()
    free, total = d.device_memory()
    block = 200 << 20
    d.DeviceArray((block // 4,)).free()
    assert _device_free() <= free - block  # room enough: kept
    d.release_cached()
    fill = d.DeviceArray(((free - total // 32) // 4,))
    left = _device_free()
    d.DeviceArray((block // 4,)).free()
    assert _device_free() >= left
    small = [d.DeviceArray((4 << 20,)) for _ in range(8)]
    for x in small:
        x.free()
    assert _device_free() >= left - (64 << 20)
    fill.free()
    d.release_cached()


def test_a_refused_allocation_is_reported_once():
    """The next call launches kernels and succeeds, whoever asked for the memory."""
    x = d.DeviceArray.from_numpy(np.arange(6, dtype=np.float32).reshape(3, 2))
    with pytest.raises(d.DnpeffError, match="out of memory"):
        d.DeviceArray((1 << 44,))
    G = d.DeviceArray((2, 2))
    d.binding.op_gram(x, G)
    assert np.array_equal(G.numpy(), [[20, 26], [26, 35]])
    with pytest.raises(d.DnpeffError, match="out of memory"):
        d.DeviceArray((1 << 44,))
    assert d.op_dot(x, x) == 55
