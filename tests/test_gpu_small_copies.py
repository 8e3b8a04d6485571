"""Host copies through pinned buffers (csrc/pool.hip): around one bounce buffer, around the words
kernel's limit, odd lengths, and on either side of the size from which pieces go over several threads."""

import ctypes as C

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


@pytest.mark.parametrize("counts", [[5], [1, 0, 300_001], [4096, 4097, 3]])
def test_scratch_buffers(counts):
    """Buffers handed out and taken back without a wait: what calls of the library wrote, also into a block that served before;
    parts of no bytes need no addresses."""
    lib, check = d.binding.lib, d.binding._check
    for seed in (3, 4):
        bufs, out = [], [np.full(max(n, 1), -1.0, np.float32) for n in counts]
        for n in counts:
            p = C.c_void_p()
            check(lib.dnpeff_scratch_malloc(4 * n, C.byref(p)))
            bufs.append(p)
            if n:
                check(lib.dnpeff_op_init_uniform(0, n, 1, seed, p))
        k = len(counts)
        check(lib.dnpeff_scratch_download(
            k, (C.c_void_p * k)(*(a.ctypes.data if n else None for a, n in zip(out, counts))),
            (C.c_void_p * k)(*(p.value if n else None for p, n in zip(bufs, counts))), (C.c_int64 * k)(*(4 * n for n in counts))))
        for p in bufs:
            check(lib.dnpeff_scratch_free(p))
        for a, n in zip(out, counts):
            assert list(a[:n][:64]) == [np.float32(d.uniform_at(seed, 0, i, 0, 1)) for i in range(min(n, 64))]
            assert (a[:n] >= 0).all() and (a[n:] == -1).all()
    with pytest.raises(d.DnpeffError, match="bad arguments"):
        check(lib.dnpeff_scratch_download(1, (C.c_void_p * 1)(None), (C.c_void_p * 1)(None), (C.c_int64 * 1)(4)))
