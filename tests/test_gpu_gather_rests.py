"""A H^T at ranks that four does not divide (csrc/spmm.hip, GatherDword): runs of every length around the steps that a batch of
64 entries is taken in, bit for bit the chain of fused multiply-adds in the order of the entries."""

import numpy as np
import pytest

import npeff_ref_amd as d
from npeff_ref_amd import binding as b

pytestmark = pytest.mark.gpu


def _chain(acc, a, h):
    """fmaf(a, h, acc): the product of two fp32 numbers is exact in fp64 (a sum there that lies halfway between two fp32
    numbers would be rounded twice; none of these do)."""
    return (np.float64(a) * h.astype(np.float64) + acc.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("large", [False, True])  # on either side of the line between the two lengths of a step (gather_many)
@pytest.mark.parametrize("r", [3, 50, 63, 126, 250, 510, 1001])
def test_runs_of_every_length_keep_the_order_of_their_sum(r, large):
    lens = [0, 1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 31, 33, 47, 48, 63, 64, 65, 79, 80, 95, 127, 128, 200]
    m = 300
    if large:  # more than 20 MB of rows to gather from, more than four workgroups per CU
        m = (5 << 20) // r + 1
        lens += [0] * (4 * 4 * d.device_info()[2])
    rng = np.random.default_rng(r)
    rowptr = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
    cols = np.concatenate([rng.permutation(m)[:n] for n in lens if n]).astype(np.int32)
    vals = rng.random(len(cols), dtype=np.float32)
    H = rng.random((m, r), dtype=np.float32)
    A = d.Csr.from_host(rowptr, cols, vals, m)
    on_device, out = d.DeviceArray.from_numpy(H), d.DeviceArray((len(lens), r))
    b._check(b.lib.dnpeff_op_spmm_n_variant(A._h, r, on_device.ptr, out.ptr, 1))
    want = np.zeros((len(lens), r), np.float32)
    for i in range(len(lens)):
        for e in range(rowptr[i], rowptr[i + 1]):
            want[i] = _chain(want[i], vals[e], H[cols[e]])
    assert np.array_equal(out.numpy(), want)
