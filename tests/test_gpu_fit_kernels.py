"""The kernels of the fixed-H learner at the edges of their tiles: the update of W with all steps in
one launch (16 rows per workgroup, ranks padded to multiples of 32), and the products with H whose
columns hold around the six entries of a slot.  Against fp64."""

import numpy as np
import pytest

import npeff_ref_amd as d
from oracle import oracle as orc
from conftest import random_csr

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize("n,r", [(1, 1), (15, 31), (16, 32), (17, 33), (40, 64), (33, 65), (16, 97), (31, 128),
                                 (50, 129), (18, 193), (35, 255), (48, 256), (20, 257)])
def test_fit_updates_at_the_edges_of_the_tiles(n, r):
    rng = np.random.default_rng(1000 * n + r)
    m, eps, iters = 600, 1e-7, 6
    A = random_csr(rng, n, m, 200)
    B = random_csr(rng, r, m, 60, sort_cols=True)
    cA, cH = d.Csr.from_host(*A, m), d.Csr.from_host(*B, m)
    lrn = d.Learner(cA, cH, d.LearnerParams(max_iters=iters, eps=eps, log_every_n_steps=4))
    AH, HH, sq = lrn.products()
    assert _rel(AH, orc.spsp_dense_f64(A, m, B, r)) < 2e-6
    assert _rel(HH, orc.spsp_dense_f64(B, m, B, r)) < 2e-6
    lrn.initialize()
    W0 = lrn.GetOnHost_W()
    hist = lrn.Run(log=lambda s: None)
    W64, ref64, true64 = orc.fit_f64(AH.astype(np.float64), HH.astype(np.float64), sq, W0, np.float32(eps), iters, 4)
    assert _rel(lrn.GetOnHost_W(), W64) < 5e-6
    assert len(hist) == 1
    np.testing.assert_allclose([hist[0][1], hist[0][2]], [ref64[0], true64[0]], rtol=2e-5)


@pytest.mark.parametrize("r,per_col", [(2, 2), (40, 5), (64, 30), (1000, 3)])
def test_products_with_short_and_long_columns(r, per_col):
    """Columns of 0 .. 40 entries: within a slot and beyond it, component ids of up to ten bits, rows of
    H of one and of several chunks.  Two runs give the same bits."""
    rng = np.random.default_rng(r)
    m = 5000
    lens = np.minimum(r, np.where(rng.random(m) < 0.01, 40, rng.poisson(per_col, m)))
    cols = np.repeat(np.arange(m), lens)
    comps = np.concatenate([rng.permutation(r)[:k] for k in lens])
    order = np.lexsort((cols, comps))
    rowptr = np.concatenate(([0], np.cumsum(np.bincount(comps, minlength=r)))).astype(np.int64)
    B = (rowptr, cols[order].astype(np.int32), rng.lognormal(0, 1, len(order)).astype(np.float32))
    A = random_csr(rng, 37, m, 700)
    cA, cH = d.Csr.from_host(*A, m), d.Csr.from_host(*B, m)
    AH, HH, HH2 = d.DeviceArray((37, r)), d.DeviceArray((r, r)), d.DeviceArray((r, r))
    d.op_spsp_dense(cA, cH, AH)
    d.op_spsp_dense(cH, cH, HH)
    d.op_spsp_dense(cH, cH, HH2)
    assert _rel(AH.numpy(), orc.spsp_dense_f64(A, m, B, r)) < 2e-6
    assert _rel(HH.numpy(), orc.spsp_dense_f64(B, m, B, r)) < 2e-6
    assert np.array_equal(HH.numpy(), HH2.numpy())


@pytest.mark.parametrize("r,order", [(2, "up"), (37, "up"), (70, "up"), (37, "mixed"), (37, "blocks")])
def test_h_ht_in_cuts_of_columns(r, order):
    """H H^T where the rows are cut at the same columns (17 cuts, in which only the components from the
    row's own up are added), and rows that are not in order or each in a block of columns of its own, which
    are not cut.  Some columns hold more than the six entries of a slot.  The products and sums of positive numbers are
    rounded a few times each: 2e-6.  Symmetric, and two runs give the same bits."""
    rng = np.random.default_rng(r)
    m, k = 17 * 65536 + 5, 17 * 256 + 9
    few = np.arange(0, m, m // 300)  # columns that every row has
    rows = []
    for i in range(r):
        lo, hi = (m * i // r, m * (i + 1) // r) if order == "blocks" else (0, m)
        c = np.unique(np.concatenate([few, rng.choice(hi - lo, min(k, hi - lo), replace=False) + lo]))
        rows.append(rng.permutation(c) if order == "mixed" else c)
    rowptr = np.concatenate(([0], np.cumsum([len(c) for c in rows]))).astype(np.int64)
    B = (rowptr, np.concatenate(rows).astype(np.int32), rng.lognormal(0, 1, rowptr[-1]).astype(np.float32))
    cH = d.Csr.from_host(*B, m)
    HH, HH2 = d.DeviceArray((r, r)), d.DeviceArray((r, r))
    d.op_spsp_dense(cH, cH, HH)
    d.op_spsp_dense(cH, cH, HH2)
    got = HH.numpy()
    np.testing.assert_allclose(got, orc.spsp_dense_f64(B, m, B, r), rtol=2e-6)
    assert np.array_equal(got, HH2.numpy())
    if order == "up":
        assert np.array_equal(got, got.T)
