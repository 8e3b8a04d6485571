"""Ranks above 128: the entry-balanced A^T W, X^T X on few rows, and ranks stored with zero components up to
the next multiple of 128."""

import numpy as np
import pytest

import npeff_ref_amd as d
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [132, 256, 300, 512, 520, 1024])
@pytest.mark.parametrize("n,m", [(1, 1), (3, 31), (600, 33), (257, 200)])
def test_spmm_t_balanced(n, m, r):
    """Columns inside a wave's share, cut by one, two and three of its ends, longer than a tile, empty."""
    rng = np.random.default_rng(n + m + r)
    fill = rng.choice([0.0, 0.003, 0.02, 0.3, 1.0], size=m)
    mask = rng.random((n, m)) < fill
    mask[0, 0] = True
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    ci = np.nonzero(mask)[1].astype(np.int32)
    va = rng.random(len(ci)).astype(np.float32)
    A = d.Csr.from_host(rp, ci, va, m)
    W = rng.random((n, r)).astype(np.float32)
    dW, dT = d.DeviceArray.from_numpy(W), d.DeviceArray.from_numpy(np.full((m, r), np.nan, dtype=np.float32))
    d.op_spmm_t(A, r, dW, dT)
    d.sync()
    dense = np.zeros((n, m))
    dense[mask] = va
    want = dense.T @ W.astype(np.float64)
    assert np.abs(dT.numpy() - want).max() <= 1e-5 * max(1.0, np.abs(want).max())
    A.close()


@pytest.mark.parametrize("n,r", [(1562, 256), (1563, 256), (1600, 252), (782, 512), (820, 492), (500, 1000)])
def test_spmm_t_balanced_on_a_large_factor(n, r):
    """On both sides of 1.6 MB of W, from which on the result goes past the caches."""
    m = 150
    rng = np.random.default_rng(n + r)
    mask = rng.random((n, m)) < rng.choice([0.0, 0.003, 0.3, 1.0], size=m)
    mask[0, 0] = True
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    ci = np.nonzero(mask)[1].astype(np.int32)
    va = rng.random(len(ci)).astype(np.float32)
    A = d.Csr.from_host(rp, ci, va, m)
    W = rng.random((n, r)).astype(np.float32)
    dW, dT = d.DeviceArray.from_numpy(W), d.DeviceArray.from_numpy(np.full((m + 1, r), np.nan, dtype=np.float32))
    d.op_spmm_t(A, r, dW, dT)
    d.sync()
    dense = np.zeros((n, m))
    dense[mask] = va
    want = dense.T @ W.astype(np.float64)
    got = dT.numpy()
    # (sums of up to n products of numbers below 1: n roundings of at most 2^-24 of the largest sum each)
    assert np.abs(got[:m] - want).max() <= n * 2.0 ** -24 * max(1.0, np.abs(want).max())
    assert np.isnan(got[m]).all()
    A.close()


@pytest.mark.parametrize("m", [32 * 4095, 32 * 4096, 32 * 4109 + 5])
def test_spmm_t_balanced_dealt_tiles(m):
    """Fewer, as many and more tiles than there are places to deal them from, with a rest."""
    n, r = 5, 132
    rng = np.random.default_rng(m)
    mask = rng.random((n, m)) < 0.3
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    va = rng.random(int(rp[-1])).astype(np.float32)
    A = d.Csr.from_host(rp, np.nonzero(mask)[1].astype(np.int32), va, m)
    W = rng.random((n, r)).astype(np.float32)
    dW, dT = d.DeviceArray.from_numpy(W), d.DeviceArray.from_numpy(np.full((m, r), np.nan, dtype=np.float32))
    d.op_spmm_t(A, r, dW, dT)
    d.sync()
    dense = np.zeros((n, m))
    dense[mask] = va
    assert np.abs(dT.numpy() - dense.T @ W).max() <= n * 2.0 ** -24 * n
    A.close()


@pytest.mark.parametrize("r", [132, 256, 600])
def test_spmm_t_tile_at_any_column(r):
    """Tiles on and off the groups of 32 columns: the rows of the whole product, bit for bit."""
    n, m = 600, 203
    rng = np.random.default_rng(r)
    mask = rng.random((n, m)) < rng.choice([0.0, 0.02, 0.3, 1.0], size=m)
    mask[0, 0] = True
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    ci = np.nonzero(mask)[1].astype(np.int32)
    A = d.Csr.from_host(rp, ci, rng.random(len(ci)).astype(np.float32), m)
    dW, dT = d.DeviceArray.from_numpy(rng.random((n, r)).astype(np.float32)), d.DeviceArray((m, r))
    d.op_spmm_t(A, r, dW, dT)
    d.sync()
    whole = dT.numpy()
    for c0, c1 in ((0, m), (32, 96), (64, m), (1, 32), (31, 33), (5, 200), (32, 50), (m - 1, m), (7, 7)):
        dP = d.DeviceArray.from_numpy(np.full((m, r), np.nan, dtype=np.float32))
        d.binding._check(d.lib.dnpeff_op_spmm_t_tile(A._h, r, dW.ptr, c0, c1, dP.ptr))
        d.sync()
        got = dP.numpy()
        assert np.array_equal(got[:c1 - c0], whole[c0:c1]) and np.isnan(got[c1 - c0:]).all()
    A.close()


@pytest.mark.parametrize("r", [256, 384, 512, 640, 1024])
@pytest.mark.parametrize("n", [1, 2, 7, 40])
def test_spmm_n_slices(n, r):
    """Rows without entries, of one entry, of parts of a chunk, of several chunks: the bits of the row chunks."""
    m = 9000
    rng = np.random.default_rng(n + r)
    lens = np.array([4097, 0, 1, 512, 513, 2048, 2049] + list(rng.integers(0, m, size=33)))[:n]
    ci = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lens]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    va = rng.random(len(ci)).astype(np.float32)
    A = d.Csr.from_host(rp, ci, va, m)
    H = rng.random((m, r)).astype(np.float32)
    if ci[0] != 0 and not np.any(ci == 0):
        H[0] = np.nan  # (gathered for groups without entries, and not added)
    dH = d.DeviceArray.from_numpy(H)
    outs = []
    for variant in (0, 2):
        dN = d.DeviceArray.from_numpy(np.full((n, r), np.nan, dtype=np.float32))
        d.binding._check(d.lib.dnpeff_op_spmm_n_variant(A._h, r, dH.ptr, dN.ptr, variant))
        d.sync()
        outs.append(dN.numpy())
    want = orc.spmm_n_f64(rp, ci, va, H)
    # (quarters of 512 entries added up one by one, then the parts: 600 roundings of 2^-24 of the sum at most)
    assert (np.abs(outs[0] - want) <= 600 * 2.0 ** -24 * np.abs(want)).all()
    if not np.isnan(H[0]).any():
        assert np.array_equal(outs[0], outs[1])
    A.close()


@pytest.mark.parametrize("n,r,per", [(37, 256, 999), (37, 256, 1001), (37, 384, 59), (37, 384, 61), (37, 512, 119),
                                     (37, 1024, 121), (520, 512, 599), (520, 1024, 351), (520, 640, 249), (520, 896, 251)])
def test_spmm_n_on_either_side_of_the_slices(n, r, per):
    """Short rows stay with the row chunks, and slices give the bits of those: ranks and rows around the line."""
    m = 4000
    rng = np.random.default_rng(n + r + per)
    ci = np.concatenate([rng.permutation(m)[:per] for _ in range(n)]).astype(np.int32)
    rp = np.arange(n + 1, dtype=np.int64) * per
    va = rng.random(n * per, dtype=np.float32)
    A = d.Csr.from_host(rp, ci, va, m)
    H = rng.random((m, r), dtype=np.float32)
    dH = d.DeviceArray.from_numpy(H)
    outs = []
    for variant in (0, 2):
        dN = d.DeviceArray.from_numpy(np.full((n, r), np.nan, dtype=np.float32))
        d.binding._check(d.lib.dnpeff_op_spmm_n_variant(A._h, r, dH.ptr, dN.ptr, variant))
        d.sync()
        outs.append(dN.numpy())
    want = orc.spmm_n_f64(rp, ci, va, H)
    assert (np.abs(outs[0] - want) <= 600 * 2.0 ** -24 * np.abs(want)).all()
    assert np.array_equal(outs[0], outs[1])
    A.close()


@pytest.mark.parametrize("rows", [128, 129, 160, 191, 1023])
@pytest.mark.parametrize("r", [256, 384, 512, 768])
def test_gram_on_few_rows(rows, r):
    X = np.random.default_rng(rows + r).random((rows, r)).astype(np.float32)
    dX, dG = d.DeviceArray.from_numpy(X), d.DeviceArray((r, r))
    d.op_gram(dX, dG)
    d.sync()
    want = X.astype(np.float64).T @ X
    assert (np.abs(dG.numpy() - want) / want).max() <= 2e-6


@pytest.mark.parametrize("n,m_full,k,r", [(40, 4000, 200, 129), (300, 30000, 900, 200), (1100, 60000, 2000, 301)])
def test_rank_between_the_tiles_of_128(n, m_full, k, r):
    eps = 1e-8
    A, norms = d.Csr.synth(n, m_full, k_fixed=k, seed=r)
    A.normalize_rows(norms)
    A.compact_columns(1)
    rp, ci, va = A.download()
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=4, eps=eps, seed=7, log_every=2))
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    assert W0[1, r - 1] == np.float32(d.uniform_at(7, 0, 1, r - 1, r))
    assert H0[r - 1, 3] == np.float32(d.uniform_at(7, 1, r - 1, 3, A.n_cols))
    nmf.run(log=lambda s: None)
    W64, H64, losses = orc.nmf_f64(rp, ci, va, A.n_cols, W0, H0, np.float32(eps), 4, 2)
    W, H = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    assert np.linalg.norm(W - W64) <= 1e-5 * np.linalg.norm(W64)
    assert np.linalg.norm(H - H64) <= 1e-5 * np.linalg.norm(H64)
    assert abs(nmf.computeUncachedLoss() - losses[-1]) <= 1e-5 * losses[-1]
    # the factors as callers see them are packed, and what they write to them counts
    w_dev, h_dev = nmf.device_factors()
    cols = np.array([0, A.n_cols - 1, 5], dtype=np.int32)
    assert np.array_equal(d.gather_rows(h_dev, r, cols), H[:, cols].T)
    assert np.array_equal(d.gather_rows(w_dev, r, np.arange(n)), W)
    d.binding._check(d.lib.dnpeff_dev_upload(w_dev, d.binding._ptr(W0), W0.nbytes))
    assert np.array_equal(nmf.loadWToHostSync(), W0)
    # from the host, and a step on
    nmf.set_factors(W0, H0)
    assert np.array_equal(nmf.loadWToHostSync(), W0) and np.array_equal(nmf.loadHToHostSync(), H0)
    nmf.step(4)
    assert np.array_equal(nmf.loadWToHostSync(), W) and np.array_equal(nmf.loadHToHostSync(), H)
    via_rows, via_cols = nmf.check_products()
    assert abs(via_rows - via_cols) <= 1e-5 * abs(via_rows)
    # the sparseness projection sees the rank's own components
    dW = d.DeviceArray.from_numpy(W)
    rounds = d.binding.op_sparsify_columns(dW, 3.0)
    assert nmf.sparsify_W(3.0) == rounds and np.array_equal(nmf.loadWToHostSync(), dW.numpy())
    nmf.close()
    A.close()


def test_padded_rank_sums_many_columns():
    """H^T H at a rank stored as 512, with large columns before small ones in every slice of the tiles: seen in
    the loss's <W^T W, H^T H>.  (W, and with it H, in eight of the components, one or two per tile.)"""
    n, m, r = 400, 2_000_000, 385
    rng = np.random.default_rng(r)
    rows = np.sort(rng.integers(0, n, m))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    cols = rng.permutation(m).astype(np.int32)
    vals = rng.random(m, dtype=np.float32) + np.float32(0.5)
    vals[cols < 20_000] *= np.float32(300)
    A = d.Csr.from_host(rp, cols, vals, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=1e-8, seed=5, log_every=0))
    nmf.initialize()
    held = np.array([0, 50, 100, 130, 200, 256, 300, 384])
    W = np.zeros((n, r), dtype=np.float32)
    W[:, held] = rng.random((n, len(held)), dtype=np.float32) + np.float32(0.5)
    nmf.set_factors(W, None)
    nmf.update_H()
    _, pos, _ = nmf.loss_terms()
    H = nmf.loadHToHostSync()[held].astype(np.float64)
    W = W[:, held].astype(np.float64)
    want = float(((W.T @ W) * (H @ H.T)).sum())
    assert abs(pos - want) <= 1.2e-7 * want  # (two roundings to fp32)
    nmf.close()
    A.close()


def test_padded_rank_sums_many_rows():
    """A^T W of the dense head's columns at a rank stored as 256, 2000 rows: one H update."""
    n, m, full, r = 2000, 40_000, 20_000, 150
    rng = np.random.default_rng(r)
    dense = np.zeros((n, m), dtype=np.float32)
    dense[:, :full] = rng.random((n, full), dtype=np.float32) + np.float32(0.5)
    dense[np.arange(m - full) % n, np.arange(full, m)] = 1
    dense[400:, 1:full:2] *= np.float32(1e-3)
    mask = dense != 0
    A = d.Csr.from_host(np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64),
                        np.nonzero(mask)[1].astype(np.int32), dense[mask], m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=1e-8, seed=5, log_every=0))
    assert A.head_info()[0] == full
    nmf.initialize()
    W, H = nmf.loadWToHostSync().astype(np.float64), nmf.loadHToHostSync().astype(np.float64)[:, :full]
    want = H * (W.T @ dense[:, :full]) / (W.T @ W @ H + 1e-8)
    nmf.update_H()
    err = np.linalg.norm(nmf.loadHToHostSync()[:, :full] - want) / np.linalg.norm(want)
    assert err <= 2.4e-7  # (four roundings to fp32)
    nmf.close()
    A.close()
