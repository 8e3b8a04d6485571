"""The step of small ranks (csrc/fused.hip, csrc/fused_wide.hip) against the fp64 oracle: remainders of the rank, tiles cut by
their number of entries, columns longer than a tile, empty columns and rows, and the changes between it
and the separate kernels."""

import numpy as np
import pytest

import npeff_ref_amd as d
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
EPS = 1e-8


def _matrix(n, m, seed, fill=0.02, full=3, empty_row=True):
    """Random columns; `full` of them hold every row (but the empty one), every seventh holds none."""
    rng = np.random.default_rng(seed)
    mask = rng.random((n, m)) < fill
    mask[:, :full] = True
    mask[:, 6::7] = False
    if empty_row and n > 3:
        mask[n // 2] = False
    rowptr = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    colind = np.concatenate([rng.permutation(np.flatnonzero(row)) for row in mask]).astype(np.int32)
    vals = rng.random(len(colind)).astype(np.float32)
    return rowptr, colind, vals


def _close(nmf, oracle_out):
    W64, H64, losses = oracle_out
    for got, want in ((nmf.loadWToHostSync(), W64), (nmf.loadHToHostSync(), H64)):
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    sq, pos, neg = nmf.loss_terms()  # (squared, against ||A||^2: a run may end on an exact product)
    assert abs(sq + pos - 2 * neg - losses[-1] ** 2) <= 1e-5 * sq


@pytest.mark.parametrize("n,m,r", [(3, 3, 1), (5, 63, 3), (7, 64, 4), (33, 65, 5), (70, 300, 8), (65, 257, 12),
                                   (40, 515, 13), (64, 1000, 16), (90, 130, 17), (1500, 1600, 20), (50, 129, 31),
                                   (130, 700, 33), (50, 64, 44), (77, 333, 50), (2100, 2200, 61), (69, 191, 64),
                                   (66, 66, 65), (97, 400, 80), (82, 95, 81), (300, 640, 96), (98, 129, 97),
                                   (1200, 1300, 113), (140, 65600, 128)])
def test_step_matches_the_oracle(n, m, r):
    rp, ci, va = _matrix(n, m, seed=n + r, fill=0.3 if n < 100 else 0.02)
    A = d.Csr.from_host(rp, ci, va, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=6, eps=EPS, seed=5, log_every=3))
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    nmf.run(log=lambda s: None)
    _close(nmf, orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 6, 3))
    nmf.close()
    A.close()


@pytest.mark.parametrize("r", [7, 48, 100])
def test_step_and_separate_kernels_in_turn(r, tune):
    """A run that changes from the fused step to the separate kernels and back, between and within
    iterations, keeps no product of an older factor."""
    n, m = 120, 900
    rp, ci, va = _matrix(n, m, seed=r, fill=0.05)
    A = d.Csr.from_host(rp, ci, va, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=6, eps=EPS, seed=5, log_every=0))
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    want = orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 6, 6)
    for fused in ((1, 1), (0, 0), (1, 0), (0, 1), (1, 1)):
        tune("fused_gram", fused[0])
        nmf.update_W()
        nmf.computeUncachedLoss()
        tune("fused_gram", fused[1])
        nmf.update_H()
    nmf.set_factors(nmf.loadWToHostSync(), nmf.loadHToHostSync())
    nmf.step(1)
    _close(nmf, want)
    nmf.close()
    A.close()


@pytest.mark.parametrize("r", [8, 16, 32, 66, 100])
def test_gram_of_many_columns(r):
    """H^T H as the H update leaves it, where a workgroup meets a column with large entries and then thousands
    with small ones (in one fp32 sum each of those would cost half a unit in the last place of the large
    one's square).  Seen in the loss's <W^T W, H^T H>."""
    n, m = 128, 4_000_000
    rng = np.random.default_rng(r)
    rows = np.sort(rng.integers(0, n, m))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    cols = rng.permutation(m).astype(np.int32)
    vals = rng.random(m, dtype=np.float32) + np.float32(0.5)
    vals[(cols < 65536) & (cols % 64 == 0)] *= np.float32(1000)
    A = d.Csr.from_host(rp, cols, vals, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
    nmf.initialize()
    nmf.step(1)
    _, pos, _ = nmf.loss_terms()
    W, H = nmf.loadWToHostSync().astype(np.float64), nmf.loadHToHostSync()
    G = np.zeros((r, r))
    for c0 in range(0, m, 500_000):
        part = H[:, c0:c0 + 500_000].astype(np.float64)
        G += part @ part.T
    want = float(((W.T @ W) * G).sum())
    assert abs(pos - want) <= 2.4e-7 * want  # (four roundings to fp32)
    nmf.close()
    A.close()


@pytest.mark.parametrize("r", [8, 16, 72])
def test_long_columns(r):
    """A^T W of columns that 40,000 rows hold: neither a lane group's entries nor the parts of its 15 to 127
    neighbours are all added up one by one.  (Sums, quotient and product with H round some ten times, with
    either sign: about three of 2^-24.)"""
    n, m, full = 40_000, 66_000, 6
    rng = np.random.default_rng(r)
    rows = np.concatenate([np.repeat(np.arange(n), full), rng.integers(0, n, m - full)])
    cols = np.concatenate([np.tile(np.arange(full), n), np.arange(full, m)]).astype(np.int32)
    order = np.argsort(rows, kind="stable")
    rows, cols = rows[order], cols[order]
    vals = rng.random(len(rows), dtype=np.float32) + np.float32(0.5)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    A = d.Csr.from_host(rp, cols, vals, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
    nmf.initialize()
    W, H = nmf.loadWToHostSync().astype(np.float64), nmf.loadHToHostSync()[:, :full].astype(np.float64)
    T = np.stack([W.T @ np.bincount(rows[cols == j], weights=vals[cols == j], minlength=n) for j in range(full)], axis=1)
    want = H * T / (W.T @ W @ H + EPS)
    nmf.update_H()
    err = np.linalg.norm(nmf.loadHToHostSync()[:, :full] - want) / np.linalg.norm(want)
    assert err <= 1.7e-7
    nmf.close()
    A.close()


def test_long_rows():
    """A H^T of rows whose large entries come first: those that follow in the same chunk join them in sums.  (Up
    to 24 roundings per chunk at the large entries' size, with either sign: about six of 2^-24.)"""
    n, m, r = 80, 300_000, 72
    rng = np.random.default_rng(r)
    vals = rng.random((n, m), dtype=np.float32) + np.float32(0.5)
    vals[:, :16] *= np.float32(700)
    A = d.Csr.from_host(np.arange(n + 1, dtype=np.int64) * m, np.tile(np.arange(m, dtype=np.int32), n), vals.reshape(-1), m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
    nmf.initialize()
    nmf.step(1)
    W, H = nmf.loadWToHostSync().astype(np.float64), nmf.loadHToHostSync().astype(np.float64)
    want = W * (vals.astype(np.float64) @ H.T) / (W @ (H @ H.T) + EPS)
    nmf.update_W()
    err = np.linalg.norm(nmf.loadWToHostSync() - want) / np.linalg.norm(want)
    assert err <= 4e-7
    nmf.close()
    A.close()


@pytest.mark.parametrize("r", [7, 16, 30, 64, 100])
def test_infinite_entry_stays_infinite(r):
    """<A H^T, W> with an infinite entry of H at the end of a row: infinite, with any number of lanes idle."""
    n, m = 130, 400
    for length in (1, 2, 3, 5, 33, 63, 64, 65, 130, 257):
        rp = np.arange(n + 1, dtype=np.int64) * length
        cols = np.tile(np.concatenate([np.arange(length - 1), [m - 1]]), n).astype(np.int32)
        A = d.Csr.from_host(rp, cols, np.ones(n * length, dtype=np.float32), m)
        nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
        W, H = np.ones((n, r), dtype=np.float32), np.ones((r, m), dtype=np.float32)
        H[0, m - 1] = np.inf
        nmf.set_factors(W, H)
        assert nmf.loss_terms()[2] == np.inf
        nmf.close()
        A.close()


@pytest.mark.parametrize("r,m", [(8, 140_000), (20, 70_000), (40, 40_000), (90, 20_000)])
def test_tiles_cut_where_lanes_and_groups_meet(r, m):
    """Columns that fill a tile by themselves, nearly or exactly, right before and after the columns at which a wave's lanes
    and the groups of columns end; empty ones beside them.  (Sums of up to n + r non-negative terms, a quotient and a product:
    as many roundings of 2^-24 and four.)"""
    n = 500
    rng = np.random.default_rng(r)
    length = np.ones(m, dtype=np.int64)
    for edge in (64, 128, 192, 256, 320, 512, 1024, m):
        at = np.arange(edge - 4, min(edge + 4, m))
        length[at] = rng.choice([0, 1, 16, 255, 256, n], size=len(at))
    length[700:900] = 33  # (many cuts in one group)
    cols = np.repeat(np.arange(m), length)
    rows = np.concatenate([rng.choice(n, size=k, replace=False) if k > 1 else [j % n] * k for j, k in enumerate(length)]).astype(np.int64)
    order = np.argsort(rows, kind="stable")
    rows, cols = rows[order], cols[order].astype(np.int32)
    vals = rng.random(len(rows), dtype=np.float32) + np.float32(0.5)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    A = d.Csr.from_host(rp, cols, vals, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
    nmf.initialize()
    W, H = nmf.loadWToHostSync().astype(np.float64), nmf.loadHToHostSync().astype(np.float64)
    T = np.stack([np.bincount(cols, weights=vals * W[rows, c], minlength=m) for c in range(r)])
    want = H * T / (W.T @ W @ H + EPS)
    nmf.update_H()
    got = nmf.loadHToHostSync()
    assert np.abs(got - want).max(axis=0)[length == 0].max(initial=0.0) == 0.0
    assert (np.abs(got - want) <= (n + r + 4) * 2.0 ** -24 * want).all()
    nmf.close()
    A.close()


def test_contexts_of_several_ranks_in_turn():
    """Contexts on one matrix whose ranks cut its columns into different tiles (64 to 256 columns each, 32, 32 with
    the long ones alone) and one without: each goes on where it was, bit for bit as by itself."""
    n, m, ranks = 150, 40_000, (8, 20, 50, 100, 129, 140)
    rp, ci, va = _matrix(n, m, seed=3, fill=0.01, full=40)

    def fresh(r):
        A = d.Csr.from_host(rp, ci, va, m)
        return A, d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))

    want = {}
    for r in ranks:
        A, nmf = fresh(r)
        nmf.initialize()
        nmf.step(3)
        want[r] = (nmf.loadWToHostSync(), nmf.loadHToHostSync(), nmf.computeUncachedLoss())
        nmf.close()
        A.close()
    A, first = fresh(ranks[0])
    contexts = {ranks[0]: first}
    for r in ranks[1:]:
        contexts[r] = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=5, log_every=0))
    for nmf in contexts.values():
        nmf.initialize()
    for _ in range(3):
        for nmf in contexts.values():
            nmf.update_W()
        for nmf in reversed(contexts.values()):
            nmf.update_H()
    for r, nmf in contexts.items():
        assert np.array_equal(nmf.loadWToHostSync(), want[r][0]) and np.array_equal(nmf.loadHToHostSync(), want[r][1])
        assert nmf.computeUncachedLoss() == want[r][2]
        nmf.close()
    A.close()


@pytest.mark.parametrize("n,m,r,fill", [(512, 3000, 9, 0.45), (512, 3000, 20, 0.45), (513, 3000, 20, 0.45),
                                        (257, 2500, 40, 0.3), (24, 1_100_000, 5, 1e-4)])
def test_partial_sums_on_either_side_of_their_limits(n, m, r, fill):
    """Eight and nine partial Gram matrices of W (summed by the H update, or before it), rows of five and six
    chunk sums (four are read at a time), and a factor too large to be written past the caches."""
    rp, ci, va = _matrix(n, m, seed=n + r, fill=fill)
    A = d.Csr.from_host(rp, ci, va, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=3, eps=EPS, seed=5, log_every=3))
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    nmf.run(log=lambda s: None)
    _close(nmf, orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 3, 3))
    nmf.close()
    A.close()


@pytest.mark.parametrize("n,m,r,fill", [(5, 24_003, 3, 0.9), (40, 9000, 17, 0.25), (61, 8191, 40, 0.22),
                                        (120, 6000, 100, 0.35), (9, 6000, 8, 0.32)])
def test_rows_grouped_by_xcd(n, m, r, fill):
    """Rows around the length from which their entries are grouped by XCD, an empty one, several chunks per
    row and XCD, sizes that no group of columns divides."""
    rp, ci, va = _matrix(n, m, seed=n + r, fill=fill)
    A = d.Csr.from_host(rp, ci, va, m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=4, eps=EPS, seed=5, log_every=2))
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    nmf.run(log=lambda s: None)
    _close(nmf, orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 4, 2))
    nmf.close()
    A.close()


@pytest.mark.parametrize("kind,by_xcd", [("any", True), ("one eighth", False), ("an eighth per row", False),
                                         ("one long share", False)])
def test_columns_that_load_the_xcds_unevenly(kind, by_xcd, tune, capfd):
    """Entries grouped by XCD (16 columns each in turn) where that gives every XCD and every workgroup about the same, not
    where the column ids repeat with a period of 128: all rows the same sixteen of it, every row its own, or one row alone."""
    n, m, k, r = 24, 24_000, 2000, 20
    rng = np.random.default_rng(7)
    of = (np.arange(m) >> 4) & 7
    rows = []
    for i in range(n):
        narrow = kind in ("one eighth", "an eighth per row") or (kind == "one long share" and i == 5)
        among = np.flatnonzero(of == (i % 8 if kind == "an eighth per row" else 3)) if narrow else np.arange(m)
        rows.append(rng.permutation(among)[:k])
    rp, ci = np.arange(n + 1, dtype=np.int64) * k, np.concatenate(rows).astype(np.int32)
    va = rng.random(n * k, dtype=np.float32)
    A = d.Csr.from_host(rp, ci, va, m)
    tune("verbose", 1)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=4, eps=EPS, seed=5, log_every=2))
    assert ("A H^T by XCD" in capfd.readouterr().err) == by_xcd
    tune("verbose", 0)
    nmf.initialize()
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    nmf.run(log=lambda s: None)
    _close(nmf, orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 4, 2))
    nmf.close()
    A.close()


@pytest.mark.parametrize("n,m,r,fill", [(2, 3, 1, 0.9), (16, 33, 4, 0.5), (17, 2100, 5, 0.05), (128, 640, 16, 0.04),
                                        (127, 300, 9, 0.1), (129, 300, 9, 0.1), (48, 907, 8, 0.07), (60, 500, 15, 0.08),
                                        (128, 500, 16, 0.04), (17, 1600, 5, 0.05), (8, 1900, 3, 0.05)])
def test_runs_in_one_workgroup(n, m, r, fill):
    """Runs that one workgroup's LDS holds (128 rows and 16 components at most), on either side of the line from which
    the launches are faster: several steps in one launch give the bits of as many launches of one step, and what the two
    updates of the launched step give (fp32 sums in another order, a few 1e-7 per step; past the line the same bits)."""
    rp, ci, va = _matrix(n, m, seed=n + m, fill=fill)
    A = d.Csr.from_host(rp, ci, va, m)

    def run(steps):
        nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=4, eps=EPS, seed=5, log_every=4))
        nmf.initialize()
        W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
        steps(nmf)
        out = nmf.loadWToHostSync(), nmf.loadHToHostSync(), nmf.loss_terms()
        nmf.close()
        return W0, H0, out

    W0, H0, one = run(lambda nmf: nmf.step(4))
    for got, want in zip(run(lambda nmf: [nmf.step(1) for _ in range(4)])[2], one):
        assert np.array_equal(got, want)
    two = run(lambda nmf: [(nmf.update_W(), nmf.update_H()) for _ in range(4)])[2]
    for got, want in zip(one[:2], two[:2]):
        assert np.linalg.norm(got - want) <= 5e-6 * np.linalg.norm(want)
        if n > 128 or 20 * m + 150 * n + 3 * len(ci) > 40_000:
            assert np.array_equal(got, want)
    W64, H64, losses = orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 4, 4)
    for got, want in zip(one[:2], (W64, H64)):
        assert np.linalg.norm(got - want) <= 5e-6 * np.linalg.norm(want)
    sq, pos, neg = one[2]
    assert abs(sq + pos - 2 * neg - losses[-1] ** 2) <= 1e-5 * sq
    A.close()


@pytest.mark.parametrize("n,fill,ranks", [(120, 0.35, (40, 100)), (1010, 0.42, (9, 8))])
def test_ranks_on_either_side_of_the_grouping(n, fill, ranks):
    """Contexts of two ranks on one matrix, whose rows only the first groups by XCD (40 and 100 components; 9 and 8
    where a row makes three even chunks): each gives the bits that it gives on a matrix of its own, whichever comes first."""
    m = 6000
    rp, ci, va = _matrix(n, m, seed=3, fill=fill)

    def run(A, r):
        nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=3, eps=EPS, seed=5, log_every=3))
        nmf.run(log=lambda s: None)
        out = nmf.loadWToHostSync(), nmf.loadHToHostSync()
        nmf.close()
        return out

    alone = {}
    first, second = ranks
    for r in ranks:
        A = d.Csr.from_host(rp, ci, va, m)
        alone[r] = run(A, r)
        A.close()
    for order in ((first, second, first), (second, first, second)):
        A = d.Csr.from_host(rp, ci, va, m)
        for r in order:
            for got, want in zip(run(A, r), alone[r]):
                assert np.array_equal(got, want)
        A.close()


@pytest.mark.parametrize("m,k,fused", [(2000, 120, True), (65_535, 700, True), (65_536, 700, True), (9000, 6800, True),
                                       (9000, 6850, False)])
def test_rank_64_with_many_rows(m, k, fused):
    """1024 rows and more at rank 64: a dense head where nine times the entries past 6 M are more than the cells (1030 x
    9000: 6826 entries per row), else the fused step."""
    n = 1030
    if 2 * k <= m:
        A, norms = d.Csr.synth(n, m, k_fixed=k, zipf_s=1.1, seed=8)
        A.normalize_rows(norms)
    else:
        rng = np.random.default_rng(m + k)
        cols = np.argsort(rng.random((n, m), dtype=np.float32), axis=1)[:, :k].astype(np.int32)
        A = d.Csr.from_host(np.arange(n + 1, dtype=np.int64) * k, cols.ravel(), rng.random(n * k, dtype=np.float32), m)
    rp, ci, va = A.download()
    nmf = d.MuNmf(A, d.MuNmfParams(rank=64, max_iters=2, eps=EPS, seed=5, log_every=2))
    nmf.initialize()
    assert (A.head_info()[0] == 0) == fused
    W0, H0 = nmf.loadWToHostSync(), nmf.loadHToHostSync()
    nmf.run(log=lambda s: None)
    _close(nmf, orc.nmf_f64(rp, ci, va, m, W0, H0, np.float32(EPS), 2, 2))
    nmf.close()
    A.close()


@pytest.mark.parametrize("zipf,head", [(1.6, True), (1.05, False)])
def test_rank_64_with_a_head_of_very_many_entries(zipf, head, tune):
    """66 M entries on 49,500 columns: a dense head where its columns hold 27 M more than the others and 7 to every column
    (52 M of them by a steep law), else the fused step (40 M).  Either way one step is the same to rounding."""
    n, k = 40_000, 1650
    A, norms = d.Csr.synth(n, 30 * k, k_fixed=k, zipf_s=zipf, seed=1)
    A.normalize_rows(norms)
    A.compact_columns(1)

    def run():
        nmf = d.MuNmf(A, d.MuNmfParams(rank=64, max_iters=1, eps=EPS, seed=3, log_every=1))
        nmf.initialize()
        nd = A.head_info()[0]
        nmf.step(1)
        W = nmf.loadWToHostSync()
        nmf.close()
        return nd, W

    nd, W = run()
    assert (nd > 0) == head
    A.split_dense_head(0.0)
    tune("dense_fill", 0)
    nd, W0 = run()
    assert nd == 0
    assert np.linalg.norm(W - W0) <= 1e-5 * np.linalg.norm(W0)
    A.close()
