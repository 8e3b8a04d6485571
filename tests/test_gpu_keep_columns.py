"""Dropping columns through bits and ranks (csrc/columns.hip): sizes around its words, its tiles of 4096 entries
and its ranges of marks, counters and marks, rows that are empty, end on a tile, or lose everything."""

import numpy as np
import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu


def _want(rowptr, cols, vals, kept):
    new = np.full(int(max(kept.max(initial=-1), cols.max(initial=-1))) + 1, -1, dtype=np.int64)
    new[kept] = np.arange(len(kept))
    keep = new[cols] >= 0
    before = np.concatenate([[0], np.cumsum(keep)])
    return before[rowptr], new[cols][keep], vals[keep]


def _check(A, rowptr, cols, vals, kept):
    rp, ci, va = A.download()
    wr, wc, wv = _want(rowptr, cols, vals, kept)
    assert A.n_cols == len(kept) and np.array_equal(A.kept_indices(), kept)
    assert np.array_equal(rp, wr) and np.array_equal(ci, wc) and np.array_equal(va, wv)


# (rows, columns, entries of the longest row): 600,000 columns need two ranges for two marks, the last
# case has too few entries for marks
@pytest.mark.parametrize("n,m,k", [(1, 33, 33), (3, 64, 40), (9, 31, 20), (40, 4096, 2048), (4, 100, 1024 // 16),
                                   (257, 5000, 700), (600, 600_000, 600), (5, 3_000_000, 100)])
@pytest.mark.parametrize("how", [1, 2, 3, "list", "none", "unordered"])
def test_keep_columns(n, m, k, how):
    rng = np.random.default_rng(n * 7 + k)
    lens = rng.integers(0, k + 1, n)
    lens[0] = k
    lens[n // 2 :: 5] = 0
    if n * k == 40 * 2048:
        lens[:] = 2048  # rows that end where a tile does
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = np.concatenate([rng.permutation(m)[:c] if m < 10_000 else rng.choice(m // 3, c, replace=False)
                           for c in lens] or [[]]).astype(np.int32)
    vals = rng.standard_normal(len(cols)).astype(np.float32)
    A = d.Csr.from_host(rowptr, cols, vals, m)
    if how in (1, 2, 3):
        kept = np.flatnonzero(np.bincount(cols, minlength=m) >= how)
        A.compact_columns(how)
    else:
        kept = np.flatnonzero(rng.random(m) < 0.6) if how != "none" else np.empty(0, dtype=np.int64)
        if how == "unordered":
            kept = rng.permutation(kept)
        A.retain_columns(kept.astype(np.int32))
    _check(A, rowptr, cols, vals, kept)
    A.close()
