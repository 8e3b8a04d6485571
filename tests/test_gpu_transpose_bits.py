"""The transposed copy through bits (csrc/loader.hip), range by range and row by row: rows around the words, ragged and
empty ones, against a stable sort by column; a repeated pair is refused on every way."""

import numpy as np
import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,k", [(1, 5, 5), (31, 50, 20), (32, 40, 40), (33, 7, 7), (65, 9000, 3000), (2048, 300, 30),
                                   (2049, 100, 20), (3, 70_000, 60_000)])
def test_transpose(n, m, k):
    rng = np.random.default_rng(n + m)
    lens = rng.integers(0, k + 1, n)
    lens[0] = k
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = np.concatenate([rng.permutation(m)[:c] for c in lens]).astype(np.int32)
    vals = rng.standard_normal(len(cols)).astype(np.float32)
    rows = np.repeat(np.arange(n), lens)
    order = np.argsort(cols, kind="stable")
    A = d.Csr.from_host(rowptr, cols, vals, m)
    cp, ri, tv = A.download_transpose()
    assert np.array_equal(cp, np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=m))]))
    assert np.array_equal(ri, rows[order]) and np.array_equal(tv, vals[order])
    A.close()
    cols[lens[0] - 1] = cols[0]
    if lens[0] > 1:
        A = d.Csr.from_host(rowptr, cols, vals, m)
        with pytest.raises(d.DnpeffError, match="1 column.*duplicate"):
            A.build_transpose()
        A.close()


@pytest.mark.parametrize("n,m,k", [(2049, 1 << 18, 1100), (2050, 300_001, 1500), (600, 2_000_003, 8100), (40, 20_000_000, 110_000)])
@pytest.mark.parametrize("what", ["ascending", "spoilt", "crowded"])
def test_transpose_by_ranges(n, m, k, what):
    """Rows in ascending order, with parts of a range longer than a wave, gaps of many ranges and empty rows; spoilt: a row
    has two columns the other way round; crowded: a range with more entries than its counters hold (2049 rows and more)."""
    rng = np.random.default_rng(n + m)
    cols = [np.unique(rng.integers(0, m, k)) for _ in range(n)]
    if what == "crowded":
        cols = [np.union1d(c, 4096 + rng.choice(2048, size=40, replace=False)) for c in cols]
    cols[1], cols[3], cols[n // 2] = cols[1][:0], cols[3][-5:], np.arange(5000, 5700)
    cols[n - 1] = np.unique(rng.integers(0, m, 3 * k))
    lens = np.array([len(c) for c in cols])
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = np.concatenate(cols).astype(np.int32)
    if what == "spoilt":
        at = rowptr[n - 2] + 1
        cols[at], cols[at - 1] = cols[at - 1], cols[at]
    vals = rng.standard_normal(len(cols)).astype(np.float32)
    rows = np.repeat(np.arange(n), lens)
    order = np.argsort(cols, kind="stable")
    A = d.Csr.from_host(rowptr, cols, vals, m)
    cp, ri, tv = A.download_transpose()
    assert np.array_equal(cp, np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=m))]))
    assert np.array_equal(ri, rows[order]) and np.array_equal(tv, vals[order])
    A.close()
    cols[rowptr[n - 2] + 1] = cols[rowptr[n - 2]]
    A = d.Csr.from_host(rowptr, cols, vals, m)
    with pytest.raises(d.DnpeffError, match="1 column.*duplicate"):
        A.build_transpose()
    A.close()
