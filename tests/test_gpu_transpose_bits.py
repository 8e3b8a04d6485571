"""The transposed copy through bits (csrc/loader.hip) and row by row: rows around the words, ragged and empty
ones, against a stable sort by column; a repeated pair is refused on either way."""

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
