"""Top-k through the sampled threshold (csrc/topk.hip): rows long enough to be sampled, values that the
sample misjudges, crowded buckets, and lengths around its chunks, against the full sort."""

import numpy as np
import pytest

import npeff_ref_amd as d
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _values(kind, n, count, rng):
    if kind == "lognormal":
        return np.exp(rng.normal(-8, 2, (n, count))).astype(np.float32)
    if kind == "uniform":
        return rng.random((n, count), dtype=np.float32)
    if kind == "normal":  # both signs
        return rng.standard_normal((n, count), dtype=np.float32)
    if kind == "equal":
        return np.full((n, count), 0.25, dtype=np.float32)
    if kind == "few":  # eight different values
        return rng.integers(0, 8, (n, count)).astype(np.float32)
    if kind == "hidden":  # everything large lies where no sample is taken
        x = rng.random((n, count), dtype=np.float32)
        x[:, 100:1100] += 100.0
        return x
    x = np.sort(rng.random((n, count), dtype=np.float32), axis=1)  # "sorted"
    x[:, -1] = 1e30
    return x


@pytest.mark.parametrize("kind", ["lognormal", "uniform", "normal", "equal", "few", "hidden", "sorted"])
@pytest.mark.parametrize("n,count,k", [(1, 600_000, 900), (3, 524_289, 4000), (2, 524_287, 64), (1, 65, 65), (5, 1, 1)])
def test_topk_matches_the_full_sort(kind, n, count, k):
    x = _values(kind, n, count, np.random.default_rng(count + k))
    v, i, nrm = d.topk_rows(d.DeviceArray.from_numpy(x), k)
    wv, wi, wn = orc.topk_rows(x, k)
    assert np.array_equal(v, wv) and np.array_equal(i, wi)
    assert np.allclose(nrm, wn, rtol=2e-7)


@pytest.mark.parametrize("count,k,outliers", [(600_001, 500, 60), (700_000, 40_000, 300), (1_200_000, 33_000, 5000),
                                              (1_200_000, 32_767, 0)])
def test_entries_above_all_of_the_sample(count, k, outliers):
    """Values far above the largest one sampled, where no chunk of either stride looks (64 of 2048 or of 4096
    entries): they share the first bucket, or are too many for it."""
    rng = np.random.default_rng(count + k)
    x = rng.lognormal(-8, 2, count).astype(np.float32)
    where = np.flatnonzero(np.arange(count) % 2048 >= 64)
    x[rng.choice(where, outliers, replace=False)] = rng.lognormal(20, 1, outliers).astype(np.float32)
    vals, idx, norms = d.topk_rows(d.DeviceArray.from_numpy(x[None, :]), k)
    order = np.lexsort((np.arange(count), -x))[:k]
    assert np.array_equal(idx[0], order) and np.array_equal(vals[0], x[order])
    np.testing.assert_allclose(norms[0], np.sqrt((x.astype(np.float64) ** 2).sum()), rtol=1e-7)


@pytest.mark.parametrize("count,k,kind", [(2_000_000, 40_000, "close"), (2_000_001, 700, "close"), (1_500_000, 33_000, "edge"),
                                          (1_500_000, 33_000, "gap"), (700_001, 900, "gap")])
def test_threshold_and_largest_entry_close_together(count, k, kind):
    """Candidates within one bin of the sample's histogram, on either side of a bin's end, or (gap) a run of larger
    entries between two chunks of the sample, twice its length with the larger stride."""
    rng = np.random.default_rng(count + k)
    x = (1.0 if kind == "close" else 0.9965) + 1e-3 * rng.standard_normal(count)
    if kind == "gap":
        stride = 4096 if k >= 32_768 else 2048
        x[3 * stride + 64:4 * stride] += 0.01 + 1e-3 * rng.random(stride - 64)
    x = x.astype(np.float32)
    vals, idx, norms = d.topk_rows(d.DeviceArray.from_numpy(x[None, :]), k)
    order = np.lexsort((np.arange(count), -x))[:k]
    assert np.array_equal(idx[0], order) and np.array_equal(vals[0], x[order])
    np.testing.assert_allclose(norms[0], np.sqrt((x.astype(np.float64) ** 2).sum()), rtol=1e-7)


@pytest.mark.parametrize("kind,n,count,k", [("lognormal", 2, 600_000, 65_536), ("lognormal", 1, 700_000, 262_100),
                                            ("lognormal", 10, 600_001, 38_482), ("lognormal", 1, 700_000, 524_280),
                                            ("lognormal", 1, 700_000, 524_288), ("lognormal", 3, 600_001, 300_000), ("few", 2, 524_288, 5000),
                                            ("hidden", 1, 600_000, 900), ("uniform", 1, 9, 1)])
def test_results_for_the_host_equal_those_on_the_device(kind, n, count, k):
    """One pinned buffer holds them (the second case just), or two (the fourth just), or not, or the sample's threshold does not serve."""
    x = d.DeviceArray.from_numpy(_values(kind, n, count, np.random.default_rng(k)))
    on_dev = [d.DeviceArray((n, k)), d.DeviceArray((n, k), np.int32), d.DeviceArray((n,))]
    d.binding._check(d.lib.dnpeff_topk_rows(n, count, k, x.ptr, *(a.ptr for a in on_dev)))
    for got, want in zip(d.topk_rows(x, k), on_dev):
        assert np.array_equal(got, want.numpy())
    vals, idx = np.empty((n, k), np.float32), np.empty((n, k), np.int32)
    d.binding._check(d.lib.dnpeff_topk_rows_host(n, count, k, x.ptr, vals.ctypes.data, idx.ctypes.data, None))
    assert np.array_equal(vals, on_dev[0].numpy()) and np.array_equal(idx, on_dev[1].numpy())
    for bad in (0, -1, count + 1):
        with pytest.raises(d.DnpeffError):
            d.topk_rows(x, bad)
