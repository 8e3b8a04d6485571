"""The updates' quotients at the ends of fp32: denominators that are subnormal, infinite or beyond the
reciprocal's range, and quotients that overflow, give what the division gives."""

import numpy as np
import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu

# a, w, h: scales of the matrix's values and of the factors (None: W^T W H comes to 2e38)
ENDS = {
    "subnormal eps, products of the factors below it": dict(eps=1e-40, a=1.0, w=1e-37, h=1.0),
    "quotients beyond the largest number": dict(eps=1e-30, a=1e22, w=1e-12, h=1e-20),
    "denominators beyond 2^126": dict(eps=1e-8, a=1.0, w=None, h=1.0),
    "infinite denominators": dict(eps=1e-8, a=1.0, w=1e20, h=1.0),
}


def _expected(x, num, den, eps):
    """x * (num / (den + eps)) with the roundings of fp32, from sums in fp64."""
    with np.errstate(all="ignore"):
        q = num.astype(np.float32) / (den.astype(np.float32) + np.float32(eps))
        return x * q


def _same(got, want):
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=1e-43)


@pytest.mark.parametrize("case", ENDS)
@pytest.mark.parametrize("r", [8, 13, 50, 64, 72, 100, 127, 200])
def test_updates_of_a_context(r, case):
    if case == "infinite denominators" and r > 64:
        pytest.skip("split operands: an infinite Gram element makes the denominators NaN, as at rank 128")
    if case.startswith("subnormal") and r > 128:
        pytest.skip("an eps below 1e-30 keeps such a rank as it is")
    n, m = 256, 400
    e = dict(ENDS[case])
    if e["w"] is None:
        e["w"] = (2e38 / (n * r)) ** 0.5
    rng = np.random.default_rng(r)
    mask = rng.random((n, m)) < 0.1
    mask[0] = True
    dense = np.where(mask, rng.random((n, m)).astype(np.float32) + np.float32(0.5), 0).astype(np.float32) * np.float32(e["a"])
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    A = d.Csr.from_host(rp, np.nonzero(mask)[1].astype(np.int32), dense[mask], m)
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, eps=e["eps"], seed=1, log_every=0))
    W = (rng.random((n, r)).astype(np.float32) + np.float32(0.5)) * np.float32(e["w"])
    H = (rng.random((r, m)).astype(np.float32) + np.float32(0.5)) * np.float32(e["h"])
    A64, W64, H64 = dense.astype(np.float64), W.astype(np.float64), H.astype(np.float64)
    with np.errstate(over="ignore"):
        G = (W64.T @ W64).astype(np.float32).astype(np.float64)
        K = (H64 @ H64.T).astype(np.float32).astype(np.float64)
        nmf.set_factors(W, H)
        nmf.update_H()
        _same(nmf.loadHToHostSync(), _expected(H, W64.T @ A64, G @ H64, e["eps"]))
        if r > 64 and e["w"] < 1e-30:  # (W in X G: the low parts of split operands are no bf16 numbers there)
            W = W / np.float32(e["w"])
            W64 = W.astype(np.float64)
        nmf.set_factors(W, H)
        nmf.update_W()
        _same(nmf.loadWToHostSync(), _expected(W, A64 @ H64.T, W64 @ K, e["eps"]))
    nmf.close()
    A.close()


@pytest.mark.parametrize("r,rows", [(128, 200), (256, 300), (384, 256)])
def test_updates_by_themselves(r, rows):
    """The kernels of ranks 128 and above on rows of every kind side by side."""
    rng = np.random.default_rng(r)
    X = rng.random((rows, r)).astype(np.float32) + np.float32(0.5)
    G = np.eye(r, dtype=np.float32)
    num = rng.random((rows, r)).astype(np.float32) + np.float32(0.5)
    X[0::5] *= np.float32(1e-40)  # subnormal den
    num[0::10] *= np.float32(1e-39)
    X[1::5] *= np.float32(1e-20)  # quotient overflows
    num[1::5] *= np.float32(1e22)
    X[2::5] *= np.float32(1.2e38)  # den above 2^126
    num[2::5] *= np.float32(1e38)
    X[3::5] = 0  # den = 0
    num[3::10] = 0
    want = _expected(X, num, X.astype(np.float64), 0.0)
    dX, dG, dn, dO, dK = [d.DeviceArray.from_numpy(a) for a in (X, G, num, np.zeros_like(X), G)]
    if r == 128:
        d.op_xg_mu_gram(dX, dG, dn, 0.0, dO, dK)
    else:
        d.op_xg_mu(dX, dG, dn, 0.0, dO)
    d.sync()
    got = dO.numpy()
    keep = np.ones(rows, bool)
    keep[0::5] = False  # (X itself is subnormal there: the matrix cores may take it as zero)
    _same(got[keep], want[keep])
