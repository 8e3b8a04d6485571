"""What a context takes from the device stays within dnpeff_plan_estimate."""

import ctypes as C

import pytest

import npeff_ref_amd as d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [8, 50, 100, 128, 200, 256, 300])
@pytest.mark.parametrize("n,m_full,k", [(500, 2_000_000, 8192), (1500, 500_000, 4096)])
def test_estimate_is_an_upper_bound(n, m_full, k, r):
    A, norms = d.Csr.synth(n, m_full, k_fixed=k, zipf_s=1.1, seed=r)
    A.normalize_rows(norms)
    A.compact_columns(1)
    A.sq_norm()
    free, total = d.device_memory()
    nmf = d.MuNmf(A, d.MuNmfParams(rank=r, max_iters=1, seed=3, log_every=0))
    nmf.initialize()
    nmf.step(1)
    nmf.computeUncachedLoss()
    nmf.device_factors()
    taken = free - d.device_memory()[0]
    n_dense, z_sparse = A.head_info()
    e = d.plan_estimate(n, A.n_cols, z_sparse, n_dense, r, False, total_bytes=total)
    # the row-major copy was there before (and stays, whole, beside a head); the reserve is for what allocations round up
    bound = sum(e.values()) - e["reserve"] - 8.0 * z_sparse + (8.0 * z_sparse if n_dense else 0.0)
    assert taken <= bound + 64 * 2**20
    nmf.close()
    A.close()
