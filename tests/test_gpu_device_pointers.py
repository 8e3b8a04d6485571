"""Factors read and written through the pointers of MuNmf.device_factors: between any two calls the next one
works on what is there, whatever the context has kept of the factor before."""

import ctypes as C

import numpy as np
import pytest

import npeff_ref_amd as d
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
EPS = 1e-8


class Run:
    def __init__(self, n, m, r):
        rng = np.random.default_rng(n + m + r)
        mask = rng.random((n, m)) < 0.06
        mask[:, :2] = True
        self.n, self.m, self.r, self.rng = n, m, r, rng
        self.rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
        self.ci = np.nonzero(mask)[1].astype(np.int32)
        self.va = rng.random(len(self.ci)).astype(np.float32)
        self.A = d.Csr.from_host(self.rp, self.ci, self.va, m)
        self.nmf = d.MuNmf(self.A, d.MuNmfParams(rank=r, max_iters=1, eps=EPS, seed=3, log_every=0))
        self.nmf.initialize()
        self.nmf.step(2)
        self.nmf.computeUncachedLoss()

    def close(self):
        self.nmf.close()
        self.A.close()

    def factors(self):
        return self.nmf.loadWToHostSync(), self.nmf.loadHToHostSync()

    def new_W(self):
        return self.rng.random((self.n, self.r)).astype(np.float32) + np.float32(0.1)

    def new_H(self):
        return self.rng.random((self.r, self.m)).astype(np.float32) + np.float32(0.1)

    def write(self, ptr, a):
        a = np.ascontiguousarray(a)
        d.binding._check(d.lib.dnpeff_dev_upload(C.c_void_p(ptr), d.binding._ptr(a), a.nbytes))

    def loss_is_that_of(self, W, H):
        want, _ = orc.loss_f64(self.rp, self.ci, self.va, self.m, W, H)
        assert abs(self.nmf.computeUncachedLoss() - want) <= 1e-5 * want

    def step_is_that_of(self, W, H, W_between=None, H_between=None):
        """After an iteration from (W, H), a factor written between its two updates as given."""
        W64, _, _ = orc.nmf_f64(self.rp, self.ci, self.va, self.m, W, H, np.float32(EPS), 1, 1)
        if W_between is not None:
            W64 = W_between
        dense = np.zeros((self.n, self.m))
        dense[np.repeat(np.arange(self.n), np.diff(self.rp)), self.ci] = self.va
        H_in = (H if H_between is None else H_between).astype(np.float64)
        W64 = W64.astype(np.float64)
        H64 = H_in * (W64.T @ dense) / ((W64.T @ W64) @ H_in + EPS)
        for got, want in zip(self.factors(), (W64, H64)):
            assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


RANKS = [5, 16, 50, 100, 128, 129, 200, 256]


@pytest.mark.parametrize("r", RANKS)
@pytest.mark.parametrize("n,m", [(300, 700)])
def test_written_between_calls(n, m, r):
    t = Run(n, m, r)
    w, h = t.nmf.device_factors()
    # several writes through pointers asked for once, a loss after each
    for _ in range(2):
        W, H = t.new_W(), t.nmf.loadHToHostSync()
        t.write(w, W)
        t.loss_is_that_of(W, H)
        H = t.new_H()
        t.write(h, H.T)
        t.loss_is_that_of(W, H)
    # and without a loss in between, straight into an iteration
    H = t.new_H()
    t.write(h, H.T)
    t.nmf.step(1)
    t.step_is_that_of(W, H)
    # W, and W and H, between the two updates of an iteration
    for both in (False, True):
        W, H = t.factors()
        t.nmf.update_W()
        w, h = t.nmf.device_factors()
        W1, H1 = t.new_W(), t.new_H() if both else None
        t.write(w, W1)
        if both:
            t.write(h, H1.T)
        t.nmf.update_H()
        t.step_is_that_of(W, H, W_between=W1, H_between=H1)
        t.loss_is_that_of(*t.factors())
    t.close()


@pytest.mark.parametrize("r", [16, 100, 129, 200, 256])
def test_pointers_follow_what_changes_the_factors_in_place(r):
    n, m = 60, 400
    t = Run(n, m, r)
    w, h = t.nmf.device_factors()

    def show(W, H):
        assert np.array_equal(d.gather_rows(w, r, np.arange(n)), W)
        assert np.array_equal(d.gather_rows(h, r, np.arange(m)), H.T)

    W, H = t.new_W(), t.new_H()
    t.nmf.set_factors(W, None)
    t.nmf.set_factors(None, H)
    show(W, H)
    t.loss_is_that_of(W, H)
    # one written through its pointer, the other set from the host
    W, H = t.new_W(), t.new_H()
    t.write(h, H.T)
    t.nmf.set_factors(W, None)
    show(W, H)
    t.loss_is_that_of(W, H)
    t.write(w, W)
    t.nmf.sparsify_W(3.0)
    W = t.nmf.loadWToHostSync()
    show(W, H)
    t.loss_is_that_of(W, H)
    t.nmf.initialize()
    show(*t.factors())
    # W's pointer alone: H keeps what is at hand of it
    t.nmf.step(1)
    W, H = t.factors()
    ptr = C.c_void_p()
    d.binding._check(d.lib.dnpeff_nmf_device_factors(t.nmf._h, C.byref(ptr), None))
    W = t.new_W()
    t.write(ptr.value, W)
    t.loss_is_that_of(W, H)
    t.close()
