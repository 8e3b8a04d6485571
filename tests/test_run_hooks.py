"""The logged windows of MuNmf.run and Learner.Run go through a step and a loss that replace the classes' own."""

import npeff_ref_amd as d
from npeff_ref_amd import binding as b


class _NoLibrary:
    def __getattr__(self, name):
        raise AssertionError(f"{name} was called")


def _quiet(_line):
    pass


def _bare(cls, params, monkeypatch):
    """An object without a context, and no library to call."""
    monkeypatch.setattr(b, "lib", _NoLibrary())
    monkeypatch.setattr(b, "sync", lambda: None)
    obj = cls.__new__(cls)
    obj._h, obj._initialized, obj.params = None, True, params
    return obj


class _Nmf(d.MuNmf):
    def step(self, n_steps=1):
        self.steps = getattr(self, "steps", []) + [n_steps]

    def computeUncachedLoss(self):
        return 7.0 - len(self.steps)


class _Learner(d.Learner):
    step = _Nmf.step

    def losses(self):
        return 7.0 - len(self.steps), 8.0


def test_subclass_of_the_factorisation(monkeypatch):
    nmf = _bare(_Nmf, d.MuNmfParams(rank=2, max_iters=25, log_every=10), monkeypatch)
    history = nmf.run(log=_quiet)
    assert nmf.steps == [10, 10, 5]
    assert [(step, loss) for step, loss, _ in history] == [(10, 6.0), (20, 5.0)]
    assert all(ms >= 0.0 for _, _, ms in history)


def test_subclass_of_the_learner(monkeypatch):
    learner = _bare(_Learner, d.LearnerParams(max_iters=20, log_every_n_steps=10), monkeypatch)
    assert [h[:3] for h in learner.Run(log=_quiet)] == [(10, 6.0, 8.0), (20, 5.0, 8.0)]
    assert learner.steps == [10, 10]


def test_a_method_of_the_object_and_one_put_into_the_class(monkeypatch):
    nmf = _bare(d.MuNmf, d.MuNmfParams(rank=2, max_iters=10, log_every=10), monkeypatch)
    steps = []
    nmf.step, nmf.computeUncachedLoss = steps.append, lambda: 1.5
    assert [h[:2] for h in nmf.run(log=_quiet)] == [(10, 1.5)]
    del nmf.step
    monkeypatch.setattr(d.MuNmf, "step", lambda self, n_steps=1: steps.append(-n_steps))
    nmf.run(log=_quiet)
    assert steps == [10, -10]
