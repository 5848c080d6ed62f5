"""CPU tests of what the launch autotuner times and under which key it keeps a plan (a stand-in for
the stepper; the timing itself needs the GPU)."""

import pytest

from openem_amd import autotune, scenes, solver, tables


class _Stepper:
    """Steps nothing; its library chooses ``default`` and a plan takes what ``cost`` says."""

    default = ("fused", 2)
    cost = staticmethod(lambda form, chunk: 1.0)

    def __init__(self, tabs, device=0, dft_batch=16, form=None, chunk=0):
        self.launch = dict(zip(("form", "chunk"), (form, chunk) if form else self.default))

    def run(self, n):
        pass

    def timed_run(self, n):
        return n * self.cost(self.launch["form"], self.launch["chunk"])

    def close(self):
        pass


@pytest.fixture
def stepper(monkeypatch):
    monkeypatch.setattr(solver, "Stepper", _Stepper)
    monkeypatch.setattr(autotune, "_cache", {})
    monkeypatch.delenv("OEM_TUNE_CACHE", raising=False)
    return _Stepper


def _tabs(**kw):
    return tables.build(scenes.mini_scene(**{**dict(shape=(14, 12, 40), num_steps=40), **kw}))


@pytest.mark.parametrize("default", [("fused", 2), ("fused", 3), ("fused", 5), ("fused", 8),
                                     ("sweeps", 4), ("sweeps", 1)])
@pytest.mark.parametrize("magnetic", [False, True])
def test_the_librarys_own_plan_is_timed(stepper, monkeypatch, default, magnetic):
    monkeypatch.setattr(stepper, "default", default)
    monkeypatch.setattr(stepper, "cost", staticmethod(lambda f, c: 1.0 if (f, c) == default else 2.0))
    plan = autotune.tune(_tabs(magnetic_dipole=magnetic), steps=8, warmup=2)
    assert f"{default[0]}/{default[1]}" in plan["timings"]
    assert (plan["form"], plan["chunk"]) == default
    if magnetic:
        assert all(k.startswith(default[0]) for k in plan["timings"])


def test_small_marches_are_timed_with_few_planes():
    small = autotune.candidates(_tabs(), "fused")
    assert {c for f, c in small if f == "fused"} >= {2, 4, 6, 8}
    assert len(small) == len(set(small))
