"""CPU tests of what the launch autotuner times and under which key it keeps a plan (a stand-in for
the stepper; the timing itself needs the GPU)."""

import json
from dataclasses import replace

import numpy as np
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


def test_a_scene_with_h_points_takes_no_plan_of_one_without(stepper, monkeypatch):
    monkeypatch.setattr(stepper, "cost", staticmethod(lambda f, c: 1.0 if f == "fused" else 2.0))
    assert autotune.tune(_tabs(), steps=8, warmup=2)["form"] == "fused"
    monkeypatch.setattr(stepper, "default", ("sweeps", 4))     # the library's choice with H points
    assert autotune.tune(_tabs(magnetic_dipole=True), steps=8, warmup=2)["form"] == "sweeps"


def test_key_holds_the_coefficients_kind():
    sc = scenes.mini_scene(shape=(48, 40, 40), num_steps=20, lorentz_on=False)
    rng = np.random.default_rng(7)              # more distinct cells than classes
    e = [2.0 + rng.uniform(0, 2, size=sc.shape) for _ in range(3)]
    dense = tables.build(replace(sc, eps_ex=e[0], eps_ey=e[1], eps_ez=e[2]))
    assert dense.material_classes() is None
    assert autotune.shape_key(dense) != autotune.shape_key(tables.build(sc))


def test_stored_plans_of_other_kernels_are_not_used(stepper, monkeypatch, tmp_path):
    tabs = _tabs()
    pml = tuple((a.pml_lo, a.pml_hi) for a in tabs.axes)
    old = {"form": "sweeps", "chunk": 64, "ms_per_step": 1.0, "timings": {}}
    f = tmp_path / "plans.json"
    f.write_text(json.dumps({f"{tuple(tabs.shape)}|r|{pml}": old}))
    monkeypatch.setenv("OEM_TUNE_CACHE", str(f))
    monkeypatch.setattr(stepper, "cost", staticmethod(lambda f, c: 1.0 if f == "fused" else 2.0))
    plan = autotune.tune(tabs, steps=8, warmup=2)
    assert plan["form"] == "fused"
    assert json.loads(f.read_text())[autotune.shape_key(tabs)] == plan      # stored beside the old one
    monkeypatch.setattr(autotune, "_cache", {})
    assert autotune.tune(tabs, steps=8, warmup=2) == plan
