"""GPU tests of launches of more work-groups than the chip holds at once, where point lists, snapshots,
objective points and gradient entries go with the work-groups only while few of those have any
(chunks of one plane make such launches of small scenes), and of the fused transposes on a grid whose
adjoint fields leave the caches.  The separate launches do the same arithmetic on the same values, so
everything agrees bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import adjoint, scenes, tables
from openem_amd.model import FieldMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
N = 21
SHAPE = (400, 24, 44)                  # 3 tiles a plane: 1200 work-groups of one plane, 1024 resident


# the work-groups that have points: 3 (a plane of x), all (a plane of z), at most 96, 170; the bound is an
# eighth of them, 150
@pytest.mark.parametrize("mons,own_launch", [
    ([("plane", 0, 100)], False),
    ([("plane", 2, 20)], True),
    ([("box", (10, 3, 3), (32, 20, 30))], False),
    ([("box", (10, 3, 3), (170, 1, 1))], True),
    ([("plane", 0, 100), ("plane", 2, 20)], True),
])
@pytest.mark.parametrize("tfsf", [False, True])
def test_lists_of_a_large_launch(gpu_lib, monkeypatch, mons, own_launch, tfsf):
    monkeypatch.setenv("OEM_CHUNK", "1")
    if tfsf:                           # faces in nearly every work-group: the lists are launched
        sc = scenes.tfsf_box_scene(shape=SHAPE, num_steps=N, scatterer=True)
    else:
        sc = scenes.mini_scene(shape=SHAPE, num_steps=N, pml_xy=True, lorentz_on=False)
    f = np.array([2.5e14, 3e14])
    sc = replace(sc, flux_monitors=[FluxMonitor(f"p{q}", m[1], m[2], +1, f)
                                    for q, m in enumerate(mons) if m[0] == "plane"],
                 field_monitors=[FieldMonitor(f"b{q}", f, m[1], m[2])
                                 for q, m in enumerate(mons) if m[0] == "box"])
    tabs = tables.build(sc)
    e0 = np.random.default_rng(2).standard_normal(SHAPE).astype(np.float32)

    def run():
        st = Stepper(tabs, dft_batch=8, form="sweeps")
        try:
            st.write_field(0, e0)
            calls = st.profile_run(5)["dft_snap"][1]
            st.run(N - 5)
            return calls, ([st.read_field(c) for c in range(6)]
                           + [st.read_monitor(i) for i in range(len(tabs.monitors))])
        finally:
            st.close()

    calls, got = run()
    monkeypatch.setenv("OEM_TAIL", "0")
    all_calls, want = run()
    assert all_calls > 0 and (calls > 0) == (own_launch or tfsf)
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def _gradients(monkeypatch, sc, name, n_design, **kw):
    t = tables.build(sc)
    m = t.monitors[[m.name for m in t.monitors].index(name)]
    rng = np.random.default_rng(4)
    K = rng.standard_normal((4, m.n1, m.n2)) + 1j * rng.standard_normal((4, m.n1, m.n2))
    cell = rng.choice(int(np.prod(sc.shape)), n_design, replace=False)
    comp = rng.integers(3, size=n_design)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("OEM_ADJ_FUSE", fuse)
        out.append(adjoint.overlap_power_gradient(sc, name, K, comp, cell, **kw))
    a, b = out
    assert np.isfinite(b.grad).all() and np.abs(b.grad).max() > 0
    assert a.J == b.J and np.array_equal(a.grad, b.grad)


# objective on a plane of x (few work-groups) or of z (all), few or many design entries, so that both,
# the objective alone or neither go with the 1200 work-groups (512 resident, 150 the bound)
@pytest.mark.parametrize("axis", [0, 2])
@pytest.mark.parametrize("n_design", [40, 2000])
def test_adjoint_tail_of_a_large_launch(gpu_lib, monkeypatch, axis, n_design):
    monkeypatch.setenv("OEM_ADJ_CHUNK", "1")
    sc = scenes.mini_scene(shape=SHAPE, num_steps=60, nf=2, field_box=False, lorentz_on=False,
                           pml_xy=True)
    sc = replace(sc, flux_monitors=[FluxMonitor("T", axis, SHAPE[axis] // 2, +1,
                                                sc.flux_monitors[0].freqs)])
    _gradients(monkeypatch, sc, "T", n_design)


def test_fused_transposes_past_the_caches(gpu_lib, monkeypatch):
    """4.5 M cells: 217 MB of adjoint fields and psi in both sets, stored past the caches."""
    sc = scenes.mini_scene(shape=(310, 130, 112), num_steps=300, nf=2, field_box=False,
                           lorentz_on=False, pml_xy=True)
    assert 48 * np.prod(sc.shape) > 200 << 20
    _gradients(monkeypatch, sc, "T", 60)


# 303,000 points go with the sweeps' work-groups, 343,000 (more than 320,000 items) keep their launch,
# and so do many of a design (3 x 110,592) in the fused transposes
@pytest.mark.parametrize("side,own_launch", [(67, False), (70, True)])
def test_most_points_of_a_table(gpu_lib, monkeypatch, side, own_launch):
    monkeypatch.delenv("OEM_CHUNK", raising=False)
    sc = scenes.mini_scene(shape=(80, 78, 76), num_steps=N, pml_xy=True, lorentz_on=False,
                           field_box=False)
    f = np.array([2.5e14])
    sc = replace(sc, flux_monitors=[], field_monitors=[FieldMonitor("b", f, (2, 2, 2), (side,) * 3)])
    tabs = tables.build(sc)
    out = []
    for tail in ("1", "0"):
        monkeypatch.setenv("OEM_TAIL", tail)
        st = Stepper(tabs, dft_batch=8, form="sweeps")
        try:
            calls = st.profile_run(5)["dft_snap"][1]
            st.run(N - 5)
            out.append([st.read_field(c) for c in range(6)] + [st.read_monitor(0)])
        finally:
            st.close()
        assert (calls > 0) == (own_launch or tail == "0")
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_large_design_of_the_fused_transposes(gpu_lib, monkeypatch):
    sc = scenes.mini_scene(shape=(60, 56, 60), num_steps=100, nf=2, field_box=False, lorentz_on=False)
    t = tables.build(sc)
    m = t.monitors[[m.name for m in t.monitors].index("T")]
    rng = np.random.default_rng(4)
    K = rng.standard_normal((4, m.n1, m.n2)) + 1j * rng.standard_normal((4, m.n1, m.n2))
    i, j, k = np.meshgrid(*[np.arange(4, 52)] * 3, indexing="ij")
    cell = np.tile(((i * 56 + j) * 60 + k).ravel(), 3)
    comp = np.repeat(np.arange(3), i.size)
    assert cell.size > 320000
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("OEM_ADJ_FUSE", fuse)
        out.append(adjoint.overlap_power_gradient(sc, "T", K, comp, cell))
    assert np.abs(out[1].grad).max() > 0 and np.array_equal(out[0].grad, out[1].grad)
