"""GPU tests of flat and thin scenes (few cells along z or y): the rule that keeps them off the tiled
kernels whose lanes they would leave idle, and the values of both forms on them."""

import numpy as np
import pytest
import torch

from openem_amd import _lib, adjoint, cpml, grid, model, scenes, tables, waveform
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
D = 20e-9


def _scene(shape, steps=40):
    """Boxes and an Ez dipole, PML on every axis of 40 cells and more, periodic on the others."""
    bnd = ["PML" if n >= 40 else "Periodic" for n in shape]
    axes = [grid.Axis(np.arange(n + 1) * D, b, b) for n, b in zip(shape, bnd)]
    dt = cpml.courant_dt((D, D, D))
    rng = np.random.default_rng(1)
    eps = np.ones(shape)
    for _ in range(6):
        lo = [int(rng.integers(0, max(1, n - 1))) for n in shape]
        eps[tuple(slice(a, a + max(1, n // 3)) for a, n in zip(lo, shape))] = rng.uniform(1.5, 10)
    wf = waveform.sample(waveform.GaussianPulse(2.5e14, 1e14), dt, steps)
    sides = [(a, s) for a in range(3) if bnd[a] == "PML" for s in ("lo", "hi")]
    fl = [model.FluxMonitor(f"f{a}", a, shape[a] - 14, +1, np.array([2.5e14]))
          for a in range(3) if shape[a] >= 40]
    return model.Scene(grid=grid.Grid(*axes), dt=dt, num_time_steps=steps, eps_ex=eps, eps_ey=eps,
                       eps_ez=eps, pml=scenes.pml_faces(dt, (D, D, D), sides, 8), flux_monitors=fl,
                       dipoles=[model.PointDipole(2, np.array([tuple(n // 2 for n in shape)]),
                                                  np.ones(1), wf)])


# the share of the march's lanes in use: 0.03, 0.24, 0.25, 0.37, 0.14, 0.51 with over half a million of
# them; under that, and above three fifths
@pytest.mark.parametrize("shape,form", [
    ((300, 300, 1), "sweeps"), ((150, 150, 8), "sweeps"), ((500, 500, 8), "sweeps"),
    ((400, 400, 12), "sweeps"), ((1000, 1, 1000), "sweeps"),
    ((200, 200, 33), "sweeps"),
    ((64, 64, 1), "fused"), ((48, 1, 48), "fused"), ((50, 50, 33), "fused"),
    ((250, 250, 28), "fused"), ((80, 70, 66), "fused")])
def test_default_form_by_lane_use(gpu_lib, monkeypatch, shape, form):
    for v in ("OEM_FUSE", "OEM_CHUNK"):
        monkeypatch.delenv(v, raising=False)
    st = Stepper(tables.build(_scene(shape)))
    try:
        assert st.launch["form"] == form
    finally:
        st.close()


@pytest.mark.parametrize("shape", [(45, 41, 1), (45, 1, 41), (1, 45, 41), (48, 2, 50), (43, 44, 4)])
def test_both_forms_agree_on_flat_scenes(gpu_lib, shape):
    sc = _scene(shape)
    e0 = np.random.default_rng(3).standard_normal((6,) + shape).astype(np.float32)
    out = []
    for form in ("fused", "sweeps"):
        st = Stepper(tables.build(sc), dft_batch=8, form=form)
        try:
            for c in range(6):
                st.write_field(c, e0[c] * (1.0 if c < 3 else 1 / 377))
            st.run(37)
            out.append([st.read_field(c) for c in range(6)]
                       + [st.read_monitor(i) for i in range(len(sc.flux_monitors))])
        finally:
            st.close()
    for a, b in zip(*out):
        assert np.isfinite(b).all() and np.array_equal(a, b)


def _setup_bytes(shape):
    """Device memory that oem_adjoint_setup takes (the fused transposes keep a second field set)."""
    st = Stepper(tables.build(_scene(shape)), form="sweeps")
    try:
        cell = np.array([int(np.prod(shape)) // 2], np.int32)
        comp = np.array([2], np.int32)
        co = adjoint.design_coefficients(st.tabs, comp, cell)
        before = torch.cuda.mem_get_info()[0]
        _lib.check(st.lib, st.lib.oem_adjoint_setup(st.ctx, 1, _lib.ptr(comp), _lib.ptr(cell),
                                                    *[_lib.ptr(x) for x in co], 4))
        return before - torch.cuda.mem_get_info()[0]
    finally:
        st.close()


# the share of the fused transposes' lanes in use: 0.12, 0.23, 0.37, 0.25 with more than two million
# of them; 0.12 with fewer, 0.73
@pytest.mark.parametrize("shape,fused", [
    ((1000, 1000, 1), False), ((700, 700, 2), False), ((1000, 1000, 3), False),
    ((8000, 1, 128), False), ((400, 400, 1), True), ((500, 500, 6), True)])
def test_transposes_form_by_lane_use(gpu_lib, monkeypatch, shape, fused):
    monkeypatch.delenv("OEM_ADJ_FUSE", raising=False)
    default = _setup_bytes(shape)
    monkeypatch.setenv("OEM_ADJ_FUSE", "0")
    two = _setup_bytes(shape)
    second = 24 * int(np.prod(shape))               # the set's bytes; allocations round up to 2 MiB
    assert (default - two > second / 2) == fused, (default, two, second)


# few rows, few cells a row: where the halo row, the wrap and the clamp of a tile meet
@pytest.mark.parametrize("shape", [(45, 41, 1), (45, 1, 41), (60, 2, 50), (1, 45, 41), (43, 44, 3),
                                   (50, 3, 2)])
def test_fused_transposes_on_flat_grids(gpu_lib, monkeypatch, shape):
    sc = _scene(shape, steps=60)
    rng = np.random.default_rng(5)
    cell = rng.choice(int(np.prod(shape)), 30, replace=False)
    comp = rng.integers(3, size=30)
    m = tables.build(sc).monitors[0]
    K = rng.standard_normal((4, m.n1, m.n2)) + 1j * rng.standard_normal((4, m.n1, m.n2))
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("OEM_ADJ_FUSE", fuse)
        out.append(adjoint.overlap_power_gradient(sc, sc.flux_monitors[0].name, K, comp, cell))
    a, b = out
    assert np.isfinite(b.grad).all() and np.abs(b.grad).max() > 0
    assert a.J == b.J and np.array_equal(a.grad, b.grad)
