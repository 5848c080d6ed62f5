"""GPU tests of flat and thin scenes (few cells along z or y): the rule that keeps them off the tiled
kernels whose lanes they would leave idle, and the values of both forms on them."""

import numpy as np
import pytest

from openem_amd import cpml, grid, model, scenes, tables, waveform
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


# the share of the march's lanes in use: 0.03, 0.24, 0.25, 0.37, 0.14 with over half a million of
# them; under that, and above a half
@pytest.mark.parametrize("shape,form", [
    ((300, 300, 1), "sweeps"), ((150, 150, 8), "sweeps"), ((500, 500, 8), "sweeps"),
    ((400, 400, 12), "sweeps"), ((1000, 1, 1000), "sweeps"),
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
