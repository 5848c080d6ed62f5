"""GPU tests of the end of a step: E-side points applied inside the fused march, small time monitors
sampled by the closing launch, and the step counter moved once per captured block.  The separate
launches (OEM_TAIL=0) and eager stepping (OEM_NO_GRAPH=1) do the same arithmetic on the same
values, so everything agrees bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import scenes, tables
from openem_amd.model import FieldMonitor, FieldTimeMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
N = 45                      # 8-step blocks: five captured, five steps of their own


def _run(tabs, form):
    st = Stepper(tabs, dft_batch=8, form=form)
    try:
        st.run(N)
        return ([st.read_field(c) for c in range(6)]
                + [st.read_monitor(i) for i in range(len(tabs.monitors))]
                + [st.read_time_monitor(i) for i in range(len(tabs.scene.field_time_monitors))])
    finally:
        st.close()


def _scene(cells, n_tm, cplx=False):
    """Ez and Ex dipoles of one point each at ``cells`` (two on a cell given twice)."""
    if cplx:
        sc = scenes.bloch_cell_scene(nxy=16, nz=70, n_pml=6, num_steps=N, nf=2, with_tfsf=False,
                                     n_cyl=2)
        wf = scenes.waveform.sample(scenes.waveform.GaussianPulse(4e14, 2e14), sc.dt, N)
    else:
        sc = scenes.mini_scene(shape=(16, 17, 70), num_steps=N, plane_wave_on=False)
        wf = sc.dipoles[0].waveform
    f = sc.flux_monitors[0].freqs
    dips = [scenes.PointDipole(2 * (q % 2), np.array([c]), np.array([1.0 + q]), wf)
            for q, c in enumerate(cells)]
    tms = [FieldTimeMonitor(f"t{q}", (0, 2, 4), (2 + q, 3, 30), (4, 4, 5), 1, N, 2, 30)
           for q in range(n_tm)]
    return replace(sc, dipoles=dips, flux_monitors=[FluxMonitor("z", 2, 34, +1, f)],
                   field_monitors=[FieldMonitor("b", f, (4, 4, 30), (6, 6, 8))],
                   field_time_monitors=tms)


# a cell twice; the first and last rows and cells of a tile (7 and 14 rows, 64 and 32 lanes), chunk
# ends, the grid's corners; more points than the march takes (10)
CELLS = {
    "same_cell": [(8, 8, 34), (8, 8, 34), (8, 8, 34)],
    "tile_edges": [(1, 6, 63), (2, 7, 64), (3, 13, 63), (2, 14, 33), (1, 16, 69), (14, 1, 1)],
    "ten": [(3 + q, 4, 30 + q) for q in range(10)],
    "one": [(8, 8, 34)],
}


@pytest.mark.parametrize("form", ["fused", "sweeps"])
@pytest.mark.parametrize("n_tm", [0, 1, 3])
@pytest.mark.parametrize("name", sorted(CELLS))
def test_folded_step_end_equals_separate_launches(gpu_lib, monkeypatch, name, n_tm, form):
    tabs = tables.build(_scene(CELLS[name], n_tm))
    got = _run(tabs, form)
    monkeypatch.setenv("OEM_NO_GRAPH", "1")
    eager = _run(tabs, form)
    monkeypatch.setenv("OEM_TAIL", "0")
    want = _run(tabs, form)
    for a, e, b in zip(got, eager, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b) and np.array_equal(e, b)


def test_folded_points_on_complex_fields(gpu_lib, monkeypatch):
    tabs = tables.build(_scene(CELLS["tile_edges"], 2, cplx=True))
    got = _run(tabs, "fused")
    monkeypatch.setenv("OEM_TAIL", "0")
    want = _run(tabs, "fused")
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)
