"""GPU tests of the point corrections, snapshots and design recordings that the work-groups of the
two sweeps do for their own cells after the march.  The launches they replace (OEM_TAIL=0) do the
same arithmetic on the same values, so everything agrees bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import adjoint, scenes, tables
from openem_amd.model import FieldMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
N = 45                      # 8-step blocks: five captured, five steps of their own


def _run(tabs):
    st = Stepper(tabs, dft_batch=8, form="sweeps")
    try:
        st.run(N)
        return ([st.read_field(c) for c in range(6)]
                + [st.read_monitor(i) for i in range(len(tabs.monitors))])
    finally:
        st.close()


def _check(monkeypatch, sc, chunk=None):
    if chunk:
        monkeypatch.setenv("OEM_CHUNK", str(chunk))
    tabs = tables.build(sc)
    got = _run(tabs)
    monkeypatch.setenv("OEM_NO_GRAPH", "1")
    eager = _run(tabs)
    monkeypatch.setenv("OEM_TAIL", "0")
    want = _run(tabs)
    for a, e, b in zip(got, eager, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b) and np.array_equal(e, b)


def _planes(sc, n):
    """Flux planes on every axis (n in all, through tile and chunk edges) and a box."""
    f = sc.flux_monitors[0].freqs
    nx, ny, nz = sc.eps_ex.shape
    at = [(2, 16), (0, 7), (1, 8), (0, 8), (2, nz - 16), (1, 15), (0, nx - 8), (2, 21), (1, 9), (0, 12)]
    return replace(sc, flux_monitors=[FluxMonitor(f"p{q}", a, m, +1, f) for q, (a, m) in enumerate(at[:n])],
                   field_monitors=[FieldMonitor("b", f, (5, 6, 14), (13, 11, nz - 28))])


# rows of whole waves and rows that are not; the chunk the rule gives, one plane, a remainder, all
@pytest.mark.parametrize("chunk", [None, 1, 7, 26])
@pytest.mark.parametrize("nz", [44, 64])
def test_lists_and_snapshots_by_work_group(gpu_lib, monkeypatch, nz, chunk):
    sc = scenes.tfsf_box_scene(shape=(26, 24, nz), num_steps=N, scatterer=True)
    _check(monkeypatch, _planes(sc, 4), chunk)


# more monitors than the sweep takes (8); more lists on a side than it takes (4)
@pytest.mark.parametrize("n_mon,n_src", [(7, 1), (10, 4), (3, 6)])
def test_more_lists_than_the_sweeps_take(gpu_lib, monkeypatch, n_mon, n_src):
    sc = scenes.tfsf_box_scene(shape=(26, 24, 44), num_steps=N)
    src = sc.tfsf_sources[0]
    sc = replace(sc, tfsf_sources=[replace(src, jxy=(1.0 + q, 0.5 * q)) for q in range(n_src)])
    _check(monkeypatch, _planes(sc, n_mon))


def test_complex_fields(gpu_lib, monkeypatch):
    sc = scenes.bloch_cell_scene(nxy=24, nz=70, n_pml=6, num_steps=N, nf=2, n_cyl=2)
    _check(monkeypatch, _planes(sc, 3))


@pytest.mark.parametrize("record_bytes", [None, 0])
def test_design_recording_by_work_group(gpu_lib, monkeypatch, record_bytes):
    sc = scenes.waveguide_scene(shape=(30, 24, 22), n_pml=6, width_cells=6, thick_cells=4,
                                fwidth_rel=0.3, num_steps=120, nf=1)
    cell = np.arange(13 * 24 * 22 + 9 * 22 + 9, 16 * 24 * 22, 37)[:30]
    comp = np.arange(cell.size) % 3
    kw = {} if record_bytes is None else dict(record_bytes=record_bytes, checkpoint_every=48)
    got = adjoint.mode_power_gradient(sc, "fwd", comp, cell, **kw)
    monkeypatch.setenv("OEM_TAIL", "0")
    want = adjoint.mode_power_gradient(sc, "fwd", comp, cell, **kw)
    assert np.abs(want.grad).max() > 0 and np.array_equal(got.grad, want.grad)
