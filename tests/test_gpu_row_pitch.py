"""GPU test of padded device rows (the layout of scenes of the fused step's size whose rows would
start inside a 128-byte line; OEM_ROW_PAD=1 forces it on the small scenes here).

The step reads and writes the same cells in the same order of operations, so everything equals
the dense layout (OEM_ROW_PAD=0) bit for bit; the energies are float64 sums of the same terms in
another order (at most 1e5 terms: n * 2^-53 = 1e-11 of their sum)."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import adjoint, scenes, tables
from openem_amd.model import FieldTimeMonitor, FluxTimeMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu


def _soup(shape, **kw):
    sc = scenes.mini_scene(shape=shape, num_steps=41, pml_xy=True, plane_wave_on=False,
                           magnetic_dipole=True, **kw)
    g = sc.grid
    span = tuple((float(g.axes[t].edges[0]), float(g.axes[t].edges[-1])) for t in (0, 1))
    return replace(sc, field_time_monitors=[
        FieldTimeMonitor("all", tuple(range(6)), (1, 2, 6), (6, 5, 14), 2, 40, 3, 12)],
        flux_time_monitors=[FluxTimeMonitor("f", 2, 20, 1, 0, 41, 2, 20, t_bounds=span)])


CASES = {
    # rows of 1 cell over, 1 under and just a multiple of 32; poles of two counts (CSR)
    "real_33": lambda: _soup((10, 12, 33)),
    "real_63_csr": lambda: _soup((9, 11, 63)),
    "real_64": lambda: _soup((9, 8, 64), lorentz_on=False),
    "real_97_pec": lambda: _soup((9, 8, 97), pec_on=True),
    "bloch_49": lambda: scenes.bloch_cell_scene(nxy=12, nz=49, n_pml=6, num_steps=41, nf=3),
}


@pytest.mark.parametrize("fuse", ["0", "1"])
@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_padded_rows_change_nothing(gpu_lib, monkeypatch, name, dense, fuse):
    sc = CASES[name]()
    tabs = tables.build(sc)
    monkeypatch.setenv("OEM_FUSE", fuse)
    rng = np.random.default_rng(4)
    e0 = rng.standard_normal(sc.shape).astype(np.complex64 if tabs.bloch else np.float32) * 1e-3
    out = []
    for pad in ("1", "0"):
        monkeypatch.setenv("OEM_ROW_PAD", pad)
        st = Stepper(tabs, dft_batch=8, dense_materials=dense)
        try:
            st.write_field(1, e0)
            assert np.array_equal(st.read_field(1), e0)
            st.run(41)
            st.setup_energy()
            out.append(([st.read_field(c) for c in range(6)]
                        + [st.read_monitor(i) for i in range(len(tabs.monitors))]
                        + [st.read_time_monitor(i) for i in range(len(sc.field_time_monitors))]
                        + [st.read_flux_time_monitor(i) for i in range(len(sc.flux_time_monitors))],
                       st.energy()))
        finally:
            st.close()
    (a, ea), (b, eb) = out
    for x, y in zip(a, b):
        assert np.abs(y).max() > 0 and np.array_equal(x, y)
    assert np.allclose(ea, eb, rtol=1e-11, atol=0)


@pytest.mark.parametrize("poles", [False, True])
def test_padded_rows_keep_the_gradient(gpu_lib, monkeypatch, poles):
    sc = (scenes.pole_guide_scene(num_steps=120, two_materials=True) if poles else
          scenes.waveguide_scene(shape=(30, 24, 22), n_pml=6, width_cells=6, thick_cells=4,
                                 fwidth_rel=0.3, num_steps=120, nf=1))
    ny, nz = sc.shape[1:]
    i, j, k = np.meshgrid([16, 18], [ny // 2 - 1, ny // 2 + 1], [nz // 2, nz // 2 + 1], indexing="ij")
    cell = ((i * ny + j) * nz + k).ravel()
    comp = np.arange(cell.size) % 3
    out = []
    for pad in ("1", "0"):
        monkeypatch.setenv("OEM_ROW_PAD", pad)
        out.append(adjoint.mode_power_gradient(sc, "fwd", comp, cell, checkpoint_every=50,
                                               record_bytes=0))
    assert np.abs(out[1].grad).max() > 0
    assert out[0].J == out[1].J and np.array_equal(out[0].grad, out[1].grad)
