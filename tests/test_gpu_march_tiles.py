"""GPU tests of the fused march's tile shapes and of the rule that picks the march for small
scenes.

The last strip of a row is 32 lanes wide (tiles of 14 rows) when at most 32 cells are left, and a
small scene's stores are plain.  The arithmetic of a cell does not depend on the tile, so fields
and phasors equal the two sweeps' bit for bit at every edge of the tiling."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import scenes, tables
from openem_amd.model import FieldMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu

# rows of one 32-wide strip alone, exactly full, one cell over (a 64-wide strip), one 64-wide and
# a 32-wide strip of 1, 31 or 32 cells, and 33 over; row counts around 7 and 14
SHAPES = [(5, 15, 20), (5, 14, 32), (4, 13, 33), (4, 7, 65), (5, 29, 95), (4, 28, 96), (4, 8, 97)]


@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_tile_edges_equal_the_sweeps(gpu_lib, shape, dense):
    sc = scenes.mini_scene(shape=shape, n_pml=3, num_steps=33, lorentz_on=shape[2] > 30,
                           field_box=False, nf=2)
    nx, ny, nz = shape
    f = sc.flux_monitors[0].freqs
    sc = replace(sc, flux_monitors=[FluxMonitor("z", 2, (nz - 1) // 32 * 32 or nz // 2, +1, f),
                                    FluxMonitor("y", 1, min(ny - 1, 14), +1, f)],
                 field_monitors=[FieldMonitor("b", f, (1, 0, nz // 2), (2, ny, nz - nz // 2))])
    tabs = tables.build(sc)
    e0 = np.random.default_rng(5).standard_normal((3,) + shape).astype(np.float32)
    out = []
    for form in ("fused", "sweeps"):
        st = Stepper(tabs, dft_batch=8, form=form, dense_materials=dense)
        try:
            for c in range(3):
                st.write_field(c, e0[c])
            st.run(33)
            out.append([st.read_field(c) for c in range(6)]
                       + [st.read_monitor(i) for i in range(len(tabs.monitors))])
        finally:
            st.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_complex_tiles_equal_the_sweeps(gpu_lib):
    sc = scenes.bloch_cell_scene(nxy=15, nz=90, n_pml=6, num_steps=24, nf=2, with_tfsf=False,
                                 n_cyl=2)
    tabs = tables.build(sc)
    rng = np.random.default_rng(3)
    e0 = (rng.standard_normal(sc.shape) + 1j * rng.standard_normal(sc.shape)).astype(np.complex64)
    out = []
    for form in ("fused", "sweeps"):
        st = Stepper(tabs, dft_batch=8, form=form)
        try:
            st.write_field(0, e0)
            st.run(24)
            out.append([st.read_field(c) for c in range(6)]
                       + [st.read_monitor(i) for i in range(len(tabs.monitors))])
        finally:
            st.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_default_form_by_size_and_point_lists(gpu_lib, monkeypatch):
    """The march for a scene whose two field sets stay in the cache, the sweeps for one with a
    magnetic point list (its results keep the sweeps' rounding) or between the two sizes."""
    monkeypatch.delenv("OEM_FUSE", raising=False)
    for kw, form in ((dict(shape=(10, 12, 40)), "fused"),
                     (dict(shape=(10, 12, 40), magnetic_dipole=True), "sweeps"),
                     (dict(shape=(160, 160, 170), lorentz_on=False), "sweeps")):
        sc = scenes.mini_scene(num_steps=2, field_box=False, **kw)
        st = Stepper(tables.build(sc))
        assert st.launch["form"] == form, kw
        st.close()
