"""GPU test of the DFT replay (one launch over the monitors, frequencies in groups of 1, 2, 4 or 8,
16 snapshots in flight).

A batch of T steps only regroups the float64 sums, so every T agrees with T = 1 (one snapshot per
replay) to the rounding of 45 float64 additions: 45 * 45 * 2^-53 = 2.3e-13 of the largest term, and
the largest accumulator is at least a tenth of it here."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import scenes, serving, tables
from openem_amd.model import FieldMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
STEPS = 45


def _scene(nf, cplx):
    if cplx:
        sc = scenes.bloch_cell_scene(nxy=9, nz=60, n_pml=6, num_steps=STEPS, nf=2, with_tfsf=False,
                                     n_cyl=2)
    else:
        sc = scenes.mini_scene(shape=(10, 12, 40), num_steps=STEPS, plane_wave_on=False)
    f = np.linspace(2e14, 4e14, nf)
    k = sc.shape[2] // 2
    # 9 monitors: more than one launch takes; a box of 270 or 243 points and single-point boxes
    flux = [FluxMonitor(f"p{q}", q % 3, 3 + q, +1, f[:1 + q % nf]) for q in range(6)]
    boxes = [FieldMonitor("b", f, (0, 0, k), (9, 9, 3)), FieldMonitor("one", f, (1, 1, k), (1, 1, 1)),
             FieldMonitor("row", f, (0, 2, k), (1, 1, 9))]
    return replace(sc, flux_monitors=flux, field_monitors=boxes)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nf", [1, 2, 3, 5, 8, 9, 17])
def test_batches_regroup_the_same_sums(gpu_lib, nf, cplx):
    sc = _scene(nf, cplx)
    tabs = tables.build(sc)
    e0 = np.random.default_rng(6).standard_normal(sc.shape).astype(np.complex64 if cplx else np.float32)
    out = {}
    for T in (1, 2, 7, 16, 17, 33, 64):
        st = Stepper(tabs, dft_batch=T)
        try:
            st.write_field(1, e0)
            st.run(STEPS)
            out[T] = [st.read_monitor(i) for i in range(len(tabs.monitors))]
        finally:
            st.close()
    for T, got in out.items():
        for a, b in zip(got, out[1]):
            assert np.abs(b).max() > 0
            assert np.abs(a - b).max() <= 2.3e-12 * np.abs(b).max(), T


@pytest.mark.parametrize("nf", [3, 9])
def test_pool_replay_equals_the_standalone_replay(gpu_lib, nf):
    tabs = tables.build(_scene(nf, False))
    st = Stepper(tabs)
    st.run(STEPS)
    want = [st.read_monitor(i) for i in range(len(tabs.monitors))]
    st.close()
    pool = serving.Pool(64 << 20)
    st = Stepper(tabs, pool=pool)
    pool.run_to_completion([st])
    got = [st.read_monitor(i) for i in range(len(tabs.monitors))]
    st.close()
    pool.close()
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)
