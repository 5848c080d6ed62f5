"""GPU tests of the DFT replay of batches that are no multiple of the snapshots it keeps in flight
(a run's last batch, a dft_batch that is not 16)."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import scenes, tables
from openem_amd.model import FieldMonitor, FluxMonitor
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu


def _large(cplx):
    """Monitors whose accumulators bound the replay: a box of 2 x 400 x 400 cells at 8 frequencies;
    four complex planes of 200 x 200 at 21."""
    if cplx:
        sc = scenes.bloch_cell_scene(nxy=200, nz=60, n_pml=6, num_steps=200, nf=21, with_tfsf=False,
                                     n_cyl=2)
        f = sc.flux_monitors[0].freqs
        return replace(sc, flux_monitors=[FluxMonitor(f"p{q}", 2, 12 + 9 * q, +1, f) for q in range(4)],
                       field_monitors=[])
    sc = scenes.mini_scene(shape=(20, 400, 400), num_steps=200, lorentz_on=False, plane_wave_on=False,
                           field_box=False)
    f = np.linspace(2e14, 4e14, 8)
    return replace(sc, flux_monitors=[], field_monitors=[FieldMonitor("b", f, (9, 0, 0), (2, 400, 400))])


@pytest.mark.parametrize("cplx", [False, True])
def test_a_shorter_batch_costs_less(gpu_lib, cplx):
    """Ten steps replayed snapshot by snapshot took as long as sixteen (1.04 and 1.00 of them)."""
    st = Stepper(tables.build(_large(cplx)))
    try:
        st.run(16)
        ms = {n: min(st.profile_run(n)["dft_flush"][0] for _ in range(6)) for n in (16, 10)}
    finally:
        st.close()
    assert ms[10] < 0.95 * ms[16], ms


@pytest.mark.parametrize("cplx", [False, True])
def test_any_batch_length_adds_in_step_order(gpu_lib, cplx):
    """A batch of n steps from cleared accumulators is the same float64 sum for every dft_batch of n
    and more, in one batch: 0 + (v1 p1 + ... + vn pn), bit for bit."""
    if cplx:
        sc = scenes.bloch_cell_scene(nxy=9, nz=60, n_pml=6, num_steps=70, nf=2, with_tfsf=False, n_cyl=2)
    else:
        sc = scenes.mini_scene(shape=(10, 12, 40), num_steps=70, plane_wave_on=False)
    f = np.linspace(2e14, 4e14, 11)
    sc = replace(sc, flux_monitors=[FluxMonitor("p", 2, 20, +1, f)],
                 field_monitors=[FieldMonitor("b", f[:3], (0, 0, 18), (9, 9, 3))])
    tabs = tables.build(sc)
    e0 = np.random.default_rng(6).standard_normal(sc.shape).astype(np.complex64 if cplx else np.float32)
    for n in (1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 31, 63):
        out = []
        for T in (n, 64):
            st = Stepper(tabs, dft_batch=T)
            try:
                st.write_field(1, e0)
                st.run(n)
                out.append([st.read_monitor(i) for i in range(2)])
            finally:
                st.close()
        for a, b in zip(*out):
            assert np.abs(b).max() > 0 and np.array_equal(a, b), n
