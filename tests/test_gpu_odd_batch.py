"""GPU tests of captured blocks of an odd number of steps on the fused path, where a block ends with
the other field set than it began with."""

import numpy as np
import pytest

from openem_amd import scenes, tables
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu


def _all(st):
    return [st.read_field(c) for c in range(6)] + [st.read_monitor(i) for i in range(len(st.tabs.monitors))]


@pytest.mark.parametrize("calls", [(50,), (7, 43), (5, 5, 5, 35), (16, 17, 17)])
@pytest.mark.parametrize("T", [1, 5, 15])
@pytest.mark.parametrize("cplx", [False, True])
def test_odd_blocks_equal_eager_steps(gpu_lib, monkeypatch, cplx, T, calls):
    sc = (scenes.bloch_cell_scene(nxy=12, nz=50, n_pml=6, num_steps=50, nf=2, n_cyl=2, with_tfsf=False)
          if cplx else scenes.mini_scene(shape=(12, 14, 40), num_steps=50))
    tabs = tables.build(sc)
    e0 = np.random.default_rng(7).standard_normal(sc.shape).astype(np.complex64 if cplx else np.float32)
    out = []
    for ng in ("0", "1"):
        monkeypatch.setenv("OEM_NO_GRAPH", ng)
        st = Stepper(tabs, dft_batch=T, form="fused")
        try:
            st.write_field(1, e0)
            for n in calls:
                st.run(n)
            out.append(_all(st))
        finally:
            st.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_odd_blocks_replay_a_graph(gpu_lib):
    """A step of launches of its own took 1.2 times a replayed one on this scene."""
    tabs = tables.build(scenes.mini_scene(shape=(12, 14, 40), num_steps=4000, lorentz_on=False,
                                          field_box=False))
    ms = {}
    for T in (16, 15):
        st = Stepper(tabs, dft_batch=T, form="fused")
        try:
            st.run(2 * T)
            ms[T] = min(st.timed_run(480) for _ in range(6))
        finally:
            st.close()
    assert ms[15] < 1.1 * ms[16], ms
