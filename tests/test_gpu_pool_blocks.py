"""GPU test of the serving pool's blocks: each combination of launches that the running scenes need
is a captured block of its own.  Scenes of every combination, joining and leaving one pool at
different blocks, keep the bits of the two sweeps run alone (the same kernels' arithmetic)."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import scenes, serving, tables
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu


def _scenes():
    m = dict(shape=(9, 10, 40), field_box=False)
    plain = scenes.mini_scene(num_steps=40, dipole_on=False, lorentz_on=False, **m)
    out = [plain,                                                                # sweeps, monitors
           replace(plain, flux_monitors=[]),                                     # sweeps alone
           scenes.mini_scene(num_steps=33, lorentz_on=False, **m),               # folded dipoles
           scenes.mini_scene(num_steps=17, dipole_on=False, **m),                # poles
           scenes.mini_scene(num_steps=50, magnetic_dipole=True, **m),           # H points, poles
           scenes.tfsf_box_scene(shape=(20, 19, 40), num_steps=31),              # both sides' faces
           scenes.waveguide_scene(shape=(30, 20, 18), n_pml=5, width_cells=6, thick_cells=4,
                                  num_steps=16, nf=1)]                           # mode points
    return [tables.build(s) for s in out]


def test_every_kind_of_block_keeps_the_sweeps_bits(gpu_lib):
    tabs = _scenes()
    want = []
    for t in tabs:
        st = Stepper(t, form="sweeps")
        st.run(t.n_total)
        want.append([st.read_field(c) for c in range(6)]
                    + [st.read_monitor(i) for i in range(len(t.monitors))])
        st.close()
    pool = serving.Pool(256 << 20)
    sts = [Stepper(t, pool=pool) for t in tabs]
    # one scene after the other joins at the next block, then all run out
    for st in sts:
        pool.attach(st)
        pool.launch(1)
    while pool.stats()["running"]:
        pool.launch(1)
    pool.wait(0)
    for t, st, ref in zip(tabs, sts, want):
        got = [st.read_field(c) for c in range(6)] + [st.read_monitor(i) for i in range(len(t.monitors))]
        st.close()
        for a, b in zip(got, ref):
            assert np.array_equal(a, b)
        assert max(np.abs(b).max() for b in ref) > 0
    pool.close()
