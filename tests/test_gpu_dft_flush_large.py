"""GPU tests of DFT monitors whose replay takes more than one launch, up to more threads than one grid
dimension holds (2^32)."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from openem_amd import _lib, cpml, grid, model, tables
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
D = 20e-9
STEPS = 4


def _axis_tables(a, n):
    """Tables of an axis of n periodic cells (from a scene that is one cell across)."""
    shape = [1, 1, 1]
    shape[a] = n
    eps = np.ones(shape)
    axes = [grid.Axis(np.arange(m + 1) * D, "Periodic", "Periodic") for m in shape]
    sc = model.Scene(grid=grid.Grid(*axes), dt=cpml.courant_dt((D, D, D)), num_time_steps=STEPS,
                     eps_ex=eps, eps_ey=eps, eps_ez=eps)
    return tables.build(sc)


class _Vacuum(SimpleNamespace):
    """Step tables of n^3 cells of vacuum with one box monitor per (origin, box), one frequency."""

    def material_classes(self):
        lut = np.zeros((1, 8), np.float32)
        lut[0, :6] = [1.0, 0.5, 1.0, 0.5, 1.0, 0.5]          # (ca, cb) per component
        return np.zeros(self.shape, np.uint16), lut


def _tabs(n, boxes):
    t = [_axis_tables(a, n) for a in range(3)]
    ph = np.linspace(-1, 1, STEPS * 4).reshape(STEPS, 1, 4)
    mons = [SimpleNamespace(kind="box", nf=1, phase=ph, origin=o, box=b) for o, b in boxes]
    return _Vacuum(shape=(n, n, n), n_total=STEPS, ch=0.5, cw=t[0].cw, bloch=False, disp=None,
                   axes=[t[a].axes[a] for a in range(3)], plane_srcs=[], dipoles=[], tfsf=[], modes=[],
                   monitors=mons, scene=SimpleNamespace(field_time_monitors=[], flux_time_monitors=[]))


def _read(st, i):
    m = st.tabs.monitors[i]
    re, im = np.empty((2, 6) + tuple(m.box))
    _lib.check(st.lib, st.lib.oem_read_monitor(st.ctx, st.mon_ids[i], _lib.ptr(re), _lib.ptr(im), re.size))
    return re, im


def test_a_box_of_two_launches_equals_its_parts(gpu_lib):
    n, m = 360, 356                               # 45 M points: 1.06 M blocks, 2^20 a launch
    e0 = np.random.default_rng(2).standard_normal((n, n, n), np.float32)
    out = []
    for parts in (1, 4):
        w = m // parts
        st = Stepper(_tabs(n, [((2 + q * w, 2, 2), (w, m, m)) for q in range(parts)]), dft_batch=1)
        try:
            st.write_field(2, e0)
            st.run(1)
            out.append([_read(st, q) for q in range(parts)])
        finally:
            st.close()
    for c in range(2):
        whole = out[0][0][c]
        for q in range(4):
            part = out[1][q][c]
            assert np.abs(part[2]).max() > 0
            assert np.array_equal(whole[:, q * (m // 4):(q + 1) * (m // 4)], part)


def test_a_box_of_more_than_2_32_threads(gpu_lib):
    n = 896                                       # 6 x 716 M values: 2^32 + 2^22
    need = 120 << 30
    if torch.cuda.mem_get_info()[0] < need:
        pytest.skip(f"needs {need >> 30} GiB of device memory")
    box = (894, 894, n)
    assert 6 * box[0] * box[1] * box[2] > 1 << 32
    st = Stepper(_tabs(n, [((1, 1, 0), box)]), dft_batch=1)
    try:
        st.run(2)
        assert st.step_index == 2
    finally:
        st.close()
