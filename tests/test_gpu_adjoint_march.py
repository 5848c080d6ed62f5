"""GPU tests of the two transposed updates as one march, with the next step's objective points and
eps gradient in its tail.  The two kernels and the launches they replace (OEM_ADJ_FUSE=0) round
every value the same way, so the gradients agree bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from openem_amd import adjoint, scenes, tables

pytestmark = pytest.mark.gpu
N = 60


def _gradients(monkeypatch, sc, chunk=None, **kw):
    t = tables.build(sc)
    m = t.monitors[[m.name for m in t.monitors].index("T")]
    rng = np.random.default_rng(4)
    K = rng.standard_normal((4, m.n1, m.n2)) + 1j * rng.standard_normal((4, m.n1, m.n2))
    cell = rng.choice(int(np.prod(sc.shape)), 60, replace=False)
    comp = rng.integers(3, size=60)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("OEM_ADJ_FUSE", fuse)
        if chunk and fuse == "1":
            monkeypatch.setenv("OEM_ADJ_CHUNK", str(chunk))
        else:
            monkeypatch.delenv("OEM_ADJ_CHUNK", raising=False)
        out.append(adjoint.overlap_power_gradient(sc, "T", K, comp, cell, **kw))
    a, b = out
    assert np.isfinite(b.grad).all() and np.abs(b.grad).max() > 0
    assert a.J == b.J and np.array_equal(a.grad, b.grad)


def _mini(shape, **kw):
    return scenes.mini_scene(shape=shape, num_steps=N, nf=2, field_box=False, **kw)


# whole and broken last tiles, fewer grid rows than a tile has, the longest row taken (128), one past
# it (the two kernels), every boundary, poles (the gradient then keeps its launch), classes in LDS
# (9 x 7: 317 of them) and in global memory
@pytest.mark.parametrize("chunk", [None, 1, 3, 99])
@pytest.mark.parametrize("shape,kw", [
    ((9, 7, 40), dict()),
    ((16, 17, 70), dict(pml_xy=True, lorentz_on=False)),
    ((13, 12, 64), dict(periodic_xy=False, lorentz_on=False, sigma_on=True)),
    ((10, 12, 127), dict(lorentz_on=False, nonuniform_z=True)),
    ((10, 9, 128), dict(lorentz_on=False, pec_on=False)),
    ((10, 9, 129), dict(lorentz_on=False)),
])
def test_march_equals_the_two_kernels(gpu_lib, monkeypatch, shape, kw, chunk):
    _gradients(monkeypatch, _mini(shape, **kw), chunk)


def test_dense_coefficients_and_segments(gpu_lib, monkeypatch):
    sc = _mini((48, 40, 40), lorentz_on=False)
    rng = np.random.default_rng(7)          # more distinct cells than classes
    e = [2.0 + rng.uniform(0, 2, size=sc.shape) for _ in range(3)]
    sc = replace(sc, eps_ex=e[0], eps_ey=e[1], eps_ez=e[2])
    _gradients(monkeypatch, sc, checkpoint_every=17, record_bytes=0)


@pytest.mark.parametrize("nx", [6, 250])
def test_chunk_of_the_two_kernels(gpu_lib, monkeypatch, nx):
    """Small grids take chunks of fewer planes; every chunk gives the same gradient."""
    monkeypatch.setenv("OEM_ADJ_FUSE", "0")
    sc = _mini((nx, 12, 44), lorentz_on=False)
    rng = np.random.default_rng(4)
    t = tables.build(sc)
    m = t.monitors[[m.name for m in t.monitors].index("T")]
    K = rng.standard_normal((4, m.n1, m.n2)) + 0j
    cell = rng.choice(int(np.prod(sc.shape)), 40, replace=False)
    comp = rng.integers(3, size=40)
    got = adjoint.overlap_power_gradient(sc, "T", K, comp, cell)
    monkeypatch.setenv("OEM_ADJ_CHUNK", "8")
    want = adjoint.overlap_power_gradient(sc, "T", K, comp, cell)
    assert np.abs(want.grad).max() > 0 and np.array_equal(got.grad, want.grad)
