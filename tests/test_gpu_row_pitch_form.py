"""GPU tests of which scenes get padded device rows: those of the fused step's size that the fused
step will march.  The rows show in the device memory that a context takes."""

import ctypes as C

import numpy as np
import pytest
import torch

from openem_amd import _lib, scenes, tables
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _defaults(monkeypatch):
    for v in ("OEM_FUSE", "OEM_ROW_PAD"):
        monkeypatch.delenv(v, raising=False)


def _bytes(lib, shape, form=None, cplx=0, write=None):
    """Device bytes of a context of ``shape`` that holds its fields (and set its form)."""
    d = _lib.Dims(nx=shape[0], ny=shape[1], nz=shape[2], n_steps=4, dft_batch=16, ch=1.0, cw=1.0,
                  complex_fields=cplx)
    ctx = C.c_void_p()
    before = torch.cuda.mem_get_info()[0]
    _lib.check(lib, lib.oem_ctx_create(C.byref(d), 0, C.byref(ctx)))
    try:
        if write is not None:
            _lib.check(lib, lib.oem_write_field(ctx, 0, _lib.ptr(write), write.size))
        if form is not None:
            _lib.check(lib, lib.oem_set_step_form(ctx, form))
        if write is not None:
            back = np.empty_like(write)
            _lib.check(lib, lib.oem_read_field(ctx, 0, _lib.ptr(back), back.size))
            assert np.array_equal(back, write)
        return before - torch.cuda.mem_get_info()[0]
    finally:
        _lib.check(lib, lib.oem_ctx_destroy(ctx))


def _fields(shape, nz, cplx=0):
    return 24 * (1 + cplx) * shape[0] * shape[1] * nz


TOL = 16 << 20          # granules of the allocations; every pad below is larger


@pytest.mark.parametrize("shape,cplx,form,nz", [
    ((400, 300, 210), 0, None, 224), ((400, 300, 210), 0, 2, 224),      # marched: rows of whole lines
    ((400, 300, 210), 0, 1, 210),                                       # the sweeps were asked for
    ((600, 600, 502), 0, None, 502),          # a field set past 4 GiB: the march cannot step it
    ((400, 400, 566), 1, None, 566),
])
def test_rows_are_padded_for_the_march_alone(gpu_lib, shape, cplx, form, nz):
    _bytes(gpu_lib, (64, 64, 64))
    got = _bytes(gpu_lib, shape, form, cplx)
    assert abs(got - _fields(shape, nz, cplx)) < TOL, (got, _fields(shape, nz, cplx))


def test_rows_follow_the_environment_and_the_last_form(gpu_lib, monkeypatch):
    shape = (400, 300, 210)
    _bytes(gpu_lib, (64, 64, 64))
    monkeypatch.setenv("OEM_FUSE", "0")
    assert abs(_bytes(gpu_lib, shape) - _fields(shape, 210)) < TOL
    assert abs(_bytes(gpu_lib, shape, 2) - _fields(shape, 224)) < TOL


@pytest.mark.parametrize("form", [1, 2])
def test_written_fields_stay(gpu_lib, monkeypatch, form):
    if form == 2:
        monkeypatch.setenv("OEM_FUSE", "0")          # dense rows at first
    shape = (240, 220, 210)
    w = np.random.default_rng(1).standard_normal(int(np.prod(shape)), np.float32)
    _bytes(gpu_lib, shape, form, write=w)


def test_sweeps_on_dense_rows_equal_the_march(gpu_lib):
    sc = scenes.box_soup_scene(shape=(230, 220, 210), n_pml=8, n_boxes=12, num_steps=12, nf=2)
    tabs = tables.build(sc)
    out = []
    for form in ("sweeps", "fused"):
        st = Stepper(tabs, form=form)
        try:
            st.run(12)
            out.append([st.read_field(c) for c in range(6)] + [st.read_monitor(0)])
        finally:
            st.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)
