"""GPU tests of small scenes on a nearly full device: the fused step's second field set is optional
below the size from which every scene takes it, and a failed allocation is reported once."""

import gc

import numpy as np
import pytest
import torch

from openem_amd import _lib, scenes, tables
from openem_amd.solver import Stepper

pytestmark = pytest.mark.gpu
N = 20


def _free():
    gc.collect()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def _fill(leave):
    """Blocks that leave about ``leave`` bytes of the device (the large one frees some of its own
    bookkeeping, so the rest goes in smaller ones)."""
    hold = [torch.empty(_free() - (4 << 30), dtype=torch.uint8, device="cuda")]
    while (left := torch.cuda.mem_get_info()[0] - leave) >= 4 << 20:
        hold.append(torch.empty(left, dtype=torch.uint8, device="cuda"))
    return hold


def _run(st):
    try:
        st.run(N)
        return [st.read_field(c) for c in range(6)]
    finally:
        st.close()


def test_small_scene_without_room_for_two_field_sets(gpu_lib, monkeypatch):
    for v in ("OEM_FUSE", "OEM_CHUNK"):
        monkeypatch.delenv(v, raising=False)
    sc = scenes.mini_scene(shape=(140, 138, 136), num_steps=N, pml_xy=True, lorentz_on=False,
                           field_box=False)
    tabs = tables.build(sc)
    field_set = 24 * int(np.prod(sc.shape))
    want = _run(Stepper(tabs))                       # also loads what the device keeps loaded
    before = _free()
    st = Stepper(tabs, form="sweeps")
    one = before - _free()
    st.close()
    st = Stepper(tabs)
    assert st.launch["form"] == "fused"
    st.close()
    # one field set and its tables fit, half a set is left
    hold = _fill(one + field_set // 2)
    try:
        st = Stepper(tabs)
        form = st.launch["form"]
    finally:
        del hold
        _free()
    assert form == "sweeps"
    for a, b in zip(_run(st), want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_a_failed_allocation_is_reported_once(gpu_lib):
    sc = scenes.mini_scene(shape=(16, 17, 40), num_steps=N)
    st = Stepper(tables.build(sc))
    big = tables.build(scenes.mini_scene(shape=(140, 138, 136), num_steps=N, field_box=False))
    hold = _fill(32 << 20)
    try:
        with pytest.raises(_lib.OpenEMError) as e:
            Stepper(big)
        assert e.value.code == _lib.OEM_ENOMEM
    finally:
        del hold
        _free()
    assert np.abs(_run(st)[2]).max() > 0            # the other context's launches did not fail
