"""kernel_variant 0's passes hold 14 work fields; with the kernels per subroutine
7 do.  Whatever fits with 7 has to fit: when an allocation fails, handles change
over, the one that allocates or another, with a recorded run or between steps,
and their results stay the oracle's bits.  The memory of the GPU is filled but
for a few fields of 16 MiB."""
import ctypes
import threading

import numpy as np
import pytest

from hicar_amd import _lib
from hicar_amd.advection import Advection, _ptr
from test_gpu_parity import random_domain
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

NX, NY, NZ = 256, 64, 256  # a field of the mass grid: 16 MiB
FIELD = 4 * NX * NY * NZ


class Filler:
    """Device memory taken until about `fields` fields are free."""

    def __init__(self):
        self.hip = Hip().h
        self.bufs = []

    def free_bytes(self):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def leave(self, fields):
        chunk = 16 << 30
        while chunk >= 2 << 20:
            room = self.free_bytes() - int(fields * FIELD)
            if room < chunk:
                chunk //= 2
                continue
            p = ctypes.c_void_p()
            if self.hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(chunk)) == 0:
                self.bufs.append(p)
            else:
                self.hip.hipGetLastError()
                chunk //= 2
        assert abs(self.free_bytes() - fields * FIELD) < FIELD

    def close(self):
        for p in self.bufs:
            self.hip.hipFree(p)
        self.bufs.clear()


@pytest.fixture
def filler():
    f = Filler()
    yield f
    f.close()


def domain(seed, nspec):
    return random_domain(NX, NY, NZ, seed, 2, True, True, nspec=nspec)


def passes_in_place(st):
    """Whether a step takes the passes in place (it is not counted)."""
    st.profile(True)
    st.advect(0.0)
    k = st.kernel_stats()
    st.profile(False)
    return "fused_first_pass" in k


def assert_bits(d, ref):
    for n in ref:
        np.testing.assert_array_equal(d.species[n].view(np.uint32), ref[n].view(np.uint32), err_msg=n)


# a handle takes 6 fields, 9 inputs, its species, and 14 or 7
def test_a_handle_that_fits_with_seven(oracle32, filler):
    case = domain(11, 2)
    d, o = case.domain, case.options
    ref = oracle32.run(d, o, 20.0, 2, 2, 2, {n: a.copy() for n, a in d.species.items()})
    filler.leave(6 + 9 + 2 + 7 + 3)
    st = Advection(d, o)
    try:
        st.run(20.0, 2, 2, 2)
        st.download()
        assert_bits(d, ref)
        assert not passes_in_place(st)
    finally:
        st.close()


@pytest.mark.parametrize("variant", [0, 1])
def test_another_handle_gets_the_memory(oracle32, filler, variant):
    a, b = domain(12, 1), domain(13, 1)
    b.options.kernel_variant = variant
    ref_a = oracle32.run(a.domain, a.options, 20.0, 4, 1, 2,
                         {n: q.copy() for n, q in a.domain.species.items()})
    ref_b = oracle32.run(b.domain, b.options, 15.0, 1, 0, 0,
                         {n: q.copy() for n, q in b.domain.species.items()})
    # variant 1: 12 coefficients, a second species buffer, a pass buffer
    need_b = 6 + 9 + 1 + (7 if variant == 0 else 12 + 1 + 1)
    filler.leave(6 + 9 + 1 + 7 + need_b + 3)
    st = Advection(a.domain, a.options)
    try:
        st.set_graph(True)
        st.run(20.0, 2, 1, 2)
        sb = Advection(b.domain, b.options)
        try:
            sb.run(15.0, 1, 0, 0)
            sb.download()
            st.run(20.0, 2, 1, 2)  # the graph was recorded over buffers that are gone
            st.download()
        finally:
            sb.close()
        assert_bits(a.domain, ref_a)
        assert_bits(b.domain, ref_b)
        assert not passes_in_place(st)
    finally:
        st.close()


def test_a_handle_steps_while_another_takes_the_memory(oracle32, filler):
    a, b = domain(14, 1), domain(15, 1)
    steps = 40
    want = Advection(a.domain, a.options)
    want.run(20.0, steps, 0, 0)
    init = {n: q.copy() for n, q in a.domain.species.items()}
    want.download()
    ref = {n: q.copy() for n, q in a.domain.species.items()}
    want.close()
    for n, q in init.items():
        a.domain.species[n][...] = q
    filler.leave(6 + 9 + 1 + 7 + 6 + 9 + 1 + 7 + 3)
    st = Advection(a.domain, a.options)
    err = []

    def go():
        try:
            for _ in range(steps):
                st.advect(20.0)
            st.sync()
        except Exception as e:  # noqa: BLE001
            err.append(e)
    t = threading.Thread(target=go)
    try:
        t.start()
        sb = Advection(b.domain, b.options)
        t.join()
        sb.close()
        assert not err, err
        st.download()
        assert_bits(a.domain, ref)
    finally:
        t.join()
        st.close()


def test_what_does_not_fit_with_seven_is_refused(oracle32, filler):
    case = domain(16, 2)
    d, o = case.domain, case.options
    filler.leave(6 + 9 + 2 + 7 - 3)
    with pytest.raises(_lib.IcarAdvError) as e:
        Advection(d, o)
    assert e.value.code == _lib.ENOMEM
    filler.close()
    st = Advection(d, o)  # the failure leaves nothing behind
    try:
        assert passes_in_place(st)
    finally:
        st.close()


# A new FP32 species finds room for its buffer, not for the second one that the
# fused path keeps; one bound again in 16 bits finds room for its buffer (half a
# field), not for the field it is converted through.
@pytest.mark.parametrize("nspec,storage,room", [(1, _lib.STORE_F32, 1.5), (2, _lib.STORE_F16, 0.3)])
def test_a_species_that_does_not_fit_is_not_bound(oracle32, filler, nspec, storage, room):
    case = domain(17, nspec)
    d, o = case.domain, case.options
    o.kernel_variant = 1
    late = np.ones_like(d.species["s0"])
    keep = {n: a.copy() for n, a in d.species.items()}
    ref = oracle32.run(d, o, 20.0, 2, 1, 2, {"s0": keep["s0"]})
    st = Advection(d, o)
    try:
        filler.leave(room)
        with pytest.raises(_lib.IcarAdvError) as e:
            st._check(st.lib.icar_adv_bind_species(st.h, 1, _ptr(late), storage, 0))
        assert e.value.code == _lib.ENOMEM
        st.run(20.0, 2, 1, 2)
        st.download()
    finally:
        st.close()
    assert_bits(d, ref)
    assert np.all(late == 1)
    if nspec == 2:
        np.testing.assert_array_equal(d.species["s1"], keep["s1"])
