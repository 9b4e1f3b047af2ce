"""A handle without species: advect() and run() form the step's winds, return 0
and leave the diagnostics their numbers, and a species bound afterwards is
advected."""
import numpy as np
import pytest

from hicar_amd import _lib, synthetic
from hicar_amd.advection import Advection, _ptr
from test_gpu_parity import random_domain

pytestmark = pytest.mark.gpu


def bind_late(st, d, name, arr):
    st._check(st.lib.icar_adv_bind_species(st.h, 0, _ptr(arr), _lib.STORE_F32, 0))
    d.species[name] = arr
    st.names = [name]
    st.upload(fields=False)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("step", ["advect", "run", "graph"])
def test_mpdata_without_species(oracle32, step, variant, order):
    case = random_domain(37, 21, 6, 5 + order, order, True, True, nspec=1)
    d, o = case.domain, case.options
    o.kernel_variant = variant
    q = d.species.pop("s0")
    o.vars_to_advect = []
    U, V, W = oracle32.compute_wind(d, 20.0, True)
    want = [np.abs(U[1:-1, :, 1:]).max(), np.abs(V[1:, :, 1:-1]).max(),
            np.abs(W / oracle32.arr(d.advection_dz))[1:-1, :, 1:-1].max()]
    st = Advection(d, o)
    try:
        if step == "advect":
            st.advect(20.0)
        else:
            st.set_graph(step == "graph")
            for _ in range(2):
                st.run(20.0, 2, 2, 2)
        np.testing.assert_array_equal(st.max_courant(), np.array(want, np.float64))
        bind_late(st, d, "s0", q)
        o.vars_to_advect = ["s0"]
        ref = oracle32.run(d, o, 12.5, 2, 2, 2, {"s0": q.copy()})
        st.run(12.5, 2, 2, 2)
        st.download()
    finally:
        st.close()
    np.testing.assert_array_equal(q.view(np.uint32), ref["s0"].view(np.uint32))


@pytest.mark.parametrize("step", ["advect", "run", "graph"])
@pytest.mark.parametrize("h,v,fc,rk3", [(5, 3, 1, True), (1, 1, 0, False)])
def test_std_without_species(oracle32, h, v, fc, rk3, step):
    case = synthetic.config_std(nx=37, ny=29, nz=8, steps=1, nspecies=1, h_order=h, v_order=v,
                                flux_corr=fc, rk3=rk3, cfl=0.4)
    d, o = case.domain, case.options
    name, q = next(iter(d.species.items()))
    d.species.clear()
    o.vars_to_advect = []
    Um, Vm, Wm, _ = oracle32.std_compute_wind(d, case.dt, o.parameters.advect_density)
    inner = (slice(1, -1), slice(None), slice(1, -1))
    want = (np.abs(Um[1:-1, :, 1:-1]).max(), np.abs(Vm[1:-1, :, 1:-1]).max(),
            np.abs(Wm / d.advection_dz.astype(np.float32))[inner].max())
    st = Advection(d, o)
    try:
        if step == "advect":
            st.advect(case.dt)
        else:
            st.set_graph(step == "graph")
            for _ in range(2):
                st.run(case.dt, 2)
        np.testing.assert_array_equal(st.max_courant(), np.array(want, np.float64))
        bind_late(st, d, name, q)
        o.vars_to_advect = [name]
        ref = {name: q.copy()}
        for _ in range(2):
            ref = oracle32.std_advect(d, o, 0.5 * case.dt, ref)
        st.run(0.5 * case.dt, 2)
        st.download()
    finally:
        st.close()
    np.testing.assert_array_equal(q.view(np.uint32), ref[name].view(np.uint32))
