"""The fused kernels read a domain's time step from a table in device memory.  A
new time step is set there in order with the steps still queued: steps enqueued
one after another with changing dt, without a wait between them, give the bits
of the same steps with one."""
import numpy as np
import pytest

from hicar_amd.advection import Advection, Ensemble
from test_gpu_parity import random_domain

pytestmark = pytest.mark.gpu

DTS = [20.0, 20.0, 20.0, 7.5, 20.0, 12.5, 12.5, 3.0]


def assert_bits(a, b):
    for n in b:
        np.testing.assert_array_equal(a[n].view(np.uint32), b[n].view(np.uint32), err_msg=n)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_queued_steps_keep_their_time_step(oracle32, order):
    case = random_domain(150, 90, 12, 31 + order, order, True, True, nspec=4)
    d, o = case.domain, case.options
    o.kernel_variant = 1
    ref = {n: a.copy() for n, a in d.species.items()}
    for dt in DTS:
        ref = oracle32.advect(d, o, dt, ref)
    st = Advection(d, o)
    try:
        for dt in DTS:
            st.advect(dt)
        st.download()
    finally:
        st.close()
    assert_bits(d.species, ref)


# 64 time steps are set per launch: one domain, just under, at and over a launch
@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_queued_ensemble_runs_keep_their_time_steps(oracle32, n):
    cases = [random_domain(5 + k % 7, 4 + k % 5, 3 + k % 3, 900 + k, 2, True, True, nspec=1)
             for k in range(n)]
    dts = np.array([[10.0 + k % 9, 4.0 + k % 4, 10.0 + k % 9] for k in range(n)], np.float32).T
    refs = []
    for k, c in enumerate(cases):
        c.options.kernel_variant = 1
        ref = {m: a.copy() for m, a in c.domain.species.items()}
        for row in dts:
            ref = oracle32.run(c.domain, c.options, row[k], 2, 1, 2, ref)
        refs.append(ref)
    members = [Advection(c.domain, c.options) for c in cases]
    ens = Ensemble(members)
    try:
        for row in dts:
            ens.run(row, 2, 1, 2)
        ens.sync()
        for m, c, ref in zip(members, cases, refs):
            m.download()
            assert_bits(c.domain.species, ref)
    finally:
        ens.close()
        for m in members:
            m.close()
