"""The fused kernels read a domain's time step from a table in device memory.  A
new time step is set there in order with the steps still queued: steps enqueued
one after another with changing dt, without a wait between them, give the bits
of the same steps with one, and a recorded run replays with the time step it was
recorded with."""
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


# the steps between leave order 1's and 2's home buffers as they were, so that
# the third run is a replay
@pytest.mark.parametrize("order,between", [(1, 2), (2, 2), (3, 1)])
def test_replay_after_steps_with_another_dt(oracle32, order, between):
    case = random_domain(61, 33, 8, 57 + order, order, True, True, nspec=2)
    d, o = case.domain, case.options
    o.kernel_variant = 1
    ref = {n: a.copy() for n, a in d.species.items()}
    st = Advection(d, o)
    try:
        st.set_graph(True)
        for _ in range(2):
            st.run(20.0, 2, 1, 2)
            ref = oracle32.run(d, o, 20.0, 2, 1, 2, ref)
            for _ in range(between):
                st.advect(6.0)
                ref = oracle32.advect(d, o, 6.0, ref)
        st.run(20.0, 2, 1, 2)
        ref = oracle32.run(d, o, 20.0, 2, 1, 2, ref)
        st.download()
    finally:
        st.close()
    assert_bits(d.species, ref)


def test_ensemble_replay_after_a_run_with_another_dt(oracle32):
    cases = [random_domain(30 + 9 * k, 20, 6, 70 + k, 2, True, True, nspec=2) for k in range(3)]
    refs = []
    for c in cases:
        c.options.kernel_variant = 1
        refs.append({m: a.copy() for m, a in c.domain.species.items()})
    members = [Advection(c.domain, c.options) for c in cases]
    ens = Ensemble(members)
    try:
        for dt, graph in ((20.0, True), (6.0, False), (20.0, True)):
            ens.run([dt] * 3, 2, 1, 2, graph=graph)
            refs = [oracle32.run(c.domain, c.options, dt, 2, 1, 2, r) for c, r in zip(cases, refs)]
        ens.sync()
        for m, c, ref in zip(members, cases, refs):
            m.download()
            assert_bits(c.domain.species, ref)
    finally:
        ens.close()
        for m in members:
            m.close()
