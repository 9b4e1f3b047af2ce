"""Negative values, zeros of both signs, infinities and NaN in the passes of
MPDATA, which replace the reference's maxima, selects and quotients by forms
that hold for ordinary values and fall back for the rest: bit for bit the
kernels per subroutine (a NaN being a NaN), and negative values and zeros the
oracle's values.  The sign of a zero is not held to the oracle, nor what is not
finite: the Fortran's MAX and MIN leave both open.  The same IEEE operations on
both sides, so the tolerance is zero."""
import numpy as np
import pytest

from hicar_amd.advection import Advection
from test_gpu_parity import random_domain

pytestmark = pytest.mark.gpu

STEPS = 2
# a tile of the corrective pass writes 60 columns and 16 or 8 rows, one of the
# donor-cell pass 62 and 8
SHAPE = (125, 35, 9)


def case_of(order, fct, specials, seed=3):
    case = random_domain(*SHAPE, seed, order, fct, True, nspec=4)
    d = case.domain
    r = np.random.default_rng(seed + order)
    d.species["s0"][...] -= np.float32(0.4)  # both signs
    q = d.species["s1"]
    q[...] = np.where(r.random(q.shape) > 0.7, q, np.where(r.random(q.shape) > 0.5, 0.0, -0.0))
    d.species["s2"][...] *= np.where(r.random(q.shape) > 0.5, 1.0, -1.0)
    for n, v in enumerate(specials):  # mid tile, on both sides of the tiles' edges, ground and top
        for j, k, i in ((10, 4, 30), (15, 0, 59), (16, 8, 60), (7, 3, 61), (8, 5, 62), (33, 2, 1)):
            d.species["s3"][j, k, (i + 3 * n) % SHAPE[0]] = v
    return case


def gpu(case, variant):
    d = case.domain
    init = {n: a.copy() for n, a in d.species.items()}
    case.options.kernel_variant = variant
    st = Advection(d, case.options)
    try:
        st.run(case.dt, STEPS, 1, 2)
        st.download()
        return {n: a.copy() for n, a in d.species.items()}
    finally:
        st.close()
        for n, a in init.items():
            d.species[n][...] = a


def assert_values(got, ref):
    for n in ref:
        nan = np.isnan(ref[n])
        np.testing.assert_array_equal(np.isnan(got[n]), nan, err_msg=n)
        np.testing.assert_array_equal(got[n].view(np.uint32)[~nan], ref[n].view(np.uint32)[~nan],
                                      err_msg=n)


def per_subroutine(monkeypatch, case):
    monkeypatch.setenv("ICAR_ADV_PASS_KERNELS", "0")
    ref = gpu(case, 0)
    monkeypatch.delenv("ICAR_ADV_PASS_KERNELS")
    return ref


@pytest.mark.parametrize("specials", [(), (np.nan,), (np.inf,), (-np.inf, np.nan), (3e38, -3e38)],
                         ids=str)
@pytest.mark.parametrize("fct", [True, False])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("variant", [0, 1])
def test_special_values(oracle32, monkeypatch, variant, order, fct, specials):
    case = case_of(order, fct, specials)
    got = gpu(case, variant)
    assert_values(got, per_subroutine(monkeypatch, case))
    if not specials:
        ref = oracle32.run(case.domain, case.options, case.dt, STEPS, 1, 2)
        for n in ref:
            np.testing.assert_array_equal(got[n], ref[n], err_msg=n)
