"""Ring conditions of all species in one launch, and enforce_limits of all
species in one launch, at the smallest and at odd sizes, for every pair of
conditions and a mix of storage kinds: the bits are those of the reference's
order (x sides, then y sides) applied species by species."""
import numpy as np
import pytest

from hicar_amd import _lib
from hicar_amd.advection import Advection
from hicar_amd.domain import Domain, Options

pytestmark = pytest.mark.gpu

KINDS = [_lib.STORE_F32, _lib.STORE_BF16, _lib.STORE_F16, _lib.STORE_BF16_SR]


def handle(nx, ny, nz, variant, seed=5):
    r = np.random.default_rng(seed)
    o = Options()
    o.kernel_variant = variant
    d = Domain(nx, ny, nz, 1000.0, halo=1)
    names = [f"s{n}" for n in range(5)]
    o.vars_to_advect = names
    vals = {n: r.normal(0.0, 1.0, d.shape) for n in names}
    vals["s1"].flat[:6] = [-0.0, 0.0, np.nan, np.inf, -np.inf, -1e-30]
    d.set_var_lists(o, vals)
    if variant == 1:
        for n, k in zip(names, KINDS):
            d.storage[n] = (k, 0)
    return d, o, names


@pytest.mark.parametrize("bc_x,bc_y", [(1, 0), (2, 0), (0, 2), (1, 2), (2, 2)])
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 3, 5), (3, 6, 3), (67, 5, 7), (300, 41, 4)])
@pytest.mark.parametrize("variant", [0, 1])
def test_ring_conditions_match_oracle(oracle32, variant, shape, bc_x, bc_y):
    d, o, names = handle(*shape, variant)
    st = Advection(d, o)
    try:
        st.download()  # the stored values (16-bit kinds round)
        ref = {n: d.species[n].copy() for n in names}
        for n in names:
            oracle32.apply_bc(ref[n], bc_x, bc_y)
        st.apply_bc(bc_x, bc_y)
        st.download()
    finally:
        st.close()
    for n in names:
        np.testing.assert_array_equal(d.species[n].view(np.uint32), ref[n].view(np.uint32),
                                      err_msg=n)


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 7, 3), (67, 5, 7), (128, 33, 8)])
@pytest.mark.parametrize("variant", [0, 1])
def test_enforce_limits_of_every_kind(shape, variant):
    d, o, names = handle(*shape, variant, seed=6)
    st = Advection(d, o)
    try:
        st.download()
        with np.errstate(invalid="ignore"):
            ref = {n: np.where(d.species[n] < 0, np.float32(0), d.species[n]) for n in names}
        st.enforce_limits()
        st.download()
    finally:
        st.close()
    for n in names:
        nan = np.isnan(ref[n])
        np.testing.assert_array_equal(np.isnan(d.species[n]), nan, err_msg=n)
        np.testing.assert_array_equal(d.species[n].view(np.uint32)[~nan],
                                      ref[n].view(np.uint32)[~nan], err_msg=n)


@pytest.mark.parametrize("variant", [0, 1])
def test_run_equals_single_steps_after_the_winds_change(variant):
    """run() forms the Courant numbers once; new winds or another dt between
    runs take effect in the next run."""
    from test_gpu_parity import random_domain

    def go(whole):
        case = random_domain(37, 21, 6, 41, 2, True, True, nspec=2)
        case.options.kernel_variant = variant
        d = case.domain
        st = Advection(d, case.options)
        try:
            for n, dt in enumerate((case.dt, case.dt, 0.5 * case.dt)):
                if whole:
                    st.run(dt, 3, 1, 2)
                else:
                    for _ in range(3):
                        st.run(dt, 1, 1, 2)
                d.u[...] *= np.float32(0.9 - 0.1 * n)
                st.upload(fields=True, species=False)
            st.download()
            return {k: a.copy() for k, a in d.species.items()}
        finally:
            st.close()
    a, b = go(True), go(False)
    for n in a:
        np.testing.assert_array_equal(a[n].view(np.uint32), b[n].view(np.uint32), err_msg=n)
