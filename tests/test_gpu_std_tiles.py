"""The standard scheme's column marches at the edges of their tiles and of
their quotients' range, bit for bit against the FP32 oracle (zero tolerance:
both sides do the same IEEE operations).  A stage updates 63 columns by 8 or
16 rows per block, the limiter 61 by 5 or 13 (one or two rows per wave, by the
size of the launch), and columns are cut into chunks.  The quotients' fast
form holds for numerators of at least 2^-96 and winds of at least 2^-100, so
the species reach far below that in some columns, zeros next to them, and one
case has winds under the bound (the general form throughout).  Infinities and
NaN must spread as the reference spreads them."""
import numpy as np
import pytest

from hicar_amd import synthetic
from hicar_amd.advection import Advection

pytestmark = pytest.mark.gpu

# tile width, height, levels, species: the last two are large enough for two
# rows per wave in the limiter, or in both kernels
TILES = [(61, 5, 4, 2), (62, 6, 9, 1), (63, 8, 3, 2), (64, 9, 6, 2), (122, 13, 13, 1),
         (127, 17, 5, 1), (190, 65, 5, 16), (367, 105, 3, 16)]
ORDERS = [(5, 3, 1, True), (3, 5, 1, False), (5, 5, 0, True)]


def tile_case(tile, h, v, fc, rk3):
    wi, hj, nz, ns = tile
    if v == 5:
        nz = max(nz, 4)

    def make(nx, ny, nlev):
        return synthetic.config_std(nx=nx, ny=ny, nz=nlev, steps=1, h_order=h, v_order=v,
                                    flux_corr=fc, rk3=rk3, cfl=1.0 if rk3 else 0.4)
    halo = make(16, 16, 4).domain.halo
    case = make(wi + 2 * halo, hj + 2 * halo, nz)
    d, o = case.domain, case.options
    assert (d.ite - d.its + 1, d.jte - d.jts + 1) == (wi, hj)
    r = np.random.default_rng(wi + hj + nz)
    o.vars_to_advect = [f"s{n}" for n in range(ns)]
    vals = {}
    for n, name in enumerate(o.vars_to_advect):
        q = r.lognormal(-9, 1.5, d.shape) * (r.random(d.shape) > 0.4)
        if n % 2 == 0:  # some columns far below the range and below FP32's normal numbers
            q[:, :, d.nx // 3:d.nx // 2] *= 1e-30
            q[: d.ny // 2, :, : d.nx // 4] *= 1e-38
        vals[name] = q
    d.set_var_lists(o, vals)
    return case


def check(oracle32, case):
    d = case.domain
    ref = oracle32.std_advect(d, case.options, case.dt, {n: a.copy() for n, a in d.species.items()})
    st = Advection(d, case.options)
    try:
        st.advect(case.dt)
        st.download()
    finally:
        st.close()
    for n in ref:
        nan = np.isnan(ref[n])
        np.testing.assert_array_equal(np.isnan(d.species[n]), nan, err_msg=n)
        np.testing.assert_array_equal(d.species[n].view(np.uint32)[~nan],
                                      ref[n].view(np.uint32)[~nan], err_msg=n)


@pytest.mark.parametrize("h,v,fc,rk3", ORDERS)
@pytest.mark.parametrize("tile", TILES, ids=lambda t: "x".join(map(str, t)))
def test_std_tiles_and_ranges_match_oracle(oracle32, tile, h, v, fc, rk3):
    check(oracle32, tile_case(tile, h, v, fc, rk3))


@pytest.mark.parametrize("h,v,fc,rk3", ORDERS)
def test_std_winds_below_the_range_match_oracle(oracle32, h, v, fc, rk3):
    case = tile_case((70, 20, 5, 2), h, v, fc, rk3)
    case.domain.v[...] *= np.float32(1e-36)
    check(oracle32, case)


@pytest.mark.parametrize("h,v,fc,rk3", ORDERS)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_std_infinities_and_nan_spread_like_the_oracle(oracle32, value, h, v, fc, rk3):
    case = tile_case((70, 20, 8, 2), h, v, fc, rk3)
    d = case.domain
    d.species["s0"][d.ny // 2, 3, d.nx // 2] = value
    d.species["s1"][6, 0, 30] = value
    check(oracle32, case)
