"""A NaN or an infinity in the base state reaches the second RK3 stage further
than it reaches the base state's upwind fluxes, and through faces without a
quotient (first order, and the faces next to the ground and the top).  The
limiter must spread it as the reference does, bit for bit (the same IEEE
operations and the Fortran's selects on both sides): at several levels, in the
middle of a tile and in the cells on both sides of a tile's edge."""
import numpy as np
import pytest

from test_gpu_std_tiles import check, tile_case

pytestmark = pytest.mark.gpu

NZ = 12


@pytest.mark.parametrize("h,v", [(1, 1), (1, 3), (5, 1), (5, 3), (3, 5)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("level", [0, 2, 4, 5, 8, NZ - 1])
def test_limiter_spreads_what_is_no_number(oracle32, level, value, h, v):
    case = tile_case((70, 20, NZ, 3), h, v, 1, True)
    d = case.domain
    halo = d.its - d.ims
    # two columns east and rows north of the first tile (61 columns, 5 or 13 rows)
    d.species["s0"][halo + 13, level, halo + 61] = value
    d.species["s1"][halo + 4, level, halo + 60] = value
    d.species["s2"][d.ny // 2, level, d.nx // 2] = value
    check(oracle32, case)
