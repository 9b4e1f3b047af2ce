"""The donor-cell kernel's tiles bit for bit against the FP32 oracle: widths and
heights at the edges of its 62 x 8 tiles, one to nine species (groups of two
and, on a grid that fills the GPU, of four with an uneven last one), chunks of
one level and of several, and operands outside the range
of its fast quotients (tiny and huge values, a divisor out of range).  Both
sides do the same IEEE operations, so the tolerance is zero."""
import numpy as np
import pytest

from hicar_amd.advection import MpdataAdvection
from test_gpu_parity import fresh_species, random_domain

pytestmark = pytest.mark.gpu

SHAPES = [(61, 7, 3, 1), (62, 8, 4, 2), (63, 9, 5, 3), (64, 16, 4, 5), (125, 17, 60, 9),
          (372, 196, 5, 13)]


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("rough", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_donor_cell_tiles_match_oracle(oracle32, shape, order, rough):
    nx, ny, nz, nspec = shape
    case = random_domain(nx, ny, nz, 4000 + nx + 5 * ny + nz, order, True, True, nspec=nspec)
    if rough:
        r = np.random.default_rng(nx + nz)
        for i, n in enumerate(case.domain.species):
            q = case.domain.species[n]
            q[...] *= r.random(q.shape) < 0.6
            q[:, nz // 2:, :] *= np.float32([1e-25, 1e-36, 1e20, 1e30][i % 4])
        case.domain.jacobian[ny // 2, 0, nx // 2] *= np.float32(2.0 ** 40)
    case.steps = 2
    ref = oracle32.run(case.domain, case.options, case.dt, case.steps, 0, 0, fresh_species(case))
    case.options.kernel_variant = 1
    st = MpdataAdvection(case.domain, case.options)
    try:
        st.run(case.dt, case.steps, 0, 0)
        st.download()
    finally:
        st.close()
    for n in ref:
        np.testing.assert_array_equal(case.domain.species[n].view(np.uint32),
                                      ref[n].view(np.uint32), err_msg=n)
