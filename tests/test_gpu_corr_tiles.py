"""The corrective kernel's two tile heights and its choice of quotient, bit for
bit against the FP32 oracle: grids whose height and width lie at the edges of
the 60x16 and 60x8 tiles, whole and chunked columns, and species whose values
lie inside the ranges the fast quotient is taken in, at their ends, outside
them in some levels and columns only, and below FP32's normal range.  Both
sides do the same IEEE operations, so the tolerance is zero."""
import numpy as np
import pytest

from hicar_amd.advection import MpdataAdvection
from test_gpu_parity import fresh_species, random_domain

pytestmark = pytest.mark.gpu

SHAPES = [(61, 7, 4, 1), (60, 8, 3, 1), (63, 9, 9, 2), (122, 17, 13, 3), (59, 25, 8, 1),
          (185, 40, 9, 2)]  # the last has tiles and levels away from every edge


def spread(case, seed):
    """Species 0 ordinary with zeros; 1 tiny in the upper levels and in one
    corner (the levels below stay in range); 2 large, with isolated values
    beyond the range's top; 3 next to the ends of both ranges."""
    r = np.random.default_rng(seed)
    q = [case.domain.species[n] for n in case.domain.species]
    shape = q[0].shape
    q[0][...] *= (r.random(shape) < 0.7)
    q[1][...] *= 1e-4
    q[1][:, shape[1] // 2:, :] *= np.float32(1e-25)
    q[1][:4, :, :5] *= np.float32(1e-38)
    q[2][...] *= np.float32(1e9)
    q[2][r.random(shape) < 0.002] = np.float32(3e10)
    ends = np.array([2.0 ** -76, 2.0 ** -75, 16.0, 15.9, 2.0 ** -46, 1e-20, 0.0], np.float32)
    q[3][...] = ends[r.integers(0, len(ends), shape)]


@pytest.mark.parametrize("cfg", [3, 6, 7])
@pytest.mark.parametrize("order,fct", [(2, True), (3, True), (2, False)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_corrective_tiles_and_ranges_match_oracle(oracle32, monkeypatch, shape, order, fct, cfg):
    nx, ny, nz, ksplit = shape
    case = random_domain(nx, ny, nz, 9000 + nx + 7 * ny + nz, order, fct, True, nspec=4)
    spread(case, nx * ny + nz)
    ref = oracle32.run(case.domain, case.options, case.dt, case.steps, 0, 0, fresh_species(case))
    monkeypatch.setenv("ICAR_ADV_CORR_CFG", str(cfg))
    monkeypatch.setenv("ICAR_ADV_KSPLIT", str(ksplit))
    case.options.kernel_variant = 1
    st = MpdataAdvection(case.domain, case.options)
    try:
        st.run(case.dt, case.steps, 0, 0)
        st.download()
        assert st.launch_config()[0] == cfg
    finally:
        st.close()
    for n in ref:
        np.testing.assert_array_equal(case.domain.species[n].view(np.uint32),
                                      ref[n].view(np.uint32), err_msg=n)
