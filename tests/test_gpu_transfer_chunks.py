"""How a host transfer is cut into chunks: arrays that share one, arrays of a
chunk each and arrays cut into several, with FP32 and 16-bit species
interleaved (these pass through one conversion buffer).  What comes back is
what went up, rounded to the species' storage; the conversions round to
nearest even on both sides, so the comparison is exact."""
import numpy as np
import pytest

from hicar_amd import _lib
from hicar_amd.advection import MpdataAdvection
from hicar_amd.domain import Domain, Options

pytestmark = pytest.mark.gpu


def rounded(a, storage, pow2):
    if storage == _lib.STORE_F32:
        return a
    x = a * np.float32(2.0 ** -pow2)
    if storage == _lib.STORE_F16:
        x = x.astype(np.float16).astype(np.float32)
    else:  # the upper half of the bits, to nearest even
        u = x.view(np.uint32)
        x = ((u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).astype(np.uint32).view(np.float32)
    return x * np.float32(2.0 ** pow2)


@pytest.mark.parametrize("shape,nspec", [((160, 100, 10), 14), ((257, 129, 40), 4), ((601, 203, 40), 3)],
                         ids=["shared", "whole", "cut"])
def test_interleaved_storage_round_trip(shape, nspec):
    nx, ny, nz = shape
    r = np.random.default_rng(nx)
    d, o = Domain(nx, ny, nz, 1000.0), Options()
    for n in d.FIELDS:
        getattr(d, n)[...] = r.uniform(0.5, 1.5, getattr(d, n).shape)
    names = [f"s{i}" for i in range(nspec)]
    o.vars_to_advect = names
    d.set_var_lists(o, {n: r.uniform(0.0, 2.0, d.shape) for n in names})
    kinds = (_lib.STORE_F32, _lib.STORE_BF16, _lib.STORE_F16)
    for i, n in enumerate(names):
        d.storage[n] = (kinds[i % 3], -2 if i % 3 else 0)
    o.kernel_variant = 1
    st = MpdataAdvection(d, o)
    try:
        for turn in range(2):
            want = {n: rounded(d.species[n], *d.storage[n]) for n in names}
            fields = {n: getattr(d, n).copy() for n in d.FIELDS}
            st.upload(fields=True, species=True)
            for n in names:
                d.species[n][...] = -1.0
            for n in d.FIELDS:
                getattr(d, n)[...] = -1.0
            st.download(species=True, fields=True)
            for n in names:
                np.testing.assert_array_equal(d.species[n], want[n], err_msg=n)
            for n in d.FIELDS:
                np.testing.assert_array_equal(getattr(d, n), fields[n], err_msg=n)
            for n in names:
                d.species[n][...] = r.uniform(0.0, 2.0, d.shape)
    finally:
        st.close()
