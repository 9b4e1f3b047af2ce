"""The wind balance, the time-step bound and the lateral forcing bit for bit
against the FP32 oracle where their kernels' loops end: rows of whole and
ragged waves of 64 columns, columns of whole and ragged batches of four
levels, and a balance that reaches the domain's edge.  The same operations on
both sides (maxima do not depend on the order), so the tolerance is zero."""
import numpy as np
import pytest

from hicar_amd import synthetic
from hicar_amd.advection import MpdataAdvection
from test_gpu_dyn import cols, windy_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("adv", [True, False])
@pytest.mark.parametrize("halo", [1, 2])
@pytest.mark.parametrize("shape", [(16, 9, 3), (64, 12, 4), (65, 21, 5), (128, 8, 8), (257, 30, 9)],
                         ids=lambda s: "x".join(map(str, s)))
def test_dynamics_at_loop_ends(oracle32, shape, halo, adv):
    nx, ny, nz = shape
    case = windy_case(31 + nx, nx=nx, ny=ny, nz=nz)
    d, o = case.domain, case.options
    d.halo = halo
    d.its, d.ite = d.ims + halo, d.ime - halo
    d.jts, d.jte = d.jms + halo, d.jme - halo
    o.parameters.advect_density = adv
    o.kernel_variant = 1
    dzl = synthetic.dz_levels(nz).astype(np.float32)
    w_ref = oracle32.balance_w(d, adv, *cols(d))
    r = np.random.default_rng(nx + nz)
    q = d.species["qv"]
    q[...] = r.uniform(0.5, 2.0, d.shape)
    fhi = r.uniform(0.5, 2.0, d.shape).astype(np.float32)
    tend = r.uniform(-1e-4, 1e-4, d.shape).astype(np.float32)
    filt = oracle32.relax_filter(nx, ny, halo, 1, 1, 1, 1)
    q_ref, _ = oracle32.apply_forcing(q.copy(), fhi, tend, filt, 37.5)
    st = MpdataAdvection(d, o)
    try:
        st.balance_w()
        st.download(species=False, fields=True)
        np.testing.assert_array_equal(d.w.view(np.uint32), w_ref.view(np.uint32))
        tile = (d.its - d.ims, d.ite - d.ims, d.jts - d.jms, d.jte - d.jms)
        ref = np.float32(oracle32.compute_dt(d, dzl, 0.9, 3, *tile))
        assert ref >= 0.1 and np.float32(st.compute_dt(0.9, 3, dzl)) == ref
        st.set_relax_filter(1, 1, 1, 1, halo=halo)
        st.set_forcing("qv", fhi, tend)
        st.apply_forcing(37.5)
        st.download()
    finally:
        st.close()
    np.testing.assert_array_equal(d.species["qv"].view(np.uint32), q_ref.view(np.uint32))
