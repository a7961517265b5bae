"""The adjoint solve's fused vector steps: the block diagonal (no sweeps, and
odd periodic lengths) and one to three half-fused sweeps lead to the same
gradient, on grids of one and of many workgroups and of odd sizes; a zero
right-hand side ends before the first iteration."""
import numpy as np
import pytest

from tests import hc_cases as HC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,periodic", [((8, 6), [1, 0]), ((33, 31), [0, 0]), ((31, 40), [1, 0]), ((130, 66), [1, 0]),
                                        ((600, 512), [1, 0])])
def test_sweeps_agree(ml, gpu_ctx, wl, n, periodic):
    case = wl.heat_flux(n=n, steps=1, seed=4)
    case["periodic"] = periodic
    op = HC.gpu_setup(ml, gpu_ctx, case)
    rng = np.random.default_rng(n[0])
    dev = lambda x: ml.DeviceArray(gpu_ctx, x.shape, host=x)
    old = case["phi"].copy()
    new = old + 1e-3 * rng.standard_normal(old.shape)
    g = rng.standard_normal(old.shape)
    dt = case["dt"]
    dold, dnew, dg = dev(old), dev(new), dev(g)
    ref = None
    for nu1 in (0, 1, 3):
        out = dev(np.zeros_like(old))
        gst, st = op.adjoint_step(dnew, dold, dt, dg, out, opts=ml.default_opts(eps=1e-13, max_iter=2000, nu1=nu1))
        assert st.exit_status == 1, (nu1, st.exit_status)
        o = HC.valid(n, out.get())
        if ref is None:
            ref = (o, gst)
            continue
        # residuals of 1e-13 |g|; J^T = 1 + positive terms is no worse
        # conditioned than 1e4 at these time steps
        assert np.max(np.abs(o - ref[0])) <= 1e-9 * np.max(np.abs(ref[0]))
        assert abs(gst - ref[1]) <= 1e-9 * max(abs(ref[1]), 1.0)
    zero = dev(np.zeros_like(old))
    out = dev(np.ones_like(old))
    gst, st = op.adjoint_step(dnew, dold, dt, zero, out, opts=ml.default_opts(eps=1e-13, max_iter=5, nu1=1))
    assert (st.exit_status, st.iterations, gst) == (8, 0, 0.0)
    assert np.all(HC.valid(n, out.get()) == 0.0)
    op.close()
