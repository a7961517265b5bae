"""The 3D colour passes that work straight from memory, where they can go
wrong: odd rows without a partner cell, rows and planes that do not fill a
block of threads, two cells along a periodic direction, cells with up to
three walls, both halves of the first (out of place) pass, and the
prolongation before the first pass.  The FP64 forms equal the oracle bit for
bit; the FP32 form ends at the FP64 solution."""
import numpy as np
import pytest

from oracle import mlref as O
from tests import hc_cases as HC
from tests.test_gpu_hc_pairs import _setup
from tests.test_gpu_hc_parity import WALLS

pytestmark = pytest.mark.gpu

SIZES = {
    "odd_walls": dict(n=(13, 15, 17), periodic=[0, 0, 0], bc=WALLS),
    "one_more_than_a_block": dict(n=(130, 9, 3), periodic=[0, 0, 0], bc=WALLS),
    "two_periodic": dict(n=(2, 40, 30), periodic=[1, 1, 1]),
    "flat": dict(n=(40, 2, 26), periodic=[0, 1, 0], bc=WALLS),
    "rows_of_48": dict(n=(48, 20, 12)),
    "periodic": dict(n=(32, 16, 16), periodic=[1, 1, 1]),
}


@pytest.mark.parametrize("name", sorted(SIZES))
@pytest.mark.parametrize("iters,acoef", [(1, True), (3, False)])
def test_hc_passes(ml, gpu_ctx, wl, name, iters, acoef):
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, SIZES[name], acoef)
    phi, rhs = case["phi"].copy(), case["phi"].copy()
    ref = O.hc_gsrb(g, p, bc, 1.0, a, -case["dt"], b, phi.copy(), rhs, iters=iters)
    d = ml.DeviceArray(gpu_ctx, phi.shape, host=phi)
    op.relax(0, d, ml.DeviceArray(gpu_ctx, rhs.shape, host=rhs), iters)
    assert HC.bitwise_equal(HC.valid(case["n"], d.get()), HC.valid(case["n"], ref))
    op.close()


@pytest.mark.parametrize("n,periodic", [((24, 32, 16), [1, 0, 0]), ((48, 16, 24), [0, 0, 0]), ((16, 16, 32), [1, 1, 1])])
@pytest.mark.parametrize("precision", ["fp64", "fp32_refined"])
def test_hc_cycles(ml, gpu_ctx, wl, n, periodic, precision):
    """Solves with prolongation, odd and even numbers of passes per visit."""
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, dict(n=n, periodic=periodic), False)
    old = case["phi"].copy()
    new = old.copy()
    kw = dict(max_iter=4, nu1=1, nu2=2) if precision == "fp64" else dict(max_iter=60, eps=1e-13, hang=-1.0)
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(**kw))
    dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
    prec = ml.PRECISION_FP64 if precision == "fp64" else ml.PRECISION_FP32_REFINED
    st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"],
                     opts=ml.default_opts(precision=prec, **kw))
    out = dn.get()
    if precision == "fp64":
        assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
        assert HC.bitwise_equal(HC.valid(n, out), HC.valid(n, new))
    else:
        # residuals 1e-13 of the first on both sides: the states agree to
        # the 1e-9 stated for the refined form
        for m in range(2):
            assert HC.rel_err(HC.valid(n, out)[m], HC.valid(n, new)[m]) <= 1e-9
    op.close()


@pytest.mark.parametrize("name", sorted(SIZES))
@pytest.mark.parametrize("iters,acoef,ccoef", [(1, False, True), (3, True, False)])
def test_vc_passes(ml, gpu_ctx, name, iters, acoef, ccoef):
    spec = SIZES[name]
    n, per = spec["n"], spec.get("periodic", [1, 0, 0])
    dx = 1.0 / max(n)
    bc = {(d, s, 0): ((d + s) % 2, 0.0) for d in range(3) if not per[d] for s in (0, 1)}
    g = O.make_grid(n, dx, per)
    rng = np.random.default_rng(sum(n))
    b = [rng.uniform(0.5, 1.5, O.face_shape(g, d, 1)) for d in range(3)]
    a = rng.uniform(0.5, 1.5, O.cell_shape(g, 1)) if acoef else None
    c = rng.uniform(0.0, 20.0, O.cell_shape(g, 1)) if ccoef else None
    phi, rhs = np.zeros(O.cell_shape(g, 1)), np.zeros(O.cell_shape(g, 1))
    O.valid(g, phi)[...] = rng.standard_normal(O.valid(g, phi).shape)
    O.valid(g, rhs)[...] = rng.standard_normal(O.valid(g, rhs).shape)
    ref = O.lin_gsrb(g, 1, O.make_bc(bc), 1.0, a, -2e-3, c, b, phi.copy(), rhs, iters=iters)
    op = ml.VCOp(gpu_ctx, list(n), dx, list(per), ml.make_bc(bc))
    dev = lambda x: None if x is None else ml.DeviceArray(gpu_ctx, x.shape, host=x)
    da, db, dc, d = dev(a), [dev(x) for x in b], dev(c), dev(phi)
    op.set_coefs(da, db, dc, 1.0, -2e-3)
    op.relax(0, d, dev(rhs), iters)
    assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, d.get())), np.ascontiguousarray(HC.valid(n, ref)))
    op.close()


@pytest.mark.parametrize("n,per", [((36, 28, 20), (1, 0, 0)), ((26, 22, 34), (0, 0, 0)), ((32, 16, 24), (1, 1, 1))])
@pytest.mark.parametrize("nu1,nu2", [(1, 1), (2, 3)])
def test_vc_cycles(ml, gpu_ctx, n, per, nu1, nu2):
    """Solves: a zero first guess on the way down, the coarse correction
    added in the first pass on the way up, iterations replayed from a graph."""
    dx = 1.0 / max(n)
    bc = {(d, s, 0): (0, 0.0) for d in range(3) if not per[d] for s in (0, 1)}
    g = O.make_grid(n, dx, per)
    rng = np.random.default_rng(sum(n))
    b = [rng.uniform(0.5, 1.5, O.face_shape(g, d, 1)) for d in range(3)]
    rhs = np.zeros(O.cell_shape(g, 1))
    O.valid(g, rhs)[...] = rng.standard_normal(O.valid(g, rhs).shape)
    kw = dict(max_iter=5, nu1=nu1, nu2=nu2, bottom=3, eps=1e-14, hang=1e-14, norm_thresh=1e-14)
    phi = np.zeros(O.cell_shape(g, 1))
    so = O.lin_mg_solve(g, 1, O.make_bc(bc), 1.0, None, -2e-3, None, b, phi, rhs, opts=O.default_opts(**kw))
    op = ml.VCOp(gpu_ctx, list(n), dx, list(per), ml.make_bc(bc))
    dev = lambda x: ml.DeviceArray(gpu_ctx, x.shape, host=x)
    db = [dev(x) for x in b]
    op.set_coefs(None, db, None, 1.0, -2e-3)
    drhs = dev(rhs)
    for _ in range(3):
        dphi = dev(np.zeros_like(phi))
        st = op.solve(dphi, drhs, opts=ml.default_opts(**kw))
        assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
        assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, dphi.get())), np.ascontiguousarray(HC.valid(n, phi)))
    op.close()
