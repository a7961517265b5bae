"""GPU (FP64) parity of the single-workgroup V-cycle of the linear operator
over the kinds of level it holds: odd rows (a thread's two cells may share a
colour), cells with two and more walls, one to five levels, with and without
the a and c coefficients, and BiCGStab bottoms of one wavefront, of two cells
a thread and in between.  The arithmetic and the order of every sum are the
oracle's, so solves agree in every bit."""
import numpy as np
import pytest

from oracle import mlref as O
from tests import hc_cases as HC

pytestmark = pytest.mark.gpu

# n, periodic directions, wall types (Neumann 1, Dirichlet 0 with a value)
LEVELS = {
    "odd_rows_walls": ((31, 20), (0, 0)),
    "thin_walls": ((2, 400), (0, 0)),
    "one_row": ((300, 1), (1, 0)),
    "nine_by_seven": ((9, 7), (0, 0)),
    "deep": ((32, 32), (1, 1)),
    "coarsest_13x5": ((52, 20), (0, 0)),
    "3d_odd_walls": ((9, 7, 5), (0, 0, 0)),
    "3d_column": ((4, 4, 64), (1, 0, 0)),
    "3d_tiled": ((24, 16, 12), (0, 1, 0)),
}


@pytest.mark.parametrize("name", sorted(LEVELS))
@pytest.mark.parametrize("acoef,ccoef,bicgstab", [(False, False, 1), (True, False, 0), (False, True, 1), (True, True, 1)])
def test_single_workgroup_cycles(ml, gpu_ctx, name, acoef, ccoef, bicgstab):
    n, per = LEVELS[name]
    dim = len(n)
    dx = 1.0 / max(n)
    bc = {(d, s, 0): ((d + s) % 2, 0.3 * s) for d in range(dim) if not per[d] for s in (0, 1)}
    g = O.make_grid(n, dx, list(per) + [0] * (3 - dim))
    rng = np.random.default_rng(sum(n))
    b = [np.zeros(O.face_shape(g, d, 1)) for d in range(dim)]
    for f in b:
        f[...] = rng.uniform(0.5, 1.5, f.shape)
    cell = lambda lo, hi: rng.uniform(lo, hi, O.cell_shape(g, 1))
    a = cell(0.5, 1.5) if acoef else None
    c = cell(0.0, 20.0) if ccoef else None
    alpha, beta = 1.0, -2e-3
    rhs = np.zeros(O.cell_shape(g, 1))
    O.valid(g, rhs)[...] = rng.standard_normal(O.valid(g, rhs).shape)
    kw = dict(max_iter=3, nu1=1, nu2=3, bottom=2, eps=1e-14, hang=1e-14, norm_thresh=1e-14, bottom_solver=bicgstab,
              bottom_max_iter=12)
    phi = np.zeros(O.cell_shape(g, 1))
    so = O.lin_mg_solve(g, 1, O.make_bc(bc), alpha, a, beta, c, b, phi, rhs, opts=O.default_opts(**kw))
    op = ml.VCOp(gpu_ctx, list(n), dx, list(per), ml.make_bc(bc))
    dev = lambda x: None if x is None else ml.DeviceArray(gpu_ctx, x.shape, host=x)
    db, da, dc = [dev(x) for x in b], dev(a), dev(c)
    op.set_coefs(da, db, dc, alpha, beta)
    dphi = dev(np.zeros_like(phi))
    st = op.solve(dphi, dev(rhs), opts=ml.default_opts(**kw))
    assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, dphi.get())), np.ascontiguousarray(HC.valid(n, phi)))
    op.close()


@pytest.mark.parametrize("n", [(1024, 128), (1024, 132), (1056, 128), (40, 4360), (1504, 776)])
def test_residual_norms_of_many_workgroups(ml, gpu_ctx, n):
    """The stopping rule sees the largest residual of every workgroup: grids
    of 512 workgroups (which report one by one), just above (in groups of
    unequal size) and several thousand, the largest value in the first, a
    middle and the last workgroup, solve after solve on one operator."""
    dx = 1.0 / n[0]
    g = O.make_grid(n, dx, [1, 0, 0])
    b = [np.ones(O.face_shape(g, d, 1)) for d in range(2)]
    bc = {(1, s, 0): (0, 0.0) for s in (0, 1)}
    op = ml.VCOp(gpu_ctx, list(n), dx, [1, 0], ml.make_bc(bc))
    dev = lambda x: ml.DeviceArray(gpu_ctx, x.shape, host=x)
    db = [dev(x) for x in b]
    op.set_coefs(None, db, None, 1.0, -1e-7)
    kw = dict(max_iter=2, nu1=1, nu2=1, bottom=2, eps=1e-15, hang=1e-15, norm_thresh=1e-15)
    rng = np.random.default_rng(n[1])
    for spot in ((0, 0), (n[0] // 2, n[1] // 2), (n[0] - 1, n[1] - 1)):
        rhs = np.zeros(O.cell_shape(g, 1))
        v = O.valid(g, rhs)
        v[...] = 1e-3 * rng.standard_normal(v.shape)
        v[(0,) * (v.ndim - 2) + spot[::-1]] = 7.0
        phi = np.zeros(O.cell_shape(g, 1))
        so = O.lin_mg_solve(g, 1, O.make_bc(bc), 1.0, None, -1e-7, None, b, phi, rhs, opts=O.default_opts(**kw))
        dphi = dev(np.zeros_like(phi))
        st = op.solve(dphi, dev(rhs), opts=ml.default_opts(**kw))
        assert st.initial_residual == so.initial_residual == 7.0
        assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    op.close()


def test_replayed_solves_follow_the_coefficients(ml, gpu_ctx):
    """Solves of one operator on the same arrays replay their iterations, and a
    batch keeps its tables; the a and c terms may come and go between them with
    alpha and beta as before."""
    n, per = (64, 48), (1, 0)
    dx = 1.0 / n[0]
    bc = {(1, s, 0): (0, 0.0) for s in (0, 1)}
    g = O.make_grid(n, dx, list(per) + [0])
    rng = np.random.default_rng(8)
    b = [rng.uniform(0.5, 1.5, O.face_shape(g, d, 1)) for d in range(2)]
    a, c = rng.uniform(0.5, 1.5, O.cell_shape(g, 1)), rng.uniform(0.0, 20.0, O.cell_shape(g, 1))
    rhs = np.zeros(O.cell_shape(g, 1))
    O.valid(g, rhs)[...] = rng.standard_normal(O.valid(g, rhs).shape)
    kw = dict(max_iter=4, nu1=1, nu2=2, bottom=3, eps=1e-14, hang=1e-14, norm_thresh=1e-14)
    op = ml.VCOp(gpu_ctx, list(n), dx, list(per), ml.make_bc(bc))
    dev = lambda x: None if x is None else ml.DeviceArray(gpu_ctx, x.shape, host=x)
    db, drhs, dphi = [dev(x) for x in b], dev(rhs), dev(np.zeros_like(rhs))
    batch = ml.VCBatch(gpu_ctx, [op])
    for ac, cc in ((None, None), (None, c), (a, c), (a, None), (None, None)):
        phi = np.zeros_like(rhs)
        so = O.lin_mg_solve(g, 1, O.make_bc(bc), 1.0, ac, -2e-3, cc, b, phi, rhs, opts=O.default_opts(**kw))
        op.set_coefs(dev(ac), db, dev(cc), 1.0, -2e-3)
        for solve in (op.solve, lambda p, r, opts: batch.solve([p], [r], opts)[0]):
            dphi.set(np.zeros_like(rhs))
            st = solve(dphi, drhs, opts=ml.default_opts(**kw))
            assert (st.iterations, st.exit_status) == (so.iterations, so.exit_status)
            assert st.final_residual == so.final_residual
            assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, dphi.get())), np.ascontiguousarray(HC.valid(n, phi)))
    batch.close()
    op.close()
