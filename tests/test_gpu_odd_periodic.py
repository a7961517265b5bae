"""Relaxation with an odd periodic length: the two cells at its seam share a
colour, and each sees the other as of the start of the pass.  Levels of more
than 1024 cells (smaller ones are refused), each direction odd in turn and
several at once; every value is the CPU oracle's, bit for bit."""
import numpy as np
import pytest

from oracle import mlref as O
from tests import hc_cases as HC
from tests.test_gpu_hc_pairs import _setup
from tests.test_gpu_hc_parity import WALLS

pytestmark = pytest.mark.gpu

GRIDS3 = {
    "x": dict(n=(33, 20, 12), periodic=[1, 0, 0], bc=WALLS),
    "y": dict(n=(20, 33, 12), periodic=[1, 1, 0], bc=WALLS),
    "z": dict(n=(12, 20, 33), periodic=[0, 0, 1], bc=WALLS),
    "all": dict(n=(15, 13, 11), periodic=[1, 1, 1]),
    "one_cell": dict(n=(40, 1, 30), periodic=[1, 1, 0], bc=WALLS),
    "rows_beyond_a_block": dict(n=(131, 9, 3), periodic=[1, 0, 1], bc=WALLS),
}

# above 512^2 cells rows stream in blocks of 252 columns: the seam inside a
# block, one cell into the last one, at the march's end (tiles instead)
STREAMS2 = {
    "x": dict(n=(1031, 520), periodic=[1, 0], bc=WALLS),
    "x_last_block_of_one": dict(n=(757, 400), periodic=[1, 1]),
    "y": dict(n=(600, 601), periodic=[0, 1], bc=WALLS),
    "both": dict(n=(1031, 517), periodic=[1, 1]),
}

# regions of 32 positions: the seam at even and odd places of a region, in the
# halo of one core and inside the next, rows hardly wider than core and halo,
# several seams in a region (rows below 18 cells in a sweep, 24 in four)
PAIRS2 = {
    "%dx%d_%d%d" % (n + tuple(per)): dict(n=n, periodic=per, bc=None if per[1] else WALLS)
    for n, per in [((33, 40), [1, 0]), ((59, 30), [1, 0]), ((81, 64), [1, 0]), ((85, 33), [1, 1]), ((129, 47), [1, 1]),
                   ((64, 35), [1, 1]), ((48, 53), [0, 1]), ((31, 66), [1, 0]), ((29, 47), [1, 1]), ((25, 48), [1, 0]),
                   ((23, 90), [1, 0]), ((17, 80), [1, 0]), ((7, 200), [1, 1]), ((200, 9), [1, 1])]
}


def _hc_relax(ml, ctx, wl, spec, iters, acoef, how="relax"):
    case, g, p, bc, b, a, op = _setup(ml, ctx, wl, spec, acoef)
    phi, rhs = case["phi"].copy(), case["phi"].copy()
    ref = O.hc_gsrb(g, p, bc, 1.0, a, -case["dt"], b, phi.copy(), rhs, iters=iters)
    d = ml.DeviceArray(ctx, phi.shape, host=phi)
    getattr(op, how)(0, d, ml.DeviceArray(ctx, rhs.shape, host=rhs), iters)
    assert HC.bitwise_equal(HC.valid(case["n"], d.get()), HC.valid(case["n"], ref))
    op.close()


@pytest.mark.parametrize("name", sorted(GRIDS3))
@pytest.mark.parametrize("iters,acoef", [(1, True), (4, False)])
def test_hc_3d(ml, gpu_ctx, wl, name, iters, acoef):
    _hc_relax(ml, gpu_ctx, wl, GRIDS3[name], iters, acoef)


@pytest.mark.parametrize("spec", [GRIDS3["x"], PAIRS2["129x47_11"], STREAMS2["x"]], ids=["3d", "pairs", "streams"])
def test_hc_solve(ml, gpu_ctx, wl, spec):
    """A single level of more than 1024 cells: the solve is its bottom's
    relaxations."""
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, spec, False)
    old = case["phi"].copy()
    new = old.copy()
    kw = dict(max_iter=3, bottom=7)
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(**kw))
    dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
    st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"], opts=ml.default_opts(**kw))
    assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    assert HC.bitwise_equal(HC.valid(case["n"], dn.get()), HC.valid(case["n"], new))
    op.close()


@pytest.mark.parametrize("spec", [GRIDS3["all"], PAIRS2["59x30_10"]], ids=["3d", "pairs"])
def test_hc_without_allocation(ml, gpu_ctx, wl, spec):
    for iters in (1, 2, 5):
        _hc_relax(ml, gpu_ctx, wl, spec, iters, False, "relax_noalloc")


@pytest.mark.parametrize("name", sorted(PAIRS2))
@pytest.mark.parametrize("iters,acoef", [(1, True), (2, False), (4, True), (5, False)])
def test_hc_2d_pairs(ml, gpu_ctx, wl, name, iters, acoef):
    _hc_relax(ml, gpu_ctx, wl, PAIRS2[name], iters, acoef)


@pytest.mark.parametrize("name", sorted(STREAMS2))
@pytest.mark.parametrize("iters,acoef", [(1, True), (3, False)])
def test_hc_2d_streams(ml, gpu_ctx, wl, name, iters, acoef):
    _hc_relax(ml, gpu_ctx, wl, STREAMS2[name], iters, acoef)


def _vc_case(ml, ctx, spec, acoef, ccoef):
    n = spec["n"]
    dim, per = len(n), spec.get("periodic", [1] + [0] * (len(n) - 1))
    dx = 1.0 / max(n)
    bc = {(d, s, 0): ((d + s) % 2, 0.0) for d in range(dim) if not per[d] for s in (0, 1)}
    g = O.make_grid(n, dx, list(per) + [0] * (3 - dim))
    rng = np.random.default_rng(sum(n))
    b = [rng.uniform(0.5, 1.5, O.face_shape(g, d, 1)) for d in range(dim)]
    a = rng.uniform(0.5, 1.5, O.cell_shape(g, 1)) if acoef else None
    c = rng.uniform(0.0, 20.0, O.cell_shape(g, 1)) if ccoef else None
    phi, rhs = np.zeros(O.cell_shape(g, 1)), np.zeros(O.cell_shape(g, 1))
    O.valid(g, phi)[...] = rng.standard_normal(O.valid(g, phi).shape)
    O.valid(g, rhs)[...] = rng.standard_normal(O.valid(g, rhs).shape)
    op = ml.VCOp(ctx, list(n), dx, list(per), ml.make_bc(bc))
    dev = lambda x: None if x is None else ml.DeviceArray(ctx, x.shape, host=x)
    op.set_coefs(dev(a), [dev(x) for x in b], dev(c), 1.0, -2e-3)
    return n, g, O.make_bc(bc), a, b, c, phi, rhs, op, dev


def _vc_relax(ml, ctx, spec, iters, acoef, ccoef):
    n, g, bc, a, b, c, phi, rhs, op, dev = _vc_case(ml, ctx, spec, acoef, ccoef)
    ref = O.lin_gsrb(g, 1, bc, 1.0, a, -2e-3, c, b, phi.copy(), rhs, iters=iters)
    d = dev(phi)
    op.relax(0, d, dev(rhs), iters)
    assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, d.get())), np.ascontiguousarray(HC.valid(n, ref)))
    op.close()


def _vc_solve(ml, ctx, spec):
    """A single level of more than 1024 cells, iterations replayed from a
    graph: the solve is its bottom's relaxations."""
    n, g, bc, a, b, c, phi, rhs, op, dev = _vc_case(ml, ctx, spec, False, True)
    kw = dict(max_iter=5, bottom=7, eps=1e-14, hang=1e-14, norm_thresh=1e-14)
    new = np.zeros_like(phi)
    so = O.lin_mg_solve(g, 1, bc, 1.0, None, -2e-3, c, b, new, rhs, opts=O.default_opts(**kw))
    drhs = dev(rhs)
    for _ in range(2):
        d = dev(np.zeros_like(phi))
        st = op.solve(d, drhs, opts=ml.default_opts(**kw))
        assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
        assert HC.bitwise_equal(np.ascontiguousarray(HC.valid(n, d.get())), np.ascontiguousarray(HC.valid(n, new)))
    op.close()


@pytest.mark.parametrize("name", sorted(GRIDS3))
@pytest.mark.parametrize("iters,acoef,ccoef", [(1, False, True), (4, True, False)])
def test_vc_3d(ml, gpu_ctx, name, iters, acoef, ccoef):
    _vc_relax(ml, gpu_ctx, GRIDS3[name], iters, acoef, ccoef)


def test_vc_3d_solve(ml, gpu_ctx):
    _vc_solve(ml, gpu_ctx, GRIDS3["y"])


TILES2 = {
    "x": dict(n=(45, 44), periodic=[1, 0], bc=WALLS),
    "y": dict(n=(44, 45), periodic=[0, 1], bc=WALLS),
    "both": dict(n=(67, 35), periodic=[1, 1]),
    "short": dict(n=(3, 400), periodic=[1, 0], bc=WALLS),
}


@pytest.mark.parametrize("name", sorted(TILES2))
@pytest.mark.parametrize("iters,acoef,ccoef", [(1, False, True), (6, True, False)])
def test_vc_2d_tiles(ml, gpu_ctx, name, iters, acoef, ccoef):
    _vc_relax(ml, gpu_ctx, TILES2[name], iters, acoef, ccoef)


@pytest.mark.parametrize("name", sorted(STREAMS2))
@pytest.mark.parametrize("iters,acoef,ccoef", [(1, False, True), (3, True, False)])
def test_vc_2d_streams(ml, gpu_ctx, name, iters, acoef, ccoef):
    _vc_relax(ml, gpu_ctx, STREAMS2[name], iters, acoef, ccoef)


@pytest.mark.parametrize("spec", [TILES2["both"], STREAMS2["x"]], ids=["tiles", "streams"])
def test_vc_2d_solve(ml, gpu_ctx, spec):
    _vc_solve(ml, gpu_ctx, spec)
