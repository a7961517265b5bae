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


def test_hc_3d_solve(ml, gpu_ctx, wl):
    """A single level of more than 1024 cells: the solve is its bottom's
    relaxations."""
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, GRIDS3["x"], False)
    old = case["phi"].copy()
    new = old.copy()
    kw = dict(max_iter=3, bottom=7)
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(**kw))
    dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
    st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"], opts=ml.default_opts(**kw))
    assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    assert HC.bitwise_equal(HC.valid(case["n"], dn.get()), HC.valid(case["n"], new))
    op.close()
