"""The 2D (H, Theta) relaxation over 32x32 regions (one cell of each colour
per thread), its fused forms on the way down and up of a FAS cycle, and the
closure's prepared products, at the places where they can go wrong: region
and tile edges, periodic lengths below a region and odd ones (the cells at
the seam share a colour), pairs across the seam and beside walls, pass
counts that split into several launches, states at the regime boundaries.
Every value is the CPU oracle's, bit for bit."""
import numpy as np
import pytest

from oracle import mlref as O
from tests import hc_cases as HC
from tests.test_gpu_hc_parity import WALLS, _case, _mixed_state

pytestmark = pytest.mark.gpu

SIZES = {
    "one_region_walls": dict(n=(33, 32), periodic=[0, 0], bc=WALLS),
    "odd_walls": dict(n=(61, 47), periodic=[0, 0], bc=WALLS),
    "odd_periodic_x": dict(n=(45, 44)),
    "odd_periodic_both": dict(n=(67, 35), periodic=[1, 1]),
    "short_periodic_x": dict(n=(6, 200)),
    "short_periodic_y": dict(n=(180, 10), periodic=[0, 1], bc=WALLS),
    "periodic_32": dict(n=(32, 40), periodic=[1, 1]),
    "no_derived_bc": dict(n=(59, 40), periodic=[0, 0], apply_bc=0),
}


def _setup(ml, ctx, wl, spec, acoef):
    case = _case(wl, **spec)
    case["phi"] = _mixed_state(case, 17)
    g, p, bc = HC.oracle_setup(case)
    b = HC.bcoef_from_state(case)
    op = HC.gpu_setup(ml, ctx, case)
    a = None
    if acoef:
        a = np.ones_like(case["phi"])
        HC.valid(case["n"], a)[:] = 1.0 + 0.3 * np.random.default_rng(5).random(HC.valid(case["n"], a).shape)
    op.set_coefs(ml.DeviceArray(ctx, a.shape, host=a) if acoef else None,
                 [ml.DeviceArray(ctx, x.shape, host=x) for x in b], 1.0, -case["dt"])
    return case, g, p, bc, b, a, op


@pytest.mark.parametrize("name", sorted(SIZES))
@pytest.mark.parametrize("iters,acoef", [(1, False), (3, True), (5, False)])
def test_relax_regions(ml, gpu_ctx, wl, name, iters, acoef):
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, SIZES[name], acoef)
    phi, rhs = case["phi"].copy(), case["phi"].copy()
    ref = O.hc_gsrb(g, p, bc, 1.0, a, -case["dt"], b, phi.copy(), rhs, iters=iters)
    d = ml.DeviceArray(gpu_ctx, phi.shape, host=phi)
    op.relax(0, d, ml.DeviceArray(gpu_ctx, rhs.shape, host=rhs), iters)
    out = d.get()
    assert HC.bitwise_equal(HC.valid(case["n"], out), HC.valid(case["n"], ref))
    op.close()


@pytest.mark.parametrize("n,periodic", [((104, 72), [1, 0]), ((64, 48), [0, 0]), ((8, 256), [1, 1]),
                                        ((36, 36), [0, 0]), ((44, 52), [1, 0])])
@pytest.mark.parametrize("nu1,nu2", [(1, 4), (2, 1), (5, 6)])
def test_fused_cycles(ml, gpu_ctx, wl, n, periodic, nu1, nu2):
    """Whole solves whose levels run the fused launches: halo 3 and 5 on the
    way down, 9 on the way up, and smoothing counts that need two launches."""
    spec = dict(n=n, periodic=periodic, bc=WALLS if periodic == [0, 0] else None)
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, spec, n == (64, 48))
    old = case["phi"].copy()
    new = old.copy()
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(max_iter=4, nu1=nu1, nu2=nu2))
    dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
    st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"],
                     opts=ml.default_opts(max_iter=4, nu1=nu1, nu2=nu2))
    out = dn.get()
    assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    assert HC.bitwise_equal(HC.valid(n, out), HC.valid(n, new))
    op.close()


@pytest.mark.parametrize("n", [(308, 308), (352, 352), (512, 512), (320, 800)])
@pytest.mark.parametrize("nu2", [4, 2])
def test_fused_cycles_of_many_workgroups(ml, gpu_ctx, wl, n, nu2):
    """The last launch of a cycle takes the residual norm and applies the
    stopping rule: above 512 workgroups (cores of 14 or 22 cells) they report
    in groups, numbered over both directions of the grid."""
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, dict(n=n), False)
    old = case["phi"].copy()
    new = old.copy()
    kw = dict(max_iter=3, nu2=nu2)
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(**kw))
    for _ in range(2):
        dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
        st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"], opts=ml.default_opts(**kw))
        assert (st.iterations, st.exit_status) == (so.iterations, so.exit_status)
        assert (st.initial_residual, st.final_residual) == (so.initial_residual, so.final_residual)
        assert HC.bitwise_equal(HC.valid(n, dn.get()), HC.valid(n, new))
    op.close()


PARAMS = {
    "default": {},
    "heat_ratio": dict(specificHeatRatio=1.7, thetaEutectic=0.2, ThetaEutectic=0.1, waterDistributionCoeff=0.1),
    "heat_ratio_low": dict(specificHeatRatio=0.4, thetaEutectic=-0.3, compositionRatio=12.5),
    "no_latent_heat": dict(stefan=0.0),
    "negative_partition": dict(waterDistributionCoeff=-1e-3),
    "tiny": dict(stefan=1e-40, compositionRatio=3.0),
}


@pytest.mark.parametrize("name", sorted(PARAMS))
def test_closure_at_regime_edges(ml, gpu_ctx, wl, name):
    """Enthalpies on the eutectic and liquidus energies, a few units in the
    last place beside them and within the products' margin, concentrations at
    -CR, infinities and NaN: the closure equals the oracle's."""
    n = (256, 250)
    case = _case(wl, n=n)
    case["params"].update(PARAMS[name])
    q = dict(stefan=5.0, compositionRatio=2.0, waterDistributionCoeff=1e-5, specificHeatRatio=1.0, thetaEutectic=0.0,
             ThetaEutectic=0.0)
    q.update(case["params"])
    St, CR, c, te, Te = (q[k] for k in ("stefan", "compositionRatio", "specificHeatRatio", "thetaEutectic",
                                        "ThetaEutectic"))
    rng = np.random.default_rng(3)
    phi = np.zeros(case["phi"].shape)
    v = HC.valid(n, phi)
    shp = v[0].shape
    C = rng.uniform(-1.3 * CR - 0.1, 0.6, shp)
    k = rng.integers(0, 12, shp)
    C = np.where(k == 0, -CR, np.where(k == 1, np.nextafter(-CR, -9.0), np.where(k == 2, np.nextafter(-CR, 9.0), C)))
    he = (CR + C) / (CR + Te) * (St + te * (1 - c)) + c * te
    hl = St - C + te + Te
    ulp = lambda x, m: x * (1.0 + m * 2.0 ** -53 * rng.integers(-4, 5, shp))
    H = np.choose(rng.integers(0, 7, shp), [ulp(he, 1), he + 1e-13 * rng.uniform(-1, 1, shp), ulp(hl, 1),
                                            rng.uniform(-2, 8, shp), he + (hl - he) * 1e-6 * rng.random(shp),
                                            np.full(shp, te * c), rng.uniform(-2, 8, shp)])
    special = rng.random(shp)
    H = np.where(special < 0.002, np.inf, np.where(special < 0.004, -np.inf, np.where(special < 0.005, np.nan, H)))
    C = np.where((special > 0.99) & (special < 0.992), np.nan, C)
    v[0], v[1] = H, C
    g, p, bc = HC.oracle_setup(case)
    op = HC.gpu_setup(ml, gpu_ctx, case)
    with np.errstate(invalid="ignore"):
        ref = O.hc_diffused_var(g, p, bc, phi.copy())
    out = ml.DeviceArray(gpu_ctx, phi.shape)
    op.diffused_var(0, ml.DeviceArray(gpu_ctx, phi.shape, host=phi), out)
    a, r = HC.valid(n, out.get()), HC.valid(n, ref)
    assert np.array_equal(np.isnan(a), np.isnan(r))
    ok = ~np.isnan(r)
    assert HC.bitwise_equal(a[ok], r[ok])
    op.close()


SMALL = {
    "odd_rows_walls": dict(n=(31, 20), periodic=[0, 0], bc=WALLS),
    "thin_walls": dict(n=(2, 400), periodic=[0, 0], bc=WALLS),
    "one_row": dict(n=(300, 1), periodic=[1, 0], bc=WALLS),
    "deep": dict(n=(32, 32), periodic=[1, 1]),
    "long": dict(n=(8, 128)),
    "3d_odd_walls": dict(n=(9, 7, 5), periodic=[0, 0, 0], bc=WALLS),
    "3d_column": dict(n=(4, 4, 64), periodic=[1, 0, 0], bc=WALLS),
    "3d_periodic": dict(n=(16, 8, 8), periodic=[1, 1, 1]),
    "3d_tiled": dict(n=(24, 16, 12)),
}


@pytest.mark.parametrize("name", sorted(SMALL))
@pytest.mark.parametrize("bottom,nu1,acoef", [(40, 1, False), (3, 2, True), (0, 0, False)])
def test_single_workgroup_cycles(ml, gpu_ctx, wl, name, bottom, nu1, acoef):
    """The V-cycle of one workgroup on every kind of level it holds: odd rows
    (a thread's two cells may share a colour), cells with two and more walls,
    one to five levels, a bottom that ends at its fixed point or not at all."""
    case, g, p, bc, b, a, op = _setup(ml, gpu_ctx, wl, SMALL[name], acoef)
    n = case["n"]
    old = case["phi"].copy()
    new = old.copy()
    kw = dict(max_iter=3, nu1=nu1, nu2=3, bottom=bottom)
    so = O.hc_be_step(g, p, bc, a, b, case["dt"], new, old, opts=O.default_opts(**kw))
    dn = ml.DeviceArray(gpu_ctx, old.shape, host=old)
    st = op.solve_be(dn, ml.DeviceArray(gpu_ctx, old.shape, host=old), case["dt"], opts=ml.default_opts(**kw))
    out = dn.get()
    assert (st.iterations, st.exit_status, st.final_residual) == (so.iterations, so.exit_status, so.final_residual)
    assert HC.bitwise_equal(HC.valid(n, out), HC.valid(n, new))
    op.close()
