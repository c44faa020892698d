"""Values below 2^-126, where FP32 rounds to multiples of 2^-149 and a sum of
products, a residual and a quotient may each be rounded there: sweeps from a nonzero
x, V-cycles and solves of LDS-resident boxes and of taller trees, both smoothers and
the stored-coefficient preconditioner, equal to the oracle's bit for bit.  Cell sizes
that are powers of two and not, and small and large ones."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

SCENES = {
    "children": dict(kind=po.SCENE_UNIFORM, uniform_level=1, has_solid=0),
    "roots": dict(kind=po.SCENE_UNIFORM, uniform_level=0, nroot=[3, 2, 1], has_solid=0),
    "uniform": dict(kind=po.SCENE_UNIFORM, uniform_level=2, has_solid=0),
    "band": dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], band_r=0.15),
}
SIZES = [0.125, 0.1, 2.0 ** -20, 3.0 * 2.0 ** 20]


def pair(scene, h0):
    o = po.Oracle(h0=h0, seed=9, **SCENES[scene])
    lev, crd, typ, _ = o.topology()
    return o, ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())), typ, o.celltypes()


def tiny(shape, bits, seed):
    """Whole multiples of 2^-149 of at most `bits` bits."""
    v = np.random.default_rng(seed).integers(-(1 << bits), (1 << bits) + 1, shape)
    return v.astype(np.float32) * np.float32(2.0 ** -149)


@pytest.mark.parametrize("scene", ["uniform", "band"])
@pytest.mark.parametrize("h0", SIZES)
@pytest.mark.parametrize("bits", [3, 10, 20])
def test_sweeps_from_a_subnormal_guess(scene, h0, bits):
    o, P, typ, ctype = pair(scene, h0)
    x, f = tiny(ctype.shape, bits, 1), tiny(ctype.shape, bits, 2)
    x[ctype != ca.INTERIOR] = 0
    for level in range(P.max_level + 1):
        for sweep in ("red", "black", "jacobi"):
            for X in (o, P):
                X.set(po.CH_Z, x)
                X.set(po.CH_TMP, f)
            if sweep == "jacobi":
                o.jacobi_sweep(level, po.CH_Z, po.CH_TMP, 2.0 / 3.0)
                ca.JacobiSweep(P, level, ca.CH_Z, ca.CH_TMP, 2.0 / 3.0)
            else:
                o.gs_color(level, po.CH_Z, po.CH_TMP, int(sweep == "black"))
                ca.GaussSeidelColor(P, level, ca.CH_Z, ca.CH_TMP, int(sweep == "black"))
            got, ref = P.get(ca.CH_Z), o.get(po.CH_Z).astype(np.float32)
            assert np.array_equal(got, ref), (level, sweep, int((got != ref).sum()), float(np.abs(got - ref).max()) * 2.0 ** 149)


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("h0", SIZES)
@pytest.mark.parametrize("smoother,nu", [(ca.SMOOTH_RBGS, 2), (ca.SMOOTH_RBGS, 1), (ca.SMOOTH_JACOBI, 2)])
def test_vcycles_of_subnormal_right_hand_sides(scene, h0, smoother, nu):
    o, P, typ, ctype = pair(scene, h0)
    leaf = typ == po.LEAF
    for bits in (10, 20, 23):
        f = tiny(ctype.shape, bits, bits)
        f[(ctype != ca.INTERIOR) | ~leaf[:, None]] = 0
        o.set(po.CH_R, f)
        P.set(ca.CH_R, f)
        o.vcycle(po.CH_Z, po.CH_R, po.CH_AP, nu, 10, smoother, 2.0 / 3.0)
        ca.GMGSolver().VCycle(P, ca.CH_Z, ca.CH_R, nu, 10, smoother, 2.0 / 3.0)
        assert np.array_equal(P.get(ca.CH_Z)[leaf], o.get(po.CH_Z).astype(np.float32)[leaf]), bits


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("h0", SIZES)
@pytest.mark.parametrize("solver", ["rbgs", "jacobi", "amg"])
def test_solves_of_subnormal_right_hand_sides(scene, h0, solver):
    o, P, typ, ctype = pair(scene, h0)
    leaf = typ == po.LEAF
    f = tiny(ctype.shape, 22, 5)
    f[(ctype != ca.INTERIOR) | ~leaf[:, None]] = 0
    o.set(po.CH_B, f)
    P.set(ca.CH_B, f)
    if solver == "amg":
        o.amg_prepare()
        ro = o.amg_solve(max_iters=9, tol=1e-6, level_iters=2, coarsest_iters=10)
        S = ca.AMGSolver()
        S.prepareTypesAndCoeffs(P)
        S.solve(P, False, 9, 1e-6, 2, 10, 1, False)
        r = S.last_batch[0]
    else:
        smoother = ca.SMOOTH_RBGS if solver == "rbgs" else ca.SMOOTH_JACOBI
        ro = o.solve(max_iters=9, tol=1e-6, level_iters=2, coarsest_iters=10, smoother=smoother)
        S = ca.GMGSolver()
        S.solve(P, False, 9, 1e-6, 2, 10, 1, False, smoother=smoother)
        r = S.last
    assert np.array_equal([r["iters"], r["rr"], r["bb"]], [ro["iters"], ro["rr"], ro["bb"]], equal_nan=True)
    assert np.array_equal(P.get(ca.CH_X)[leaf], o.get(po.CH_X).astype(np.float32)[leaf], equal_nan=True)


@pytest.mark.parametrize("coarsening", [2.0 ** -115, 2.0 ** -60, 2.0 ** 60, 2.0 ** 110])
def test_reciprocals_of_extreme_diagonals(coarsening):
    """Stored coefficients scaled per level far from 1, so that a diagonal lies beyond
    the range of the fast reciprocal: the LDS-resident levels against the same levels by
    grid-wide launches, which divide."""
    o, P, typ, ctype = pair("children", 0.125)
    leaf = typ == po.LEAF
    f = np.random.default_rng(6).standard_normal(ctype.shape).astype(np.float32)
    f[(ctype != ca.INTERIOR) | ~leaf[:, None]] = 0
    S = ca.AMGSolver(one_over_alpha=coarsening)
    S.prepareTypesAndCoeffs(P)
    d = S.coefficients(P)[3][typ == po.NONLEAF]
    assert (d != 0).any() and np.all((np.abs(d) < 2.0 ** -100) | (np.abs(d) > 2.0 ** 100)) == (coarsening not in (2.0 ** -60, 2.0 ** 60))
    out = []
    for shift in (0, 2):
        P.set_schedule(coarse_shift=shift)
        P.set(ca.CH_B, f)
        S.solve(P, False, 3, 1e-6, 1, 4, 1, False)
        r = S.last_batch[0]
        out.append(([r["iters"], r["rr"]], P.get(ca.CH_P)[leaf], P.get(ca.CH_X)[leaf]))
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.isfinite(out[0][1]).all() and out[0][1].any()
