"""Infinities and NaN in a right-hand side, and cell sizes at which a row's diagonal
is 0 or infinite (its coefficients 1 / h^2 underflow or overflow), leave what the FP32
division leaves: V-cycles of boxes whose levels are all LDS-resident, of taller ones
and of a tree with GHOST tiles, and sweeps of every level, equal to the oracle's."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

SCENES = {
    "root": dict(kind=po.SCENE_UNIFORM, uniform_level=0, has_solid=0),
    "children": dict(kind=po.SCENE_UNIFORM, uniform_level=1, has_solid=0),
    "roots": dict(kind=po.SCENE_UNIFORM, uniform_level=0, nroot=[3, 2, 1], has_solid=0),
    "uniform": dict(kind=po.SCENE_UNIFORM, uniform_level=2, has_solid=0),
    "band": dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], band_r=0.15),
}
SIZES = [0.125, 0.3, 2.0 ** 78, 2.0 ** -70]  # D of about 6 h, 0, infinite


def pair(scene, h0):
    o = po.Oracle(h0=h0, seed=5, **SCENES[scene])
    lev, crd, typ, _ = o.topology()
    return o, ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())), typ, o.celltypes()


def field(typ, ctype, values, seed):
    """N(0,1) on the INTERIOR cells of LEAF tiles, three of them the given values."""
    rng = np.random.default_rng(seed)
    f = rng.standard_normal(ctype.shape).astype(np.float32)
    inside = (ctype == ca.INTERIOR) & (typ == po.LEAF)[:, None]
    f[~inside] = 0
    cells = np.argwhere(inside)
    for (t, c), v in zip(cells[[0, len(cells) // 2, -1]], values):
        f[t, c] = v
    return f


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("h0", SIZES)
@pytest.mark.parametrize("smoother,nu,coarsest", [(ca.SMOOTH_JACOBI, 1, 0), (ca.SMOOTH_JACOBI, 2, 4), (ca.SMOOTH_RBGS, 1, 0),
                                                  (ca.SMOOTH_RBGS, 1, 2), (ca.SMOOTH_RBGS, 2, 4)])
def test_vcycles_of_infinite_right_hand_sides(scene, h0, smoother, nu, coarsest):
    o, P, typ, ctype = pair(scene, h0)
    leaf = typ == po.LEAF
    for values in ((np.inf, 1.0, -np.inf), (1.0, np.nan, 1.0)):
        f = field(typ, ctype, values, 3)
        o.set(po.CH_R, f)
        P.set(ca.CH_R, f)
        o.vcycle(po.CH_Z, po.CH_R, po.CH_AP, nu, coarsest, smoother, 2.0 / 3.0)
        ca.GMGSolver().VCycle(P, ca.CH_Z, ca.CH_R, nu, coarsest, smoother, 2.0 / 3.0)
        assert np.array_equal(P.get(ca.CH_Z)[leaf], o.get(po.CH_Z).astype(np.float32)[leaf], equal_nan=True), values


@pytest.mark.parametrize("scene", ["uniform", "band"])
@pytest.mark.parametrize("h0", SIZES)
def test_sweeps_of_infinite_right_hand_sides(scene, h0):
    o, P, typ, ctype = pair(scene, h0)
    x = np.random.default_rng(4).standard_normal(ctype.shape).astype(np.float32)
    x[ctype != ca.INTERIOR] = 0
    f = np.random.default_rng(5).standard_normal(ctype.shape).astype(np.float32)
    for value in (np.inf, -np.inf, np.nan):
        f[:, 219] = value  # cell (3, 3, 3) of every tile
        f[:, 292] = value  # cell (4, 4, 4)
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
                assert np.array_equal(P.get(ca.CH_Z), o.get(po.CH_Z).astype(np.float32), equal_nan=True), (value, level, sweep)
