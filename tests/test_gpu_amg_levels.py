"""The grid-wide levels of the stored-coefficient V-cycle: the residual pass that
restricts, the rhs of LEAF tiles with GHOST children on every level (LDS-resident
ones included), rows at the grid's edge, and the pass that hands z over with its
r.z partials -- solves equal to the oracle's bit for bit."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

SCENES = {
    "uniform": dict(kind=po.SCENE_UNIFORM, uniform_level=2),
    "two_roots": dict(kind=po.SCENE_UNIFORM, uniform_level=1, nroot=[1, 2, 1], has_solid=0),
    "band": dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], solid_r=0.1),
    "plane_from_roots": dict(kind=po.SCENE_PLANE, plane_level=[2, 1], nroot=[1, 1, 2], has_solid=0),
    "plane_coarse": dict(kind=po.SCENE_PLANE, plane_level=[3, 1]),
    "vortex": dict(kind=po.SCENE_VORTEX, nroot=[1, 1, 2], vortex_level=[4, 2], seed=3),
}


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("nu,coarsest", [(1, 10), (2, 10), (3, 4), (0, 10)])
def test_amg_solve_on_every_kind_of_level(name, nu, coarsest):
    o = po.Oracle(**SCENES[name])
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    b = o.get(po.CH_B)
    o.amg_prepare()
    S = ca.AMGSolver()
    S.prepareTypesAndCoeffs(P)
    leaf = typ == po.LEAF
    for iters in (2, 12):
        o.set(po.CH_B, b)
        P.set(ca.CH_B, b.astype(np.float32))
        ro = o.amg_solve(max_iters=iters, tol=1e-12, level_iters=nu, coarsest_iters=coarsest)
        S.solve(P, False, iters, 1e-12, nu, coarsest, 1, False)
        r = S.last_batch[0]
        assert np.array_equal([r["iters"], r["rr"]], [ro["iters"], ro["rr"]], equal_nan=True), iters
        assert np.array_equal(P.get(ca.CH_X)[leaf], o.get(po.CH_X).astype(np.float32)[leaf], equal_nan=True), iters
