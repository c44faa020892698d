"""Tiles without a cut face or a non-INTERIOR cell take shorter rows (one
coefficient set per tile, quotients by a prepared reciprocal, the cell size's
powers in one product where it is a power of two); the others the general ones.
Solves equal to the oracle's bit for bit where these rules meet: a power of two
as the root cell size and not, open tiles beside GHOST tiles (other coefficients
on those faces), beside solids and at the walls, one root and several; both
smoothers, every storage type, one to three iterations per level, the fused
first iteration on and off."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

SCENES = {
    "uniform": dict(kind=po.SCENE_UNIFORM, uniform_level=2, has_solid=0),
    "band": dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], band_r=0.15),
    "plane_two_roots": dict(kind=po.SCENE_PLANE, plane_level=[3, 2], nroot=[1, 1, 2], has_solid=0,
                            face_bc=[po.DIRICHLET] * 3 + [po.NEUMANN] * 3),
}


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("h0", [0.125, 0.1, 0.3])
@pytest.mark.parametrize("smoother,storage,nu", [(ca.SMOOTH_RBGS, ca.STORE_F32, 2), (ca.SMOOTH_RBGS, ca.STORE_F32, 3),
                                                 (ca.SMOOTH_RBGS, ca.STORE_BF16, 2), (ca.SMOOTH_RBGS, ca.STORE_F16, 1),
                                                 (ca.SMOOTH_JACOBI, ca.STORE_F32, 2), (ca.SMOOTH_JACOBI, ca.STORE_BF16, 3)])
def test_open_tiles_give_the_oracle_solve(scene, h0, smoother, storage, nu):
    o = po.Oracle(h0=h0, seed=7, **SCENES[scene])
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    b = o.get(po.CH_B)
    ro = o.solve(max_iters=8, tol=1e-6, level_iters=nu, coarsest_iters=10, smoother=smoother, storage=storage)
    xo = o.get(po.CH_X).astype(np.float32)[typ == po.LEAF]
    for fused16 in (-1, 0):
        P.set_level_forms(-1, fused16, -1)
        P.set(ca.CH_B, b.astype(np.float32))
        S = ca.GMGSolver()
        S.solve(P, False, 8, 1e-6, nu, 10, 1, False, smoother=smoother, storage=storage)
        assert (S.last["iters"], S.last["rr"], S.last["bb"]) == (ro["iters"], ro["rr"], ro["bb"]), fused16
        assert np.array_equal(P.get(ca.CH_X)[typ == po.LEAF], xo), fused16


def test_open_tiles_of_several_cell_sizes_in_one_batch():
    items = []
    for h0 in (0.125, 0.1, 0.25, 0.3):
        o = po.Oracle(h0=h0, seed=3, **SCENES["band"])
        lev, crd, typ, nbr = o.topology()
        items.append((o, ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()), typ))
    bs = [o.get(po.CH_B) for o, _, _ in items]
    B = ca.Problem.batch([t for _, t, _ in items])
    B.set(ca.CH_B, np.concatenate([b.astype(np.float32) for b in bs]))
    res = ca.GMGSolver().solve_batch(B, 60, 1e-6, 2, 10)
    X = B.split(B.get(ca.CH_X))
    for k, (o, _, typ) in enumerate(items):
        ro = o.solve(max_iters=60, tol=1e-6, level_iters=2, coarsest_iters=10)
        assert (res[k]["iters"], res[k]["rr"]) == (ro["iters"], ro["rr"]), k
        m = typ == po.LEAF
        assert np.array_equal(X[k][m], o.get(po.CH_X).astype(np.float32)[m]), k
