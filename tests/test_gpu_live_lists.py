"""A pool's worklists narrowed to the problems still running, while others stop:
problems of different sizes and tolerances' worth of iterations in one handle
large enough for stream launches, some done at once (b = 0), solved twice (the
handle's own lists come back), in every storage type, with checks at a stride,
as a refinement (inner solves in which whole problems take no part) -- each
result equal to the problem solved alone."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

KINDS = [dict(kind=po.SCENE_UNIFORM, uniform_level=1), dict(kind=po.SCENE_SPHERE_BAND, band_level=[5, 4, 3]),
         dict(kind=po.SCENE_UNIFORM, uniform_level=3), dict(kind=po.SCENE_PLANE, plane_level=[3, 2]),
         dict(kind=po.SCENE_VORTEX, nroot=[1, 1, 2], vortex_level=[4, 2], seed=3), dict(kind=po.SCENE_UNIFORM, uniform_level=0)]
_cache = []


def problems():
    if not _cache:
        for k, kw in enumerate(KINDS + KINDS[1:4]):
            o = po.Oracle(**dict(kw, seed=kw.get("seed", k)))
            lev, crd, typ, nbr = o.topology()
            b = o.get(po.CH_B).astype(np.float32)
            if k == 3:
                b = 0 * b
            _cache.append((ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()), b, typ == po.LEAF))
    return _cache


@pytest.mark.parametrize("storage,smoother,stride", [(ca.STORE_F32, ca.SMOOTH_RBGS, 1), (ca.STORE_BF16, ca.SMOOTH_RBGS, 1),
                                                     (ca.STORE_F16, ca.SMOOTH_RBGS, 3), (ca.STORE_F32, ca.SMOOTH_JACOBI, 2)])
def test_pool_equals_its_problems_alone(storage, smoother, stride):
    items = problems()
    B = ca.Problem.batch([t for t, _, _ in items])
    assert B.n >= 8192  # stream launches
    for _ in range(2):
        B.set(ca.CH_B, np.concatenate([b for _, b, _ in items]))
        res = ca.GMGSolver().solve_batch(B, 60, 1e-6, 2, 10, storage=storage, smoother=smoother, sync_stride=stride)
        X = B.split(B.get(ca.CH_X))
        R = B.split(B.get(ca.CH_R))
        for k, (tree, b, leaf) in enumerate(items):
            P = ca.Problem(tree)
            P.set(ca.CH_B, b)
            one = ca.GMGSolver().solve_batch(P, 60, 1e-6, 2, 10, storage=storage, smoother=smoother, sync_stride=stride)[0]
            assert (res[k]["iters"], res[k]["rr"]) == (one["iters"], one["rr"]), k
            assert np.array_equal(X[k][leaf], P.get(ca.CH_X)[leaf]), k
            assert np.array_equal(R[k][leaf], P.get(ca.CH_R)[leaf]), k
    assert len({r["iters"] for r in res}) > 2


def test_refined_pool_equals_its_problems_alone():
    items = problems()
    B = ca.Problem.batch([t for t, _, _ in items])
    B.set(ca.CH_B, np.concatenate([b for _, b, _ in items]))
    res = ca.GMGSolver().solve_refined(B, 1e-8, 1e-4, 20, 60, 2, 10, storage=ca.STORE_BF16)
    X = B.split(B.get_f64())
    for k, (tree, b, leaf) in enumerate(items):
        P = ca.Problem(tree)
        P.set(ca.CH_B, b)
        one = ca.GMGSolver().solve_refined(P, 1e-8, 1e-4, 20, 60, 2, 10, storage=ca.STORE_BF16)[0]
        assert (res[k]["iters"], res[k]["outer"]) == (one["iters"], one["outer"]), k
        assert np.array_equal(X[k][leaf], P.get_f64()[leaf]), k
