"""Problems whose every level is LDS-resident run whole CG iterations in one
launch.  Against the same solve by launches (a schedule that gives the levels
back to grid-wide ones): every channel the solve leaves, the iteration counts and
residuals, bit for bit, and the oracle's.  One root, one to eight roots, a root
with children; every storage type, both smoothers, no sweeps, no bottom
iterations; re-centred; checks at a stride; more iterations than one launch runs;
a solve continued by its cap; boxes of different sizes in one handle."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

BOXES = [((1, 1, 1), 0), ((1, 1, 1), 1), ((2, 1, 1), 0), ((1, 1, 5), 0), ((3, 2, 1), 0), ((2, 2, 2), 0)]
CHANNELS = (ca.CH_X, ca.CH_R, ca.CH_P, ca.CH_Z, ca.CH_AP)


def box(nroot, level, seed=0, **kw):
    o = po.Oracle(kind=po.SCENE_UNIFORM, nroot=list(nroot), uniform_level=level, seed=seed, **kw)
    lev, crd, typ, nbr = o.topology()
    return o, ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()), typ, o.get(po.CH_B)


def run(P, b, shift, *args, **kw):
    P.set_schedule(coarse_shift=shift)
    P.set(ca.CH_B, b.astype(np.float32))
    S = ca.GMGSolver()
    S.solve(P, False, *args, **kw)
    return (S.last["iters"], S.last["rr"], S.last["bb"], S.last["converged"])


@pytest.mark.parametrize("nroot,level", BOXES)
@pytest.mark.parametrize("smoother,storage", [(ca.SMOOTH_RBGS, ca.STORE_F32), (ca.SMOOTH_RBGS, ca.STORE_BF16),
                                              (ca.SMOOTH_RBGS, ca.STORE_F16), (ca.SMOOTH_JACOBI, ca.STORE_F32),
                                              (ca.SMOOTH_JACOBI, ca.STORE_F16)])
@pytest.mark.parametrize("pure", [False, True])
def test_one_launch_leaves_what_the_launches_leave(nroot, level, smoother, storage, pure):
    bc = dict(face_bc=[po.NEUMANN] * 6, has_solid=0) if pure else {}
    o, tree, typ, b = box(nroot, level, seed=sum(nroot), **bc)
    P = ca.Problem(tree)
    leaf = typ == po.LEAF
    for iters, tol, nu, coarsest, stride in ((40, 1e-6, 2, 10, 1), (33, 1e-30, 1, 4, 1), (16, 1e-30, 2, 10, 5), (1, 1e-6, 2, 10, 1),
                                             (200, 1e-6, 1, 10, 3), (7, 1e-6, 0, 10, 1), (5, 1e-6, 2, 10, 0)):
        kw = dict(smoother=smoother, storage=storage)
        small = run(P, b, 0, iters, tol, nu, coarsest, stride, pure, **kw)
        got = [P.get(ch)[leaf] for ch in CHANNELS]
        wide = run(P, b, 2, iters, tol, nu, coarsest, stride, pure, **kw)
        case = (iters, tol, nu, coarsest, stride)
        assert np.array_equal(small, wide, equal_nan=True), (case, small, wide)
        for ch, g in zip(CHANNELS, got):
            assert np.array_equal(g, P.get(ch)[leaf], equal_nan=True), (case, ch)
        o.set(po.CH_B, b)
        ro = o.solve(max_iters=iters, tol=tol, level_iters=nu, coarsest_iters=coarsest, sync_stride=stride, pure_neumann=pure,
                     smoother=smoother, storage=storage)
        assert small[0] == ro["iters"] and np.array_equal(got[0], o.get(po.CH_X).astype(np.float32)[leaf], equal_nan=True), case
        if small[3] or not pure:  # at its cap the oracle measures r after one more re-centring
            assert np.array_equal(small[1], ro["rr"], equal_nan=True), case


def test_boxes_of_different_sizes_in_one_handle():
    items = [box(nr, lv, seed=k) for k, (nr, lv) in enumerate(BOXES * 2)]
    B = ca.Problem.batch([t for _, t, _, _ in items])
    b = np.concatenate([it[3].astype(np.float32) for it in items])
    for storage in (ca.STORE_F32, ca.STORE_BF16):
        B.set(ca.CH_B, b)
        res = ca.GMGSolver().solve_batch(B, 60, 1e-6, 2, 10, storage=storage)
        X = B.split(B.get(ca.CH_X))
        for k, (o, _, typ, bk) in enumerate(items):
            o.set(po.CH_B, bk)
            ro = o.solve(max_iters=60, tol=1e-6, level_iters=2, coarsest_iters=10, storage=storage)
            assert (res[k]["iters"], res[k]["rr"]) == (ro["iters"], ro["rr"]), k
            m = typ == po.LEAF
            assert np.array_equal(X[k][m], o.get(po.CH_X).astype(np.float32)[m]), k
