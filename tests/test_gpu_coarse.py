"""The LDS-resident coarse levels (one workgroup per problem) at the sizes where
they can go wrong: one to eight root tiles alone (level 0 in LDS), nine (too
many: grid-wide launches), one root with its eight children (both levels in
LDS), two roots (level 1 grid-wide), boxes of every axis order, both smoothers,
every storage type, the stored-coefficient preconditioner -- each solve equal to the
oracle's bit for bit; and the arithmetic by which these kernels divide."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

BOXES = [((1, 1, 1), 0), ((1, 1, 1), 1), ((2, 1, 1), 0), ((1, 3, 1), 0), ((1, 1, 5), 0), ((3, 2, 1), 0), ((2, 2, 2), 0),
         ((3, 3, 1), 0), ((1, 1, 2), 1), ((1, 2, 1), 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("nroot,level", BOXES)
@pytest.mark.parametrize("smoother,storage", [(ca.SMOOTH_RBGS, ca.STORE_F32), (ca.SMOOTH_RBGS, ca.STORE_BF16),
                                              (ca.SMOOTH_RBGS, ca.STORE_F16), (ca.SMOOTH_JACOBI, ca.STORE_F32)])
def test_coarse_levels_give_the_oracle_solve(nroot, level, smoother, storage):
    o = po.Oracle(kind=po.SCENE_UNIFORM, nroot=list(nroot), uniform_level=level, seed=sum(nroot))
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    b = o.get(po.CH_B)
    for coarsest, nu in ((10, 2), (3, 1), (0, 1)):
        o.set(po.CH_B, b)
        P.set(ca.CH_B, b.astype(np.float32))
        ro = o.solve(max_iters=12, tol=1e-6, level_iters=nu, coarsest_iters=coarsest, smoother=smoother, storage=storage)
        S = ca.GMGSolver()
        S.solve(P, False, 12, 1e-6, nu, coarsest, 1, False, smoother=smoother, storage=storage)
        # without bottom iterations a single level's z is 0 and both solves are NaN
        same = [S.last["iters"], S.last["rr"]], [ro["iters"], ro["rr"]]
        assert np.array_equal(*same, equal_nan=True), (coarsest, nu, same)
        xo = o.get(po.CH_X).astype(np.float32)[typ == po.LEAF]
        assert np.array_equal(P.get(ca.CH_X)[typ == po.LEAF], xo, equal_nan=True), (coarsest, nu)


@pytest.mark.gpu
@pytest.mark.parametrize("nroot,level", BOXES)
def test_amg_coarse_levels_give_the_oracle_solve(nroot, level):
    o = po.Oracle(kind=po.SCENE_UNIFORM, nroot=list(nroot), uniform_level=level, seed=sum(nroot))
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    b = o.get(po.CH_B)
    o.amg_prepare()
    S = ca.AMGSolver()
    S.prepareTypesAndCoeffs(P)
    for coarsest, nu in ((10, 2), (3, 1), (0, 1)):
        o.set(po.CH_B, b)
        P.set(ca.CH_B, b.astype(np.float32))
        ro = o.amg_solve(max_iters=12, tol=1e-6, level_iters=nu, coarsest_iters=coarsest)
        S.solve(P, False, 12, 1e-6, nu, coarsest, 1, False)
        r = S.last_batch[0]
        assert np.array_equal([r["iters"], r["rr"]], [ro["iters"], ro["rr"]], equal_nan=True), (coarsest, nu, r, ro)
        xo = o.get(po.CH_X).astype(np.float32)[typ == po.LEAF]
        assert np.array_equal(P.get(ca.CH_X)[typ == po.LEAF], xo, equal_nan=True), (coarsest, nu)


def test_division_by_a_64bit_reciprocal_rounds_as_division():
    """float32(float64(a) * (1/d)) is the correctly rounded a / d, also with a
    reciprocal off by 2^-52 of itself (random significands and the ends of the range)."""
    rng = np.random.default_rng(3)
    n = 1 << 20
    sig = rng.integers(1 << 23, 1 << 24, (2, n)).astype(np.float64)
    sig[:, :4] = [[1 << 23, (1 << 24) - 1, 1 << 23, (1 << 24) - 1], [1 << 23, 1 << 23, (1 << 24) - 1, (1 << 24) - 1]]
    a = np.ldexp(sig[0], rng.integers(-60, 20, n)).astype(np.float32)
    d = np.ldexp(sig[1], rng.integers(-40, 0, n)).astype(np.float32)
    for err in (0.0, 2.0 ** -52, -(2.0 ** -52)):
        rd = (1.0 / d.astype(np.float64)) * (1.0 + err)
        q = (a.astype(np.float64) * rd).astype(np.float32)
        assert np.array_equal(q, a / d), err
