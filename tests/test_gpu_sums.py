"""The per-problem sums of the tile partials at the counts where their forms
change or run out: below, at and past one row of lanes, one batch of rows, the
line between the one-wavefront and the whole-workgroup form, one LDS chunk and
several; and several problems of different counts in one launch.  The order of
every addition is fixed, so residuals and iteration counts equal the oracle's."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu


def row_of_tiles(n, seed=5):
    o = po.Oracle(kind=po.SCENE_UNIFORM, nroot=[n, 1, 1], uniform_level=0, has_solid=0, seed=seed)
    lev, crd, typ, nbr = o.topology()
    return o, ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2048, 2049, 4097, 6144, 6145, 16384, 16385, 33000])
def test_sums_of_one_problem(n):
    o, tree = row_of_tiles(n)
    P = ca.Problem(tree)
    P.set(ca.CH_B, o.get(po.CH_B).astype(np.float32))
    ro = o.solve(max_iters=3, tol=1e-12, level_iters=1, coarsest_iters=2)
    S = ca.GMGSolver()
    S.solve(P, False, 3, 1e-12, 1, 2, 1, False)
    assert (S.last["iters"], S.last["rr"], S.last["bb"]) == (ro["iters"], ro["rr"], ro["bb"])


@pytest.mark.parametrize("counts", [(1, 64, 2049, 65), (6145, 3, 16385)])
def test_sums_of_several_problems(counts):
    items = [row_of_tiles(n, seed=n) for n in counts]
    B = ca.Problem.batch([t for _, t in items])
    B.set(ca.CH_B, np.concatenate([o.get(po.CH_B).astype(np.float32) for o, _ in items]))
    res = ca.GMGSolver().solve_batch(B, 3, 1e-12, 1, 2)
    for r, (o, _) in zip(res, items):
        ro = o.solve(max_iters=3, tol=1e-12, level_iters=1, coarsest_iters=2)
        assert (r["iters"], r["rr"], r["bb"]) == (ro["iters"], ro["rr"], ro["bb"])


@pytest.mark.parametrize("kw", [dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2]), dict(kind=po.SCENE_UNIFORM, uniform_level=1)])
def test_dot_over_every_set_of_tile_types(kw):
    """Sets of types that are a list of the handle's, others, and empty ones (a
    uniform tree has no GHOST tiles)."""
    o = po.Oracle(**kw)
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    rng = np.random.default_rng(2)
    for ch in (po.CH_P, po.CH_Z):
        v = rng.standard_normal((P.n, 512)).astype(np.float32)
        o.set(ch, v)
        P.set(ch, v)
    for types in range(1, 8):
        assert P.dot(ca.CH_P, ca.CH_Z, types) == o.dot(po.CH_P, po.CH_Z, types), types
