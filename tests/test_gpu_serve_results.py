"""The pressures a server hands over, taken from one reused buffer or handed over
with it: each result an array of its own that later results leave alone, sizes far
apart and alike, polls that find nothing in between, zeros for a request that asked
for no pressure (also after one that did)."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu

SIZES = [dict(kind=po.SCENE_UNIFORM, uniform_level=1), dict(kind=po.SCENE_UNIFORM, uniform_level=3),
         dict(kind=po.SCENE_UNIFORM, uniform_level=3, seed=4), dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2])]


def collect(S, expect):
    out = {}
    for _ in range(5000):
        S.step()
        r = S.next_result()
        if r is not None:
            out[r[0]] = r
        if len(out) == expect:
            return out
    raise AssertionError("requests did not finish")


@pytest.mark.parametrize("storage", [ca.STORE_F32, ca.STORE_BF16])
def test_results_are_arrays_of_their_own(storage):
    items = []
    for kw in SIZES:
        o = po.Oracle(**kw)
        lev, crd, typ, nbr = o.topology()
        b = o.get(po.CH_B).astype(np.float32)
        ro = o.solve(max_iters=200, tol=1e-6, level_iters=2, coarsest_iters=10, storage=storage)
        leaf = typ == po.LEAF
        items.append((ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()), b, leaf, o.get(po.CH_X).astype(np.float32)[leaf],
                      ro["iters"]))
    S = ca.Server(1 << 30, 8, storage=storage, level_iters=2, coarsest_iters=10, rel_tol=1e-6)
    ids = [S.admit(t) for t, *_ in items]
    kept = []
    for round_ in range(3):
        silent = round_ == 1
        for k, (tree, b, leaf, x, iters) in enumerate(items):
            S.submit(ids[k], b, tag=k, download=not (silent and k % 2))
        got = collect(S, len(items))
        for k, (tree, b, leaf, x, iters) in enumerate(items):
            p = got[k][3]
            assert p.shape == (tree.n, 512) and p.dtype == np.float32 and got[k][2]["iters"] == iters
            kept.append((p, leaf, None if silent and k % 2 else x))
    for p, leaf, x in kept:
        assert not p.any() if x is None else np.array_equal(p[leaf], x)
