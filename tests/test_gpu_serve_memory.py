"""A pressure that a server hands over holds memory of its own size only, also where
it is the buffer of a larger instance that is handed over."""
import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu


def test_results_hold_their_own_size():
    S = ca.Server(1 << 30, 8, level_iters=2, coarsest_iters=10, rel_tol=1e-6)
    items = []
    for nroot in ([1, 1, 1], [2, 1, 1], [3, 1, 1]):  # 73, 146 and 219 tiles
        o = po.Oracle(kind=po.SCENE_UNIFORM, uniform_level=2, nroot=nroot)
        lev, crd, typ, _ = o.topology()
        b = o.get(po.CH_B).astype(np.float32)
        tree = ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())
        o.solve(max_iters=200, tol=1e-6, level_iters=2, coarsest_iters=10)
        items.append((S.admit(tree), b, typ == po.LEAF, o.get(po.CH_X).astype(np.float32)))
    for _ in range(2):
        for k, (inst, b, _, _) in enumerate(items):
            S.submit(inst, b, tag=k)
        kept = {}
        for _ in range(5000):
            S.step()
            r = S.next_result()
            if r is not None:
                kept[r[0]] = r[3]
            if len(kept) == len(items):
                break
        for k, (_, b, leaf, x) in enumerate(items):
            p = kept[k]
            assert p.base is None and p.flags.owndata and p.shape == b.shape
            assert np.array_equal(p[leaf], x[leaf])
    S.close()
