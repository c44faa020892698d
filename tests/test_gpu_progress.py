"""How a solve ends, as the host follows the device's iterations through host
memory: no iteration allowed, a cap inside and at a stride of checks,
convergence, a zero right-hand side, problems of one handle that stop at
different iterations, and several handles at once from several threads; by graph
replay and by stream launches.  Iteration counts and residuals equal the
oracle's, and the same handle solves again afterwards."""
import threading

import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

pytestmark = pytest.mark.gpu


def scene(seed=0, **kw):
    kw.setdefault("kind", po.SCENE_UNIFORM)
    kw.setdefault("uniform_level", 2)
    o = po.Oracle(seed=seed, **kw)
    lev, crd, typ, nbr = o.topology()
    return o, ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()), o.get(po.CH_B)


@pytest.mark.parametrize("use_graph", [False, True])
def test_every_way_to_stop(use_graph):
    o, tree, b = scene()
    P = ca.Problem(tree)
    for max_iters, stride, tol, rhs in ((200, 1, 1e-6, b), (0, 1, 1e-6, b), (1, 1, 1e-6, b), (4, 3, 1e-12, b), (6, 3, 1e-12, b),
                                        (200, 3, 1e-6, b), (5, 0, 1e-6, b), (200, 1, 1e-6, 0 * b), (200, 1, 1e-6, b)):
        o.set(po.CH_B, rhs)
        P.set(ca.CH_B, rhs.astype(np.float32))
        ro = o.solve(max_iters=max_iters, tol=tol, level_iters=2, coarsest_iters=10, sync_stride=stride)
        S = ca.GMGSolver()
        S.solve(P, False, max_iters, tol, 2, 10, stride, False, use_graph=use_graph)
        assert (S.last["iters"], S.last["rr"]) == (ro["iters"], ro["rr"]), (max_iters, stride, tol)


def test_problems_that_stop_apart():
    items = [scene(seed=s, uniform_level=lv) for s, lv in ((1, 1), (2, 3), (3, 2), (4, 0))]
    B = ca.Problem.batch([t for _, t, _ in items])
    B.set(ca.CH_B, np.concatenate([b.astype(np.float32) for _, _, b in items]))
    for _ in range(2):
        res = ca.GMGSolver().solve_batch(B, 200, 1e-6, 2, 10)
        B.set(ca.CH_B, np.concatenate([b.astype(np.float32) for _, _, b in items]))
    for r, (o, _, b) in zip(res, items):
        o.set(po.CH_B, b)
        ro = o.solve(max_iters=200, tol=1e-6, level_iters=2, coarsest_iters=10)
        assert (r["iters"], r["rr"]) == (ro["iters"], ro["rr"])


def test_handles_in_several_threads():
    items = [scene(seed=s, uniform_level=1 + s % 2) for s in range(4)]
    want = [o.solve(max_iters=200, tol=1e-6, level_iters=2, coarsest_iters=10) for o, _, _ in items]
    handles = [ca.Problem(t) for _, t, _ in items]
    got = [[] for _ in items]

    def work(k):
        for rep in range(3):
            handles[k].set(ca.CH_B, items[k][2].astype(np.float32))
            S = ca.GMGSolver()
            S.solve(handles[k], False, 200, 1e-6, 2, 10, 1, False, use_graph=bool((k + rep) % 2))
            got[k].append((S.last["iters"], S.last["rr"]))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for w, g in zip(want, got):
        assert g == [(w["iters"], w["rr"])] * 3
