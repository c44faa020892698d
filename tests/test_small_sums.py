"""The LDS-resident CG's sums (k_cg_small): tile partials are handed from the
wavefronts that form them to all of them through LDS, so between a row's last read
and its next write, and between its write and the read of it, has to stand a
barrier, also from one iteration to the next.  Checked on the kernel's text, with and
without the re-centring (a wavefront that arrives late shows a missing barrier on the
device now and then only); and closed boxes whose |r|^2 at the stopping threshold is
above the number of a tile's cells, many of them in one launch, against the oracle."""
import os
import re

import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po

KERNELS = os.path.join(os.path.dirname(os.path.abspath(ca.__file__)), "csrc", "kernels.hpp")


def block(text, at):
    """The text from the brace at or after `at` to the one that closes it."""
    begin = text.index("{", at)
    depth = 0
    for k in range(begin, len(text)):
        depth += {"{": 1, "}": -1}.get(text[k], 0)
        if depth == 0:
            return begin, k + 1
    raise AssertionError("no closing brace")


@pytest.mark.parametrize("pure", [False, True])
def test_a_barrier_between_uses_of_a_row(pure):
    text = re.sub(r"//[^\n]*", "", open(KERNELS).read())
    lo, hi = block(text, text.index("void sm_solve("))
    body = text[lo:hi]
    lo, hi = block(body, body.index("for (int k = 0; k < iters"))
    loop = body[lo:hi]
    if not pure:
        at = loop.index("if (st.pure_neumann)")
        lo, hi = block(loop, at)
        loop = loop[:at] + loop[hi:]
    # the V-cycle's own barriers are left out: without sweeps it has none
    uses = re.findall(r"(__syncthreads)\(\)|S\.part\[(\w+)\]\[wave\]( =)|sm_total\(S\.part\[(\w+)\]", loop)
    events = [("barrier", None) if u[0] else ("write", u[1]) if u[2] else ("read", u[3]) for u in uses]
    assert sum(e[0] == "write" for e in events) == sum(e[0] == "read" for e in events) == (5 if pure else 3)
    since = []  # uses since the last barrier
    for kind, row in events * 2:
        if kind == "barrier":
            since = []
            continue
        assert all(r != row or k == kind == "read" for k, r in since), (kind, row, since)
        since.append((kind, row))


@pytest.mark.gpu
@pytest.mark.parametrize("nroot,level", [((1, 1, 1), 0), ((1, 1, 1), 1), ((2, 2, 2), 0)])
@pytest.mark.parametrize("smoother,nu,coarsest", [(ca.SMOOTH_RBGS, 2, 10), (ca.SMOOTH_RBGS, 1, 2), (ca.SMOOTH_JACOBI, 2, 10)])
def test_closed_boxes_with_large_right_hand_sides(nroot, level, smoother, nu, coarsest):
    o = po.Oracle(kind=po.SCENE_UNIFORM, nroot=list(nroot), uniform_level=level, seed=11, face_bc=[po.NEUMANN] * 6, has_solid=0)
    lev, crd, typ, _ = o.topology()
    leaf = typ == po.LEAF
    b = o.get(po.CH_B).astype(np.float32) * np.float32(2.0 ** 30)
    o.set(po.CH_B, b)
    ro = o.solve(max_iters=40, tol=1e-4, level_iters=nu, coarsest_iters=coarsest, pure_neumann=True, smoother=smoother)
    assert 1 < ro["iters"] < 40 and ro["bb"] * 1e-8 > 512  # the threshold is above the counts
    xo = o.get(po.CH_X).astype(np.float32)[leaf]
    B = ca.Problem.batch([ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())] * 64)
    B.set(ca.CH_B, np.concatenate([b] * 64))
    res = ca.GMGSolver().solve_batch(B, 40, 1e-4, nu, coarsest, is_pure_neumann=True, smoother=smoother)
    for r, x in zip(res, B.split(B.get(ca.CH_X))):
        assert (r["iters"], r["rr"], r["converged"]) == (ro["iters"], ro["rr"], 1)
        assert np.array_equal(x[leaf], xo)
