"""A solve that ends by an error while its kernels are queued (here an error that the
thread's earlier HIP call left and the solve reports) leaves nothing behind that the
next solve on the handle could take for its own: the device's progress words of the
failed one would say that every problem is done."""
import ctypes

import numpy as np
import pytest

import cirrus_amd as ca
import pyoracle as po
from test_gpu_device_io import DevBuf, hip

pytestmark = pytest.mark.gpu


def test_a_solve_after_a_failed_one():
    o = po.Oracle(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], seed=2)
    lev, crd, typ, _ = o.topology()
    tree = ca.Tree(o.params.h0, lev, crd, typ, o.celltypes())
    copies = 400000 // tree.n
    P = ca.Problem.batch([tree] * copies)
    h = hip()
    h.hipSetDevice.restype = ctypes.c_int
    b = np.concatenate([o.get(po.CH_B).astype(np.float32)] * copies)
    full, zero = DevBuf(h, b.nbytes), DevBuf(h, b.nbytes)
    full.put(b)
    zero.put(np.zeros_like(b))
    ro = o.solve(max_iters=40, tol=1e-6, level_iters=2, coarsest_iters=10)
    S = ca.GMGSolver()
    for _ in range(2):
        P.set_device(ca.CH_B, zero.p.value)
        assert h.hipSetDevice(9999) != 0  # refused by the runtime, which keeps the error for the thread
        with pytest.raises(ca.CirrusError):
            S.solve_batch(P, 40, 1e-6, 2, 10)
        P.set_device(ca.CH_B, full.p.value)
        res = S.solve_batch(P, 40, 1e-6, 2, 10)
        assert {(r["iters"], r["rr"], r["converged"]) for r in res} == {(ro["iters"], ro["rr"], 1)}
    full.free()
    zero.free()
