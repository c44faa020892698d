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

SCENES = {
    "uniform": dict(kind=po.SCENE_UNIFORM, uniform_level=2, has_solid=0),
    "band": dict(kind=po.SCENE_SPHERE_BAND, band_level=[4, 3, 2], band_r=0.15),
    "plane_two_roots": dict(kind=po.SCENE_PLANE, plane_level=[3, 2], nroot=[1, 1, 2], has_solid=0,
                            face_bc=[po.DIRICHLET] * 3 + [po.NEUMANN] * 3),
}


@pytest.mark.gpu
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


@pytest.mark.gpu
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


@pytest.mark.gpu
@pytest.mark.parametrize("h0", [0.125, 0.3])
def test_subnormal_quotients_round_as_division(h0):
    """A sweep from x = 0 leaves b / D; with b near the lowest FP32 values the
    quotients are subnormal, where many lie halfway between two."""
    o = po.Oracle(h0=h0, seed=7, **SCENES["band"])
    lev, crd, typ, nbr = o.topology()
    P = ca.Problem(ca.Tree(o.params.h0, lev, crd, typ, o.celltypes()))
    b = np.random.default_rng(1).integers(-1 << 14, 1 << 14, (P.n, 512)).astype(np.float32) * np.float32(2.0 ** -149)
    for level in range(P.max_level + 1):
        for sweep in ("rbgs", "jacobi"):
            for X in (o, P):
                X.set(po.CH_Z, np.zeros((P.n, 512), np.float32))
                X.set(po.CH_TMP, b)
            if sweep == "rbgs":
                o.gs_color(level, po.CH_Z, po.CH_TMP, 0)
                ca.GaussSeidelColor(P, level, ca.CH_Z, ca.CH_TMP, 0)
            else:
                o.jacobi_sweep(level, po.CH_Z, po.CH_TMP, 1.0)
                ca.JacobiSweep(P, level, ca.CH_Z, ca.CH_TMP, 1.0)
            assert np.array_equal(P.get(ca.CH_Z), o.get(po.CH_Z).astype(np.float32)), (level, sweep)


@pytest.mark.parametrize("err", [0.0, 2.0 ** -52, -(2.0 ** -52), 2.0 ** -51, -(2.0 ** -51)])
def test_subnormal_quotients_from_a_reciprocal(err):
    """The kernels' steps in numpy: a quotient below 2^-126 from a 64-bit
    reciprocal off by err, taken to the multiple of 2^-150 within 2^-49 of it,
    rounds as the exact quotient does (halfway cases made on purpose)."""
    rng = np.random.default_rng(9)
    n = 1 << 20
    d = np.ldexp(rng.integers(1 << 23, 1 << 24, n).astype(np.float64), rng.integers(-30, 2, n)).astype(np.float32)
    a = np.ldexp(rng.integers(1, 1 << 24, n).astype(np.float64), -149).astype(np.float32)  # any subnormal or small normal value
    m = n // 2  # halfway: a = d (k + 1/2) 2^-149, d a small integer times a power of two
    d[:m] = rng.integers(1, 64, m) * np.float32(0.5)
    a[:m] = (d[:m].astype(np.float64) * (rng.integers(0, 1 << 12, m) + 0.5) * 2.0 ** -149).astype(np.float32)
    rd = (1.0 / d.astype(np.float64)) * (1.0 + err)
    v = a.astype(np.float64) * rd
    q = v.astype(np.float32)
    t = (v + 1.5 * 2.0 ** -98) - 1.5 * 2.0 ** -98
    sub = (q != 0) & (np.abs(q) < np.float32(2.0 ** -126))
    q = np.where(sub & (np.abs(v - t) <= np.abs(v) * 2.0 ** -49), t.astype(np.float32), q)
    assert sub.mean() > 0.4
    assert np.array_equal(q, a / d)


@pytest.mark.parametrize("err", [0.0, 2.0 ** -53, -(2.0 ** -53)])
@pytest.mark.parametrize("low", [False, True])
def test_quotients_rounded_to_fifty_bits(err, low):
    """The branch-free form: the product with a reciprocal (one unit of its last
    place off at most) rounded to 50 bits, then to FP32."""
    rng = np.random.default_rng(10)
    n = 1 << 20
    d = np.ldexp(rng.integers(1 << 23, 1 << 24, n).astype(np.float64), rng.integers(-30, 2, n)).astype(np.float32)
    if low:
        a = np.ldexp(rng.integers(1, 1 << 24, n).astype(np.float64), -149).astype(np.float32)
        m = n // 2
        d[:m] = rng.integers(1, 64, m) * np.float32(0.5)
        a[:m] = (d[:m].astype(np.float64) * (rng.integers(0, 1 << 12, m) + 0.5) * 2.0 ** -149).astype(np.float32)
    else:
        a = np.ldexp(rng.integers(1 << 23, 1 << 24, n).astype(np.float64), rng.integers(-60, 20, n)).astype(np.float32)
    v = a.astype(np.float64) * ((1.0 / d.astype(np.float64)) * (1.0 + err))
    c = 9.0 * v
    assert np.array_equal((c - (c - v)).astype(np.float32), a / d)
