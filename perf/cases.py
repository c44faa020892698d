"""The work that programs have this library do, as cases for timing.

A case is one call (or one short round of calls) of the public Python API on a
device-resident octree.  The trees are the library's own workloads
(``cirrus_amd.workloads``) and plain boxes around them; right-hand sides are the
divergence of a seeded N(0,1) face-velocity field, as in those workloads, and
live in device memory, as a simulation's fields do (the server takes host
arrays, as its clients send them).

* ``solve``    one pressure solve: b to the handle, ``GMGSolver.solve``, x back.
* ``project``  one projection: velocities in, ``GMGSolver.project``, velocities
               and pressure back.
* ``krylov``   the pieces of a caller's own Krylov loop: z = one V-cycle of b,
               A b, and the inner products b.z and b.Ab.
* ``amg``      one solve with the stored-coefficient preconditioner.
* ``batch``    many independent trees in one handle, solved together in FP32, or
               with 16-bit V-cycle storage inside the FP64 refinement.
* ``refined``  one large tree through the mixed-precision refinement.
* ``serve``    one round of the serving loop: a warm-started request for every
               resident instance, stepped until all results are read.

``exact`` states the discrete pressure equation on the leaf cells by itself (a
sparse matrix in 64 bits) and solves it with Jacobi-preconditioned conjugate
gradients in torch.
"""
import functools
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import cirrus_amd as ca
from cirrus_amd import workloads

DEVICE = "cuda"
STORE = {"f32": ca.STORE_F32, "bf16": ca.STORE_BF16, "f16": ca.STORE_F16}
SMOOTH = {"rbgs": ca.SMOOTH_RBGS, "jacobi": ca.SMOOTH_JACOBI}
MAX_ITERS = 500
# Trees of more leaf tiles than this have no 64-bit solution here (it takes too long).
EXACT_LEAF_TILES = 8192


def listed():
    return [
        # the smallest call: a 16^3 box (9 tiles), the reference's own default settings
        dict(name="solve_uniform16", path="solve", scene="uniform", level=1, nx=1, ny=1, nz=1, nu=1, smoother="rbgs",
             storage="f32", neumann=False),
        # the plain configuration: uniform 64^3, damped Jacobi 2+2
        dict(name="solve_uniform64_jacobi", path="solve", scene="uniform", level=3, nx=1, ny=1, nz=1, nu=2,
             smoother="jacobi", storage="f32", neumann=False),
        # the headline solve: adaptive octree, 256^3 effective, RB-GS 2+2
        dict(name="solve_adaptive256", path="solve", scene="band", level=5, r=0.15, w=0.05, nx=1, ny=1, nz=1, nu=2,
             smoother="rbgs", storage="f32", neumann=False),
        # a closed box of uneven extent (3x2x1 root tiles, 96x64x32 cells): pure Neumann, re-centred every iteration
        dict(name="solve_neumann_box", path="solve", scene="uniform", level=2, nx=3, ny=2, nz=1, nu=2, smoother="rbgs",
             storage="f32", neumann=True),
        # a simulation step's projection with the reference's settings (one sweep per level)
        dict(name="project_adaptive256", path="project", scene="band", level=5, r=0.15, w=0.05, nx=1, ny=1, nz=1, nu=1),
        # one step of a caller's own Krylov loop
        dict(name="krylov_adaptive256", path="krylov", scene="band", level=5, r=0.15, w=0.05, nx=1, ny=1, nz=1, nu=2),
        # the stored-coefficient solver on a coarse/fine plane
        dict(name="amg_plane128", path="amg", scene="plane", level=4, nx=1, ny=1, nz=1, nu=2),
        # a small pool, FP32
        dict(name="batch24_f32", path="batch", scene="batch", first=0, count=24, storage="f32", refined=False),
        # float16 storage, a handful of trees
        dict(name="batch7_f16_refined", path="batch", scene="batch", first=40, count=7, storage="f16", refined=True),
        # the batched workload: 256 trees, bfloat16 storage, FP64 refinement to 1e-6
        dict(name="batch256_bf16_refined", path="batch", scene="batch", first=0, count=256, storage="bf16", refined=True),
        # the largest single tree: vortex tubes, 512x512x1024 effective, refinement to 1e-8
        dict(name="refined_vortex512_bf16", path="refined", scene="vortex", level=6, storage="bf16", nu=2),
        # the serving loop with 16 resident instances, bfloat16 storage, warm starts, FP64 refinement
        dict(name="serve16_bf16_warm", path="serve", scene="batch", first=100, count=16, storage="bf16"),
    ]


def draw(rng):
    path = rng.choice(["solve", "solve", "solve", "project", "krylov", "amg", "batch", "batch", "refined", "serve"])
    if path in ("batch", "serve"):
        count = max(2, int(round(2.0 ** rng.uniform(1.0, 6.5 if path == "batch" else 4.5))))
        storage = rng.choice(["f32", "bf16", "f16"] if path == "batch" else ["f32", "bf16"])
        case = dict(path=path, scene="batch", first=rng.randrange(0, 1000), count=count, storage=storage)
        if path == "batch":
            case["refined"] = storage != "f32" or rng.random() < 0.5
        return case
    if path == "refined":
        return dict(path=path, scene="vortex", level=rng.choice([4, 5, 5]), storage=rng.choice(["f32", "bf16", "f16"]),
                    nu=rng.choice([1, 2, 3]))
    scene = rng.choice(["uniform", "band", "band", "plane"])
    case = dict(path=path, scene=scene, nx=1, ny=1, nz=1, nu=rng.choice([1, 1, 2, 2, 3]))
    if scene == "uniform":
        case.update(level=rng.choice([1, 2, 3, 4]))
        case.update(zip(("nx", "ny", "nz"), rng.choice([(1, 1, 1), (2, 1, 1), (1, 3, 1), (2, 2, 1), (1, 1, 5), (3, 2, 1)])))
        if case["level"] == 4:
            case.update(nx=1, ny=1)
    else:
        case.update(level=rng.choice([3, 4, 4, 5, 5] if scene == "band" else [2, 3, 4]))
    if scene == "band":
        case.update(r=round(rng.uniform(0.08, 0.24), 4), w=round(0.3 * 2.0 ** -rng.uniform(case["level"] - 2, case["level"]), 4))
    if path == "solve":
        case.update(smoother=rng.choice(["rbgs", "rbgs", "rbgs", "jacobi"]), storage=rng.choice(["f32", "f32", "bf16", "f16"]),
                    neumann=scene == "uniform" and rng.random() < 0.3)
        if case["smoother"] == "jacobi":
            case.update(nu=max(2, case["nu"]))  # one damped-Jacobi sweep per level smooths too little to converge
    return case


# ---- trees -------------------------------------------------------------------
def _scene_args(case):
    s = case["scene"]
    if s == "vortex":
        return [dict(workloads.VORTEX512, vortex_level=[case["level"], case["level"] - 2])]
    if s == "batch":
        return [workloads.batch_scene_params(q)[0] for q in range(case["first"], case["first"] + case["count"])]
    kw = dict(nroot=[case["nx"], case["ny"], case["nz"]])
    if s == "uniform":
        kw.update(kind=ca.SCENE_UNIFORM, uniform_level=case["level"])
    elif s == "plane":
        kw.update(kind=ca.SCENE_PLANE, plane_level=[case["level"], case["level"] - 1])
    else:
        lv = case["level"]
        kw.update(kind=ca.SCENE_SPHERE_BAND, solid_r=case["r"], band_r=case["r"], band_w=[case["w"], 3 * case["w"]],
                  band_level=[lv, lv - 1, lv - 2])
    if case.get("neumann"):
        kw.update(face_bc=[ca.NEUMANN] * 6)
    return [kw]


def _freeze(v):
    return tuple(v) if isinstance(v, list) else v


@functools.lru_cache(maxsize=640)
def _tree(frozen):
    kw = {k: list(v) if isinstance(v, tuple) else v for k, v in frozen}
    if kw.get("kind") == ca.SCENE_VORTEX:
        return ca.Scene(**kw).tree
    t = ca.scene_tree_device(max_tiles=1 << 17, **kw)
    order = np.lexsort((t.coord[:, 2], t.coord[:, 1], t.coord[:, 0], t.level))  # the device build's order is not fixed
    return ca.Tree(t.h0, t.level[order], t.coord[order], t.type[order], t.cell_type[order])


def _trees(case):
    keys = [tuple(sorted((k, _freeze(v)) for k, v in kw.items())) for kw in _scene_args(case)]
    if len(keys) == 1:
        return [_tree(keys[0])]
    with ThreadPoolExecutor(max_workers=8) as ex:
        return list(ex.map(_tree, keys))


# ---- inputs ------------------------------------------------------------------
def _velocity(prob, trees, gen):
    """N(0,1) face velocities (channels 6-8), zero inside solids."""
    solid = torch.from_numpy(np.concatenate([t.cell_type for t in trees]) == ca.NEUMANN).to(DEVICE)
    out = []
    for c in (ca.CH_U, ca.CH_V, ca.CH_W):
        u = torch.randn((prob.n, 512), generator=gen, device=DEVICE)
        u.masked_fill_(solid, 0.0)
        prob.set_device(c, u.data_ptr())
        out.append(u)
    return out


def _rhs(prob, trees, gen):
    """The divergence of such a field, as a device tensor."""
    _velocity(prob, trees, gen)
    ca.VelocityVolumeDivergenceOnLeafs(prob, ca.CH_B)
    b = torch.empty((prob.n, 512), device=DEVICE)
    prob.get_device(ca.CH_B, b.data_ptr())
    torch.cuda.synchronize()
    return b


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    s.trees = _trees(case)
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    if case["path"] == "serve":
        return _prepare_server(s, gen)
    s.prob = ca.Problem.batch(s.trees)
    s.x = torch.empty((s.prob.n, 512), device=DEVICE)
    if case["path"] == "project":
        s.u = _velocity(s.prob, s.trees, gen)
        s.out = [torch.empty_like(u) for u in s.u]
        torch.cuda.synchronize()
    else:
        s.b = _rhs(s.prob, s.trees, gen)
    if case["path"] == "krylov":
        s.ab = torch.empty_like(s.x)
    s.solver = ca.GMGSolver()
    if case["path"] == "amg":
        s.solver = ca.AMGSolver()
        s.solver.prepareTypesAndCoeffs(s.prob)
    return s


def _prepare_server(s, gen):
    pool = ca.Problem.batch(s.trees)
    b = _rhs(pool, s.trees, gen)
    inside = torch.from_numpy(np.concatenate([t.cell_type for t in s.trees]) == ca.INTERIOR).to(DEVICE)
    noise = torch.randn(b.shape, generator=gen, device=DEVICE)
    b2 = 0.95 * b + 0.3 * b[inside].std() * noise * inside  # the next of a sequence of correlated steps
    s.rhs = [[q.copy() for q in pool.split(v.cpu().numpy())] for v in (b, b2)]
    pool.close()
    n = sum(t.n for t in s.trees)
    s.server = ca.Server(budget_bytes=int(n * 36e3) + (1 << 28), max_problems=len(s.trees), refine=True, level_iters=2,
                         storage=STORE[s.case["storage"]], rel_tol=1e-6, max_iters=MAX_ITERS)
    s.inst = [s.server.admit(t) for t in s.trees]
    s.turn = 0
    return s


# ---- one pass ----------------------------------------------------------------
def run(s):
    return _RUN[s.case["path"]](s, s.case)


def _run_solve(s, case):
    s.prob.set_device(ca.CH_B, s.b.data_ptr())
    iters, rel = s.solver.solve(s.prob, False, MAX_ITERS, 1e-6, case["nu"], 10, 1, case["neumann"],
                                smoother=SMOOTH[case["smoother"]], storage=STORE[case["storage"]])
    s.prob.get_device(ca.CH_X, s.x.data_ptr())
    return dict(x=s.x, iters=iters, rel=rel)


def _run_amg(s, case):
    s.prob.set_device(ca.CH_B, s.b.data_ptr())
    iters, rel = s.solver.solve(s.prob, False, MAX_ITERS, 1e-6, case["nu"], 10, 1, False)
    s.prob.get_device(ca.CH_X, s.x.data_ptr())
    return dict(x=s.x, iters=iters, rel=rel)


def _run_project(s, case):
    for c, u in zip((ca.CH_U, ca.CH_V, ca.CH_W), s.u):
        s.prob.set_device(c, u.data_ptr())
    res = s.solver.project(s.prob, max_iters=MAX_ITERS, level_iters=case["nu"])[0]
    for c, u in zip((ca.CH_U, ca.CH_V, ca.CH_W), s.out):
        s.prob.get_device(c, u.data_ptr())
    s.prob.get_device(ca.CH_X, s.x.data_ptr())
    return dict(x=s.x, u=s.out[0], v=s.out[1], w=s.out[2], iters=res["iters"], rel=res["rel_res"])


def _run_krylov(s, case):
    s.prob.set_device(ca.CH_P, s.b.data_ptr())
    s.solver.VCycle(s.prob, ca.CH_Z, ca.CH_P, level_iters=case["nu"])
    bz = s.prob.dot(ca.CH_P, ca.CH_Z)
    ca.FullNegativeLaplacian(s.prob, ca.CH_P, ca.CH_AP)
    bab = s.prob.dot(ca.CH_P, ca.CH_AP)
    s.prob.get_device(ca.CH_Z, s.x.data_ptr())
    s.prob.get_device(ca.CH_AP, s.ab.data_ptr())
    return dict(z=s.x, ab=s.ab, bz=bz, bab=bab)


def _run_batch(s, case):
    s.prob.set_device(ca.CH_B, s.b.data_ptr())
    storage = STORE[case["storage"]]
    if case["refined"]:
        res = s.solver.solve_refined(s.prob, 1e-6, 5e-7, 20, MAX_ITERS, 2, 10, storage=storage)
    else:
        res = s.solver.solve_batch(s.prob, MAX_ITERS, 1e-6, 2, 10, storage=storage)
    s.prob.get_device(ca.CH_X, s.x.data_ptr())
    return dict(x=s.x, iters=np.array([r["iters"] for r in res]), rel=np.array([r["rel_res"] for r in res]))


def _run_refined(s, case):
    s.prob.set_device(ca.CH_B, s.b.data_ptr())
    res = s.solver.solve_refined(s.prob, 1e-8, 1e-4, 20, MAX_ITERS, case["nu"], 10, storage=STORE[case["storage"]])[0]
    s.prob.get_device(ca.CH_X, s.x.data_ptr())
    return dict(x=s.x, iters=res["iters"], rel=res["rel_res"])


def _run_serve(s, case):
    rhs = s.rhs[s.turn & 1]
    s.turn += 1
    for k, i in enumerate(s.inst):
        s.server.submit(i, rhs[k], warm=True, tag=k)
    got = {}
    while len(got) < len(s.inst):
        s.server.step()
        while True:
            r = s.server.next_result(wait=False, with_x=True)
            if r is None:
                break
            got[r[0]] = r
    order = [got[k] for k in range(len(s.inst))]
    return dict(x=[r[3] for r in order], iters=np.array([r[2]["iters"] for r in order]))


_RUN = dict(solve=_run_solve, amg=_run_amg, project=_run_project, krylov=_run_krylov, batch=_run_batch,
            refined=_run_refined, serve=_run_serve)


# ---- what a pass cannot do without --------------------------------------------
def work(case):
    """Bytes: the caller's fields in and out once and the cell types once (an
    iterative solve may keep everything between on the chip).  Operations: the
    iterations the workloads take, each a V-cycle (2 nu sweeps and a residual
    per level) and a CG step."""
    trees = _trees(case)
    cells = 512.0 * sum(int((t.type == ca.LEAF).sum()) for t in trees)
    nu = case.get("nu", 2)
    fields = {"project": 3 + 4, "krylov": 1 + 2}.get(case["path"], 2)
    iters = {"krylov": 1, "refined": 50, "serve": 18}.get(case["path"], 20)
    vcycle = 8.0 / 7.0 * (2 * nu + 1) * 20.0
    return {"bytes": cells * (4 * fields + 1), "flops": cells * iters * (vcycle + 30.0)}


# ---- the pressure equation in 64 bits -------------------------------------------
def _key(level, g):
    return (level << 57) | (g[..., 0] << 38) | (g[..., 1] << 19) | g[..., 2]


class _Leaves:
    """The volume-weighted Poisson operator on the leaf cells: h (x_c - x_n)
    across a face between cells of one size or to the outside (x_n = 0), and
    (2/3) h_f (x_c - x_n) across the faces of the finer cell where sizes differ;
    no flux where either cell is NEUMANN; unknowns are the INTERIOR cells."""

    def __init__(self, tree):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)  # noqa: E731
        level, coord, self.type, ctype = t(tree.level).long(), t(tree.coord).long(), t(tree.type), t(tree.cell_type)
        self.tree, self.ctype, self.tile_level, self.coord = tree, ctype, level, coord
        self.leaf = torch.nonzero(self.type == ca.LEAF)[:, 0]
        c = torch.arange(512, device=DEVICE)
        loc = torch.stack([c >> 6, (c >> 3) & 7, c & 7], 1)
        lv = level[self.leaf].repeat_interleave(512)
        g = (coord[self.leaf][:, None, :] * 8 + loc[None]).reshape(-1, 3)
        ct = ctype[self.leaf].reshape(-1)
        n = len(lv)
        skeys, order = torch.sort(_key(lv, g))

        def find(l, p):
            k = torch.where((p < 0).any(-1) | (l < 0), torch.full_like(l, -1), _key(l.clamp(min=0), p.clamp(min=0)))
            at = torch.searchsorted(skeys, k).clamp(max=n - 1)
            return torch.where(skeys[at] == k, order[at], torch.full_like(at, -1))

        h = tree.h0 / torch.pow(2.0, lv.double())
        rows, cols, vals = [], [], []
        diag = torch.zeros(n, dtype=torch.float64, device=DEVICE)
        open_cell = ct != ca.NEUMANN
        inner = ct == ca.INTERIOR
        for a in range(3):
            for step in (-1, 1):
                q = g.clone()
                q[:, a] += step
                same = find(lv, q)
                coarse = torch.where(same < 0, find(lv - 1, q >> 1), torch.full_like(same, -1))
                far = torch.where(same >= 0, same, coarse)
                w = torch.where(same >= 0, h, (2.0 / 3.0) * h)
                # neither: the outside, or finer cells (their faces are added from their side)
                finer = find(lv + 1, 2 * q)
                outside = (far < 0) & (finer < 0)
                m = outside & inner
                diag[m] += h[m]
                m = (far >= 0) & open_cell
                m &= open_cell[far.clamp(min=0)]
                i, j, v = torch.nonzero(m)[:, 0], far[m], w[m]
                cross = coarse[m] >= 0
                k = inner[i]
                diag.index_add_(0, i[k], v[k])
                rows.append(i[k]); cols.append(j[k]); vals.append(-v[k])
                k = cross & inner[j]  # the coarse cell's row
                diag.index_add_(0, j[k], v[k])
                rows.append(j[k]); cols.append(i[k]); vals.append(-v[k])
        every = torch.arange(n, device=DEVICE)
        rows.append(every); cols.append(every); vals.append(diag)
        r, c, v = torch.cat(rows), torch.cat(cols), torch.cat(vals)
        v = torch.where(inner[c], v, torch.zeros_like(v))  # other cells hold 0
        self.A = torch.sparse_coo_tensor(torch.stack([r, c]), v, (n, n)).coalesce().to_sparse_csr()
        self.diag, self.inner = diag, inner

    def gather(self, field):
        return field[self.leaf].reshape(-1).double()

    def scatter(self, v, ghosts=False):
        out = torch.zeros((self.tree.n, 512), dtype=torch.float64, device=DEVICE)
        out[self.leaf] = v.reshape(-1, 512)
        if ghosts:  # a ghost cell takes its parent cell's value where both are INTERIOR
            ids = {(int(l),) + tuple(c): i for i, (l, c) in enumerate(zip(self.tree.level.tolist(), self.tree.coord.tolist()))}
            gt = np.nonzero(self.tree.type == ca.GHOST)[0]
            par = np.array([ids[(int(self.tree.level[i]) - 1,) + tuple(x >> 1 for x in self.tree.coord[i].tolist())] for i in gt])
            cc = np.arange(512)
            for i, p in zip(gt, par):
                o = self.tree.coord[i] & 1
                pc = (((o[0] * 4 + (cc >> 7)) << 6) | ((o[1] * 4 + ((cc >> 4) & 3)) << 3) | (o[2] * 4 + ((cc >> 1) & 3)))
                both = (self.tree.cell_type[i] == ca.INTERIOR) & (self.tree.cell_type[p][pc] == ca.INTERIOR)
                out[i] = torch.where(torch.from_numpy(both).to(DEVICE), out[p][torch.from_numpy(pc).to(DEVICE)], 0.0)
        return out

    def solve(self, b, tol=1e-12, most=20000):
        b = torch.where(self.inner, b, torch.zeros_like(b))
        inv = torch.where(self.diag > 0, 1.0 / self.diag, torch.zeros_like(self.diag))
        x, r = torch.zeros_like(b), b.clone()
        z = inv * r
        p, rz, stop = z.clone(), torch.dot(r, z), tol * torch.linalg.vector_norm(b)
        for it in range(most):
            ap = torch.mv(self.A, p)
            alpha = rz / torch.dot(p, ap)
            x += alpha * p
            r -= alpha * ap
            if it % 25 == 0 and bool(torch.linalg.vector_norm(r) <= stop):
                return x
            z = inv * r
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
        return None


def exact(case, seed):
    trees = _trees(case)
    path = case["path"]
    if sum(int((t.type == ca.LEAF).sum()) for t in trees) > EXACT_LEAF_TILES or case.get("neumann"):
        return None  # too large; or determined up to a constant only
    s = prepare(case, seed)
    if path == "project":
        return dict(x=_pressure_of_velocity(s), u=None, v=None, w=None, iters=None, rel=None)
    if path == "serve":
        bs = [torch.from_numpy(v).to(DEVICE) for v in s.rhs[0]]
    else:
        bs = s.prob.split(s.b)
    if path == "krylov":
        L = _Leaves(trees[0])
        b = L.gather(bs[0])
        ab = torch.where(L.inner, torch.mv(L.A, b), torch.zeros_like(b))
        return dict(z=None, ab=None, bz=None, bab=float(torch.dot(b, ab)))
    xs = []
    for t, b in zip(trees, bs):
        L = _Leaves(t)
        x = L.solve(L.gather(b))
        if x is None:
            return None
        xs.append(L.scatter(x))
    if path == "serve":
        return dict(x=[x.cpu().numpy() for x in xs], iters=None)
    return dict(x=torch.cat(xs), iters=None, rel=None)


def _pressure_of_velocity(s):
    """The projection's pressure: the divergence of the velocities as the rhs."""
    for c, u in zip((ca.CH_U, ca.CH_V, ca.CH_W), s.u):
        s.prob.set_device(c, u.data_ptr())
    ca.VelocityVolumeDivergenceOnLeafs(s.prob, ca.CH_B)
    b = torch.empty_like(s.x)
    s.prob.get_device(ca.CH_B, b.data_ptr())
    torch.cuda.synchronize()
    L = _Leaves(s.trees[0])
    x = L.solve(L.gather(b))
    return None if x is None else L.scatter(x, ghosts=True)
