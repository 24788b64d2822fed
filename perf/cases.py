"""The work that a program using panopaea_amd has it do, as cases that can be timed.

Eight kinds, each through the package's public calls:

- "dec":       the Manifold2d operators of one 2D grid, one call each;
- "explicit":  the step's explicit operators by themselves (advection of cells
               and faces, divergence, the pressure operator, projection);
- "scene":     one step of the reference example's scene (f64, obstacle mask,
               identity-preconditioned CG with the absolute stop test);
- "step":      pano_fluid_step with the Jacobi or the multigrid preconditioner;
- "solve":     the preconditioned CG on a given right-hand side;
- "mixed":     the FP64 solve by FP32 inner iterations;
- "batch":     steps of many uneven 2D grids together, then their states;
- "serve":     projection requests through the server, from submit to fetch.

Device fields are torch tensors that the calls are given the addresses of, as
a program that keeps its data in torch would do. listed() names the cases,
draw() gives others of the same ranges, prepare() makes what a program has in
hand before the call, run() is one pass, exact() the same pass in 64 bits by
plain torch and numpy.
"""
import ctypes
import math
import random

import numpy as np
import torch

import panopaea_amd as pa
from panopaea_amd import _lib
from panopaea_amd import scenes
from panopaea_amd import workloads as W

OPEN_TOP = 32  # the z+ side open, every other side a wall


def listed():
    return [
        # A handful of operator calls on a small grid: what a program that builds its own solver
        # out of Manifold2d calls waits for is the launches.
        dict(name="dec_2d_130x97_f64", kind="dec", ny=130, nx=97, f64=True),
        # The explicit operators on an odd 3D grid, f32, a side open: odd rows, ragged tiles.
        dict(name="explicit_3d_odd_f32", kind="explicit", nz=125, ny=131, nx=193, f64=False, bc=OPEN_TOP, cells=1.0),
        # The reference's example program: 128^2, f64, obstacle, at most 100 plain CG iterations.
        dict(name="scene_128_f64", kind="scene", n=128),
        # The repository's smallest step workload: 128^2 closed box, Jacobi, hundreds of iterations.
        dict(name="step_2d_128_jacobi_f32", kind="step", nz=1, ny=128, nx=128, f64=False, bc=0, precond="jacobi",
             levels=0, tol=1e-6),
        # The same in f64 on a ragged, larger grid (no power of two, odd width).
        dict(name="step_2d_150x203_jacobi_f64", kind="step", nz=1, ny=150, nx=203, f64=True, bc=0, precond="jacobi",
             levels=0, tol=1e-6),
        # A large single 2D grid with multigrid: the largest 2D side the serving mix asks for.
        dict(name="step_2d_1024_mg_f32", kind="step", nz=1, ny=1024, nx=1024, f64=False, bc=0, precond="mg",
             levels=4, tol=1e-6),
        # A small smoke plume (previews, tests): the same launches as the large one, little work in each.
        dict(name="step_3d_64_mg_f32", kind="step", nz=64, ny=64, nx=64, f64=False, bc=OPEN_TOP, precond="mg",
             levels=4, tol=1e-6),
        # The flagship step: the 256^3 smoke plume.
        dict(name="step_3d_256_mg_f32", kind="step", nz=256, ny=256, nx=256, f64=False, bc=OPEN_TOP, precond="mg",
             levels=4, tol=1e-6),
        # A pressure solve in f64, the reference's own precision, to a tight tolerance.
        dict(name="solve_3d_128_mg_f64", kind="solve", nz=128, ny=128, nx=128, f64=True, bc=OPEN_TOP, precond="mg",
             levels=4, tol=1e-10),
        # The largest problem: 512^3 cells to 1e-10 by FP32 solves inside an FP64 loop.
        dict(name="mixed_512", kind="mixed", nz=512, ny=512, nx=512, bc=0),
        # The batch of 64 uneven 2D grids, its 20 steps, and every grid's state afterwards.
        dict(name="batch_64_2d", kind="batch", count=64, steps=20),
        # Two dozen requests of the serving mix (2D squares to 1024, 3D cubes to 256), host to host.
        dict(name="serve_24_mixed", kind="serve", count=24, mix=11),
    ]


def _logint(rng, lo, hi, step=1):
    """An integer in [lo, hi], a multiple of `step`, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["dec", "explicit", "scene", "step_jacobi", "step_mg2", "step_mg3", "solve", "solve_jacobi",
                       "mixed", "batch", "serve"])
    f64 = rng.random() < 0.4
    if kind == "dec":
        return dict(kind="dec", ny=_logint(rng, 16, 2048), nx=_logint(rng, 16, 2048), f64=f64)
    if kind == "explicit":
        # departures from a fraction of a cell to a few cells
        cells = rng.uniform(0.2, 3.0)
        if rng.random() < 0.4:
            return dict(kind="explicit", nz=1, ny=_logint(rng, 16, 2048), nx=_logint(rng, 16, 2048), f64=f64,
                        bc=rng.randrange(16), cells=cells)
        return dict(kind="explicit", nz=_logint(rng, 12, 200), ny=_logint(rng, 12, 200), nx=_logint(rng, 12, 200),
                    f64=f64, bc=rng.randrange(64), cells=cells)
    if kind == "scene":
        return dict(kind="scene", n=rng.randint(96, 192))
    if kind == "step_jacobi":
        return dict(kind="step", nz=1, ny=_logint(rng, 24, 300), nx=_logint(rng, 24, 300), f64=f64,
                    bc=rng.choice([0, 0, 8, 1]), precond="jacobi", levels=0, tol=1e-6)
    if kind == "step_mg2":
        return dict(kind="step", nz=1, ny=_logint(rng, 64, 1536, 8), nx=_logint(rng, 64, 1536, 8), f64=f64,
                    bc=rng.choice([0, 0, 8]), precond="mg", levels=4, tol=1e-6)
    if kind == "step_mg3":
        return dict(kind="step", nz=_logint(rng, 32, 224, 8), ny=_logint(rng, 32, 224, 8),
                    nx=_logint(rng, 32, 224, 8), f64=False, bc=rng.choice([0, OPEN_TOP]), precond="mg", levels=4,
                    tol=1e-6)
    if kind == "solve":
        if rng.random() < 0.3:
            return dict(kind="solve", nz=1, ny=_logint(rng, 64, 1024, 8), nx=_logint(rng, 64, 1024, 8), f64=True,
                        bc=rng.choice([0, 8]), precond="mg", levels=4, tol=1e-10)
        return dict(kind="solve", nz=_logint(rng, 32, 192, 8), ny=_logint(rng, 32, 192, 8),
                    nx=_logint(rng, 32, 192, 8), f64=True, bc=rng.choice([0, OPEN_TOP]), precond="mg", levels=4,
                    tol=1e-10)
    if kind == "solve_jacobi":
        return dict(kind="solve", nz=_logint(rng, 12, 72), ny=_logint(rng, 12, 72), nx=_logint(rng, 12, 72), f64=f64,
                    bc=rng.choice([0, OPEN_TOP]), precond=rng.choice(["jacobi", "identity"]), levels=0,
                    tol=1e-9 if f64 else 1e-5)
    if kind == "mixed":
        return dict(kind="mixed", nz=_logint(rng, 64, 320, 8), ny=_logint(rng, 64, 320, 8),
                    nx=_logint(rng, 64, 320, 8), bc=rng.choice([0, OPEN_TOP]))
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(3, 64), steps=rng.randint(5, 20))
    return dict(kind="serve", count=rng.randint(2, 24), mix=rng.randrange(1 << 16))


# ---- what a program has in hand ---------------------------------------------------------


class Field:
    """A torch tensor as a field of a grid: what the package's calls take."""

    def __init__(self, grid, n, dtype=None):
        self.grid = grid
        self.n = int(n)
        self.ctx = grid._ctx()
        self.dtype = np.dtype(dtype or grid.dtype)
        kind = {"float32": torch.float32, "float64": torch.float64, "uint8": torch.uint8}[self.dtype.name]
        self.t = torch.zeros(self.n, dtype=kind, device="cuda")
        torch.cuda.synchronize()  # the package's calls run on a stream of their own
        self.ptr = ctypes.c_void_p(self.t.data_ptr())

    def set(self, values):
        self.t.copy_(torch.as_tensor(values, device="cuda").reshape(-1))
        torch.cuda.synchronize()
        return self


class State:
    pass


def _bc(mask):
    return tuple((mask >> i) & 1 for i in range(6))


def _grid(case, f64=None):
    f64 = case.get("f64", True) if f64 is None else f64
    dtype = np.float64 if f64 else np.float32
    if case.get("nz", 1) > 1:
        return pa.Grid3d((case["nz"], case["ny"], case["nx"]), dtype, bc=_bc(case["bc"]))
    return pa.Grid2d((case["ny"], case["nx"]), dtype, bc=_bc(case.get("bc", 0)))


def _dims(case):
    d = case.get("nz", 1)
    return (d, case["ny"], case["nx"])


def _faces_count(d, h, w):
    return (h + 1) * w + h * (w + 1) if d == 1 else (d + 1) * h * w + d * (h + 1) * w + d * h * (w + 1)


def _density(d, h, w, seed):
    """A few smooth puffs of smoke, made from the seed: values in [0, 1]."""
    rng = random.Random(1000003 * seed + 17)
    z, y, x = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5 for n in (d, h, w))
    rho = torch.zeros((d, h, w), dtype=torch.float64, device="cuda")
    for _ in range(4):
        s = rng.uniform(0.05, 0.15) * w
        ez, ey, ex = (torch.exp(-(v - rng.uniform(0.2, 0.8) * n) ** 2 / (2 * s * s))
                      for v, n in ((z, d), (y, h), (x, w)))
        rho += ez[:, None, None] * ey[None, :, None] * ex[None, None, :]
    return rho.clamp_(max=1.0).reshape(-1)


def _velocity(grid, seed, n_modes, k_max, amplitude=1.0):
    """A smooth seeded velocity, as the repository's workloads start from."""
    f = Field(grid, grid.num_elem_1())
    pa.gen_bandlimited_faces_device(f, seed, n_modes, k_max, amplitude)
    grid._ctx().synchronize()
    return f


def _modes(case):
    # the mode counts of the 2D and the 3D workloads
    return (32, 16.0) if case.get("nz", 1) > 1 else (16, 8.0)


def _preconditioner(case):
    if case["precond"] == "mg":
        return pa.Multigrid(case["levels"], 2)
    return pa.Jacobi() if case["precond"] == "jacobi" else pa.Identity()


def _step_config(case):
    dt = 0.5 / case["nx"]
    kw = {}
    if case.get("nz", 1) > 1:  # the smoke plume: a source sphere near the bottom, buoyancy
        kw = dict(buoyancy=1.0, src_radius=0.08 * case["nx"],
                  src_center=(0.1 * case["nz"], case["ny"] / 2.0, case["nx"] / 2.0))
    return pa.StepConfig(dt=dt, preconditioner=_preconditioner(case), tol=case["tol"], tol_kind="rel",
                         max_iterations=4000, **kw)


def _explicit_dt(case):
    # departures of about case["cells"] cells at the velocity's peaks (16 to 32 modes of amplitude 1)
    return case["cells"] / (6.0 if case.get("nz", 1) > 1 else 5.0)


def _batch_grids(case):
    return W.batch_grids(dict(W.BATCH64_2D, count=case["count"]))


def _serve_grids(case):
    """Sizes of the serving mix: 70% 2D squares, 30% 3D cubes, in their order of arrival."""
    wl, rng, out = W.SERVE, random.Random(case["mix"]), []
    for _ in range(case["count"]):
        two = rng.random() < wl["p2d"]
        lo, hi = wl["n2d"] if two else wl["n3d"]
        n = lo + wl["step"] * rng.randrange((hi - lo) // wl["step"] + 1)
        dims = (n, n) if two else (n, n, n)
        out.append(dict(dims=dims, dt=0.5 / n, bc=_bc(0 if two else OPEN_TOP)))
    return out


def prepare(case, seed):
    s = State()
    s.case, s.kind = case, case["kind"]
    globals()["_prepare_" + s.kind](s, case, seed)
    pa.default_context().synchronize()
    torch.cuda.synchronize()
    return s


def _prepare_dec(s, case, seed):
    s.grid = g = _grid(dict(case, nz=1))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n0, n1, n2 = g.num_elem_0(), g.num_elem_1(), g.num_elem_2()
    s.v, s.e, s.c = Field(g, n0), Field(g, n1), Field(g, n2)
    for f in (s.v, s.e, s.c):
        f.t.normal_(generator=gen)
    s.out = {k: Field(g, n) for k, n in
             dict(v_dual=n0, v_primal=n0, e_dual=n1, e_primal=n1, c_dual=n2, d0=n1, d1=n2, g_dual=n1, g=n1,
                  lap=n2).items()}


def _prepare_explicit(s, case, seed):
    s.grid = g = _grid(case)
    s.dt = _explicit_dt(case)
    s.vel = _velocity(g, seed, *_modes(case))
    s.rho = Field(g, g.num_elem_2()).set(_density(*_dims(case), seed))
    s.p = Field(g, g.num_elem_2()).set(_density(*_dims(case), seed + 1))
    s.op = pa.PoissonOperator(g, s.dt)
    s.rho2, s.b, s.q = (Field(g, g.num_elem_2()) for _ in range(3))
    s.vel2 = Field(g, g.num_elem_1())


def _prepare_scene(s, case, seed):
    n = case["n"]
    s.grid = g = pa.Grid2d((n, n), np.float64)
    s.dt = 0.05  # the example's step, threshold and iteration limit
    s.mask = Field(g, g.num_elem_1(), np.uint8).set(scenes.obstacle_mask(n, n))
    s.op = pa.PoissonOperator(g, s.dt, s.mask)
    s.vel = _velocity(g, seed, 16, 8.0)
    s.rho = Field(g, g.num_elem_2()).set(_density(1, n, n, seed))
    (y0, y1), (x0, x1) = scenes.INFLOW_ROWS, scenes.INFLOW_COLS
    s.rho.t.view(n, n)[y0:y1, x0:x1] = 1.0
    s.vel.t[:(n + 1) * n].view(n + 1, n)[y0:y1, x0:x1] = 20.0
    s.rho2, s.b, s.p, s.r, s.a, s.s = (Field(g, g.num_elem_2()) for _ in range(6))
    s.vel2 = Field(g, g.num_elem_1())


def _prepare_step(s, case, seed):
    s.grid = g = _grid(case)
    s.cfg = _step_config(case)
    s.vel = _velocity(g, seed, *_modes(case))
    s.rho = Field(g, g.num_elem_2()).set(_density(*_dims(case), seed))
    s.rho2, s.p = Field(g, g.num_elem_2()), Field(g, g.num_elem_2())
    s.vel2 = Field(g, g.num_elem_1())


def _prepare_solve(s, case, seed):
    s.grid = g = _grid(case)
    vel = _velocity(g, seed, *_modes(case))
    s.pre = _preconditioner(case)
    s.op = pa.PoissonOperator(g, 0.5 / case["nx"])
    s.b, s.x, s.r, s.a, s.s = (Field(g, g.num_elem_2()) for _ in range(5))
    pa.neg_divergence(s.b, vel)
    g._ctx().synchronize()


def _prepare_mixed(s, case, seed):
    # rough data: b = -div u of independent uniform face values
    s.grid = g = _grid(case, f64=True)
    u = Field(g, g.num_elem_1())
    pa.gen_uniform_faces_device(u, seed)
    s.b, s.x = Field(g, g.num_elem_2()), Field(g, g.num_elem_2())
    pa.neg_divergence(s.b, u)
    g._ctx().synchronize()


def _batch_state(g, i, seed):
    """Host density and velocity of grid i."""
    h, w = g["dims"]
    grid = pa.Grid2d(g["dims"], np.float32, bc=g["bc"])
    vel = _velocity(grid, 64 * seed + i, 16, 8.0).t.cpu().numpy()
    return _density(1, h, w, 64 * seed + i).float().cpu().numpy(), vel


def _prepare_batch(s, case, seed):
    grids = _batch_grids(case)
    s.batch = pa.Batch(grids, tol=1e-6)
    cells = [g["dims"][0] * g["dims"][1] for g in grids]
    faces = [_faces_count(1, *g["dims"]) for g in grids]
    s.co, s.fo = (np.concatenate([[0], np.cumsum(v)]) for v in (cells, faces))
    s.rho, s.vel = np.zeros(s.co[-1], np.float32), np.zeros(s.fo[-1], np.float32)
    for i, g in enumerate(grids):
        s.batch.set_state(i, *_batch_state(g, i, seed))


def _serve_faces(g, i, seed):
    three = len(g["dims"]) == 3
    grid = (pa.Grid3d if three else pa.Grid2d)(g["dims"], np.float32, bc=g["bc"])
    return _velocity(grid, 64 * seed + i, *((32, 16.0) if three else (16, 8.0))).t.cpu().numpy()


def _prepare_serve(s, case, seed):
    s.grids = _serve_grids(case)
    s.faces = [_serve_faces(g, i, seed) for i, g in enumerate(s.grids)]
    s.server = pa.Server(hbm_budget=8 << 30)


# ---- one pass --------------------------------------------------------------------------


def run(s):
    return globals()["_run_" + s.kind](s)


def _run_dec(s):
    g, o = s.grid, s.out
    g.hodge_0_primal(o["v_dual"], s.v)
    g.hodge_2_dual(o["v_primal"], s.v)
    g.hodge_1_primal(o["e_dual"], s.e)
    g.hodge_1_dual(o["e_primal"], s.e)
    g.derivative_0_primal(o["d0"], s.v)
    g.derivative_1_primal(o["d1"], s.e)
    # the Laplacian of a cell field, operator by operator
    g.hodge_2_primal(o["c_dual"], s.c)
    g.derivative_0_dual(o["g_dual"], o["c_dual"])
    g.hodge_1_dual(o["g"], o["g_dual"])
    g.derivative_1_primal(o["lap"], o["g"])
    return {k: f.t for k, f in o.items()}


def _run_explicit(s):
    pa.advect(s.rho2, s.rho, s.dt, s.vel)
    pa.advect_mac(s.vel2, s.vel, s.dt, s.vel)
    pa.neg_divergence(s.b, s.vel2)
    s.op(s.q, s.p)
    pa.project(s.vel2, s.p, s.dt)
    return [s.rho2.t, s.vel2.t, s.b.t, s.q.t]


def _run_scene(s):
    pa.advect(s.rho2, s.rho, s.dt, s.vel)
    pa.advect_mac(s.vel2, s.vel, s.dt, s.vel)
    pa.neg_divergence(s.b, s.vel2, s.mask)
    info = pa.precond_conjugate_gradient(pa.Identity(), s.p, s.b, 100, 0.1, s.r, s.a, s.s, s.op, tol_kind="abs",
                                         remove_mean=0)
    pa.project(s.vel2, s.p, s.dt)
    return dict(rho=s.rho2.t, vel=s.vel2.t, b=s.b.t, p=s.p.t, iterations=int(info.iterations))


def _run_step(s):
    info = pa.fluid_step(s.grid, s.cfg, s.rho, s.vel, s.rho2, s.vel2, s.p)
    return dict(rho=s.rho2.t, vel=s.vel2.t, p=s.p.t, iterations=int(info.iterations))


def _run_solve(s):
    info = pa.precond_conjugate_gradient(s.pre, s.x, s.b, 4000, s.case["tol"], s.r, s.a, s.s, s.op, tol_kind="rel")
    return dict(x=s.x.t, iterations=int(info.iterations))


def _run_mixed(s):
    info = pa.poisson_solve_mixed(s.x, s.b, dt=1.0, preconditioner=pa.Multigrid(4, 2), inner_tol=1e-4,
                                  outer_tol=1e-10)
    return dict(x=s.x.t, outer=int(info.outer_iterations), inner=int(info.inner_iterations))


def _run_batch(s):
    its = [s.batch.step() for _ in range(s.case["steps"])]
    get = _lib.lib().pano_batch_get_state
    for i in range(s.case["count"]):  # into the program's own arrays
        _lib.check(get(s.batch.handle, i, s.rho.ctypes.data + 4 * int(s.co[i]), s.vel.ctypes.data + 4 * int(s.fo[i])))
    return dict(rho=s.rho, vel=s.vel, iterations=np.array(its, np.int32))


def _run_serve(s):
    ids = [s.server.submit(g, faces=f) for g, f in zip(s.grids, s.faces)]
    got = {}

    def done(rid):
        got[rid] = s.server.fetch(rid) + (s.server.status(rid)["iterations"],)
        s.server.release(rid)

    s.server.run_until_idle(on_done=done)
    return dict(vel=[got[r][0] for r in ids], p=[got[r][1] for r in ids],
                iterations=np.array([got[r][2] for r in ids], np.int32))


# ---- what a pass cannot do without -------------------------------------------------------


def work(case):
    """Bytes: each input read once and each output written once. Operations: those of one
    evaluation of each output; for a solve, one fast direct solve (about 50 per cell)."""
    kind = case["kind"]
    el = 8 if case.get("f64", kind in ("scene", "mixed")) else 4
    if kind == "batch":
        c = sum(g["dims"][0] * g["dims"][1] for g in _batch_grids(case))
        return {"bytes": 4.0 * 6 * c, "flops": 150.0 * c * case["steps"]}
    if kind == "serve":
        c = f = 0
        for g in _serve_grids(case):
            d = tuple(g["dims"])
            c += math.prod(d)
            f += _faces_count(*((1,) + d if len(d) == 2 else d))
        return {"bytes": 4.0 * (2 * f + c), "flops": 70.0 * c}
    d, h, w = (1, case["n"], case["n"]) if kind == "scene" else _dims(case)
    c, f = d * h * w, _faces_count(d, h, w)
    if kind == "dec":
        v = (h + 1) * (w + 1)
        return {"bytes": float(el) * ((v + f + c) + (2 * v + 5 * f + 3 * c)), "flops": 10.0 * c}
    adv = 30.0 if d == 1 else 60.0  # an interpolated value and its departure point
    if kind == "explicit":
        return {"bytes": float(el) * (2 * f + 5 * c), "flops": adv * (c + f) + 20.0 * c}
    if kind == "scene":
        return {"bytes": float(el) * (2 * f + 4 * c) + f, "flops": adv * (c + f) + 70.0 * c}
    if kind == "step":
        return {"bytes": float(el) * (2 * f + 3 * c), "flops": adv * (c + f) + 70.0 * c}
    return {"bytes": float(el) * 2 * c, "flops": 50.0 * c}


# ---- the same in 64 bits -----------------------------------------------------------------


def exact(case, seed):
    return globals()["_exact_of_" + case["kind"]](case, seed)


def _split(f, d, h, w):
    """(z, y, x) face components of a flat face array, as 3D arrays (z None in 2D)."""
    nz = (d + 1) * h * w if d > 1 else 0
    ny = d * (h + 1) * w
    z = f[:nz].view(d + 1, h, w) if d > 1 else None
    return z, f[nz:nz + ny].view(d, h + 1, w), f[nz + ny:].view(d, h, w + 1)


def _join(z, y, x):
    return torch.cat([t.reshape(-1) for t in (z, y, x) if t is not None])


def _gather(q, axes):
    """Multilinear interpolation of q at the (lower index, upper index, weight) of each axis."""
    n1, n2 = q.shape[1], q.shape[2]
    flat, out = q.reshape(-1), 0.0
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                wt = 1.0
                for k, hi in zip((0, 1, 2), (a, b, c)):
                    wt = wt * (axes[k][2] if hi else 1.0 - axes[k][2])
                out = out + wt * flat[(axes[0][a] * n1 + axes[1][b]) * n2 + axes[2][c]]
    return out


def _mean4(q, axis_pair, lo, hi):
    """Sum over a face pair along axis_pair and the two cells lo, hi along the other axis, / 4."""
    ax, other = axis_pair
    n = q.shape[ax] - 1
    s = q.narrow(ax, 0, n) + q.narrow(ax, 1, n)
    return (s.index_select(other, lo) + s.index_select(other, hi)) / 4.0


def _cell_axis(p, n):
    if n == 1:
        z = torch.zeros_like(p, dtype=torch.long)
        return z, z, torch.zeros_like(p)
    p = torch.clamp(p - 0.5, min=0.0).clamp_(max=n - 1.00001)
    i = torch.floor(p)
    return i.long(), (i + 1).long().clamp_(max=n - 1), p - i


def _face_axis(p, off, nmax):
    i = torch.floor(p - off).clamp_(0, nmax + 1)
    return i.long().clamp(max=nmax), (i + 1).long().clamp(max=nmax), (p - off - i).clamp(0, 1)


def _exact_advect(rho, vel, d, h, w, dt):
    """Semi-Lagrangian advection of cells and faces by the same velocity; flat f64 tensors in and out."""
    vz, vy, vx = _split(vel, d, h, w)
    dev = vel.device
    idx = lambda n: torch.arange(n, device=dev, dtype=torch.float64)  # noqa: E731
    cz, cy, cx = idx(d)[:, None, None], idx(h)[None, :, None], idx(w)[None, None, :]
    zero = torch.zeros((), dtype=torch.float64, device=dev)
    ux, uy = (vx[:, :, :-1] + vx[:, :, 1:]) / 2, (vy[:, :-1] + vy[:, 1:]) / 2
    uz = (vz[:-1] + vz[1:]) / 2 if d > 1 else zero
    shape = (d, h, w)
    full = lambda t, sh: t.expand(sh).contiguous()  # noqa: E731
    r = rho.view(shape)
    rho2 = _gather(r, [_cell_axis(full(cz + 0.5 - dt * uz, shape), d), _cell_axis(cy + 0.5 - dt * uy, h),
                       _cell_axis(cx + 0.5 - dt * ux, w)])

    def pair(n):  # cells on the two sides of each of n + 1 faces, clamped
        a = torch.arange(n + 1, device=dev)
        return a.clamp(max=n - 1), (a - 1).clamp(min=0)

    def zaxis(p, sh):
        return _face_axis(full(p, sh), 0.5, d - 1) if d > 1 else _cell_axis(full(p, sh) * 0, 1)

    fx, fy, fz = idx(w + 1)[None, None, :], idx(h + 1)[None, :, None], idx(d + 1)[:, None, None]
    # x faces
    sh = (d, h, w + 1)
    ay = _mean4(vy, (1, 2), *pair(w))
    az = _mean4(vz, (0, 2), *pair(w)) if d > 1 else zero
    x2 = _gather(vx, [zaxis(cz + 0.5 - dt * az, sh), _face_axis(full(cy + 0.5 - dt * ay, sh), 0.5, h - 1),
                      _face_axis(full(fx - dt * vx, sh), 0.0, w)])
    # y faces
    sh = (d, h + 1, w)
    ax = _mean4(vx, (2, 1), *pair(h))
    az = _mean4(vz, (0, 1), *pair(h)) if d > 1 else zero
    y2 = _gather(vy, [zaxis(cz + 0.5 - dt * az, sh), _face_axis(full(fy - dt * vy, sh), 0.0, h),
                      _face_axis(full(cx + 0.5 - dt * ax, sh), 0.5, w - 1)])
    z2 = None
    if d > 1:
        sh = (d + 1, h, w)
        ax, ay = _mean4(vx, (2, 0), *pair(d)), _mean4(vy, (1, 0), *pair(d))
        z2 = _gather(vz, [_face_axis(full(fz - dt * vz, sh), 0.0, d),
                          _face_axis(full(cy + 0.5 - dt * ay, sh), 0.5, h - 1),
                          _face_axis(full(cx + 0.5 - dt * ax, sh), 0.5, w - 1)])
    return rho2.reshape(-1), _join(z2, y2, x2)


def _exact_neg_div(vel, d, h, w):
    vz, vy, vx = _split(vel, d, h, w)
    div = vy[:, 1:] - vy[:, :-1] + vx[:, :, 1:] - vx[:, :, :-1]
    if d > 1:
        div = div + vz[1:] - vz[:-1]
    return -div.reshape(-1)


def _gradient(p, d, h, w, bc):
    """Dual derivative of the cell field on every face: 0 on walls, p = 0 outside open sides."""
    p = p.view(d, h, w)
    out = []
    for axis, lo, hi in ((0, 4, 5), (1, 2, 3), (2, 0, 1)):
        if axis == 0 and d == 1:
            out.append(None)
            continue
        first, last = p.narrow(axis, 0, 1), p.narrow(axis, p.shape[axis] - 1, 1)
        g = torch.cat([-first * (1.0 if bc >> lo & 1 else 0.0), p.narrow(axis, 0, p.shape[axis] - 1) -
                       p.narrow(axis, 1, p.shape[axis] - 1), last * (1.0 if bc >> hi & 1 else 0.0)], axis)
        out.append(g)
    return out


def _exact_apply(p, d, h, w, bc, dt):
    gz, gy, gx = _gradient(p, d, h, w, bc)
    # the operator is dt times minus the divergence of minus the gradient
    return -dt * _exact_neg_div(_join(gz, gy, gx), d, h, w)


def _exact_project(vel, p, d, h, w, bc, dt):
    g = _gradient(p, d, h, w, bc)
    out = []
    for axis, (u, q) in enumerate(zip(_split(vel, d, h, w), g)):
        if u is None:
            out.append(None)
            continue
        r = u + dt * q
        lo, hi = ((4, 5), (2, 3), (0, 1))[axis]
        if not bc >> lo & 1:
            r.narrow(axis, 0, 1).zero_()
        if not bc >> hi & 1:
            r.narrow(axis, r.shape[axis] - 1, 1).zero_()
        out.append(r)
    return _join(*out)


def _basis(n, lo, hi, dev):
    """Eigenvectors (columns) and eigenvalues of the 1D operator with walls or open sides."""
    j = torch.arange(n, dtype=torch.float64, device=dev)[:, None]
    k = torch.arange(n, dtype=torch.float64, device=dev)[None, :]
    if not lo and not hi:
        th = math.pi * k / n
        V = torch.cos(th * (j + 0.5))
    elif lo and hi:
        th = math.pi * (k + 1) / (n + 1)
        V = torch.sin(th * (j + 1))
    else:
        th = math.pi * (2 * k + 1) / (2 * n + 1)
        V = torch.cos(th * ((n - 1 - j if lo else j) + 0.5))
    return V / V.norm(dim=0, keepdim=True), (2.0 - 2.0 * torch.cos(th)).reshape(-1)


def _exact_solve(b, d, h, w, bc, dt):
    """The pressure of dt A p = b by diagonalisation (of zero mean in a closed box)."""
    dev = b.device
    Vz, lz = _basis(d, bc >> 4 & 1, bc >> 5 & 1, dev) if d > 1 else (torch.ones((1, 1), dtype=torch.float64,
                                                                                device=dev), torch.zeros(
        1, dtype=torch.float64, device=dev))
    Vy, ly = _basis(h, bc >> 2 & 1, bc >> 3 & 1, dev)
    Vx, lx = _basis(w, bc & 1, bc >> 1 & 1, dev)
    t = b.view(d * h, w) @ Vx
    t = torch.stack([Vy.T @ m for m in t.view(d, h, w)])
    t = (Vz.T @ t.view(d, h * w)).view(d, h, w)
    lam = lz[:, None, None] + ly[None, :, None] + lx[None, None, :]
    t = torch.where(lam > 1e-12, t / (dt * lam).clamp_(min=1e-300), torch.zeros_like(t))
    t = (Vz @ t.view(d, h * w)).view(d, h, w)
    t = torch.stack([Vy @ m for m in t])
    return (t.view(d * h, w) @ Vx.T).reshape(-1)


def _exact_of_dec(case, seed):
    s = prepare(case, seed)
    h, w = case["ny"], case["nx"]
    v, e, c = (f.t.double() for f in (s.v, s.e, s.c))
    V = v.view(h + 1, w + 1)

    def star(side, corner):
        # the example's vertex star: its side factors, and its corner factor at the corners it reaches;
        # vertices it does not write keep what was there (zero)
        o = torch.zeros_like(V)
        o[1:-1, 1:-1] = V[1:-1, 1:-1]
        for y, x in ((0, 0), (0, w - 1), (h - 1, 0), (h - 1, w - 1)):
            o[y, x] = V[y, x] * corner
        for sl in ((0, slice(1, -1)), (h, slice(1, -1)), (slice(1, -1), 0), (slice(1, -1), w)):
            o[sl] = V[sl] * side
        o[1:-1, 1:-1] = V[1:-1, 1:-1]
        return o.reshape(-1)

    ny = (h + 1) * w
    ey, ex = e[:ny].view(h + 1, w), e[ny:].view(h, w + 1)

    def d1(y, x):
        return (y[:-1] - y[1:] - x[:, :-1] + x[:, 1:]).reshape(-1)

    C = c.view(h, w)
    gy, gx = torch.zeros_like(ey), torch.zeros_like(ex)
    gy[1:-1] = -(C[1:] - C[:-1])
    gx[:, 1:-1] = C[:, :-1] - C[:, 1:]
    j = lambda a, b: torch.cat([a.reshape(-1), b.reshape(-1)])  # noqa: E731
    return dict(v_dual=star(0.5, 0.25), v_primal=star(2.0, 4.0), e_dual=j(ey, -ex), e_primal=j(-ey, ex), c_dual=c,
                d0=j(V[:, 1:] - V[:, :-1], V[1:] - V[:-1]), d1=d1(ey, ex), g_dual=j(gy, gx), g=j(-gy, gx),
                lap=d1(-gy, gx))


def _exact_of_explicit(case, seed):
    s = prepare(case, seed)
    D, bc = _dims(case), case["bc"] & (63 if case["nz"] > 1 else 15)
    rho, vel, p = s.rho.t.double(), s.vel.t.double(), s.p.t.double()
    rho2, vel2 = _exact_advect(rho, vel, *D, s.dt)
    b = _exact_neg_div(vel2, *D)
    return [rho2, _exact_project(vel2, p, *D, bc, s.dt), b, _exact_apply(p, *D, bc, s.dt)]


def _exact_of_scene(case, seed):
    # the solve stops far from its solution: what it computes has no value of its own
    s = prepare(case, seed)
    n = case["n"]
    rho2, vel2 = _exact_advect(s.rho.t, s.vel.t, 1, n, n, s.dt)
    b = _exact_neg_div(torch.where(s.mask.t != 0, vel2, torch.zeros_like(vel2)), 1, n, n)
    return dict(rho=rho2, vel=None, b=b, p=None, iterations=None)


def _exact_step_fields(rho, vel, d, h, w, bc, dt, buoyancy=0.0, sphere=None):
    if sphere is not None:
        cz, cy, cx, r = sphere
        z, y, x = (torch.arange(n, device=rho.device, dtype=torch.float64) + 0.5 for n in (d, h, w))
        inside = ((z - cz) ** 2)[:, None, None] + ((y - cy) ** 2)[None, :, None] + ((x - cx) ** 2)[None, None, :]
        rho = torch.where(inside.reshape(-1) <= r * r, torch.ones_like(rho), rho)
    rho2, vel2 = _exact_advect(rho, vel, d, h, w, dt)
    if d > 1 and buoyancy:
        z2, r = _split(vel2, d, h, w)[0], rho.view(d, h, w)
        z2[1:-1] += dt * buoyancy * 0.5 * (r[:-1] + r[1:])
        if bc >> 4 & 1:
            z2[0] += dt * buoyancy * 0.5 * r[0]
        if bc >> 5 & 1:
            z2[-1] += dt * buoyancy * 0.5 * r[-1]
    p = _exact_solve(_exact_neg_div(vel2, d, h, w), d, h, w, bc, dt)
    return rho2, _exact_project(vel2, p, d, h, w, bc, dt), p


def _exact_of_step(case, seed):
    s = prepare(case, seed)
    bc = case["bc"] & (63 if case["nz"] > 1 else 15)
    sphere = tuple(s.cfg.src_center) + (s.cfg.src_radius,) if s.cfg.src_radius > 0 else None
    rho, vel, p = _exact_step_fields(s.rho.t.double(), s.vel.t.double(), *_dims(case), bc, s.cfg.dt, s.cfg.buoyancy,
                                     sphere)
    # in a closed box the pressure is known up to a constant only
    return dict(rho=rho, vel=vel, p=p if bc else None, iterations=None)


def _exact_solve_case(case, seed, dt):
    s = prepare(case, seed)
    bc = case["bc"] & (63 if case["nz"] > 1 else 15)
    return _exact_solve(s.b.t.double(), *_dims(case), bc, dt) if bc else None


def _exact_of_solve(case, seed):
    x = _exact_solve_case(case, seed, 0.5 / case["nx"])
    return None if x is None else dict(x=x, iterations=None)


def _exact_of_mixed(case, seed):
    x = _exact_solve_case(case, seed, 1.0)
    return None if x is None else dict(x=x, outer=None, inner=None)


def _exact_of_batch(case, seed):
    rho, vel = [], []
    for i, g in enumerate(_batch_grids(case)):
        h, w = g["dims"]
        r, v = (torch.from_numpy(a).double().cuda() for a in _batch_state(g, i, seed))
        for _ in range(case["steps"]):
            r, v, _p = _exact_step_fields(r, v, 1, h, w, 0, g["dt"])
        rho.append(r)
        vel.append(v)
    return dict(rho=torch.cat(rho), vel=torch.cat(vel), iterations=None)


def _exact_of_serve(case, seed):
    vel, p = [], []
    for i, g in enumerate(_serve_grids(case)):
        d = tuple(g["dims"])
        three = len(d) == 3
        D, bc = (d if three else (1,) + d), (OPEN_TOP if three else 0)
        u = torch.from_numpy(_serve_faces(g, i, seed)).double().cuda()
        q = _exact_solve(_exact_neg_div(u, *D), *D, bc, g["dt"])
        vel.append(_exact_project(u, q, *D, bc, g["dt"]))
        p.append(q if three else None)
    return dict(vel=vel, p=p, iterations=None)
