"""Small identity and Jacobi solves end inside their one kernel (its counts say
so: one begun, none given up), also with more workgroups than a wave has lanes,
and through the step; polls that
give up at once are counted as given up, and where the rule sends a solve to
the launches nothing is counted."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu

OPEN_TOP = (0, 0, 0, 0, 0, 1)
# (1, 3): one workgroup; 128^2: 64; the others more than 64 (512^2 and 64^3 the most)
CASES = [((1, 3), (1, 0, 0, 0, 0, 0), "f4"), ((128, 128), (0,) * 6, "f4"), ((257, 256), (0,) * 6, "f8"),
         ((365, 363), (0, 0, 0, 1, 0, 0), "f4"), ((512, 512), (0,) * 6, "f4"), ((63, 65, 64), OPEN_TOP, "f8"),
         ((64, 64, 64), OPEN_TOP, "f4"), ((66, 65, 64), OPEN_TOP, "f4")]


def grid(dims, bc, dt):
    return (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, dt, bc=bc)


def run(ctx, g, solve):
    n0, a0 = ctx.cluster_counts()
    out = solve()
    n1, a1 = ctx.cluster_counts()
    return out, (n1 - n0, a1 - a0)


def cg(g, max_it=60):
    max_it = min(max_it, (g.cells + 1) // 2)  # an exact solution leaves nothing to divide by
    b = np.random.default_rng(g.cells).standard_normal(g.cells).astype(g.dtype)
    x, r, a, s = (g.new_simplex_2() for _ in range(4))
    pa.precond_conjugate_gradient(pa.Jacobi(), x, g.new_simplex_2().upload(b), max_it, 1e-30, r, a, s,
                                  pa.PoissonOperator(g, 0.05))
    return x.download()


@pytest.mark.parametrize("dims,bc,dt", CASES)
def test_gpu_cluster_ends_in_one_kernel(ctx, dims, bc, dt, monkeypatch):
    print("cluster counts", dims, bc, dt, flush=True)
    g = grid(dims, bc, dt)
    x1, n = run(ctx, g, lambda: cg(g))
    assert n == (1, 0)
    x2, n = run(ctx, g, lambda: cg(g))
    assert n == (1, 0) and np.array_equal(x1, x2)
    monkeypatch.setenv("PANO_CG_CLUSTER", "0")
    assert run(ctx, g, lambda: cg(g))[1] == (0, 0)


def test_gpu_cluster_step_counts(ctx):
    g = grid((300, 260), (0,) * 6, "f4")
    rho, vel, rho2, vel2 = g.new_simplex_2(), g.new_simplex_1(), g.new_simplex_2(), g.new_simplex_1()
    vel.upload(np.random.default_rng(1).standard_normal(g.num_elem_1()).astype("f4"))
    cfg = pa.StepConfig(dt=0.01, preconditioner=pa.Jacobi(), tol=1e-4, tol_kind="rel", max_iterations=2000)
    info, n = run(ctx, g, lambda: pa.fluid_step(g, cfg, rho, vel, rho2, vel2))
    assert info.converged and n == (1, 0)


def test_gpu_cluster_given_up_and_too_large(ctx, monkeypatch):
    g = grid((257, 256), (0,) * 6, "f4")
    x0, n = run(ctx, g, lambda: cg(g))
    assert n == (1, 0)
    monkeypatch.setenv("PANO_CG_CLUSTER", "1")  # more than 64 workgroups never all answer the first poll
    x1, n = run(ctx, g, lambda: cg(g))
    assert n == (1, 1)
    monkeypatch.setenv("PANO_CG_CLUSTER", "0")
    assert np.array_equal(x1, cg(g))
    monkeypatch.delenv("PANO_CG_CLUSTER")
    # once in a row: the next solve is one kernel again; it ends
    x2, n = run(ctx, g, lambda: cg(g))
    assert n == (1, 0) and np.array_equal(x2, x0)
    for dims in ((8, 2049), (1025, 1024)):  # a row too wide, too many cells
        big = grid(dims, (0,) * 6, "f4")
        assert run(ctx, big, lambda: cg(big, 3))[1] == (0, 0)


def test_gpu_cluster_stays_with_the_launches(monkeypatch):
    """Given up twice in a row, the next solve takes the launches, after three
    times the next three; a context of its own, as its state lasts."""
    own = pa.Context(0)
    g = pa.Grid2d((257, 256), "f4", ctx=own)
    seen = []
    monkeypatch.setenv("PANO_CG_CLUSTER", "1")
    for k in range(9):
        x, n = run(own, g, lambda: cg(g, 20))
        seen.append(n)
        if k == 7:
            monkeypatch.delenv("PANO_CG_CLUSTER")
    up, no, ok = (1, 1), (0, 0), (1, 0)
    assert seen == [up, up, no, up, no, no, no, up, no]  # the eighth: four in a row
    for _ in range(6):
        assert run(own, g, lambda: cg(g, 20))[1] == no
    assert run(own, g, lambda: cg(g, 20))[1] == ok  # back to one kernel
    assert run(own, g, lambda: cg(g, 20))[1] == ok
