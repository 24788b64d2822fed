"""The identity and Jacobi solves of small grids as one kernel
(PANO_CG_CLUSTER=0: the launches): the same iteration count, a solution that
meets the stop test in the oracle's operator, and, where its workgroups do not
all answer (PANO_CG_CLUSTER=1: polls give up at once), the launches' solution
bit for bit. Bounds: both loops round the same expressions and differ in the
order of FP64 sums only, so a stop test may fall one iteration apart and
the true residual is the recursive one up to the fields' rounding: 20 tol in
f32, 10 tol in f64, as for the other solves, or, where x is so large against b
that its rounding alone is more (long rows that end in an open side), that of
the launches."""
import numpy as np
import pytest

import panopaea_amd as pa
from oracle import oracle as o
from panopaea_amd import scenes

pytestmark = pytest.mark.gpu

OPEN_TOP = (0, 0, 0, 0, 0, 1)
CASES = [((1, 3), (1, 0, 0, 0), "f4", "jacobi"),            # one workgroup, fewer cells than a wave
         ((5, 7), (0,) * 4, "f8", "identity"),
         ((16, 16), (0, 0, 1, 0), "f4", "identity"),        # exactly one workgroup
         ((16, 17), (0,) * 4, "f4", "jacobi"),              # two, the second nearly empty
         ((9, 300), (0,) * 4, "f8", "jacobi"),              # rows wider than a workgroup's cells
         ((2, 2048), (0, 1, 0, 0), "f4", "jacobi"),         # the widest rows, no interior row
         ((1100, 3), (0,) * 4, "f8", "jacobi"),             # many short rows
         ((129, 128), (0, 0, 0, 1), "f4", "identity"),      # one row past 256 threads: 512
         ((151, 217), (0,) * 4, "f4", "jacobi"),            # 32767 cells: the last of 512 threads
         ((181, 182), (0,) * 4, "f8", "identity"),          # 1024 threads
         ((365, 363), (0, 0, 0, 1), "f4", "jacobi"),        # two cells per thread
         ((600, 700), (0, 1, 0, 1), "f8", "jacobi"),        # four
         ((8, 9, 10), (0,) * 6, "f4", "jacobi"),
         ((2, 3, 400), OPEN_TOP, "f8", "jacobi"),           # planes smaller than a workgroup
         ((3, 40, 40), (0, 0, 0, 0, 1, 0), "f4", "identity"),
         ((63, 65, 64), OPEN_TOP, "f8", "jacobi"),
         ((66, 65, 64), OPEN_TOP, "f4", "jacobi")]          # past one cell per thread in 3D


def solve(g, pre, b, tol, mask=None, remove_mean=-1, tol_kind="rel", max_it=3000):
    x, r, a, s = (g.new_simplex_2() for _ in range(4))
    info = pa.precond_conjugate_gradient({"jacobi": pa.Jacobi(), "identity": pa.Identity()}[pre], x,
                                         g.new_simplex_2().upload(b), max_it, tol, r, a, s,
                                         pa.PoissonOperator(g, 0.05, mask), tol_kind=tol_kind,
                                         remove_mean=remove_mean)
    return x.download(), r.download(), info


@pytest.mark.parametrize("dims,bc,dt,pre", CASES)
def test_gpu_cluster_solve(ctx, dims, bc, dt, pre, monkeypatch):
    print("cluster", dims, bc, dt, pre, flush=True)
    bc6 = tuple(bc) + (0,) * (6 - len(bc))
    g = (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, dt, bc=bc6)
    P = o.params(dims, bc=bc6, dt=0.05)
    b = o.neg_div(P, np.random.default_rng(sum(dims)).standard_normal(g.num_elem_1())).astype(dt)
    tol = 1e-6 if dt == "f4" else 1e-9
    monkeypatch.setenv("PANO_CG_CLUSTER", "0")
    x0, r0, i0 = solve(g, pre, b, tol)
    monkeypatch.setenv("PANO_CG_CLUSTER", "1")
    xs, rs, _ = solve(g, pre, b, tol)
    monkeypatch.delenv("PANO_CG_CLUSTER")
    x1, r1, i1 = solve(g, pre, b, tol)
    xa, ra, ia = solve(g, pre, b, tol)
    assert i0.converged and i1.converged and abs(i0.iterations - i1.iterations) <= 1
    assert np.array_equal(xa, x1) and np.array_equal(ra, r1) and ia.iterations == i1.iterations
    if g.cells > 64 * 256:  # 64 workgroups and more never all answer the first poll
        assert np.array_equal(xs, x0) and np.array_equal(rs, r0)
    bu = b.astype(np.float64) - (b.astype(np.float64).mean() if not any(bc) else 0.0)
    e1, e0 = (np.abs(o.poisson(P, x.astype(np.float64)) - bu).max() / np.abs(bu).max() for x in (x1, x0))
    assert e1 < max((20 if dt == "f4" else 10) * tol, 2 * e0)
    assert np.abs(r1).max() == i1.r_linf


@pytest.mark.parametrize("dt", ["f4", "f8"])
def test_gpu_cluster_masked_and_limits(ctx, dt, monkeypatch):
    """The obstacle scene's solve (stopped by the limit), a limit of one, b = 0 and a NaN."""
    n = 128
    g = pa.Grid2d((n, n), dt)
    m = scenes.obstacle_mask(n, n)
    mask = pa.face_mask(g, m)
    u = g.new_simplex_1().upload(np.random.default_rng(3).standard_normal(g.num_elem_1()))
    bd = g.new_simplex_2()
    pa.neg_divergence(bd, u, mask)
    b = bd.download()
    for max_it in (1, 2, 5, 100):
        monkeypatch.setenv("PANO_CG_CLUSTER", "0")
        x0, r0, i0 = solve(g, "identity", b, 1e-30, mask, 0, "abs", max_it)
        monkeypatch.delenv("PANO_CG_CLUSTER")
        x1, r1, i1 = solve(g, "identity", b, 1e-30, mask, 0, "abs", max_it)
        assert i1.iterations == i0.iterations == max_it and not i1.converged
        # max_it roundings of each field and sum, each amplified at most by the condition of the shift
        eps = np.finfo(dt).eps
        assert np.abs(x1 - x0).max() <= 100 * max_it * eps * np.abs(x0).max()
    x, _, i = solve(g, "jacobi", 0 * b, 1e-6)
    assert i.converged and i.iterations == 0 and not x.any()
    b[5] = np.nan
    with pytest.raises(pa.PanoError):
        solve(g, "jacobi", b, 1e-6, remove_mean=0)
