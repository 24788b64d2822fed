"""A multigrid level's legs as one launch each against the separate kernels
(PANO_MG_FUSED=0): the same V-cycle bit for bit, f32 and f64, 2D and 3D, at
sizes around the tiles' edges (3D tiles of 16 x 8 cells by 8 planes, or by 2
where at most 256 of those cover the level; 2D 64 x 16 cells) and with every
kind of boundary. In f64 the solve around it takes the same iterations."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu

OPEN = (1, 0, 0, 1, 0, 1)
CASES = [((2, 2, 4), (0,) * 6, 2), ((4, 2, 6), OPEN, 2), ((2, 8, 16), (0, 0, 0, 0, 1, 1), 2),
         ((10, 10, 18), (0,) * 6, 2), ((18, 30, 46), (0, 0, 0, 0, 0, 1), 2),
         ((32, 32, 32), OPEN, 3), ((64, 32, 32), (0,) * 6, 2), ((66, 32, 32), OPEN, 2),  # thin tiles, the most of them, thick
         ((64, 64, 68), (0, 1, 1, 0, 1, 0), 3), ((100, 92, 108), (0,) * 6, 3),
         ((2, 4), (0,) * 4, 2), ((16, 64), (1, 0, 0, 1), 3), ((18, 66), (0,) * 4, 2), ((130, 200), (0, 0, 0, 1), 2),
         ((1024, 1024), (0,) * 4, 4), ((1032, 1024), (0, 1, 0, 0), 4)]   # either side of the f32 2D limit


def vcycle(g, r, levels):
    z = g.new_simplex_2()
    pa.precond_apply(pa.Multigrid(levels, 2), z, g.new_simplex_2().upload(r), dt=0.4)
    return z.download()


@pytest.mark.parametrize("dt", ["f4", "f8"])
@pytest.mark.parametrize("dims,bc,levels", CASES)
def test_gpu_leg_bitwise(ctx, dims, bc, levels, dt, monkeypatch):
    print("leg", dims, bc, levels, dt, flush=True)
    bc = tuple(bc) + (0,) * (6 - len(bc))
    g = (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, dt, bc=bc)
    r = np.random.default_rng(sum(dims)).standard_normal(g.cells).astype(dt)
    zl = vcycle(g, r, levels)
    assert np.isfinite(zl).all()
    assert np.array_equal(zl, vcycle(g, r, levels))
    monkeypatch.setenv("PANO_MG_FUSED", "0")
    assert np.array_equal(zl, vcycle(g, r, levels))


@pytest.mark.parametrize("dims,bc", [((64, 64, 64), (0, 0, 0, 0, 0, 1)), ((40, 48, 104), (0,) * 6),
                                     ((136, 264), (0,) * 6)])
def test_gpu_leg_solve_f64(ctx, dims, bc, monkeypatch):
    g = (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, "f8", bc=bc)
    u = g.new_simplex_1().upload(np.random.default_rng(1).standard_normal(g.num_elem_1()))
    b = g.new_simplex_2()
    pa.neg_divergence(b, u)

    def solve():
        x, r, a, s = (g.new_simplex_2() for _ in range(4))
        info = pa.precond_conjugate_gradient(pa.Multigrid(4, 2), x, b, 200, 1e-10, r, a, s,
                                             pa.PoissonOperator(g, 0.05), tol_kind="rel")
        return x.download(), info

    x1, i1 = solve()
    monkeypatch.setenv("PANO_MG_FUSED", "0")
    x0, i0 = solve()
    # the z.r sums are added in another order: a rounding of sigma per iteration
    assert i1.converged and i1.iterations == i0.iterations
    assert np.abs(x1 - x0).max() <= 1e-9 * np.abs(x0).max()
