"""The refinement's start from x = 0 and its corrections: a right-hand side of
0, inner solves that end at their iteration limit (their last step is then
still to add), with and without the mean's removal, and what x holds before
the call. The tolerance is the mixed solve's own stop test with the factor 1.5
for the rounding of the second operator."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu


def grid(dims, bc):
    return (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, np.float64, bc=bc)


@pytest.mark.parametrize("dims,bc", [((18, 26), (0,) * 6), ((20, 28, 36), (0, 0, 0, 0, 0, 1)),
                                     ((8, 136, 496), (0,) * 6)])
@pytest.mark.parametrize("max_inner", [1, 3, 200])
def test_gpu_mixed_corrections(ctx, dims, bc, max_inner):
    g = grid(dims, bc)
    b = np.random.default_rng(len(dims) + max_inner).standard_normal(g.cells)
    x = g.new_simplex_2().upload(np.full(g.cells, np.nan))
    info = pa.poisson_solve_mixed(x, g.new_simplex_2().upload(b), preconditioner=pa.Multigrid(2, 2), inner_tol=1e-4,
                                  outer_tol=1e-10, max_outer=400, max_inner=max_inner)
    assert info.converged
    q = g.new_simplex_2()
    pa.PoissonOperator(g, 1.0)(q, x)
    r = (b if any(bc) else b - b.mean()) - q.download()
    assert np.abs(r).max() <= 1.5e-10 * np.abs(b).max()


@pytest.mark.parametrize("dims,bc", [((18, 26), (0,) * 6), ((20, 28, 36), (0, 0, 0, 0, 0, 1))])
def test_gpu_mixed_zero_right_hand_side(ctx, dims, bc):
    g = grid(dims, bc)
    x = g.new_simplex_2().upload(np.full(g.cells, 7.0))
    info = pa.poisson_solve_mixed(x, g.new_simplex_2().upload(np.zeros(g.cells)), preconditioner=pa.Multigrid(2, 2))
    assert info.converged and info.outer_iterations == 0 and info.inner_iterations == 0
    assert not x.download().any()
