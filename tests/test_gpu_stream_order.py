"""The operator and FP64 residual on fields larger than the 256 MB memory-side
cache, whose tiles are taken in chunks: a grid whose tile count is no multiple
of the chunk group, with plane runs that end past the grid.

The tolerance is that of the mixed solve's own stop test, max|b - A x| <= tol
max|b|, as the solve measures it with these kernels, against the operator of
the natural layout (which keeps its order); the factor 1.5 covers the rounding
of the second operator, as in the small sizes' test."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,bc,levels", [((262, 508, 512), (0, 0, 0, 0, 0, 1), 2), ((264, 416, 664), (0,) * 6, 4)])
def test_gpu_mixed_residual_on_large_fields(dims, bc, levels):
    g = pa.Grid3d(dims, np.float64, bc=bc)
    faces, b, x, q = g.new_simplex_1(), g.new_simplex_2(), g.new_simplex_2(), g.new_simplex_2()
    pa.gen_uniform_faces_device(faces, 3)
    pa.neg_divergence(b, faces)
    faces.free()
    info = pa.poisson_solve_mixed(x, b, dt=1.0, preconditioner=pa.Multigrid(levels, 2), inner_tol=1e-4, outer_tol=1e-9)
    assert info.converged and info.outer_iterations <= 6
    pa.PoissonOperator(g, 1.0)(q, x)
    bh = b.download()
    if not any(bc):
        bh -= bh.mean()
    res = np.abs(bh - q.download()).max()
    assert res <= 1.5e-9 * np.abs(bh).max(), res
    for f in (b, x, q):
        f.free()
