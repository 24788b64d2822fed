"""The 3D operator in runs of planes against the oracle's, at plane counts
around a run, ragged rows and every side's condition. f64 within 1e-12 of the
largest value (the same expressions; the bound is 4500 roundings), f32 against
the FP64 result within 2e-6 (16 roundings)."""
import numpy as np
import pytest

import panopaea_amd as pa
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float32, 2e-6), (np.float64, 1e-12)])
@pytest.mark.parametrize("dims", [(2, 3, 5), (3, 1, 70), (4, 9, 64), (5, 4, 65), (7, 6, 2), (9, 5, 129)])
@pytest.mark.parametrize("bc", [(0,) * 6, (1, 0, 0, 1, 0, 1), (0, 1, 1, 0, 1, 0)])
def test_gpu_poisson_plane_runs(ctx, dims, bc, dtype, tol):
    g = pa.Grid3d(dims, dtype, bc=bc)
    p = np.random.default_rng(sum(dims)).standard_normal(g.cells).astype(dtype)
    q = g.new_simplex_2()
    pa.PoissonOperator(g, 0.7)(q, g.new_simplex_2().upload(p))
    ref = o.poisson(o.params(dims, bc=bc, dt=0.7), p.astype(np.float64))
    assert np.abs(q.download() - ref).max() <= tol * np.abs(ref).max()
