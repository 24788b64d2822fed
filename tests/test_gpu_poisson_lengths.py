"""The 3D operator on either side of the limits of its run lengths (tiles of
single planes, one per plane here: f32 runs of 1 and 4 planes, f64 of 1, 2 and
4), with every remainder of the last run. Bounds as for the other run tests:
f64 1e-12 of the largest value, f32 against the FP64 result 2e-6."""
import numpy as np
import pytest

import panopaea_amd as pa
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol,planes", [(np.float32, 2e-6, (1023, 1024, 1025, 1026, 1027)),
                                              (np.float64, 1e-12, (2047, 2048, 2049, 16383, 16384, 16385, 16386, 16387))])
@pytest.mark.parametrize("bc", [(0,) * 6, (1, 0, 0, 1, 0, 1)])
def test_gpu_poisson_run_lengths(ctx, dtype, tol, planes, bc):
    for d in planes:
        dims = (d, 3, 5)
        print("operator", dims, bc, dtype.__name__, flush=True)
        g = pa.Grid3d(dims, dtype, bc=bc)
        p = np.random.default_rng(d).standard_normal(g.cells).astype(dtype)
        q = g.new_simplex_2()
        pa.PoissonOperator(g, 0.7)(q, g.new_simplex_2().upload(p))
        ref = o.poisson(o.params(dims, bc=bc, dt=0.7), p.astype(np.float64))
        assert np.abs(q.download() - ref).max() <= tol * np.abs(ref).max()
