"""The coarsest level of 2D multigrid (matrix products on the matrix cores: one
workgroup up to 64 x 64 cells, four tiled launches beyond) against the
oracle's V-cycle, at coarsest sizes around the tiles' and the variants' edges.
Bound: in f32 the coarse values are rounded once from FP64 sums of at most
n^2 terms whose error is far below f32's, so the V-cycles differ by the f32
sweeps' roundings, 1e-5 of the largest value; in f64 by the sums' order and the
two bases' rounding, 1e-9 as for the other V-cycles. In a closed box the
constant is arbitrary up to rounding and is taken out."""
import numpy as np
import pytest

import panopaea_amd as pa
from oracle import oracle as o

pytestmark = pytest.mark.gpu

COARSE = [(1, 3), (3, 1), (8, 8), (15, 16), (16, 17), (17, 33), (32, 32), (33, 31), (48, 20), (64, 64), (63, 5),
          (65, 64), (64, 66), (80, 130), (3, 255), (256, 16), (129, 97)]


@pytest.mark.parametrize("dt", ["f4", "f8"])
@pytest.mark.parametrize("ny,nx", COARSE)
def test_gpu_coarse_2d(ctx, ny, nx, dt):
    dims = (2 * ny, 2 * nx)
    for bc in ((0,) * 6, (0, 1, 0, 0, 0, 0), (1, 1, 1, 0, 0, 0)):
        print("coarse 2D", dims, dt, bc, flush=True)
        g = pa.Grid2d(dims, dt, bc=bc)
        r = np.random.default_rng(ny * nx).standard_normal(g.cells).astype(dt)
        if not any(bc):
            r -= r.mean()
        z = g.new_simplex_2()
        pa.precond_apply(pa.Multigrid(2, 2), z, g.new_simplex_2().upload(r), dt=0.4)
        ez, zz = o.mg_vcycle(o.params(dims, bc=bc, dt=0.4, levels=2), r).astype(np.float64), z.download()
        if not any(bc):
            zz, ez = zz - zz.mean(dtype=np.float64), ez - ez.mean()
        assert np.abs(zz - ez).max() < (1e-5 if dt == "f4" else 1e-9) * np.abs(ez).max()
