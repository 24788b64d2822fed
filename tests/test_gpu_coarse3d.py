"""The 3D coarsest level's matrix products on the matrix cores: against the
one-workgroup-per-plane passes (PANO_FDM_SPLIT=0), which form the same chains
of fused multiply-adds, bit for bit, at the edges of the 16-wide tiles and of
the one-workgroup form (16 cells per axis); and, for planes past those passes'
4096 cells, by the convergence of a solve (tolerance: the solve's own, with
the factor 1.5 for the rounding of the second operator)."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims,bc", [
    ((32, 32, 32), (0,) * 6),                 # 16^3: the largest one-workgroup level
    ((6, 18, 30), (0, 1, 0, 0, 1, 0)),        # 3 x 9 x 15 in one workgroup
    ((4, 4, 4), (0,) * 6),                    # 2^3
    ((34, 32, 32), (0, 0, 0, 0, 0, 1)),       # 17 planes: three launches
    ((30, 66, 10), (0,) * 6),                 # 15 x 33 x 5: 5 columns, a row past two tiles
    ((10, 34, 98), (1, 0, 0, 0, 0, 1)),       # 5 x 17 x 49
    ((128, 16, 126), (0, 0, 1, 0, 0, 0))])    # 64 x 8 x 63
def test_gpu_coarse3d_bitwise(ctx, dims, bc, dtype, monkeypatch):
    print("coarse 3d", dims, bc, dtype.__name__, flush=True)
    g = pa.Grid3d(dims, dtype, bc=bc)
    r = np.random.default_rng(sum(dims)).standard_normal(g.cells)
    if not any(bc):
        r -= r.mean()
    src, out = g.new_simplex_2().upload(r.astype(dtype)), []
    for flag in ("1", "0"):
        monkeypatch.setenv("PANO_FDM_SPLIT", flag)
        z = g.new_simplex_2()
        pa.precond_apply(pa.Multigrid(2, 2), z, src, dt=0.3)
        out.append(z.download())
    assert np.all(np.isfinite(out[0]))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("dims,bc", [((16, 140, 162), (0,) * 6), ((6, 512, 34), (0, 0, 0, 1, 0, 1)),
                                     ((512, 6, 510), (1, 0, 0, 0, 0, 0))])
def test_gpu_coarse3d_large_planes(ctx, dims, bc):
    g = pa.Grid3d(dims, np.float64, bc=bc)
    b = np.random.default_rng(sum(dims)).standard_normal(g.cells)
    x, q = g.new_simplex_2(), g.new_simplex_2()
    info = pa.precond_conjugate_gradient(pa.Multigrid(2, 2), x, g.new_simplex_2().upload(b), 40, 1e-10,
                                         *(g.new_simplex_2() for _ in range(3)), pa.PoissonOperator(g, 1.0),
                                         tol_kind="rel")
    assert info.converged
    pa.PoissonOperator(g, 1.0)(q, x)
    r = (b if any(bc) else b - b.mean()) - q.download()
    assert np.abs(r).max() <= 1.5e-10 * np.abs(b).max()
