"""The 3D coarsest level's matrix products with axes past 64 cells (16 waves per
workgroup; the y and z products split over workgroups where there are few)
against the one-workgroup-per-plane passes (PANO_FDM_SPLIT=0), which form the
same chains of fused multiply-adds: the same V-cycle bit for bit, at the edges of
the 64-cell groups and of the numbers of workgroups that decide."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("coarse,bc", [
    ((64, 4, 4), (0,) * 6), ((65, 4, 4), (0, 0, 0, 0, 0, 1)),    # z: four tiles, five
    ((256, 8, 16), (0,) * 6), ((129, 3, 6), (1, 0, 0, 0, 1, 0)),
    ((66, 40, 51), (0,) * 6), ((66, 41, 50), (0, 0, 0, 1, 0, 0)),   # 128 and 129 workgroups in z
    ((8, 256, 8), (0,) * 6), ((3, 130, 18), (0, 1, 0, 0, 0, 0)),    # y: split
    ((63, 65, 8), (0,) * 6), ((64, 65, 8), (0, 0, 1, 0, 0, 0)),     # the last that is, and not
    ((2, 66, 17), (0, 0, 0, 0, 1, 1)),                           # two tiles of columns
    ((7, 4, 248), (0,) * 6), ((5, 62, 66), (1, 0, 0, 0, 0, 1)),      # x
    ((17, 65, 63), (0, 0, 0, 0, 0, 1))])
def test_gpu_coarse3d_long_axes(ctx, coarse, bc, dtype, monkeypatch):
    dims = tuple(2 * n for n in coarse)
    print("coarse 3d", coarse, bc, dtype.__name__, flush=True)
    assert coarse[2] * coarse[1] <= 4096 and coarse[2] * coarse[0] <= 4096  # what the other passes take
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
