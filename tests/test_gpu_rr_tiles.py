"""The tiles of the one-pass residual + restriction (64 x 8 and 32 x 16 coarse
cells) against the separate residual and restriction kernels
(PANO_MG_FUSED=0): the same V-cycle bit for bit, at ragged edges of both tile
shapes, into the red-black and the natural (coarsest) layout, with odd chunks."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu

CASES = [((256, 240, 144), (0, 0, 0, 0, 0, 1), 4),  # 72 coarse columns: narrow tiles
         ((256, 244, 144), (0, 1, 1, 0, 0, 0), 2),  # narrow, into the coarsest level, ragged rows
         ((140, 250, 240), (0,) * 6, 2),            # wide, into the coarsest level, ragged both ways
         ((512, 16, 1024), (1, 0, 0, 0, 1, 0), 4),  # wide, one row of tiles
         ((600, 200, 72), (0,) * 6, 3)]             # 36 coarse columns: one ragged wide tile


@pytest.mark.parametrize("dims,bc,levels", CASES)
def test_gpu_residual_restriction_tiles_bitwise(ctx, dims, bc, levels, monkeypatch):
    print("rr tiles", dims, bc, levels, flush=True)
    g = pa.Grid3d(dims, np.float32, bc=bc)
    r = np.random.default_rng(dims[1]).standard_normal(g.num_elem_2()).astype(np.float32)
    if not any(bc):
        r -= r.mean(dtype=np.float64).astype(np.float32)
    src, out = g.new_simplex_2().upload(r), {}
    for fused in (True, False):
        if fused:
            monkeypatch.delenv("PANO_MG_FUSED", raising=False)
        else:
            monkeypatch.setenv("PANO_MG_FUSED", "0")
        z = g.new_simplex_2()
        pa.precond_apply(pa.Multigrid(levels, 2), z, src, dt=0.4)
        out[fused] = z.download()
    assert np.all(np.isfinite(out[True]))
    assert np.array_equal(out[True], out[False])
