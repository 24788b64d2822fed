"""The velocity advected by itself with chunks of one plane and of two: either
side of the number of workgroups that decides (two tiles per plane: 318 planes
are 318 workgroups of two planes, 319 and 320 are 320), against the
per-component kernels (PANO_ADV_FUSED=0) bit for bit."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 3, 70), (317, 30, 30), (318, 30, 30), (319, 30, 30), (320, 30, 30),
                                  (23, 66, 31)])
@pytest.mark.parametrize("bc", [(0,) * 6, (0, 1, 0, 0, 1, 1)])
def test_gpu_advect_mac_planes(ctx, dims, bc, monkeypatch):
    print("advect_mac planes", dims, bc, flush=True)
    g = pa.Grid3d(dims, np.float32, bc=bc)
    v = g.new_simplex_1().upload(np.random.default_rng(sum(dims)).uniform(-1, 1, g.num_elem_1()))

    def run():
        out = []
        for dt in (0.4, 3.1, 40.0):
            a = g.new_simplex_1()
            pa.advect_mac(a, v, dt, v)
            out.append(a.download())
        return out

    one = run()
    monkeypatch.setenv("PANO_ADV_FUSED", "0")
    for x, y in zip(one, run()):
        assert np.array_equal(x, y)
