"""The velocity advected by itself on 3D f32 grids in one pass, against the
per-component kernels (PANO_ADV_FUSED=0) bit for bit, at sizes around its
tiles (32 x 16 or 64 x 8 cells, chunks of 2 to 16 planes), with departures of
a fraction of a cell and of several; the same for a step, which also advects
the density."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu

CASES = [(2, 1, 1), (3, 5, 7), (2, 16, 32), (17, 17, 33), (16, 8, 64), (5, 40, 40), (9, 33, 65), (40, 15, 31),
         (130, 70, 97), (33, 260, 130)]


@pytest.mark.parametrize("dims", CASES)
def test_gpu_advect_mac_one_pass(ctx, dims, monkeypatch):
    print("advect_mac", dims, flush=True)
    g = pa.Grid3d(dims, np.float32, bc=(0, 0, 0, 0, 0, 1))
    rng = np.random.default_rng(sum(dims))
    v = g.new_simplex_1().upload(rng.uniform(-1, 1, g.num_elem_1()))
    w = g.new_simplex_1().upload(rng.uniform(-1, 1, g.num_elem_1()))
    rho = g.new_simplex_2().upload(rng.random(g.cells))
    cfg = pa.StepConfig(dt=0.7, preconditioner=pa.Jacobi(), max_iterations=1, buoyancy=0.3, src_radius=2.0,
                        src_center=(1.0, 2.0, 3.0))

    def run():
        out = []
        for dt in (0.3, 2.7, 50.0):
            a, b = g.new_simplex_1(), g.new_simplex_1()
            pa.advect_mac(a, v, dt, v)
            pa.advect_mac(b, w, dt, v)  # another field than the velocity: the component kernels
            out += [a.download(), b.download()]
        r2, v2 = g.new_simplex_2(), g.new_simplex_1()
        pa.fluid_step(g, cfg, rho, v, r2, v2)
        return out + [r2.download(), v2.download()]

    one = run()
    monkeypatch.setenv("PANO_ADV_FUSED", "0")
    for x, y in zip(one, run()):
        assert np.array_equal(x, y)
