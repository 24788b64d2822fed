"""The fetched pressure in natural order on either side of the size at which the
host puts it in order (65536 cells): the fetched velocity is u + dt d0*(p) of it
along every axis (f32, the projection's own expression), a second fetch gives the
same bits, and either output may be left out."""
import ctypes

import numpy as np
import pytest

import panopaea_amd as pa
from panopaea_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 16), (256, 256), (256, 264), (8, 8, 8), (32, 32, 64), (40, 32, 64)])
def test_gpu_server_pressure_order(ctx, dims):
    print("server order", dims, flush=True)
    q = dict(dims=dims, dt=0.5 / dims[-1], bc=(0,) * 6)
    g = (pa.Grid2d if len(dims) == 2 else pa.Grid3d)(dims, np.float32)
    u = np.random.default_rng(dims[0]).standard_normal(g.num_elem_1()).astype(np.float32)
    S = pa.Server(hbm_budget=1 << 30, max_active=4, mg_levels=3)
    rid = S.submit(q, faces=u)
    S.run_until_idle()
    f, p = S.fetch(rid)
    P, dt = p.reshape(dims), np.float32(q["dt"])
    uz, uy, ux = g.split_faces(u)
    vz, vy, vx = g.split_faces(f)
    assert np.array_equal(vx[..., 1:-1], ux[..., 1:-1] + dt * (P[..., :-1] - P[..., 1:]))
    assert np.array_equal(vy[..., 1:-1, :], uy[..., 1:-1, :] + dt * (P[..., :-1, :] - P[..., 1:, :]))
    if len(dims) == 3:
        assert np.array_equal(vz[1:-1], uz[1:-1] + dt * (P[:-1] - P[1:]))
    f2, p2 = np.zeros_like(f), np.zeros_like(p)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p) if a is not None else None
    sig = _lib._SIGS["pano_server_fetch"][0]
    cast = lambda a, t: ctypes.cast(ptr(a), t) if a is not None else None
    L = _lib.lib()
    _lib.check(L.pano_server_fetch(S.handle, rid, cast(f2, sig[2]), None))
    _lib.check(L.pano_server_fetch(S.handle, rid, None, cast(p2, sig[3])))
    assert np.array_equal(f, f2) and np.array_equal(p, p2)
    S.close()
