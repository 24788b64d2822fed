"""A grid with more partial sums than the narrow finalize step takes (past 8192:
264 x 256 x 272 cells) beside small ones: the bits of each are those of the
request alone, whatever the width of the others' reductions."""
import numpy as np
import pytest

import panopaea_amd as pa

pytestmark = pytest.mark.gpu

GRIDS = [dict(dims=(264, 256, 272), dt=0.5 / 256, bc=(0, 0, 0, 0, 0, 1)), dict(dims=(64, 96), dt=0.5 / 96),
         dict(dims=(256, 256, 256), dt=0.5 / 256, bc=(0, 0, 0, 0, 0, 1)), dict(dims=(40, 48, 56), dt=0.5 / 56)]


def serve(ids):
    S = pa.Server(hbm_budget=8 << 30, max_active=8)
    rid = [S.submit(GRIDS[i], seed=3 + i) for i in ids]
    S.run_until_idle()
    out = [(S.status(r), *S.fetch(r)) for r in rid]
    S.close()
    return out


def test_gpu_server_finalize_widths(ctx):
    print("server finalize", GRIDS, flush=True)
    together = serve(range(len(GRIDS)))
    for i, (st, f, p) in enumerate(together):
        (st1, f1, p1), = serve([i])
        assert st["converged"] == 1 and st["iterations"] == st1["iterations"], (st, st1)
        assert np.array_equal(f, f1) and np.array_equal(p, p1), GRIDS[i]
