"""The library's own launch shapes of the forecast (a context whose shape was not
set): blocks of four steps, strips of any height and row length, with and without
forcing, against the FP64 oracle and, bit for bit, against single-step tiles.

The tolerance is the one of the other forecast tests: a few ulp of FP32 per step."""
import numpy as np
import pytest

from test_gpu_lbm import TOL_F, _ensemble, _rel

pytestmark = pytest.mark.gpu
STEPS = 11  # whole launches of two, three and four steps, each with a remainder


@pytest.mark.parametrize("forced", [False, True])
@pytest.mark.parametrize("nx,ny,M", [
    (4, 4, 1),        # blocks: the region wraps around the grid several times
    (17, 9, 3),       # blocks with ragged edges
    (64, 64, 8),      # blocks
    (1030, 16, 2),    # blocks: rows too long for a strip
    (250, 131, 20),   # three-step strips, ragged rows and a short last strip
    (512, 19, 40),    # three-step strips of the longest row
    (128, 96, 64),    # three-step strips, a tuned height
    (600, 40, 24),    # two-step strips
    (1031, 1021, 1),  # forcing phases past the table
    (16500, 8, 1),    # forcing phases of a row past their FP32 quotient
])
def test_default_shape(lb, orc, nx, ny, M, forced):
    cfg = lb.preset("ref" if forced else "baseline")
    cfg.nx, cfg.ny, cfg.obs_stride = nx, ny, 1
    if not forced:
        cfg.loc_scale, cfg.loc_cutoff = 1.0, 1.0
    cfg.variant = lb.VARIANT_MIXED
    print(f"case: default shape {nx}x{ny} M={M} forced={forced}", flush=True)
    with _ensemble(lb, cfg, M) as ctx, lb.Context(cfg, M) as one:
        f0 = ctx.get_all_states()
        one.set_all_states(f0)
        ctx.forecast(STEPS)
        got = ctx.get_all_states()
        # single-step tiles: ragged grids take them for any tile count, others for two
        tiles = ((nx + 63) // 64) * ((ny + 15) // 16) * M
        one.set_tuning(2 if tiles % 2 == 0 or nx % 64 or ny % 16 else 3, 8)
        one.forecast(STEPS)
        np.testing.assert_array_equal(got, one.get_all_states())
    f = f0[:2].astype(np.float64)
    for s in range(STEPS):
        f = orc.lbm_step(cfg, f, s)
    err = _rel(got[:2], f)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err < TOL_F
