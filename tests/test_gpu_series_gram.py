"""The Gram matrix of the analysis by series (f16 parts, chunks of 32 local sites, one to
three variables of a site dealt to blocks of 32 observations) at the edges of its tiles and
chunks against the FP64 oracle, and what lies past its range."""
import numpy as np
import pytest

from conftest import small_cfg
from test_gpu_letkf import TOLS, _osse, _rel

pytestmark = pytest.mark.gpu

# Two f16 parts leave 2^-22 of an operand, the FP32 sums over at most 300 observations
# sqrt(300) 2^-24 of the matrix: below 2e-6 together, times a condition number up to 10 in
# the part of the increment that the observations determine.
TOL = 2e-5


@pytest.mark.parametrize("M,obs_vars,stride,cutoff,passes", [
    (2, 3, 4, 3.0, 3),     # one site or none
    (16, 1, 4, 7.0, 3),    # a few sites, one variable
    (16, 3, 4, 9.0, 3),    # 16 sites: the second block of the chunk empty or one site
    (17, 7, 4, 9.0, 3),    # three variables, members past a tile
    (31, 7, 4, 13.0, 3),   # around 32 sites
    (33, 3, 4, 13.0, 3),
    (45, 1, 4, 18.5, 3),   # around 64 sites
    (63, 7, 4, 18.5, 3),
    (64, 3, 2, 11.0, 3),   # three chunks
    (8, 3, 1, 4.2, 3),     # every node observed
    (33, 7, 4, 9.0, 1),
    (64, 3, 4, 13.0, 1),
])
def test_gram_shapes(lb, orc, M, obs_vars, stride, cutoff, passes):
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=stride, loc_scale=cutoff / 3.0, loc_cutoff=cutoff,
                    obs_sigma_u=0.02, obs_vars=obs_vars, gram_passes=passes)
    cfg.ny = 40
    print(f"case: gram M={M} vars={obs_vars} stride={stride} cutoff={cutoff} passes={passes}", flush=True)
    ens, nat = _osse(lb, cfg, M)
    with ens, nat:
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        fb = ens.get_all_states().astype(np.float64)
        ens.analysis(yo)
        fa = ens.get_all_states().astype(np.float64)
    fo = fb.copy()
    orc.letkf_analysis(cfg, fo, yo.astype(np.float64))
    err = _rel(fa - fb, fo - fb)
    print(f"  increment rel {err:.2e}", flush=True)
    assert err < (TOL if passes == 3 else TOLS["mixed1"][1])


@pytest.mark.parametrize("M", [8, 32])
@pytest.mark.parametrize("sigma", [1e-7, 1e-12])
def test_past_the_range(lb, M, sigma):
    # rows of dY past the range of f16, and a matrix whose squared columns pass FP32's: the
    # sweeps take every gridpoint, as when all are dumped, and stay finite
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=4, loc_scale=3.0, loc_cutoff=9.0, obs_sigma_u=sigma)
    cfg.ny = 40
    print(f"case: range M={M} sigma={sigma}", flush=True)
    ens, nat = _osse(lb, cfg, M)
    with ens, nat:
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        fb = ens.get_all_states()
        ens.analysis(yo)
        fa = ens.get_all_states()
        ens.set_all_states(fb)
        ens.set_dump(0, cfg.nx * cfg.ny)
        ens.analysis(yo)
        fs = ens.get_all_states()
    assert np.isfinite(fa).all()
    np.testing.assert_array_equal(fa, fs)


def test_density_that_cancels(lb):
    # populations of either sign whose sum is exactly zero are observed with a finite
    # velocity, c (-0.25 - 0.25) over half a unit in the last place of 0.25
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=8, loc_scale=3.0, loc_cutoff=7.0)
    with lb.Context(cfg, 1) as ctx:
        f = np.full((9, 64, 64), 1.0 / 9, np.float32)
        f[:, 16, 24] = 0.0
        f[0, 16, 24], f[8, 16, 24] = 0.25, -0.25
        ctx.set_state(0, f)
        y = ctx.observe(0, seed=11, counter=3, noise=False)
    assert np.isfinite(y).all()
    assert np.abs(y).max() == np.float32(cfg.c * 0.5 / 2.0**-27)
