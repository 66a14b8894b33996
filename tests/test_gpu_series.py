"""The analysis by series (condition number of the local problem up to 1023) and by
sweeps (above) on both sides of the line and with both in one analysis, at member counts
at the edges of the 16-member tiles, against the FP64 oracle.

The tolerance is the mixed variant's (the sweeps' split-bf16 Gram matrix sets it)."""
import numpy as np
import pytest

from conftest import small_cfg
from test_gpu_letkf import TOLS, _osse, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,sigma", [(2, 0.01), (16, 0.02), (16, 0.0015), (17, 0.006), (32, 0.004), (33, 0.01),
                                     (64, 0.006), (64, 0.0012)])
def test_series_and_sweeps(lb, orc, M, sigma):
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=8, loc_scale=6.0, loc_cutoff=20.0, obs_sigma_u=sigma)
    cfg.ny = 40
    cfg.loc_cutoff = 19.0
    print(f"case: series M={M} sigma={sigma}", flush=True)
    ens, nat = _osse(lb, cfg, M)
    with ens, nat:
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        fb = ens.get_all_states().astype(np.float64)
        ens.analysis(yo)
        fa = ens.get_all_states().astype(np.float64)
        # the same analysis with every gridpoint dumped: the sweeps do all of it
        ens.set_all_states(fb.astype(np.float32))
        ens.set_dump(0, cfg.nx * cfg.ny)
        ens.analysis(yo)
        fs = ens.get_all_states().astype(np.float64)
        ev = ens.get_dump()[2]
    fo = fb.copy()
    orc.letkf_analysis(cfg, fo, yo.astype(np.float64))
    kappa = ev[:, -1] / ev[:, 0]
    err, err_s = _rel(fa - fb, fo - fb), _rel(fs - fb, fo - fb)
    print(f"  condition {kappa.min():.3g}..{kappa.max():.3g}  increment rel {err:.2e}  by sweeps alone {err_s:.2e}",
          flush=True)
    assert err < TOLS["mixed3"][1]


@pytest.mark.parametrize("M,sigma", [(2, 0.01), (16, 0.02), (16, 0.0015), (16, 2e-4), (17, 0.006), (33, 0.01),
                                     (64, 0.0012)])
def test_plain_series_and_eigensolve(lb, orc, M, sigma):
    # the PLAIN analysis: FP32 Gram matrix, the rest in FP64; series up to condition 65500.
    # Beyond ~1000 the rounding of C alone (6e-8 of its norm) moves the result by more than
    # the variant's tolerance: 6e-8 times the condition bounds it.
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=8, loc_scale=6.0, loc_cutoff=19.0, obs_sigma_u=sigma,
                    variant=lb.VARIANT_PLAIN)
    cfg.ny = 40
    print(f"case: plain series M={M} sigma={sigma}", flush=True)
    ens, nat = _osse(lb, cfg, M)
    with ens, nat:
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        fb = ens.get_all_states().astype(np.float64)
        ens.analysis(yo)
        fa = ens.get_all_states().astype(np.float64)
    fo = fb.copy()
    ev = orc.letkf_analysis(cfg, fo, yo.astype(np.float64), 0, cfg.nx * cfg.ny)[2]
    kappa = (ev[:, -1] / ev[:, 0]).max()
    err = _rel(fa - fb, fo - fb)
    print(f"  condition up to {kappa:.3g}  increment rel {err:.2e}", flush=True)
    assert err < max(TOLS["plain"][1], 6e-8 * kappa)


@pytest.mark.parametrize("variant", ["plain", "mixed"])
def test_nan_member_is_reported(lb, variant):
    # a NaN at an observed node: every gridpoint that uses the observation becomes NaN, and
    # the next synchronising call says so
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=8, loc_scale=3.0, loc_cutoff=7.0,
                    variant=lb.VARIANT_PLAIN if variant == "plain" else lb.VARIANT_MIXED)
    print(f"case: NaN {variant}", flush=True)
    ens, nat = _osse(lb, cfg, 8, spin=0)
    with ens, nat:
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        f = ens.get_state(3)
        f[:, 16, 24] = np.nan
        ens.set_state(3, f)
        with pytest.raises(lb.LbmLetkfError) as e:
            ens.analysis(yo)
        assert e.value.status == lb.ERR_NUMERIC
        fa = ens.get_all_states()
    assert np.isnan(fa[:, :, 16, 24]).all() and np.isnan(fa[:, :, 16 + 6, 24]).all()
    assert np.isfinite(fa[:, :, 16 + 9, 24]).all() and np.isfinite(fa[:, :, 40:, 40:]).all()
