"""Perturbations and innovations of the observed ensemble, a group of 16, 32 or 64 lanes per
observation: member counts at the edges of the groups, a number of observations that fills
no whole workgroup.  dY and dyo are FP64 differences rounded once to FP32."""
import numpy as np
import pytest

from conftest import small_cfg
from test_gpu_letkf import _osse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [2, 16, 17, 32, 33, 64])
def test_observed_ensemble(lb, M):
    cfg = small_cfg(lb, "baseline", n=64, obs_stride=8, loc_scale=2.0, loc_cutoff=6.0)
    sites = np.arange(5, 64 * 64, 311, dtype=np.int32)  # 14 sites, 28 observations
    print(f"case: observed ensemble M={M}", flush=True)
    ens, nat = _osse(lb, cfg, M, spin=4)
    with ens, nat:
        ens.set_obs_sites(sites)
        nat.set_obs_sites(sites)
        yo = nat.observe(0, seed=11, counter=3, noise=True)
        f = ens.get_all_states().astype(np.float64).reshape(M, 9, -1)[:, :, sites]
        ens.analysis(yo)
        dy, dyo = ens.get_obs_ensemble()
    rho = f.sum(1)
    u = cfg.c * ((f[:, 2] + f[:, 5] + f[:, 8]) - (f[:, 0] + f[:, 3] + f[:, 6])) / rho
    v = cfg.c * ((f[:, 6] + f[:, 7] + f[:, 8]) - (f[:, 0] + f[:, 1] + f[:, 2])) / rho
    hx = np.stack([u, v], axis=2).reshape(M, -1).T  # [site, variable][member]
    mean = hx.mean(1)
    # the FP64 sums may differ by a few units of 1e-16, far below half a unit of FP32
    np.testing.assert_allclose(dy, hx - mean[:, None], rtol=2.0**-23, atol=1e-15)
    np.testing.assert_allclose(dyo, yo.ravel().astype(np.float64) - mean, rtol=2.0**-23, atol=1e-15)
