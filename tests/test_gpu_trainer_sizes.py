"""Loss and gradient of the closure's trainer at sample counts around its groupings (16
samples per wavefront step, 64 per workgroup step, 512 workgroups), and the Adam update
against the same formula in numpy.  Tolerances as in test_gpu_closure.py."""
import numpy as np
import pytest

from test_gpu_closure import NP, _params, _samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 512 * 64 + 5])
def test_loss_grad_counts(lb, orc, n):
    cfg = lb.preset("baseline")
    rng = np.random.default_rng(n)
    smp, p = _samples(rng, n, cfg.closure_strain_scale, cfg.closure_nu_scale), _params(rng)
    wn = 1.0 / float(np.mean(smp[:, 20].astype(np.float64) ** 2 + smp[:, 21].astype(np.float64) ** 2))
    print(f"case: trainer n={n}", flush=True)
    with lb.Trainer(cfg, n) as tr:
        tr.set_samples(smp)
        tr.set_params(p)
        loss, g = tr.loss_grad(w_norm=wn)
    loss_o, g_o = orc.closure_loss_grad(p, smp, cfg.closure_nu_scale, wn)
    assert loss == pytest.approx(loss_o, rel=1e-5)
    assert np.linalg.norm(g - g_o) / np.linalg.norm(g_o) < 1e-4


def test_adam_step(lb):
    cfg = lb.preset("baseline")
    rng = np.random.default_rng(3)
    smp, p = _samples(rng, 100, cfg.closure_strain_scale, cfg.closure_nu_scale), _params(rng)
    with lb.Trainer(cfg, 100) as tr:
        tr.set_samples(smp)
        tr.set_params(p)
        loss, g = tr.loss_grad()
        hist = tr.train(100, 1, 1e-3)
        q = tr.get_params()
    assert hist[0] == pytest.approx(loss, rel=1e-6)  # the same samples, permuted
    # the first update is lr g / (|g| + eps) with the bias corrections
    big = np.abs(g) > 1e-3 * np.abs(g).max()  # where the sign and eps play no part
    np.testing.assert_allclose((p - q)[:NP][big], (1e-3 * np.sign(g))[big], rtol=2e-2)
