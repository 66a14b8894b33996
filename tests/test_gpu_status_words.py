"""The status words of many contexts at once (they come in pages of 64): each context
reports its own, also after others have been closed and made again."""
import numpy as np
import pytest

from conftest import small_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 66])
def test_each_context_reports_its_own(lb, n):
    cfg = small_cfg(lb, "baseline", n=16, obs_stride=4, loc_scale=1.0, loc_cutoff=3.0)
    cfg.ny = 16
    print(f"case: status words n={n}", flush=True)
    ctxs = [lb.Context(cfg, 2) for _ in range(n)]
    try:
        for k in range(0, n, 3):  # the words of closed contexts are taken again
            ctxs[k].close()
            ctxs[k] = lb.Context(cfg, 2)
        for c in ctxs:
            for m in range(2):
                c.init_member(m, 100 + m)
        yo = ctxs[0].observe(0, seed=1, counter=1, noise=True)
        bad = {0, n - 1}
        for k in sorted(bad):
            f = ctxs[k].get_state(1)
            f[:, 4, 8] = np.nan
            ctxs[k].set_state(1, f)
        for k, c in enumerate(ctxs):
            if k in bad:
                with pytest.raises(lb.LbmLetkfError) as e:
                    c.analysis(yo)
                assert e.value.status == lb.ERR_NUMERIC
                c.synchronize()  # reported once
            else:
                c.analysis(yo)
    finally:
        for c in ctxs:
            c.close()
