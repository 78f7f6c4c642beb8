"""mh_adjoint_backward_ms: recomputation and reverse stages alone. The cotangent's way to the device is
not in it, so the figure of one step is that of a step, however long the transfer takes."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import problems

pytestmark = pytest.mark.gpu


def test_backward_time_without_transfers():
    cfg = problems.kh_config(1024)
    cfg.max_cfl = 0.4
    q0 = problems.kh_band(cfg)
    lam = np.random.default_rng(3).standard_normal(cfg.shape)
    best = {}
    with M.HydroContext(cfg) as ctx:
        for steps in (1, 6):
            ctx.upload(q0)
            ctx.fill_bcs()
            ctx.adjoint_forward(steps, 1)
            for _ in range(4):
                ctx.adjoint_backward(lam.copy())
                best[steps] = min(best.get(steps, 1e9), ctx.adjoint_backward_ms())
    # a step's reverse sweep and recomputation are the same work in both; the upload of 34 MB and the
    # host's copy of it are several steps' worth
    assert best[1] * 6 < 1.5 * best[6], best
