"""The FP64 signal speed where its square overflows (a density near the smallest numbers under a large
pressure): infinite, so that there is no time step, as the oracle has it."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd", [1, 2, 3])
def test_step_size_with_an_infinite_sound_speed(orc, nd):
    """An infinite signal speed leaves no time step."""
    cfg = Config(num_dim=nd, nx=70, ny=9 if nd > 1 else 1, nz=8 if nd > 2 else 1, ng=3, bc=("wall",) * max(4, 2 * nd),
                 reconstruction="fog", riemann_solver="rusanov", time_stepper="rk2", max_cfl=0.3, max_time=1e30,
                 output_delta=1e30)
    q = np.zeros(cfg.shape)
    q[0], q[-1] = 1.0, 2.5
    at = (nd > 2) * 5, (nd > 1) * 5, 40
    q[(0,) + at], q[(-1,) + at] = 1e-170, 1e170
    sim = orc.OracleSim(cfg)
    sim.set_q(q)
    sim.fill_bcs()
    assert sim.compute_dt(0.0, 0.0) == 0.0
    with M.HydroContext(cfg) as ctx:
        ctx.upload(q)
        ctx.fill_bcs()
        assert ctx.compute_dt(0.0, 0.0) == 0.0
