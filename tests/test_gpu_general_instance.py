"""The FP64 stage with a gravity source on launches of at most and of more than one wavefront per SIMD,
which run different instances: both the oracle's bits, mirrored and copied ghosts alike."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [("periodic",) * 4, ("periodic", "periodic", "wall", "symmetric")])
def test_fp64_gravity_both_instances(orc, bc):
    # 11 strips of columns, 189 rows: 95 spans of two rows are 1045 wavefronts, 93 spans 1023
    cfg = Config(num_dim=2, nx=640, ny=189, ng=3, bc=bc, reconstruction="weno5z", riemann_solver="hllc",
                 time_stepper="ssprk3", max_cfl=0.3, max_time=1e30, output_delta=1e30, gravity=(0.2, -0.1, 0.0))
    rng = np.random.default_rng(5)
    shape = cfg.shape[1:]
    rho, p = 1.0 + 0.4 * rng.random(shape), 1.0 + 0.4 * rng.random(shape)
    v = [0.3 * rng.standard_normal(shape) for _ in range(2)]
    q0 = np.stack([rho, rho * v[0], rho * v[1], p / (cfg.gamma - 1) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2)])
    sim = orc.OracleSim(cfg)
    sim.set_q(q0)
    sim.fill_bcs()
    t, prev, _ = sim.run(max_steps=2)
    for span_rows in (2, 3, 0):
        with M.HydroContext(cfg, span_rows=span_rows) as ctx:
            ctx.upload(q0)
            ctx.fill_bcs()
            assert ctx.run(2) == (t, prev)
            np.testing.assert_array_equal(ctx.download(), sim.get_q())
