"""How the 3-D march deals the planes' columns to wavefronts (march_columns): planes that share a
wavefront, planes with strips of their own, last groups of fewer wavefronts, against the oracle
bit for bit."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config, problems

pytestmark = pytest.mark.gpu

# (nx, ny, nz): several planes per wavefront; one wavefront and a bit per plane; exact multiples of
# 62 (own strips); as many wavefronts either way (own strips); between
SHAPES = [(7, 12, 9), (63, 8, 13), (62, 9, 10), (124, 8, 5), (56, 9, 7), (130, 10, 6)]
KINDS = [dict(reconstruction="weno5z", riemann_solver="hllc", bc=("periodic",) * 6),
         dict(reconstruction="weno5z", riemann_solver="hllc", bc=("wall", "zerograd", "zerograd", "wall", "periodic", "periodic")),
         dict(reconstruction="muscl", slope_limiter="minmod", riemann_solver="hll", bc=("zerograd",) * 6),
         dict(reconstruction="fog", riemann_solver="rusanov", bc=("symmetric", "wall") * 3)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", range(len(KINDS)))
def test_3d_columns_bitwise(orc, kind, shape):
    nx, ny, nz = shape
    cfg = Config(num_dim=3, nx=nx, ny=ny, nz=nz, ng=3, x_dim=nx / 32.0, max_cfl=0.3, time_stepper="ssprk3",
                 **KINDS[kind])
    q0 = problems.blast_3d(cfg, seed=kind + 21, p_ratio=2.0)
    sim = orc.OracleSim(cfg)
    sim.set_q(q0)
    sim.fill_bcs()
    t, p, _ = sim.run(max_steps=4)
    with M.HydroContext(cfg) as ctx:
        ctx.upload(q0)
        ctx.fill_bcs()
        assert ctx.run(4) == (t, p)
        np.testing.assert_array_equal(ctx.download(), sim.get_q())
    # spans of one row, of all rows
    for rows in (1, ny):
        with M.HydroContext(cfg, span_rows=rows) as ctx:
            ctx.upload(q0)
            ctx.fill_bcs()
            ctx.run(4)
            np.testing.assert_array_equal(ctx.download(), sim.get_q())
