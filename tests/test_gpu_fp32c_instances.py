"""The compensated form's steps do not depend on which copy of a stage runs: ghosts read from their sources
or filled (a context with a hook that does nothing) give the same bits, for PPM with every limiter, solver
and option (WENO5-Z + HLLC: test_gpu_ghost_sources)."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", ["wall", "periodic"])
@pytest.mark.parametrize("kind", ["plain", "floors", "tracers", "3d"])
@pytest.mark.parametrize("solver", ["rusanov", "hll", "hllc"])
@pytest.mark.parametrize("limiter", ["vanleer", "monotonizedcentral", "minmod"])
def test_ppm_bits(limiter, solver, kind, bc):
    nd = 3 if kind == "3d" else 2
    cfg = Config(num_dim=nd, nx=131 if nd == 2 else 40, ny=20, nz=9 if nd > 2 else 1, ng=3, x_dim=2.0,
                 bc=(bc,) * (2 * nd), reconstruction="ppm", slope_limiter=limiter, riemann_solver=solver,
                 time_stepper="ssprk3", max_cfl=0.3, max_time=1e30, output_delta=1e30,
                 num_tracers=2 if kind == "tracers" else 0)
    floors = (1e-3, 1e-3) if kind == "floors" else (0.0, 0.0)
    rng = np.random.default_rng(3)
    shape = cfg.shape[1:]
    rho, p = 1.0 + 0.4 * rng.random(shape), 1.0 + 0.4 * rng.random(shape)
    v = [0.3 * rng.standard_normal(shape) for _ in range(nd)]
    q = [rho, *(rho * a for a in v), p / (cfg.gamma - 1) + 0.5 * rho * sum(a * a for a in v)]
    q0 = np.stack(q + [rho * rng.random(shape) for _ in range(cfg.num_tracers)])
    out = []
    for hook in (None, lambda view: None):
        with M.HydroContext(cfg, precision_form=M.FP32C, rho_floor=floors[0], p_floor=floors[1]) as ctx:
            ctx.set_user_bc(hook)
            ctx.upload(q0)
            ctx.fill_bcs()
            out.append((ctx.run(3), ctx.download()))
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
