"""The tracer march at the edges of its strips and spans, every reconstruction, fluxes of both signs
side by side, ghosts read from their sources or filled, against the oracle bit for bit."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu

# a strip has 62, 60 or 58 output columns (stencil order 0, 1, 2)
SIZES = [(3, 3), (57, 9), (58, 4), (59, 31), (61, 5), (117, 12), (125, 40)]
SCHEMES = [("fog", "minmod"), ("muscl", "minmod"), ("muscl", "vanleer"), ("muscl", "monotonizedcentral"),
           ("ppm", "minmod"), ("ppm", "vanleer"), ("ppm", "monotonizedcentral"), ("weno5z", "minmod")]
FACES = [("periodic",) * 4, ("wall", "zerograd", "symmetric", "wall"), ("zerograd", "symmetricoutflowdiode", "wall", "wall")]


@pytest.mark.parametrize("scheme", range(len(SCHEMES)))
@pytest.mark.parametrize("size", range(len(SIZES)))
def test_tracers_bitwise(orc, scheme, size):
    recon, limiter = SCHEMES[scheme]
    nx, ny = SIZES[size]
    cfg = Config(num_dim=2, nx=nx, ny=ny, ng=3, x_dim=nx / 64.0, bc=FACES[(scheme + size) % len(FACES)],
                 reconstruction=recon, slope_limiter=limiter, riemann_solver="hllc", time_stepper="rk2", max_cfl=0.3,
                 max_time=1e30, output_delta=1e30, num_tracers=1 + size % 3)
    rng = np.random.default_rng(8 * scheme + size)
    shape = cfg.shape[1:]
    rho, p = 1.0 + 0.4 * rng.random(shape), 1.0 + 0.4 * rng.random(shape)
    v = [0.3 * rng.standard_normal(shape) for _ in range(2)]
    q0 = np.stack([rho, *(rho * a for a in v), p / (cfg.gamma - 1) + 0.5 * rho * sum(a * a for a in v)]
                  + [rho * rng.standard_normal(shape) for _ in range(cfg.num_tracers)])
    sim = orc.OracleSim(cfg)
    sim.set_q(q0)
    sim.fill_bcs()
    t, prev, _ = sim.run(max_steps=2)
    with M.HydroContext(cfg) as ctx:
        ctx.upload(q0)
        ctx.fill_bcs()
        assert ctx.run(2) == (t, prev)
        np.testing.assert_array_equal(ctx.download(), sim.get_q())
