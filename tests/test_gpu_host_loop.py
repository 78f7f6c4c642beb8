"""Host-driven stepping (mh_compute_dt, mh_time_step): a step after mh_compute_dt leaves the maximum
signal speed behind, so the next mh_compute_dt does not rescan the state; whatever changes the state
or the clock in between makes it rescan. Every dt and state against the oracle, bit for bit; 1-D
grids read copied ghosts from their sources."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config, problems

pytestmark = pytest.mark.gpu


def _cfg(nd, bc, stepper):
    kw = dict(reconstruction="weno5z", riemann_solver="hllc", time_stepper=stepper, max_cfl=0.3, max_time=1e30,
              output_delta=1e30)
    if nd == 1:
        return Config(num_dim=1, nx=131, ng=3, bc=(bc, bc, "wall", "wall"), **kw)
    if nd == 2:
        return Config(num_dim=2, nx=65, ny=40, ng=3, bc=(bc,) * 4, **kw)
    return Config(num_dim=3, nx=20, ny=18, nz=17, ng=3, bc=(bc,) * 6, **kw)


def _state(cfg, seed):
    if cfg.num_dim == 3:
        return problems.blast_3d(cfg, seed=seed, p_ratio=2.0)
    rng = np.random.default_rng(seed)
    shape = cfg.shape[1:]
    rho = 1.0 + 0.2 * rng.random(shape)
    v = [0.3 * rng.standard_normal(shape) for _ in range(cfg.num_dim)]
    p = 1.0 + 0.3 * rng.random(shape)
    return np.stack([rho, *(rho * a for a in v), p / (cfg.gamma - 1) + 0.5 * rho * sum(a * a for a in v)])


@pytest.mark.parametrize("nd", [1, 2, 3])
@pytest.mark.parametrize("bc", ["periodic", "zerograd", "wall"])
@pytest.mark.parametrize("stepper", ["rk2", "ssprk3", "ssprk4"])
def test_host_loop_bitwise(orc, nd, bc, stepper):
    cfg = _cfg(nd, bc, stepper)
    q0, q1 = _state(cfg, 3), _state(cfg, 4)

    def steps(sim, step, dt_of, put):
        """A loop with the things a driver may do between steps; returns every dt."""
        dts = []
        put(q0)
        for k in range(10):
            dts.append(dt_of())
            if k == 2:
                dts.append(dt_of())  # asked twice
            step(dts[-1] * (0.5 if k == 4 else 1.0))
            if k == 5:
                step(dts[-1] * 0.25)  # a step without asking
            if k == 7:
                put(q1)  # another state
        dts.append(dt_of())
        return dts

    sim = orc.OracleSim(cfg)

    def put_oracle(q):
        sim.set_q(q)
        sim.fill_bcs()

    want = steps(sim, sim.time_step, lambda: sim.compute_dt(0.0, 0.0), put_oracle)
    with M.HydroContext(cfg) as ctx:
        def put(q):
            ctx.upload(q)
            ctx.fill_bcs()

        got = steps(ctx, ctx.time_step, lambda: ctx.compute_dt(0.0, 0.0), put)
        assert got == want
        np.testing.assert_array_equal(ctx.download(), sim.get_q())
        # mh_run goes on from the maximum that the last step left, and from a scan
        ctx.run(2)
        q = ctx.download()
        ctx.upload(sim.get_q())
        ctx.run(2)
        np.testing.assert_array_equal(ctx.download(), q)
