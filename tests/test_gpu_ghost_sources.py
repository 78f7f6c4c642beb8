"""Stages that read wall, symmetric, zero-gradient and periodic ghosts from their source cells, face by
face: bit for bit the oracle's (FP64), and bit for bit a context with a hook that does nothing, whose
stages read filled ghosts (both forms, tracers, gravity). Ghosts that a caller uploaded and did not
fill are read as they are by the first stage."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu

FACES = [("wall", "symmetric"), ("zerograd", "wall"), ("symmetric", "zerograd"), ("wall", "wall"), ("periodic",) * 2]
# (nd, sizes): no more interior cells than ghosts, one wavefront's columns and a few more, several strips
GRIDS = [(1, (3,)), (1, (64,)), (1, (190,)), (2, (3, 3)), (2, (62, 5)), (2, (131, 20)), (3, (3, 4, 3)),
         (3, (66, 7, 5))]


def _cfg(nd, n, first, **more):
    bc = tuple(f for a in range(nd) for f in FACES[(first + a) % len(FACES)])
    n = tuple(n) + (1,) * (3 - nd)
    return Config(num_dim=nd, nx=n[0], ny=n[1], nz=n[2], ng=3, x_dim=n[0] / 64.0,
                  bc=bc + ("wall",) * max(0, 4 - 2 * nd), reconstruction="weno5z", riemann_solver="hllc",
                  time_stepper="ssprk3", max_cfl=0.3, max_time=1e30, output_delta=1e30, **more)


def _state(cfg, seed):
    """A rough flow that runs into the faces, every cell set on its own (ghosts too)."""
    rng = np.random.default_rng(seed)
    shape = cfg.shape[1:]
    rho, p = 1.0 + 0.4 * rng.random(shape), 1.0 + 0.4 * rng.random(shape)
    v = [0.3 * rng.standard_normal(shape) for _ in range(cfg.num_dim)]
    q = [rho, *(rho * a for a in v), p / (cfg.gamma - 1) + 0.5 * rho * sum(a * a for a in v)]
    return np.stack(q + [rho * rng.random(shape) for _ in range(cfg.num_tracers)])


@pytest.mark.parametrize("first", range(len(FACES)))
@pytest.mark.parametrize("grid", range(len(GRIDS)))
@pytest.mark.parametrize("fill", [True, False])
def test_oracle_bitwise(orc, grid, first, fill):
    cfg = _cfg(*GRIDS[grid], first)
    q0 = _state(cfg, 10 * grid + first)
    if not fill and cfg.num_dim > 1 and set(cfg.bc[:2 * cfg.num_dim]) <= {"periodic", "zerograd"}:
        pytest.skip("ghosts always read from their sources")
    sim = orc.OracleSim(cfg)
    sim.set_q(q0)
    if fill:
        sim.fill_bcs()
    t, p, _ = sim.run(max_steps=3)
    for host_loop in (False, True):
        with M.HydroContext(cfg) as ctx:
            ctx.upload(q0)
            if fill:
                ctx.fill_bcs()
            if host_loop:
                assert M.run_to_time(ctx, max_steps=3)[0] == t
            else:
                assert ctx.run(3) == (t, p)
            np.testing.assert_array_equal(ctx.download(), sim.get_q())


@pytest.mark.parametrize("first", range(len(FACES)))
@pytest.mark.parametrize("kind", ["fp64_tracers", "fp32c", "fp32c_floors", "fp32c_tracers", "fp32c_3d"])
def test_sources_equal_filled_ghosts(first, kind):
    nd, n = (3, (40, 9, 8)) if kind.endswith("3d") else (2, (131, 20))
    more = dict(num_tracers=2, gravity=(0.0, -0.1, 0.0)) if kind.endswith("tracers") else {}
    cfg = _cfg(nd, n, first, **more)
    form = M.FP64 if kind.startswith("fp64") else M.FP32C
    floors = (1e-3, 1e-3) if kind.endswith("floors") else (0.0, 0.0)
    q0 = _state(cfg, first)
    out = []
    for hook in (None, lambda view: None):
        with M.HydroContext(cfg, precision_form=form, rho_floor=floors[0], p_floor=floors[1]) as ctx:
            ctx.set_user_bc(hook)
            ctx.upload(q0)
            ctx.fill_bcs()
            out.append((ctx.run(3), ctx.download()))
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
