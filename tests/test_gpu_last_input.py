"""EOS fields of the last stage's input after steps that read ghosts from their sources, which leave that
input's ghosts unfilled: equal to those after the same stages one by one (mh_stage fills every stage's
ghosts), for every face kind and way of stepping, and where a hook or a table is installed in between."""
import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config
from mosscap_amd.lte_table import generate

pytestmark = pytest.mark.gpu

H_MASS, K_B = 1.6737830080950003e-27, 1.380649e-23
GRIDS = [(1, ("wall", "symmetric"), 0), (1, ("periodic", "periodic"), 0),
         (2, ("wall", "wall", "symmetric", "zerograd"), 0), (2, ("periodic",) * 2 + ("wall",) * 2, 2),
         (2, ("zerograd",) * 4, 0), (3, ("wall", "zerograd", "symmetric", "wall", "periodic", "periodic"), 0)]


def _cfg(nd, bc, tracers):
    return Config(num_dim=nd, nx=67, ny=24 if nd > 1 else 1, nz=10 if nd > 2 else 1, ng=3,
                  bc=bc + ("wall",) * max(0, 4 - 2 * nd), reconstruction="muscl", slope_limiter="minmod",
                  riemann_solver="hll", time_stepper="ssprk3", gamma=5.0 / 3.0, max_cfl=0.3, max_time=1e30,
                  output_delta=1e30, num_tracers=tracers)


def _state(cfg):
    """Partly ionised hydrogen in motion, every cell set on its own (ghosts too)."""
    rng = np.random.default_rng(12)
    shape = cfg.shape[1:]
    rho = 10 ** (-8.0 + 0.5 * rng.random(shape))
    p = rho * (K_B / H_MASS) * 1.5 * 10 ** (4.0 + 0.3 * rng.random(shape))
    v = [300.0 * rng.standard_normal(shape) for _ in range(cfg.num_dim)]
    q = [rho, *(rho * a for a in v), p / (cfg.gamma - 1) + 0.5 * rho * sum(a * a for a in v)]
    return np.stack(q + [rho * rng.random(shape) for _ in range(cfg.num_tracers)])


@pytest.mark.parametrize("then", ["read", "hook", "table"])
@pytest.mark.parametrize("entry", ["time_step", "graph", "eager", "stages_after_graph"])
@pytest.mark.parametrize("grid", range(len(GRIDS)))
@pytest.mark.parametrize("form", [M.FP64, M.FP32C])
def test_fields_of_last_stage_input(form, grid, entry, then):
    cfg = _cfg(*GRIDS[grid])
    q0 = _state(cfg)
    with M.HydroContext(cfg, precision_form=form) as a, M.HydroContext(cfg, precision_form=form) as b:
        for c in (a, b):
            c.upload(q0)
            c.fill_bcs()
        steps = 1 if entry == "time_step" else 3
        if entry == "time_step":
            a.time_step(a.compute_dt(0.0, 0.0))
        else:
            a.run(steps, use_graph=entry != "eager")
        if entry == "stages_after_graph":
            dt = a.compute_dt(0.0, 0.0)
            for s in range(3):
                a.stage(s, dt)
            steps += 1
        for k in range(steps):
            dt = b.compute_dt(0.0, 0.0)
            for s in range(3 if k + 1 < steps else 2):
                b.stage(s, dt)
        if then == "hook":
            a.set_user_bc(lambda view: None)
        if then == "table":
            a.set_tabulated_eos(generate(32, 16))
        ya, Ta = a.eos_fields(which=1)
        yb, Tb = b.eos_fields(which=0)  # its current state is the input of a's last stage
    np.testing.assert_array_equal(Ta, Tb)
    np.testing.assert_array_equal(ya, yb)
