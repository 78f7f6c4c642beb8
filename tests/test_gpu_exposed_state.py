"""A state written through mh_device_state outside a hook, between calls, with mh_fill_bcs after the write
or without: the next step size and state are the oracle's for what was written, whatever the call."""
import ctypes as C

import numpy as np
import pytest

import mosscap_amd as M
from mosscap_amd import Config

pytestmark = pytest.mark.gpu


def _pointer(ctx):
    view = M.MhDeviceView()
    assert M.lib().mh_device_state(ctx.handle, C.byref(view)) == M.MH_OK
    return view.q


def _write(ctx, ptr, q):
    """q into the state's device buffer, behind the context's back."""
    with M.HydroContext(ctx.cfg) as other:
        other.upload(q)
        other.download_device(ptr)


@pytest.mark.parametrize("how", ["graph", "eager", "host_loop"])
@pytest.mark.parametrize("bc", ["wall", "symmetric", "periodic"])
@pytest.mark.parametrize("nd", [1, 2])
@pytest.mark.parametrize("fill", [True, False])
def test_written_state(orc, nd, bc, how, fill):
    cfg = Config(num_dim=nd, nx=131, ny=20 if nd > 1 else 1, ng=3, bc=(bc,) * 4, reconstruction="weno5z",
                 riemann_solver="hllc", time_stepper="ssprk3", max_cfl=0.3, max_time=1e30, output_delta=1e30)
    rng = np.random.default_rng(8)
    shape = cfg.shape[1:]
    rho, p = 1.0 + 0.4 * rng.random(shape), 1.0 + 0.4 * rng.random(shape)
    q0 = np.stack([rho, *(0.3 * rho * rng.standard_normal(shape) for _ in range(nd)), p / (cfg.gamma - 1) + rho])
    sim = orc.OracleSim(cfg)
    sim.set_q(q0)
    sim.fill_bcs()
    with M.HydroContext(cfg) as ctx:
        ctx.upload(q0)
        ctx.fill_bcs()
        clock = [(0.0, 0.0), (0.0, 0.0)]

        def steps(n):
            t, prev, _ = sim.run(*clock[0], max_steps=n)
            clock[0] = (t, prev)
            if how == "host_loop":
                t, prev, _ = M.run_to_time(ctx, *clock[1], max_steps=n)
            else:
                t, prev = ctx.run(n, *clock[1], use_graph=how == "graph")
            clock[1] = (t, prev)
            assert clock[1] == clock[0]
            np.testing.assert_array_equal(ctx.download(), sim.get_q())

        ptr = _pointer(ctx)  # asked for once: the buffers rotate, and every third step returns to this one
        steps(2)
        steps(1)
        for k in range(4):  # each time hotter, so the old maximum signal speed allows too long a step
            q = sim.get_q()
            q[-1] *= 1.5
            if k % 2 and (nd == 1 or bc != "periodic"):  # ghosts of the caller's own
                q[:, :, :, :3] *= 1.1
            _write(ctx, ptr, q)
            sim.set_q(q)
            if fill:
                ctx.fill_bcs()
                sim.fill_bcs()
            steps(2)
            steps(1)
