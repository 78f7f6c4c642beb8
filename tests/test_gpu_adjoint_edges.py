"""Riemann VJPs of a state without pressure: the pressure's cotangent is infinite, as dc_s/dp is, with
the sign it has at a vanishing pressure, and every other entry is the one at a vanishing pressure."""
import numpy as np
import pytest

import mosscap_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,axis", [("rusanov", 0), ("rusanov", 1), ("hllc", 0), ("hllc", 1)])
@pytest.mark.parametrize("side", [0, 4])
def test_riemann_vjp_without_pressure(solver, axis, side):
    rng = np.random.default_rng(6)
    n = 4000
    w = np.empty((n, 8))
    for o in (0, 4):
        w[:, o] = 10 ** rng.uniform(-1, 1, n)
        w[:, o + 1:o + 3] = rng.normal(size=(n, 2))
        w[:, o + 3] = 10 ** rng.uniform(-4, -2, n)
    # flow apart, so that HLLC's middle pressure lies below both sides' (its other wave speeds are
    # undefined without pressure)
    w[:, 1 + axis], w[:, 5 + axis] = -2.0 - rng.random(n), 2.0 + rng.random(n)
    cot = rng.normal(size=(n, 4))
    what = {"rusanov": 2, "hllc": 6}[solver] + 2 * axis
    w[:, side + 3] = 1e-40
    near = M.probe_vjp(what, w, cot)
    w[:, side + 3] = 0.0
    at = M.probe_vjp(what, w, cot)
    speed = np.abs(near[:, side + 3]) > 1e10  # c_s takes part in the flux
    assert speed.any() and (solver == "hllc" or speed.all())
    np.testing.assert_array_equal(at[speed, side + 3], np.sign(near[speed, side + 3]) * np.inf)
    rest = [k for k in range(8) if k != side + 3]
    np.testing.assert_allclose(at[:, rest], near[:, rest], rtol=1e-12, atol=1e-12)
