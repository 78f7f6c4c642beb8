"""The FP64 functors' own division, square root and WENO5-Z (fast64.hpp) against the oracle, bit for
bit, at the scales where their shorter sequences could go wrong: tiny, denormal and zero numerators,
signed zeros, large and small fields, flat stencils next to jumps, both signs of the contact speed."""
import numpy as np
import pytest

from mosscap_amd import probe_math, probe_reconstruct, probe_riemann

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e-12, 1e-160, 1e-300, 5e-321, 1e6, 1e100, 1e150])
def test_weno5z_bitwise_over_scales(orc, scale):
    rng = np.random.default_rng(31)
    n = 40000
    s = rng.normal(size=(n, 5))
    s[: n // 4] = np.round(s[: n // 4] * 2) / 2
    jump = n // 4 + np.arange(n // 4)
    s[jump] = 1.0 + 1e-9 * s[jump]
    s[jump, 3:] += 10.0 ** rng.uniform(-12, 3, (n // 4, 1)) * (scale < 1e10)
    s *= scale
    s[-100:] = np.where(rng.random((100, 5)) < 0.5, 0.0, -0.0)
    s[-200:-100] = np.where(rng.random((100, 5)) < 0.3, 4.9e-324, 0.0)
    wl, wr = probe_reconstruct("weno5z", "minmod", s)
    ol, orr = orc.reconstruct("weno5z", "minmod", s)
    np.testing.assert_array_equal(wl, ol)
    np.testing.assert_array_equal(wr, orr)


@pytest.mark.parametrize("nd,axis", [(1, 0), (2, 1), (3, 2)])
@pytest.mark.parametrize("solver", ["hllc", "hll", "rusanov"])
def test_riemann_bitwise_over_scales(orc, solver, nd, axis):
    rng = np.random.default_rng(32)
    n = 60000
    w = [np.empty((n, 2 + nd)) for _ in range(2)]
    spread = 10.0 ** rng.uniform(-60, 60, (n, 1))
    spread[: n // 2] = 1.0
    for a in w:
        a[:, :1] = spread * 10.0 ** rng.uniform(-4, 4, (n, 1))
        a[:, -1:] = spread * 10.0 ** rng.uniform(-6, 6, (n, 1))
        a[:, 1:-1] = rng.normal(size=(n, nd))
        tiny = rng.random((n, nd))
        a[:, 1:-1] = np.where(tiny < 0.1, a[:, 1:-1] * 1e-305, np.where(tiny < 0.2, 0.0 * a[:, 1:-1], a[:, 1:-1]))
    same = slice(n // 2, n // 2 + 2000)  # a stationary or slow contact: equal pressures, equal velocities
    w[1][same, 1:] = w[0][same, 1:]
    w[0][-1000:, -1] = 0.0  # no pressure on the left: the sound speed's square root of zero
    f = probe_riemann(solver, axis, nd, 1.4, *w)
    np.testing.assert_array_equal(f, orc.riemann(solver, axis, nd, 1.4, *w))


def test_divide_ieee_at_the_edges_of_its_scaling():
    rng = np.random.default_rng(33)
    m = 1.0 + rng.random((2, 200000))
    e = rng.integers(-1074, 1024, (2, 200000)).astype(np.float64)
    a, b = m[0] * 2.0 ** (e[0] / 2) * 2.0 ** (e[0] - e[0] / 2), m[1] * 2.0 ** (e[1] / 2) * 2.0 ** (e[1] - e[1] / 2)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0, 4.9e-324, -2.2e-308, 1.7e308, 2.0 ** -970])
    a, b = np.concatenate([a, np.repeat(special, special.size)]), np.concatenate([b, np.tile(special, special.size)])
    with np.errstate(all="ignore"):
        want = a / b
    got = probe_math(0, a, b)
    np.testing.assert_array_equal(got, want)
    zero = want == 0
    np.testing.assert_array_equal(np.signbit(got[zero]), np.signbit(want[zero]))
