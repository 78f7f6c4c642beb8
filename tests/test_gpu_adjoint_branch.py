"""WENO5-Z's VJP at stencils whose outer smoothness indicators differ in their last bits or not at all:
tau's derivative takes the sign of beta0 - beta2 as the forward rounds it."""
import numpy as np
import pytest

import mosscap_amd as M

pytestmark = pytest.mark.gpu


def _betas(s):
    c = 13.0 / 12.0
    a0, b0 = s[:, 0] - 2 * s[:, 1] + s[:, 2], s[:, 0] - 4 * s[:, 1] + 3 * s[:, 2]
    a2, b2 = s[:, 2] - 2 * s[:, 3] + s[:, 4], 3 * s[:, 2] - 4 * s[:, 3] + s[:, 4]
    return c * (a0 * a0) + 0.25 * (b0 * b0), c * (a2 * a2) + 0.25 * (b2 * b2)


def test_weno_vjp_takes_the_forwards_branch():
    # a large field whose beta1 vanishes next to equal outer indicators: tau / (beta1 + eps) is then
    # large, and its derivative shows the sign
    rng = np.random.default_rng(4)
    n = 400000
    d, e = rng.normal(size=n), rng.normal(size=n)
    s = np.stack([e, 0 * d, 0 * d, 0 * d, e], axis=1)  # beta1 = 0, beta0 = beta2 up to the end cells
    s[:, 4] = np.nextafter(s[:, 4], np.where(rng.random(n) < 0.5, np.inf, -np.inf))
    b0, b2 = _betas(s)
    cot = np.tile([1.0, 0.5], (n, 1))
    hand, dual = M.probe_vjp(0, s, cot), M.probe_vjp(1, s, cot)
    assert (b0 == b2).any() and (b0 != b2).any()
    scale = np.abs(dual).max(axis=1, keepdims=True)
    np.testing.assert_allclose(hand / scale, dual / scale, rtol=0, atol=1e-11)
