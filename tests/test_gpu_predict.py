"""Kriging and triangular solves return their vector with the failure word in one
copy: one value, as many as the problem has rows, and more; buffers that grow
between calls.  Against numpy with K_nu from scipy, to n eps times this field's
condition number (below 1e3): 1e-11.
"""
import numpy as np
import pytest
from scipy.linalg import solve_triangular
from scipy.special import gamma, kv

import exageostatcpp_amd as egs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


def matern(d, nu):
    out = np.ones_like(d)
    m = d > 0
    out[m] = d[m] ** nu * kv(nu, d[m]) / (2 ** (nu - 1) * gamma(nu))
    return out


@pytest.mark.parametrize("nu", [0.5, 0.83])
@pytest.mark.parametrize("n", [1, 64, 255, 256, 257, 700])
def test_vectors(ctx, n, nu):
    r = np.random.default_rng(n)
    root = int(np.ceil(np.sqrt(n)))
    cell = np.arange(n)
    x, y = ((c + 0.5 + r.uniform(-0.4, 0.4, n)) / root for c in (cell // root, cell % root))
    z = r.standard_normal(n)
    rng = 0.8 / root
    p = egs.Problem(ctx, 0, x, y, dts=128)
    p.set_observations(z)
    theta = [1.3, rng, nu]
    p.loglik(theta)
    a = 1.3 * matern(np.hypot(x[:, None] - x, y[:, None] - y) / rng, nu)
    low = np.linalg.cholesky(a)
    w = np.linalg.solve(a, z)
    for m in (1, 128, 129, 512, 513, 2, 3000):   # padded rows: 128 to 768
        t = r.random((2, m))
        t[:, 0] = x[0], y[0]   # one target on a location
        want = 1.3 * matern(np.hypot(t[0][:, None] - x, t[1][:, None] - y) / rng, nu) @ w
        got = p.predict(theta, t[0], t[1])[0]
        assert np.max(np.abs(got - want)) <= 1e-11 * np.max(np.abs(z))
    for trans in (False, True):
        want = solve_triangular(low.T if trans else low, z, lower=not trans)
        got = p.trsm(z, trans=trans)
        assert np.max(np.abs(got - want)) <= 1e-11 * np.max(np.abs(want))
    assert p.loglik(theta)[2] == pytest.approx(w @ z, rel=1e-11)
    p.close()


def test_bivariate(ctx):
    n = 120   # 240 rows
    r = np.random.default_rng(n)
    x, y = r.random((2, n))
    p = egs.Problem(ctx, 1, x, y, dts=64)
    z = r.standard_normal(2 * n)
    p.set_observations(z)
    theta = [1.0, 1.0, 0.05, 0.6, 0.9, 0.0]   # uncorrelated: two univariate fields
    p.loglik(theta)
    for m in (1, 256, 257):
        t = r.random((2, m))
        got = p.predict(theta, t[0], t[1])[0]
        for v, nu in ((0, 0.6), (1, 0.9)):
            q = egs.Problem(ctx, 0, x, y, dts=64)
            q.set_observations(z[v::2])
            want = q.predict([1.0, 0.05, nu], t[0], t[1])[0]
            q.close()
            assert np.max(np.abs(got[v::2] - want)) <= 1e-11 * np.max(np.abs(z))
    p.close()
