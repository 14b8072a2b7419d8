"""Covariance generation of whole problems (egs_covariance) against the oracle,
entry by entry: orders with and without a closed form, separations inside the
tables of the Matern function and on both sides of them, padding and ragged
tiles, both kernels and both metrics; and kriging through the same tables.

Tolerance 1e-13 relative per entry: the oracle's own K_nu is within 1e-14, the
tables' fit within 1e-16, and a rounding of the separation (about 4e-16) grows
by the separation over the range, at most 90 inside the tables.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs
from oracle import orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


def check(ctx, kernel, loc, theta, dts, metric=0, tol=1e-13):
    p = egs.Problem(ctx, kernel, *loc, metric=metric, dts=dts)
    p.covariance(theta)
    got = p.get_matrix()
    p.close()
    n = got.shape[0]
    ref = np.tril(orc.covariance_tile(kernel, n, n, 0, 0, loc, loc, theta, metric=metric))
    big = np.abs(ref) > 1e-290
    assert np.isfinite(got).all()
    assert np.max(np.abs(got - ref)[big] / np.abs(ref)[big]) < tol
    assert np.max(np.abs(got - ref)[~big], initial=0.0) < 1e-290


@pytest.mark.parametrize("nu", [0.05, 0.3, 0.5, 0.83, 1.0, 1.5, 2.5, 3.7, 19.9, 20.5])
@pytest.mark.parametrize("rng", [0.004, 0.1, 30.0])
def test_univariate_orders_and_ranges(ctx, nu, rng):
    # range 0.004: separations to 350 (beyond the tables); 30: most below 2^-5,
    # and a pair of near-duplicates below 2^-10
    r = np.random.default_rng(int(nu * 100))
    x, y = r.random(130), r.random(130)
    x[1], y[1] = x[0] + 1e-6, y[0]
    if nu > 20 and rng > 1:
        rng = 1.0   # K_nu overflows in both at smaller separations
    # 350 ranges times the separation's rounding: 2e-13; 20 recurrence steps: 1e-12
    check(ctx, 0, (x, y), [1.7, rng, nu], 64, tol=1e-12 if nu > 20 else 2e-13 if rng < 0.01 else 1e-13)


@pytest.mark.parametrize("n,dts", [(1, 64), (63, 64), (65, 64), (192, 192), (321, 320), (500, 192), (200, 384)])
def test_tiles_and_padding(ctx, n, dts):
    r = np.random.default_rng(n)
    check(ctx, 0, (r.random(n), r.random(n)), [1.0, 0.1, 0.7], dts)


def test_three_dimensions(ctx):
    r = np.random.default_rng(3)
    check(ctx, 0, tuple(r.random((3, 140))), [1.0, 0.2, 0.9], 64)


@pytest.mark.parametrize("nu", [0.5, 0.8])
def test_great_circle_univariate(ctx, nu):
    r = np.random.default_rng(6)
    check(ctx, 0, (r.uniform(-60, 60, 130), r.uniform(-170, 170, 130)), [1.0, 900.0, nu], 64, metric=1, tol=1e-12)


@pytest.mark.parametrize("nu1,nu2", [(0.5, 1.5), (0.5, 1.0), (0.6, 0.6), (0.4, 1.3)])
@pytest.mark.parametrize("metric", [0, 1])
def test_bivariate_tables(ctx, nu1, nu2, metric):
    # no table, two, two of equal order, three
    r = np.random.default_rng(5)
    n = 97
    if metric:
        loc = (r.uniform(-60, 60, n), r.uniform(-170, 170, n))
        # sin and asin of the distance differ by ulps between the libraries
        check(ctx, 1, loc, [1.0, 2.0, 900.0, nu1, nu2, 0.4], 64, metric=1, tol=1e-12)
    else:
        check(ctx, 1, (r.random(n), r.random(n)), [1.0, 2.0, 0.1, nu1, nu2, 0.4], 64)


@pytest.mark.parametrize("kernel,theta", [(0, [1.0, 0.1, 0.8]), (1, [1.0, 2.0, 0.1, 0.4, 1.3, 0.4])])
def test_kriging_after_another_theta(ctx, kernel, theta):
    # the tables are of the last covariance parameters; kriging needs its own
    r = np.random.default_rng(8)
    loc = (r.random(150), r.random(150))
    pv = 2 if kernel else 1
    z = r.standard_normal(150 * pv)
    xm, ym = r.random(7), r.random(7)
    p = egs.Problem(ctx, kernel, *loc, dts=64)
    p.set_observations(z)
    other = list(theta)
    other[-1 if kernel == 0 else 3] += 0.2
    p.loglik(theta)
    p.loglik(other)
    got = p.predict(theta, xm, ym)[0]
    p.close()
    n = 150 * pv
    s = orc.covariance_tile(kernel, n, n, 0, 0, loc, loc, theta)
    s12 = orc.covariance_tile(kernel, 7 * pv, n, 0, 0, (xm, ym), loc, theta)
    want = s12 @ np.linalg.solve(s, z)
    assert np.max(np.abs(got - want)) < 1e-8 * np.max(np.abs(want))
