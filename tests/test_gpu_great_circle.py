"""Covariances of near locations on the sphere, against 80-bit values.

The separation of two locations with latitudes within 60 degrees is good to
about 8 eps, whatever their longitudes (difference, conversion and sine one
rounding each or two, squared and rooted, cos(latitude) to tan(60) * pi/3 eps):
an entry exp(-d) to 10 d eps + 4 eps, and through the table of another order,
whose own values are good to 6e-15, to 20 d eps + 6e-15.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
LD = np.longdouble
PI = LD(np.pi) + LD(1.2246467991473532e-16)


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


def separations(lat, lon, i, j):
    lat, lon = lat.astype(LD), lon.astype(LD)   # differences before the conversion: exact
    u, v = np.sin((lat[j] - lat[i]) * PI / 360), np.sin((lon[j] - lon[i]) * PI / 360)
    return 2 * LD(6371) * np.arcsin(np.sqrt(u * u + np.cos(lat[i] * PI / 180) * np.cos(lat[j] * PI / 180) * v * v))


def bessel_form(d, nu):
    """d^nu K_nu(d) / (2^(nu - 1) Gamma(nu)) by the trapezoidal rule, nu = 1 or 2."""
    h = LD(1) / 7
    out = LD(0.5) * np.exp(-d)
    for k in range(1, int(7 * np.arccosh(1 + 900 / float(d.min()))) + 1):
        t = k * h
        out += np.exp(-d * np.cosh(t) + nu * t) * (1 + np.exp(-2 * nu * t)) / 2
    return out * h * d ** nu / (1 if nu == 1 else 2)


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("nu", [0.5, 1.0, 2.0])
def test_near_locations(ctx, kernel, nu):
    r = np.random.default_rng(3)
    n, rng = 400, 1.0   # a cloud of a few km, far from longitude 0
    lat, lon = 51.0 + 0.02 * r.random(n), 171.0 + 0.03 * r.random(n)
    p = egs.Problem(ctx, kernel, lat, lon, metric=1, dts=320)
    p.covariance([1.0, rng, nu] if kernel == 0 else [1.0, 1.0, rng, 0.5, nu, 0.1])
    a = p.get_matrix()
    p.close()
    step = 1 + kernel   # of the bivariate field the second variable
    i, j = np.tril_indices(n, -1)
    got = a[step * i + kernel, step * j + kernel]
    assert np.all(a[np.arange(len(a)), np.arange(len(a))] == 1.0)
    d = separations(lat, lon, i, j) / LD(rng)
    want = np.exp(-d) if nu == 0.5 else bessel_form(d, int(nu))
    bound = (10 * d + 4) * EPS if nu == 0.5 else 20 * d * EPS + 6e-15
    assert np.all(np.abs(got - want) <= bound * want)
