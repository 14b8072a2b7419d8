"""Results do not depend on what recycled device memory holds.  The library's
block cache hands a mixed plan's refinement vectors blocks that a problem with
NaN observations has just released; the plan then has to refine as it does in
fresh memory: to the residual at which the refinement stops (1e-12 of the
observations), and the quadratic form to 1e-12 times the condition number of
the FP64 plan's.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs
from exageostatcpp_amd import capi

pytestmark = pytest.mark.gpu
THETA = [1.0, 0.03, 0.5]


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


@pytest.fixture
def cache():
    capi.memory_cache(1 << 30)
    yield
    capi.memory_cache(0)


def leave_nans(ctx, words):
    """Two cached blocks of `words` doubles, all NaN (the vectors of a bivariate
    problem, whose other buffers are of other sizes)."""
    assert words % 64 == 0
    r = np.random.default_rng(words)
    p = egs.Problem(ctx, 1, 100.0 * r.random(words // 2), 100.0 * r.random(words // 2), dts=64)
    p.set_observations(np.full(words, np.nan))
    assert np.isnan(p.loglik([1.0, 1.0, 2.0, 0.5, 0.5, 0.1])[0])
    p.close()


@pytest.mark.parametrize("n,dts,bands", [(950, 192, (1, 2)), (1900, 384, (1, 1)), (1150, 192, (1, 4))])
def test_refinement(ctx, cache, n, dts, bands):
    r = np.random.default_rng(n)
    x, y, z = r.random(n), r.random(n), r.standard_normal(n)
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    p.set_observations(z)
    want = p.loglik(THETA)
    low = p.get_matrix()
    t = r.random((2, 50))
    kriged = p.predict(THETA, t[0], t[1])[0]
    p.close()
    leave_nans(ctx, 5 * ((n + dts - 1) // dts) * dts)
    q = egs.Problem(ctx, 0, x, y, dts=dts)
    q.set_observations(z)
    q.set_precision(capi.PRECISION_MIXED, *bands)
    q.set_fallback(0, 0.0)
    got = q.loglik(THETA)
    assert q.refinement()["residual"] <= 1e-11
    cond = np.linalg.cond(low) ** 2
    assert abs(got[2] - want[2]) <= 1e-12 * cond * abs(want[2])
    again = q.predict(THETA, t[0], t[1])[0]
    assert np.max(np.abs(again - kriged)) <= 1e-12 * cond * np.max(np.abs(kriged))
    q.close()
