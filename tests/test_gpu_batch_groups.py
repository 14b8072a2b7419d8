"""A batch whose problems differ in what shapes their covariance launch: orders
with and without a table, bivariate and univariate, Euclidean and great circle,
2D and 3D, one tile and many.  Each result against the same problem alone: the
two paths may round in another order, which the condition of these fields (up to
1e6) makes n eps cond, 1e-9 at most.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs
from exageostatcpp_amd import capi

pytestmark = pytest.mark.gpu


def problem(ctx, kernel, n, metric, dim, seed):
    r = np.random.default_rng(seed)
    x, y = (r.random(n), r.random(n)) if metric == 0 else (10 * r.random(n), 40 + 10 * r.random(n))
    p = egs.Problem(ctx, kernel, x, y, r.random(n) if dim == 3 else None, metric=metric, dts=128)
    p.set_observations(r.standard_normal(n * (2 if kernel else 1)))
    return p


@pytest.mark.parametrize("forms", [[0], [2, 2], [0, 1, 2, 3, 4, 5, 6, 0, 2, 4]])
def test_batch_of_forms(forms):
    # kernel, metric, dim, theta
    kinds = [(0, 0, 2, [1.0, 0.1, 0.5]), (0, 0, 2, [1.2, 0.1, 0.9]), (0, 0, 3, [1.0, 0.2, 1.5]),
             (0, 1, 2, [1.0, 200.0, 0.7]), (1, 0, 2, [1.0, 1.5, 0.1, 0.5, 1.0, 0.3]),
             (1, 0, 2, [1.0, 1.0, 0.08, 0.6, 1.1, 0.2]), (1, 1, 2, [1.0, 1.0, 150.0, 0.6, 0.8, 0.2])]
    ctx = egs.Context(0)
    probs, thetas = [], []
    for i, f in enumerate(forms):
        kernel, metric, dim, theta = kinds[f]
        probs.append(problem(ctx, kernel, (40, 300, 128, 700)[i % 4], metric, dim, 10 * i + f))
        thetas.append(theta)
    alone = [p.loglik(t) for p, t in zip(probs, thetas)]
    for got, want in zip(capi.loglik_batch(probs, thetas), alone):
        assert np.all(np.abs(np.subtract(got, want)) <= 1e-9 * np.abs(want))
    for p in probs:
        p.close()
    ctx.close()


@pytest.mark.parametrize("failed_before", [False, True])
def test_predict_with_the_factor_of_a_batch(failed_before):
    """A prediction that reuses a batch's factor: nothing that an earlier
    factorization of the problem left (or did not leave) is read for it."""
    ctx = egs.Context(0)
    theta, miss = [1.0, 0.1, 0.5], np.random.default_rng(3).random((2, 20))
    p, q, fresh = (problem(ctx, 0, 300, 0, 2, s) for s in (5, 6, 5))
    if failed_before:
        with pytest.raises(egs.NotPositiveDefinite):
            p.loglik([-1.0, 0.1, 0.5])   # negative variance
    assert not any(isinstance(r, Exception) for r in capi.loglik_batch([p, q], [theta, theta]))
    want = fresh.predict(theta, *miss)[0]
    got = p.predict(theta, *miss)[0]
    assert np.max(np.abs(got - want)) <= 1e-9 * np.max(np.abs(want))
    for e in (p, q, fresh):
        e.close()
    ctx.close()
