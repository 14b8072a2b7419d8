"""Tiles above 1,152, whose diagonal tiles are factored by two launches per block
column instead of one per tile: the smallest such size, the largest but one,
one block beyond a tile, a tile's last block, a single tile; direct, replayed
from a graph, batched, and mixed.

Tolerances: the factor's backward error to 64 n eps (Higham's bound with a
small constant); values against the same field in tiles of 64 to 1e-11 (n eps
times this field's condition number), mixed within its 1e-6.
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


def field(ctx, n, dts):
    r = np.random.default_rng(n)
    p = egs.Problem(ctx, 0, r.random(n), r.random(n), dts=dts)
    p.set_observations(r.standard_normal(n))
    return p


def close(a, b, tol):
    a, b = np.asarray(a), np.asarray(b)
    assert np.max(np.abs(a - b)) <= tol * np.max(np.abs(b))


@pytest.mark.parametrize("n,dts", [(60, 1216), (1216, 1216), (1217, 1216), (3700, 1216), (2688, 1344), (3001, 1536), (1985, 1984),
                                   (4096, 1984)])
def test_fp64(ctx, n, dts):
    p = field(ctx, n, dts)
    p.covariance(THETA)
    a = p.get_matrix()
    p.potrf()
    low = p.get_matrix()
    assert np.max(np.abs(low @ low.T - (a + np.tril(a, -1).T))) < 64 * n * np.finfo(float).eps
    t = np.random.default_rng(1).random((2, 20))
    out = []
    for q in (p, field(ctx, n, 64)):
        llh = q.loglik(THETA)
        out.append((llh, q.predict(THETA, t[0], t[1])[0], q.generate_observations(THETA, seed=3)))
    for x, y in zip(*out):
        close(x, y, 1e-11)
    want = p.loglik(THETA)
    p.set_graph(True)
    for _ in range(3):
        close(p.loglik(THETA), want, 1e-12)
    p.close()
    q.close()


@pytest.mark.parametrize("sizes,dts", [([2500, 1217, 300, 1216, 64], 1216), ([2100, 1984, 1000], 1984)])
def test_batch(ctx, sizes, dts):
    probs = [field(ctx, n, dts) for n in sizes]
    got = capi.loglik_batch(probs, [THETA] * len(sizes))
    for p, n, g in zip(probs, sizes, got):
        q = field(ctx, n, 64)
        close(g, q.loglik(THETA), 1e-11)
        q.close()
        p.close()


def test_first_failing_minor_is_reported(ctx):
    p = field(ctx, 1300, 1216)
    with pytest.raises(egs.NotPositiveDefinite, match=r"leading minor 1\)"):
        p.loglik([-1.0, 0.1, 0.5])
    p.close()


def test_mixed(ctx):
    p = field(ctx, 4100, 1344)
    want = p.loglik(THETA)
    p.set_precision(capi.PRECISION_MIXED, 1, 1)
    got = p.loglik(THETA)
    p.close()
    close(got[0], want[0], 1e-6)
    close(got[2], want[2], 1e-8)
