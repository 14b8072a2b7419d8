"""The two schedules of the trailing update: tile column k + 2 updated by a launch
of its own, or by the critical stream with two panels at once, which FP64
factorizations of at least eleven tile columns begin with.  Ten to fourteen
columns, 64 x 64 updates (these tiles are too few for the 96 x 192 form), ragged
last tiles, direct and replayed from a graph; against the covariance matrix itself: 64 n eps on the factor's
backward error (Higham), and the replays equal to the first to 1e-12.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dts", [64, 192, 320])
@pytest.mark.parametrize("tiles", [10, 11, 12, 14])
@pytest.mark.parametrize("ragged", [0, 37])
def test_factor(ctx, dts, tiles, ragged):
    n = tiles * dts - ragged
    r = np.random.default_rng(n)
    x, y, z = r.random(n), r.random(n), r.standard_normal(n)
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    p.set_observations(z)
    theta = [1.0, 0.05, 0.5]
    p.covariance(theta)
    a = p.get_matrix()
    a = a + np.tril(a, -1).T
    p.potrf()
    low = p.get_matrix()
    assert np.max(np.abs(low @ low.T - a)) < 64 * n * np.finfo(float).eps
    want = p.loglik(theta)
    p.set_graph(True)
    for _ in range(3):
        got = p.loglik(theta)
        assert np.all(np.abs(np.subtract(got, want)) <= 1e-12 * np.abs(want))
    p.close()
