"""The 96 x 192-block form of the FP64 trailing update at sizes where a launch
takes it (more than 768 blocks of 64 x 64, 1,800 on the critical stream): each
tile size with one panel, and with two panels at once (eleven tile columns and
more; twelve of 960 have ten, then nine tiles in a column, 2,250 and 2,025 blocks),
ragged last tiles, direct and replayed from a graph.

A v = L (L' v) for a random v, to the bound of a Cholesky factor's backward error,
n eps |L| |L'| |v|; replays equal to the first evaluation to 1e-12.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs

pytestmark = pytest.mark.gpu
THETA = [1.0, 0.03, 0.5]


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


# the launch of the columns beyond k + 2 at the first step: tiles x (dts / 64)^2
@pytest.mark.parametrize("n,dts", [(3260, 192),      # 105 x 9
                                   (3800, 384),      # 28 x 36
                                   (4600, 576),      # 15 x 81
                                   (5700, 960),      # 6 x 225
                                   (5300, 1152),     # 3 x 324
                                   (10600, 960),     # two panels, 40 rows in the last tile
                                   (11500, 960)])    # two panels
def test_factor(ctx, n, dts):
    r = np.random.default_rng(n)
    x, y, v = r.random(n), r.random(n), r.standard_normal(n)
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    p.set_observations(r.standard_normal(n))
    want = p.loglik(THETA)
    low = p.get_matrix()
    got = low @ (low.T @ v)
    scale = np.abs(low) @ (np.abs(low.T) @ np.abs(v))
    del low
    av = np.empty(n)
    for i in range(0, n, 500):
        av[i:i + 500] = np.exp(-np.hypot(x[i:i + 500, None] - x, y[i:i + 500, None] - y) / THETA[1]) @ v
    assert np.all(np.abs(got - av) <= n * np.finfo(float).eps * scale)
    p.set_graph(True)
    for _ in range(3):
        assert np.all(np.abs(np.subtract(p.loglik(THETA), want)) <= 1e-12 * np.abs(want))
    p.close()
