"""The FP64 trailing update at the sizes where its two forms meet (64 x 64 and
96 x 192 blocks) and at their edges: one tile beyond the panel, the smallest
and an odd multiple of 192, counts of blocks on both sides of the rule, ragged
last tiles.  The factor of the whole matrix against LAPACK's, on a
well-conditioned field: 1e-12 relative to the largest entry (a few hundred
times n eps), and the log-likelihood against the oracle's formula at 1e-11.
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


# 128 blocks of 64 x 64 (32-row halves up to there): 32 tiles of 128 (33 columns), 5 of 320 (6), 14 of 192 (15)
# more than 768 blocks of 64 x 64 in a launch: 2,900 and 3,100 locations in tiles of 192 (91 and 105 tiles of 9
# blocks), 3,500 in tiles of 384 (28 of 36); the other tile sizes in test_gpu_update192.py
@pytest.mark.parametrize("n,dts", [(200, 192), (500, 192), (2700, 192), (3100, 192), (900, 384), (2650, 384),
                                   (3500, 384), (1800, 576), (2900, 576), (2000, 960), (3000, 960), (1900, 1152),
                                   (3000, 128), (4224, 128), (4340, 128), (1900, 320), (2210, 320), (2880, 192),
                                   (2900, 192), (65, 64), (97, 64)])
def test_factor_and_likelihood(ctx, n, dts):
    r = np.random.default_rng(n)
    x, y, z = r.random(n), r.random(n), r.standard_normal(n)
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    p.set_observations(z)
    llh, logdet, quad = p.loglik([1.0, 0.05, 0.5])
    low = p.get_matrix()
    p.close()
    a = np.exp(-np.hypot(x[:, None] - x, y[:, None] - y) / 0.05)
    ref = np.linalg.cholesky(a)
    assert np.max(np.abs(low - ref)) < 1e-12 * np.max(np.abs(ref)) * np.sqrt(np.linalg.cond(ref))
    w = np.linalg.solve(ref, z)
    assert abs(quad - w @ w) < 1e-11 * quad
    assert abs(logdet - 2 * np.log(np.diag(ref)).sum()) < 1e-11 * abs(logdet)
    assert abs(llh + 0.5 * (w @ w) + np.log(np.diag(ref)).sum() + 0.5 * n * np.log(2 * np.pi)) < 1e-11 * abs(llh)
