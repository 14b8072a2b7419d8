"""The rounding of the tiled Cholesky, on the diagonal of L L^T - A (80-bit sums).

A has ones on its diagonal, and what is left of them stays in [1/4, 1] for this
field, so that a subtraction from it rounds by 0.29 ulp = 0.29 * 2^-53 rms.  With
products of 32 columns or more summed first, row i has at most i / 32 of them:
up to 0.29 sqrt(n / 64) = 1.6 * 2^-53 rms over all rows for n = 1,984, and about
2^-53 come with the rounding of L itself: 3 * 2^-53 in all.  One column after another
they would be 0.29 sqrt(n / 2), 5 * 2^-53 for n = 640 and more beyond.
"""
import numpy as np
import pytest

import exageostatcpp_amd as egs
from exageostatcpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = egs.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,dts", [(640, 640), (960, 960), (1152, 1152), (1984, 1984), (1500, 320), (1500, 64), (1900, 960)])
@pytest.mark.parametrize("batch", [False, True])
def test_rounding_of_the_diagonal(ctx, n, dts, batch):
    r = np.random.default_rng(n)
    root = int(np.ceil(np.sqrt(n)))
    cell = np.arange(n)
    x, y = ((c + 0.5 + r.uniform(-0.4, 0.4, n)) / root for c in (cell // root, cell % root))
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    p.set_observations(r.standard_normal(n))
    theta = [1.0, 0.1 * 25 / root, 0.5]
    if batch:
        capi.loglik_batch([p], [theta])
    else:
        p.loglik(theta)
    low = np.tril(p.get_matrix()).astype(np.longdouble)
    p.close()
    off = (low * low).sum(1) - 1
    assert float(np.sqrt((off * off).mean())) <= 3 * 2.0 ** -53
