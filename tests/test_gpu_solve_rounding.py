"""The rounding of the forward solve: L y - z in 80 bits, for a field z of unit
variance.

A row's products are summed by blocks of 64 columns and 16 blocks at a time, so
that the sum as a whole rounds n / 1024 times, by 0.29 * 2^-53 each (its size is
between 1/2 and 2), under 2^-53 rms for these n; its groups, which are smaller,
and the product with the inverse of the diagonal block bring about as much each:
4 * 2^-53 in all.  With every product added to the running sum it would be
0.29 sqrt(n / 8) * 2^-53, 4.1 for n = 1,600, on top of the last, and more beyond.
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


@pytest.mark.parametrize("n,dts", [(1600, 320), (2500, 64), (5700, 960), (9000, 384)])
def test_forward_residual(ctx, n, dts):
    r = np.random.default_rng(n)
    root = int(np.ceil(np.sqrt(n)))
    cell = np.arange(n)
    x, y = ((c + 0.5 + r.uniform(-0.4, 0.4, n)) / root for c in (cell // root, cell % root))
    p = egs.Problem(ctx, 0, x, y, dts=dts)
    z = p.generate_observations([1.0, 5.0 / root, 0.5], seed=1)
    low, s = p.get_matrix(), p.trsm(z).astype(np.longdouble)
    p.close()
    off = np.concatenate([np.tril(low[i:i + 250], i).astype(np.longdouble) @ s for i in range(0, n, 250)]) - z
    assert float(np.sqrt((off * off).mean())) <= 4 * 2.0 ** -53
