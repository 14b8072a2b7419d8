"""The profiler counts each launch and each flop of a factorization once,
whichever launch solves a panel: the one that factors the diagonal tile (up to
128 blocks of 64 FP64 rows below it) or one of its own.
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


def expected(n, ts, bands):
    """(flops of diagonal tiles and panels, panel launches, update flops)"""
    rows = [min(ts, n - i) for i in range(0, n, ts)]
    blocks = -(-n // 64)
    factor = update = 0.0
    panels = 0
    for k, r in enumerate(rows):
        factor += r ** 3 / 3.0 + sum(rows[k + 1:]) * float(ts) ** 2
        update += sum(q * (q + 1.0) * ts + 2.0 * q * ts * sum(rows[j + 1:]) for j, q in enumerate(rows) if j > k)
        below = max(0, blocks - (k + 1) * ts // 64)
        fp64 = below if bands is None else min(below, bands[0] * ts // 64)
        panels += below > fp64 or (fp64 > 128)
    return factor, panels, update


@pytest.mark.parametrize("n,dts,bands", [(40, 64, None), (1000, 192, None), (8400, 64, None), (8256, 64, None), (10000, 960, None),
                                         (2000, 192, (1, 2)), (2000, 192, (3, 4))])
def test_flops_and_launches(ctx, n, dts, bands):
    r = np.random.default_rng(n)
    p = egs.Problem(ctx, 0, r.random(n), r.random(n), dts=dts)
    p.set_observations(r.standard_normal(n))
    if bands:
        p.set_precision(capi.PRECISION_MIXED, *bands)
        p.set_fallback(0, 0.0)
    p.profile(True)
    p.loglik([1.0, 0.03, 0.5])
    diagonal, panel = p.kernel_stats(capi.PROFILE_DIAGONAL), p.kernel_stats(capi.PROFILE_PANEL_TRSM)
    updates = [p.kernel_stats(q) for q in (capi.PROFILE_UPDATE, capi.PROFILE_UPDATE_F32, capi.PROFILE_UPDATE_16,
                                           capi.PROFILE_UPDATE_16_SELECT)]
    p.close()
    factor, panels, update = expected(n, dts, bands)
    assert diagonal["launches"] == -(-n // dts) and panel["launches"] == panels
    assert diagonal["flops"] + panel["flops"] == pytest.approx(factor, rel=1e-12)
    if bands is None:
        assert sum(u["flops"] for u in updates) == pytest.approx(update, rel=1e-12)
    assert (panel["flops"] > 0) == (panels > 0)
