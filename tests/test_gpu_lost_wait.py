"""A wait between workgroups that ends in vain: the call that meets the mark
returns an error, every kernel ends, and the factor is given up, so that the
next evaluation factors anew and succeeds with the values from before.  The
mark is set from the host; the waits themselves are met as ever.
"""
import ctypes

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


def mark(p):
    f = capi.lib().egs_test_mark_lost_wait
    f.argtypes, f.restype = [ctypes.c_void_p], ctypes.c_int
    assert f(p.handle) == 0


@pytest.mark.parametrize("call,mixed", [("predict", False), ("predict", True), ("solve_logdet_quad", False),
                                        ("solve_logdet_quad", True), ("trsm", False), ("loglik", False),
                                        ("loglik", True), ("generate_observations", False),
                                        ("generate_observations", True)])
def test_the_call_fails_and_the_next_evaluation_succeeds(ctx, call, mixed):
    n = 1150
    r = np.random.default_rng(n)
    p = egs.Problem(ctx, 0, r.random(n), r.random(n), dts=192)
    z, t = r.standard_normal(n), r.random((2, 40))
    p.set_observations(z)
    if mixed:
        p.set_precision(capi.PRECISION_MIXED, 1, 2)
    want = p.loglik(THETA)
    kriged = p.predict(THETA, t[0], t[1])[0]
    calls = {"predict": lambda: p.predict(THETA, t[0], t[1]), "solve_logdet_quad": p.solve_logdet_quad,
             "trsm": lambda: p.trsm(z)}
    mark(p)
    if call in calls:   # with the factor that is there
        with pytest.raises(egs.EGSError) as e:
            calls[call]()
        assert e.value.code == capi.ERR_HIP
        if call != "predict":
            with pytest.raises(egs.EGSError) as e:   # the factor is given up
                calls[call]()
            assert e.value.code == capi.ERR_STATE
    elif call == "loglik":   # factors anew, and the call after it has a sound factor again
        assert tuple(p.loglik(THETA)) == tuple(want)
    else:   # likewise
        assert np.all(np.isfinite(p.generate_observations(THETA, seed=1)))
        p.set_observations(z)
    assert np.array_equal(p.predict(THETA, t[0], t[1])[0], kriged)
    assert tuple(p.loglik(THETA)) == tuple(want)
    p.close()
