"""Body records in and out at the edges of the 64-body tiles and with padded records: every field back
where it was, the padding untouched."""
import ctypes

import numpy as np
import pytest

from uvlm_amd import FMMCalculator, _capi

pytestmark = pytest.mark.gpu


def dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("width", [37, 40])
def test_records_round_trip(n, width):
    rng = np.random.default_rng(n)
    b = rng.normal(size=(n, width))
    print(f"[records] n={n} width={width}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=64)
    _capi.check(g.lib.uvlm_set_bodies_aos(g._h, dp(b), n, 8 * width))
    out = np.full((n, width), 7.0)
    _capi.check(g.lib.uvlm_get_bodies_aos(g._h, dp(out), n, 8 * width))
    assert np.array_equal(out[:, :37], b[:, :37]) and (out[:, 37:] == 7.0).all()
    g.close()


@pytest.mark.parametrize("n", [1, 64, 65, 1000])
def test_arrays_round_trip(n):
    rng = np.random.default_rng(n + 1)
    X, A, S = rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.uniform(0.1, 0.2, n)
    print(f"[records] arrays n={n}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=64)
    g.set_bodies(rng.normal(size=(n + 9, 37)))  # fields of an earlier, larger set are cleared
    g.set_arrays(X, A, S)
    b = g.copyBodies2Host()
    assert np.array_equal(b[:, 9:12], X) and np.array_equal(b[:, 12:15], A) and np.array_equal(b[:, 33], S)
    assert not np.delete(b, [9, 10, 11, 12, 13, 14, 33], axis=1).any()
    g.build()
    g.calculate()
    b, a = g.copyBodies2Host(), g.arrays()
    for name, sl in (("J", slice(0, 9)), ("X", slice(9, 12)), ("alpha", slice(12, 15)), ("velocity", slice(15, 18)),
                     ("dadt", slice(18, 21)), ("sigma", 33), ("drdt", 34)):
        assert np.array_equal(a[name], b[:, sl]), name
    g.update_arrays(X=X[::-1])
    assert np.array_equal(g.arrays()["X"], X[::-1]) and np.array_equal(g.arrays()["alpha"], a["alpha"])
    g.close()
