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


def test_arrays_in_several_pieces():
    """Sets whose arrays pass the staging buffer (2^23 doubles) in more than one piece, the last of them
    ragged: every value back in its place."""
    n = 2 ** 23 // 3 + 1001
    X, A, S = (np.arange(k * n, dtype=np.float64).reshape(n, -1) + 0.25 * k for k in (3, 3, 1))
    print(f"[records] arrays in pieces n={n}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=64)
    g.set_arrays(X, A[::-1], S[:, 0])
    a = g.arrays()
    assert np.array_equal(a["X"], X) and np.array_equal(a["alpha"], A[::-1]) and np.array_equal(a["sigma"], S[:, 0])
    assert not a["J"].any() and not a["velocity"].any()
    g.update_arrays(X=A, alpha=X)
    a = g.arrays()
    assert np.array_equal(a["X"], A) and np.array_equal(a["alpha"], X)
    n = 2 ** 23 // 9 + 77
    b = np.arange(37.0 * n).reshape(n, 37)
    g.set_bodies(b)
    a = g.arrays()
    assert np.array_equal(a["J"], b[:, :9]) and np.array_equal(a["velocity"], b[:, 15:18])
    g.close()


def test_one_array_takes_room_for_itself_alone():
    """The positions alone take no room for the other arrays on the device."""
    n = 1 << 20
    g = FMMCalculator(P=4, theta=0.5, ncrit=64)
    X, out = np.zeros((n, 3)), np.zeros((n, 3))
    X[:, 1] = np.arange(n)
    g.set_arrays(X, X, np.ones(n))

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert g.lib.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0  # of the runtime the library is linked to
        return a.value

    before = free()
    print("[records] one array", flush=True)
    none = ctypes.POINTER(ctypes.c_double)()
    _capi.check(g.lib.uvlm_get_bodies_soa(g._h, n, dp(out), none, none, none, none, none, none))
    assert np.array_equal(out, X)
    assert before - free() < 24 * n * 1.25 + (4 << 20)
    g.close()
