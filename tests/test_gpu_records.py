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
