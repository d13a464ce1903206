"""Octree and lists at the sizes where the build changes path: one body, leaves of one body, leaves
below and above the largest that is ranked in LDS (1,024 bodies), coincident bodies, a cluster whose
cells share many digits, rebuilds that need fewer and more digits than the last.  Bit for bit against
the oracle."""
import numpy as np
import pytest

from uvlm_amd import FMMCalculator, make_bodies
from uvlm_amd import workloads as W
from uvlm_amd.fmm import UVLMError

pytestmark = pytest.mark.gpu


def points(n, seed, tight, same):
    rng = W.SplitMix64(seed)
    X = rng.uniform(3 * n).reshape(n, 3) * 2.0 - 1.0
    X[: n // 2] = 0.3 + tight * X[: n // 2]
    X[n // 3: n // 3 + same] = X[n // 3]
    return X


def check(g, orc, X, ncrit):
    n = X.shape[0]
    A, S = np.arange(3.0 * n).reshape(n, 3), np.full(n, 0.1)
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=4, theta=0.5, ncrit=ncrit)
    ref.init(ref_b)
    b = make_bodies(X, A, S)
    g.init(b)
    assert np.array_equal(b, ref_b)  # the permutation, input order inside the leaves
    ints, reals = ref.cells()
    gi, gr = g.cells()
    assert np.array_equal(gi, ints) and np.array_equal(gr, reals)
    for got, want in zip(g.lists(), ref.pairs()):
        want = want[np.lexsort((want[:, 1], want[:, 0]))]
        assert np.array_equal(got, want)


@pytest.mark.parametrize("n,ncrit,tight,same", [
    (1, 1, 1.0, 0), (2, 1, 1.0, 0), (65, 1, 1e-3, 0), (700, 7, 1e-5, 7), (5000, 64, 1e-2, 64), (5000, 1024, 1e-2, 0),
    (5000, 1025, 1e-2, 0), (3000, 3000, 1.0, 500), (40000, 100, 1e-4, 90), (30000, 2, 1.0, 2)])
def test_tree_and_lists(orc, n, ncrit, tight, same):
    g = FMMCalculator(P=4, theta=0.5, ncrit=ncrit)
    print(f"[tree] n={n} ncrit={ncrit}", flush=True)
    check(g, orc, points(n, n, tight, same), ncrit)
    check(g, orc, points(n, n + 1, 1.0, 0), ncrit)          # the same handle, a shallower tree
    check(g, orc, points(n, n + 2, max(0.1 * tight, 1e-5), same), ncrit)  # and a deeper one (21 levels at most)
    g.close()


def test_too_deep_is_refused():
    g = FMMCalculator(P=4, theta=0.5, ncrit=8)
    X = points(500, 1, 1e-2, 9)
    g.set_bodies(make_bodies(X, X, np.ones(500)))
    with pytest.raises(UVLMError):
        g.build()
    X = points(500, 1, 1e-2, 8)
    g.set_bodies(make_bodies(X, X, np.ones(500)))
    g.build()
    g.close()
