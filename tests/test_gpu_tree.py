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


@pytest.mark.parametrize("n,m,ncrit", [(3000, 1, 1), (20000, 2, 1), (6000, 60, 4)])
def test_long_rows(orc, n, m, ncrit):
    """Few targets against many sources: rows past the sizes that are ranked by a wavefront (1,024
    entries) and sorted in LDS (16,384), through the getList entry point, and their transposes
    through the probe adjoint's lists (run only)."""
    from uvlm_amd import _capi
    import ctypes

    X, Y = points(n, 5, 1.0, 0), points(max(m, 2), 6, 1.0, 0)[:m]
    g, h = FMMCalculator(P=4, theta=1e-3, ncrit=ncrit), FMMCalculator(P=4, theta=1e-3, ncrit=ncrit)
    trees = []
    for c, Z in ((h, Y), (g, X)):
        c.set_bodies(make_bodies(Z, Z, np.ones(len(Z))))
        c.build()
        trees.append(c.cells())
    (ti, tr), (si, sr) = trees
    print(f"[tree] long rows {len(ti)} x {len(si)} cells", flush=True)

    def ip(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))

    def dp(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))

    a, b = ctypes.c_int64(), ctypes.c_int64()
    args = (0, 1e-3, len(ti), ip(ti), dp(tr), len(si), ip(si), dp(sr))
    _capi.check(g.lib.uvlm_get_list(*args, 0, 0, ctypes.byref(a), ctypes.byref(b), None, None))
    p2p, m2l = np.zeros((a.value, 2), dtype=np.int64), np.zeros((b.value, 2), dtype=np.int64)
    _capi.check(g.lib.uvlm_get_list(*args, a.value, b.value, ctypes.byref(a), ctypes.byref(b), ip(p2p), ip(m2l)))
    # the same walk on the host, with the device's test
    want_p, want_m, front = [], [], [(0, 0)]
    if ti[0, 0] == 0 and si[0, 0] == 0:
        want_p, front = [(0, 0)], []
    while front:
        nxt = []
        for t, s in front:
            if si[s, 0] == 0 or (tr[t, 3] >= sr[s, 3] and ti[t, 0] != 0):
                kids = [(ti[t, 2] + c, s) for c in range(ti[t, 0])]
            else:
                kids = [(t, si[s, 2] + c) for c in range(si[s, 0])]
            for x, y in kids:
                d = tr[x, :3] - sr[y, :3]
                if (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) * 1e-3 * 1e-3 < (tr[x, 3] + sr[y, 3]) ** 2:
                    (want_p if ti[x, 0] == 0 and si[y, 0] == 0 else nxt).append((x, y))
                else:
                    want_m.append((x, y))
        front = nxt
    assert np.array_equal(p2p, np.array(sorted(want_p)).reshape(-1, 2))
    assert np.array_equal(m2l, np.array(sorted(want_m)).reshape(-1, 2))
    assert np.bincount(p2p[:, 0]).max() > (1024 if n < 20000 else 16384)
    W_ = np.ones((len(Y), 3))
    ga, gx = g.probe_adjoint(Y + 0.01, W_)
    ga2, gx2 = g.probe_adjoint(Y + 0.01, W_)
    assert np.array_equal(ga, ga2) and np.array_equal(gx, gx2) and np.isfinite(ga).all()
    g.close()
    h.close()


@pytest.mark.parametrize("n,ncrit", [(1, 1), (2, 1), (9, 1), (9, 8), (70, 1), (600, 3), (600, 40)])
@pytest.mark.parametrize("capacity", [None, "1"])
def test_first_steps(orc, monkeypatch, n, ncrit, capacity):
    """Traversals that end within, at and after the steps that one workgroup takes, and with
    buffers that overflow in them."""
    if capacity:
        monkeypatch.setenv("UVLM_LIST_CAPACITY", capacity)
    print(f"[first] n={n} ncrit={ncrit} capacity={capacity}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=ncrit)
    for seed in (n, n + 1):
        check(g, orc, points(n, seed, 0.5, 0), ncrit)
    g.close()


def test_get_list_of_cells_that_share_children(orc):
    """A caller's tree may hand the same children to two cells: their pairs are listed twice."""
    from uvlm_amd import _capi
    import ctypes

    # root 0 with cells 1 and 2, both with the children 3 .. 5
    ints = np.array([[2, 6, 1, 0, 0], [3, 3, 3, 0, 1], [3, 3, 3, 3, 1], [0, 1, 0, 0, 2], [0, 1, 0, 1, 2], [0, 1, 0, 2, 2]],
                    dtype=np.int64)
    reals = np.array([[0, 0, 0, 1], [0.1, 0, 0, 0.5], [-0.1, 0, 0, 0.5], [0.2, 0, 0, 0.1], [0, 0.2, 0, 0.1],
                      [0, 0, 0.2, 0.1]])
    ip = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))  # noqa: E731
    dp = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))  # noqa: E731
    g = FMMCalculator(P=4, theta=0.5, ncrit=4)
    a, b = ctypes.c_int64(), ctypes.c_int64()
    p2p, m2l = np.zeros((200, 2), dtype=np.int64), np.zeros((200, 2), dtype=np.int64)
    print("[tree] shared children", flush=True)
    _capi.check(g.lib.uvlm_get_list(0, 0.5, 6, ip(ints), dp(reals), 6, ip(ints), dp(reals), 200, 200, ctypes.byref(a),
                                    ctypes.byref(b), ip(p2p), ip(m2l)))
    want, front = [[], []], [(0, 0)]
    while front:
        nxt = []
        for t, s in front:
            if ints[s, 0] == 0 or (reals[t, 3] >= reals[s, 3] and ints[t, 0] != 0):
                kids = [(ints[t, 2] + c, s) for c in range(ints[t, 0])]
            else:
                kids = [(t, ints[s, 2] + c) for c in range(ints[s, 0])]
            for x, y in kids:
                d2 = ((reals[x, :3] - reals[y, :3]) ** 2).sum()
                if d2 * 0.25 < (reals[x, 3] + reals[y, 3]) ** 2:
                    if ints[x, 0] == 0 and ints[y, 0] == 0:
                        want[0].append((x, y))
                    else:
                        nxt.append((x, y))
                else:
                    want[1].append((x, y))
        front = nxt
    assert len(set(want[0])) < len(want[0])
    assert np.array_equal(p2p[: a.value], np.array(sorted(want[0])))
    assert np.array_equal(m2l[: b.value], np.array(sorted(want[1])).reshape(-1, 2))


def test_a_refused_tree_leaves_the_last_one():
    """A build that is refused as too deep leaves the last tree and its lists in use."""
    X = points(900, 3, 1e-2, 1)
    g = FMMCalculator(P=4, theta=0.5, ncrit=8)
    g.set_bodies(make_bodies(X, X, np.full(900, 0.1)))
    g.build()
    g.calculate()
    want = g.arrays()
    g.update_arrays(X=np.repeat(want["X"][:1], 900, 0))
    print("[tree] refused rebuild", flush=True)
    with pytest.raises(UVLMError):
        g.build()
    g.update_arrays(X=want["X"])
    g.calculate()
    got = g.arrays()
    assert np.array_equal(got["X"], want["X"]) and np.isfinite(got["velocity"]).all()
    assert np.linalg.norm(got["velocity"] - want["velocity"]) < 1e-12 * np.linalg.norm(want["velocity"])
    g.close()
