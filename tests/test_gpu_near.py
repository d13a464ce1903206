"""Near-field kernels at the sizes where their units, splits and chunks change: leaves of 1 to a few
hundred bodies, lists far longer than the others' (a coarse leaf beside a dense cluster), probe trees
with a handful of leaves, separations across every branch of the pair factors.  Against the oracle,
with the tolerances of the parity tests (FP64 1e-10, mixed 1e-6 of the FP64 values)."""
import numpy as np
import pytest

from uvlm_amd import FMMCalculator, make_bodies
from uvlm_amd import workloads as W

pytestmark = pytest.mark.gpu


def cluster(n, seed, sigma):
    """Half the bodies in a cube of edge 0.02, the others over [-1, 1]^3: leaves of the sparse half
    list hundreds of the dense half's."""
    rng = W.SplitMix64(seed)
    X = rng.uniform(3 * n).reshape(n, 3) * 2.0 - 1.0
    X[: n // 2] = 0.3 + 0.01 * X[: n // 2]
    A = rng.normal(3 * n).reshape(n, 3)
    return X, A, np.full(n, sigma) * (0.5 + rng.uniform(n))


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,ncrit,sigma", [(3, 64, 0.5), (65, 1, 0.3), (130, 64, 1e-4), (1500, 7, 0.02),
                                           (4000, 33, 0.05), (6000, 64, 0.003), (9000, 200, 0.02), (2500, 600, 0.2)])
def test_particles(orc, n, ncrit, sigma):
    X, A, S = cluster(n, n, sigma)
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=6, theta=0.5, ncrit=ncrit)
    ref.init(ref_b)
    ref.calculate()
    want = ref.bodies(n)
    out = {}
    for precision in ("fp64", "mixed"):
        print(f"[near] n={n} ncrit={ncrit} {precision}", flush=True)
        g = FMMCalculator(P=6, theta=0.5, ncrit=ncrit, precision=precision)
        g.set_bodies(make_bodies(X, A, S))
        for _ in range(2):  # the second build starts from the sorted bodies
            g.build()
            g.calculate()
        out[precision] = g.copyBodies2Host()
        assert np.array_equal(out[precision][:, 9:12], want[:, 9:12])
        g.close()
    for sl in (slice(0, 9), slice(15, 18), slice(18, 21)):
        assert rel(out["fp64"][:, sl], want[:, sl]) < 1e-10
        # n = 130: bodies a few 1e-4 apart in leaves half a unit wide.  The mixed path's FP32 offsets
        # from the leaf centre (2^-25 of up to 0.9) are then 1e-5 of such a separation, so 1e-6 is
        # not its accuracy there; only the FP64 values are checked.
        if n != 130:
            assert rel(out["mixed"][:, sl], out["fp64"][:, sl]) < 1e-6


# (a single probe sits at its cell's centre, where the oracle's L2P, like the reference's, is NaN)
@pytest.mark.parametrize("m,ncrit", [(2, 64), (5, 64), (300, 64), (300, 200)])
def test_probes(orc, m, ncrit):
    X, A, S = cluster(8000, 3, 0.02)
    pts = X[:: 8000 // m][:m] + 0.003
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=6, theta=0.5, ncrit=ncrit)
    ref.init(ref_b)
    ref.calculate()
    sb = orc.make_bodies(pts, np.zeros((m, 3)), np.ones(m))
    ref.sensor_data(sb)
    print(f"[near] probes m={m} ncrit={ncrit}", flush=True)
    g = FMMCalculator(P=6, theta=0.5, ncrit=ncrit)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    s = make_bodies(pts, np.zeros((m, 3)), np.ones(m))
    g.getSensorData(s)
    assert np.array_equal(s[:, 9:12], sb[:, 9:12])
    assert rel(s[:, 15:18], sb[:, 15:18]) < 1e-10
    g.close()


@pytest.mark.parametrize("m,n", [(1, 1), (1, 1025), (3, 700), (511, 1), (513, 2049), (1100, 1024), (16384, 333)])
def test_direct(orc, m, n):
    X, A, S = cluster(max(n, 2), 5, 0.05)
    X, A, S = X[:n], A[:n], S[:n]
    rng = W.SplitMix64(m)
    xt = 1.5 * (rng.uniform(3 * m).reshape(m, 3) * 2.0 - 1.0)
    xt[: min(m, n) // 2] = X[: min(m, n) // 2]  # coincident with sources: skipped pairs
    at = rng.normal(3 * m).reshape(m, 3)
    print(f"[near] direct m={m} n={n}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=64)
    g.set_arrays(X, A, S)
    u, J, D = g.direct(xt, at)
    u2, _, _ = g.direct(xt, want_J=False)
    wu, wJ = orc.direct(xt, X, A, S)
    wD = np.einsum("iab,ib->ia", wJ.reshape(m, 3, 3), at)
    assert rel(u, wu) < 1e-12 and rel(u2, wu) < 1e-12
    assert rel(J, wJ.reshape(m, 9)) < 1e-11 and rel(D, wD) < 1e-11
    g.close()


@pytest.mark.parametrize("n,ncrit", [(3, 64), (65, 1), (1500, 7), (4000, 33), (9000, 200)])
def test_gaussian_sums(orc, n, ncrit):
    """PSE rates and probe vorticity over the same lists; two coincident bodies among them (that
    pair is skipped by PSE and counted by the vorticity)."""
    X, A, S = cluster(n, n + 1, 0.05)
    if ncrit > 1:
        X[-1] = X[0]
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=4, theta=0.5, ncrit=ncrit)
    ref.init(ref_b)
    ref.calculate()
    ref.set_viscosity("pse", 0.3)
    ref.viscosity(0.01)
    want = ref.bodies(n)
    m = min(n, 37)
    sb = orc.make_bodies(X[:m] + 0.002, np.zeros((m, 3)), np.ones(m))
    ref.vorticity(sb)
    print(f"[near] gauss n={n} ncrit={ncrit}", flush=True)
    g = FMMCalculator(P=4, theta=0.5, ncrit=ncrit)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    g.set_viscosity("pse", 0.3)
    g.viscosity(0.01)
    out = g.copyBodies2Host()
    assert rel(out[:, 18:21], want[:, 18:21]) < 1e-10
    s = make_bodies(X[:m] + 0.002, np.zeros((m, 3)), np.ones(m))
    g.vorticity(s)
    assert np.array_equal(s[:, 9:12], sb[:, 9:12])
    assert rel(s[:, 21:24], sb[:, 21:24]) < 1e-10
    g.close()


@pytest.mark.parametrize("m,ncrit,theta", [(2, 2, 0.05), (40, 2, 0.05), (300, 8, 0.2)])
def test_probes_with_long_rows(orc, m, ncrit, theta):
    """Probe lists of thousands of sources a row: rows sorted by a workgroup, M2L lists in segments."""
    X, A, S = cluster(6000, 5, 0.02)
    pts = X[:: 6000 // m][:m] + 0.003
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=6, theta=theta, ncrit=ncrit)
    ref.init(ref_b)
    ref.calculate()
    sb = orc.make_bodies(pts, np.zeros((m, 3)), np.ones(m))
    ref.sensor_data(sb)
    print(f"[near] long rows m={m} ncrit={ncrit}", flush=True)
    g = FMMCalculator(P=6, theta=theta, ncrit=ncrit)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    for _ in range(2):  # the second pass counts the rows ahead
        s = make_bodies(pts, np.zeros((m, 3)), np.ones(m))
        g.getSensorData(s)
        assert np.array_equal(s[:, 9:12], sb[:, 9:12])
        assert rel(s[:, 15:18], sb[:, 15:18]) < 1e-10
    g.close()


@pytest.mark.parametrize("n,m,ncrit", [(40, 5, 64), (900, 37, 7)])
def test_nan_coordinates_show_in_the_vorticity(n, m, ncrit):
    """exp(NaN) is NaN: a body with a NaN coordinate shows at every probe whose list holds its leaf (with
    theta 1e-3 all of them), a NaN probe at itself alone."""
    X, A, S = cluster(n, n, 0.3)
    pts = X[:m] + 0.01

    def vorticity(X, pts):
        g = FMMCalculator(P=4, theta=1e-3, ncrit=ncrit)
        g.set_bodies(make_bodies(X, A, S))
        g.build()
        s = make_bodies(pts, np.arange(3.0 * m).reshape(m, 3), np.ones(m))
        g.vorticity(s)
        g.close()
        return s[np.argsort(s[:, 12])][:, 21:24]  # in the probes' order

    print(f"[near] NaN n={n} m={m}", flush=True)
    want = vorticity(X, pts)
    assert np.isfinite(want).all()
    bad = X.copy()
    bad[n // 2, 1] = np.nan
    assert np.isnan(vorticity(bad, pts)).all()
    badp = pts.copy()
    badp[m // 2, 0] = np.nan
    got = vorticity(X, badp)
    assert np.isnan(got[m // 2]).all() and np.isfinite(np.delete(got, m // 2, 0)).all()


@pytest.mark.parametrize("sigma", [1e-30, 1e-40, 1e-62, 1e-104, 1e-120, 1e-150])
def test_tiny_cores(orc, sigma):
    """FP64 with cores so small that powers of 1 / sigma leave the range of a double: the singular
    kernel, as the reference's formula gives it (f1 and f2 there have R alone in them).  Same bars as
    for ordinary cores."""
    n, m = 200, 40
    X, A, _ = cluster(n, 11, 1.0)
    S = np.full(n, sigma)
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=6, theta=0.5, ncrit=64)
    ref.init(ref_b)
    ref.calculate()
    want = ref.bodies(n)
    print(f"[near] sigma={sigma}", flush=True)
    g = FMMCalculator(P=6, theta=0.5, ncrit=64)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    got = g.copyBodies2Host()
    for sl in (slice(0, 9), slice(15, 18), slice(18, 21)):
        assert rel(got[:, sl], want[:, sl]) < 1e-10
    xt = np.concatenate([X[:m], X[:m] + 0.01])
    at = A[: 2 * m]
    u, J, D = g.direct(xt, at)
    wu, wJ = orc.direct(xt, X, A, S)
    assert rel(u, wu) < 1e-12 and rel(J, wJ.reshape(-1, 9)) < 1e-11
    s, w = make_bodies(X[:m] + 0.01, A[:m], np.ones(m)), orc.make_bodies(X[:m] + 0.01, A[:m], np.ones(m))
    g.vorticity(s)
    ref.vorticity(w)
    assert np.array_equal(s[:, 21:24], w[:, 21:24])  # e^{-R^2 / 2 sigma^2} = 0
    g.close()
    # both sides of the adjoint's near pairs, one leaf
    g = FMMCalculator(P=6, theta=0.5, ncrit=1024)
    g.set_arrays(X, A, S)
    g.build()
    ub, ab = A[::-1].copy(), X[::-1].copy()
    xb, alb = g.eval_vjp(ub, ab)
    arr = g.arrays()
    exb, ealb = orc.direct_vjp(arr["X"], arr["alpha"], arr["sigma"], ub, ab, "transposed")
    assert rel(xb, exb) < 1e-10 and rel(alb, ealb) < 1e-10
    g.close()


def test_bodies_without_a_core(orc):
    """sigma = 0 or NaN leaves a body without a near kernel; it still skips itself.  Two such bodies in
    leaves apart see each other through the far field alone and stay finite, in the rates, the direct
    sum and both sides of the adjoint; any other near pair is neither finite."""
    X = np.array([[0.0, 0.0, 0.0], [1.0, 1.1, 0.9]])
    A = np.array([[1.0, -0.5, 0.3], [0.2, 0.7, -0.4]])
    for S in (np.zeros(2), np.array([0.1, np.nan])):
        ref_b = orc.make_bodies(X, A, S)
        ref = orc.Calculator(P=4, theta=0.9, ncrit=1)
        ref.init(ref_b)
        ref.calculate()
        want = ref.bodies(2)
        print(f"[near] sigma={S}", flush=True)
        g = FMMCalculator(P=4, theta=0.9, ncrit=1)
        g.set_bodies(make_bodies(X, A, S))
        g.build()
        assert g.timings()["n_m2l_pairs"] > 0
        g.calculate()
        got = g.copyBodies2Host()
        assert np.isfinite(want[:, :9]).all() and np.isfinite(want[:, 15:21]).all()
        for sl in (slice(0, 9), slice(15, 18), slice(18, 21)):
            assert rel(got[:, sl], want[:, sl]) < 1e-10
        xb, ab = g.eval_vjp(A, X)
        assert np.isfinite(xb).all() and np.isfinite(ab).all()
        g.set_bodies(make_bodies(X[1:], A[1:], S[1:]))
        u, J, _ = g.direct(np.concatenate([X[1:], X[:1]]))
        assert np.all(u[0] == 0) and np.all(J[0] == 0) and not np.isfinite(u[1]).any() and not np.isfinite(J[1]).any()
        g.close()


@pytest.mark.parametrize("rows", ["0", "40", "3000"])
def test_units_without_room_for_their_partial_sums(monkeypatch, rows):
    """Lists cut again with fewer rows of partial sums, down to one unit a leaf: the same pairs in another
    order, so 1e-12 bounds the rounding of the FP64 sums with two orders to spare."""
    n, m = 6000, 300
    X, A, S = cluster(n, 8, 0.05)
    pts, w = X[:: n // m][:m] + 0.003, A[:m]

    def values():
        g = FMMCalculator(P=4, theta=0.5, ncrit=64)
        g.set_bodies(make_bodies(X, A, S))
        out = []
        for _ in range(2):  # the second build makes its units ahead
            g.build()
            g.calculate()
        g.set_viscosity("pse", 0.3)
        g.viscosity(0.01)
        out += [g.copyBodies2Host()[:, k] for k in (slice(0, 9), slice(15, 18), slice(18, 21))]
        s = make_bodies(pts, w, np.ones(m))
        g.getSensorData(s)
        out.append(s[:, 15:18])
        s = make_bodies(pts, w, np.ones(m))
        g.vorticity(s)
        out.append(s[:, 21:24])
        g.set_viscosity("inviscid", 0.0)
        out += list(g.probe_adjoint(pts, w)) + list(g.eval_vjp(A, X))
        g.close()
        return out

    want = values()
    monkeypatch.setenv("UVLM_NEAR_ROWS", rows)
    print(f"[near] rows {rows}", flush=True)
    for got, ref in zip(values(), want):
        assert rel(got, ref) < 1e-12


def groups(k, size, seed):
    """k groups of `size` bodies in different octants: k leaves at ncrit = size, lists of k entries."""
    rng = W.SplitMix64(seed)
    c = np.array([[-1.0 if i >> d & 1 else 1.0 for d in range(3)] for i in (0, 7, 1, 6, 2, 5, 3)[:k]])
    X = np.repeat(c, size, 0) * 0.5 + 0.2 * (rng.uniform(3 * k * size).reshape(-1, 3) - 0.5)
    return X, rng.normal(3 * k * size).reshape(-1, 3), np.full(k * size, 0.1) * (0.5 + rng.uniform(k * size))


def pair_factors(r2, sigma):
    """f1, f2 = 2 df1/dR^2 and f3 = 2 df2/dR^2: the power series of G below x = 2, where the closed form
    loses x^-3 of its digits to cancellation, and that form above."""
    from scipy.special import erf

    q = 0.5 / (sigma * sigma)
    x = r2 * q
    G = np.zeros((3,) + x.shape)
    near = x < 2.0
    k, c, power = 2.0 / np.sqrt(np.pi), 1.0, [np.zeros(near.sum()), np.zeros(near.sum()), np.ones(near.sum())]
    for i in range(50):  # sum (-1)^i 2 / ((2 i + 3) i!) x^i and its derivatives
        c = -c / i if i else 1.0  # (-1)^i / i!
        a = k * c * 2.0 / (2 * i + 3)
        for d, f in enumerate((1, i, i * (i - 1))):
            G[d][near] += a * f * power[2 - d]
        power = [power[1], power[2], power[2] * x[near]]
    xf = x[~near]
    e = k * np.exp(-xf)
    G[0][~near] = (erf(np.sqrt(xf)) - e * np.sqrt(xf)) * xf ** -1.5
    G[1][~near] = (e - 1.5 * G[0][~near]) / xf
    G[2][~near] = (-e - 2.5 * G[1][~near]) / xf
    c1 = q * np.sqrt(q) / (4.0 * np.pi)
    return [np.where(r2 == 0.0, 0.0, f)[..., None] for f in (G[0] * c1, 2 * G[1] * q * c1, 4 * G[2] * q * q * c1)]


def direct_vjp(X, A, S, ub, ab):
    """xbar and alphabar of sum ub.u + ab.(J^T alpha) over all pairs, in plain numpy: with r = x_i - x_j and
    Jbar_i = alpha_i (x) ab_i, e its axial vector, pair ij adds -alpha_j . (f1 (ub_i x r + e_i) + f2 (Jbar_i
    r) x r) to it."""
    n = len(X)
    xb, alb = np.zeros((n, 3)), np.zeros((n, 3))
    Jb = A[:, :, None] * ab[:, None, :]
    e = np.stack([Jb[:, 1, 2] - Jb[:, 2, 1], Jb[:, 2, 0] - Jb[:, 0, 2], Jb[:, 0, 1] - Jb[:, 1, 0]], 1)
    for c in range(0, n, 200):
        i = slice(c, c + 200)
        r = X[i, None] - X[None]
        f1, f2, f3 = pair_factors((r * r).sum(-1), np.broadcast_to(S, r.shape[:2]))
        Jr, rxa = np.einsum("iab,ijb->ija", Jb[i], r), np.cross(r, A[None])
        w, v = np.cross(ub[i, None], r) + e[i, None], np.cross(Jr, r)
        c1, c3 = (A * w).sum(-1, keepdims=True), (A * v).sum(-1, keepdims=True)
        dS = -((f2 * c1 + f3 * c3) * r + f1 * np.cross(A[None], ub[i, None]) +
               f2 * (np.einsum("iba,ijb->ija", Jb[i], rxa) + np.cross(A[None], Jr)))
        xb[i] += dS.sum(1)
        xb -= dS.sum(0)
        alb -= (f1 * w + f2 * v).sum(0)
        J, F = -np.einsum("ija,ijb->iab", f2 * rxa, r), (f1 * A).sum(1)
        for a, b, k, sign in ((0, 1, 2, 1), (1, 2, 0, 1), (2, 0, 1, 1), (1, 0, 2, -1), (2, 1, 0, -1), (0, 2, 1, -1)):
            J[:, a, b] -= sign * F[:, k]
        alb[i] += np.einsum("iab,ib->ia", J, ab[i])
    return xb, alb


@pytest.mark.parametrize("kind,n,ncrit", [("groups", 4, 40), ("groups", 7, 64), ("groups", 6, 1), ("cluster", 900, 7),
                                          ("cluster", 3000, 20), ("cluster", 3000, 100), ("cluster", 2000, 600)])
@pytest.mark.parametrize("lanes", ["64", "256"])
def test_adjoint_pairs(monkeypatch, lanes, kind, n, ncrit):
    """Both sides of the adjoint's near pairs over many leaves, with lists of a few entries (the groups) and
    of hundreds, cut into units, by workgroups of either width (256 alone above 64 bodies a leaf).  With theta 1e-3 every pair is near, so the
    direct sum's VJP is the answer: 1e-10, mixed 1e-5, the bars of the one-leaf case.  (The oracle's
    direct VJP is itself off by 1.3e-10 in the dense half of the 900: its factors cancel there.)"""
    monkeypatch.setenv("UVLM_NEAR_LANES", lanes)
    X, A, S = groups(n, ncrit, n) if kind == "groups" else cluster(n, n, 0.1)
    rng = W.SplitMix64(n + ncrit)
    ub, ab = (rng.normal(3 * len(X)).reshape(-1, 3) for _ in range(2))
    for precision, bar in (("fp64", 1e-10), ("mixed", 1e-5)):
        print(f"[near] adjoint {kind} n={n} ncrit={ncrit} {precision}", flush=True)
        g = FMMCalculator(P=4, theta=1e-3, ncrit=ncrit, precision=precision)
        g.set_arrays(X, A, S)
        g.build()
        t = g.timings()
        assert t["n_m2l_pairs"] == 0 and t["n_leaves"] > 1
        xb, alb = g.eval_vjp(ub, ab)
        arr = g.arrays()
        exb, ealb = direct_vjp(arr["X"], arr["alpha"], arr["sigma"], ub, ab)
        assert rel(xb, exb) < bar and rel(alb, ealb) < bar
        g.close()


def tube(n):
    """n bodies along a helix: leaves of a few bodies with short lists."""
    t = np.arange(n) / n
    rng = W.SplitMix64(n)
    X = np.stack([np.cos(6 * t) + 0.004 * np.cos(5000 * t), np.sin(6 * t) + 0.004 * np.sin(5000 * t), t], 1)
    return X, rng.normal(3 * n).reshape(-1, 3), np.full(n, 1e-3)


@pytest.mark.parametrize("lanes", ["64", "256", None])
@pytest.mark.parametrize("kind,n,ncrit", [("groups", 2, 1), ("groups", 4, 40), ("groups", 7, 64), ("tube", 9000, 8),
                                          ("cluster", 4000, 33)])
def test_lanes_of_a_unit(orc, monkeypatch, lanes, kind, n, ncrit):
    """The near field, the Gaussian sums and the probes with workgroups of 64 and of 256 lanes, and with
    those the lists choose (64 for the tube), on lists of 2 to hundreds of entries."""
    if lanes:
        monkeypatch.setenv("UVLM_NEAR_LANES", lanes)
    X, A, S = groups(n, ncrit, n + ncrit) if kind == "groups" else tube(n) if kind == "tube" else cluster(n, n, 0.02)
    n, theta = len(X), 1e-3 if kind == "groups" else 0.5
    pts = X[:: max(1, n // 200)] + 0.003
    m = len(pts)
    ref = orc.Calculator(P=4, theta=theta, ncrit=ncrit)
    ref.init(orc.make_bodies(X, A, S))
    ref.calculate()
    want = ref.bodies(n)
    ref.set_viscosity("pse", 0.3)
    ref.viscosity(0.01)
    pse = ref.bodies(n)
    sb = orc.make_bodies(pts, np.zeros((m, 3)), np.ones(m))
    sv = sb.copy()
    ref.sensor_data(sb)
    ref.vorticity(sv)
    print(f"[near] lanes {lanes} {kind} n={n}", flush=True)
    g = FMMCalculator(P=4, theta=theta, ncrit=ncrit)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    got = g.copyBodies2Host()
    for sl in (slice(0, 9), slice(15, 18), slice(18, 21)):
        assert rel(got[:, sl], want[:, sl]) < 1e-10
    g.set_viscosity("pse", 0.3)
    g.viscosity(0.01)
    assert rel(g.copyBodies2Host()[:, 18:21], pse[:, 18:21]) < 1e-10
    s = make_bodies(pts, np.zeros((m, 3)), np.ones(m))
    v = s.copy()
    g.getSensorData(s)
    g.vorticity(v)
    assert rel(s[:, 15:18], sb[:, 15:18]) < 1e-10 and rel(v[:, 21:24], sv[:, 21:24]) < 1e-10
    g.close()
    # mixed: FP32 pair arithmetic, the bar of test_particles
    g = FMMCalculator(P=4, theta=theta, ncrit=ncrit, precision="mixed")
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    mixed = g.copyBodies2Host()
    for sl in (slice(0, 9), slice(15, 18), slice(18, 21)):
        assert rel(mixed[:, sl], want[:, sl]) < 1e-6
    g.close()
