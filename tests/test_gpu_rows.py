"""List rows of built trees through every way they are put in order, and what is summed over them, against
the oracle: rows ranked by a wavefront (up to 256 entries), through the bit map of the source cells
(more entries, up to 229,376 source cells), by the bitonic sort (more source cells), and rows of more
than 16,384 entries, which send the lists to the radix sort.  Built trees alone take the first three; a
caller's own trees (getList) always take the radix sort."""
import numpy as np
import pytest

from uvlm_amd import FMMCalculator, make_bodies
from uvlm_amd import workloads as W

pytestmark = pytest.mark.gpu

ROW_RANK, ROW_LONG, ROW_BITS, ROWS_SORTED = 256, 16384, 229376, 3 << 20


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def line(n, length, lone):
    """n bodies evenly along a line of the given length, whose leaves list a few neighbours each, and the
    lone ones beside it, whose larger leaves list a stretch of it or all of it."""
    t = (np.arange(n) + 0.5) / n - 0.5
    X = np.stack([length * t, np.full(n, 0.013), np.full(n, -0.017)], 1)
    return np.concatenate([X, np.reshape(lone, (-1, 3))])


SORTS = {
    # a line of 10,000 leaves beside two leaves half the box wide: rows of 10,000
    "bits": (line(10000, 0.1, [[0.9, 0.9, 0.9], [-0.9, -0.9, -0.9]]), 0.5),
    # the same with rows past LDS
    "long": (line(17000, 0.1, [[0.9, 0.9, 0.9], [-0.9, -0.9, -0.9]]), 0.5),
    # 2^17 leaves and about as many cells above them; the body beside the line lists a stretch of some
    # thousand, the two close together make the box wide enough for its leaf to be small
    "bitonic": (line(1 << 17, 2.0, [[0.21, 0.035, -0.017], [0.1, -0.6, 0.4], [0.101, -0.601, 0.401]]), 0.4),
    # every leaf lists every other: rows of 129 .. 256 and of 257 entries and more
    "rank": (line(200, 1.0, []), 1e-3),
    "bits_all": (line(1500, 1.0, []), 1e-3),
}


@pytest.mark.parametrize("way", SORTS)
def test_rows_of_built_trees(orc, way):
    """Bit for bit, on the first build (the sizes read back first) and on the second (rows counted ahead)."""
    X, theta = SORTS[way]
    n = len(X)
    A, S = np.ones((n, 3)), np.full(n, 0.1)
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=4, theta=theta, ncrit=1)
    ref.init(ref_b)
    want = [w[np.lexsort((w[:, 1], w[:, 0]))] for w in ref.pairs()]
    C = len(ref.cells()[0])
    longest = max(np.bincount(w[:, 0]).max() for w in want if len(w))
    total = sum(len(w) for w in want)
    print(f"[rows] {way}: {C} cells, {total} pairs, longest row {longest}", flush=True)
    assert total <= ROWS_SORTED
    assert {"bits": ROW_RANK < longest <= ROW_LONG and C <= ROW_BITS, "long": longest > ROW_LONG,
            "bitonic": ROW_RANK < longest <= ROW_LONG and C > ROW_BITS, "rank": 128 < longest <= ROW_RANK,
            "bits_all": ROW_RANK < longest <= ROW_LONG and C <= ROW_BITS}[way]
    g = FMMCalculator(P=4, theta=theta, ncrit=1)
    for _ in range(2):
        b = make_bodies(X, A, S)
        g.init(b)
        assert np.array_equal(b, ref_b)
        for got, w in zip(g.lists(), want):
            assert np.array_equal(got, w)
    g.close()


@pytest.mark.parametrize("n", [10000, 17000])
def test_probe_rows(orc, n):
    """Probes whose rows hold every leaf of the line, below and above 16,384: velocities on the first and
    the second call, the parity bar 1e-10."""
    X = line(n, 0.1, [[0.9, 0.9, 0.9], [-0.9, -0.9, -0.9]])
    rng = W.SplitMix64(n)
    A, S = rng.normal(3 * len(X)).reshape(-1, 3), np.full(len(X), 2e-5)
    pts = np.array([[0.7, 0.6, -0.8], [-0.6, 0.8, 0.5], [0.5, -0.7, 0.6]])
    ref = orc.Calculator(P=6, theta=0.5, ncrit=1)
    ref.init(orc.make_bodies(X, A, S))
    ref.calculate()
    want = orc.make_bodies(pts, np.zeros((3, 3)), np.ones(3))
    ref.sensor_data(want)
    assert np.bincount(ref.pairs(sensor=True)[0][:, 0]).max() >= n
    print(f"[rows] probes of {n}", flush=True)
    g = FMMCalculator(P=6, theta=0.5, ncrit=1)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    for _ in range(2):
        s = make_bodies(pts, np.zeros((3, 3)), np.ones(3))
        g.getSensorData(s)
        assert np.array_equal(s[:, 9:12], want[:, 9:12])
        assert rel(s[:, 15:18], want[:, 15:18]) < 1e-10
    g.close()


@pytest.mark.parametrize("n,m,ncrit", [(900, 90, 2), (1500, 700, 2), (20, 17000, 1)])
def test_transposed_rows(orc, n, m, ncrit):
    """The probe adjoint over transposed lists of up to 256 entries a row, of more, and of more than 16,384.
    With theta 1e-3 every pair is near, so the gradients are the direct sum's: the bar of the near-field
    adjoint, 1e-10."""
    rng = W.SplitMix64(n + m)
    X = rng.uniform(3 * n).reshape(n, 3) * 2.0 - 1.0
    A, S = rng.normal(3 * n).reshape(n, 3), np.full(n, 0.1)
    pts, w = rng.uniform(3 * m).reshape(m, 3) * 2.0 - 1.0, rng.normal(3 * m).reshape(m, 3)
    print(f"[rows] transposed n={n} m={m}", flush=True)
    g = FMMCalculator(P=4, theta=1e-3, ncrit=ncrit)
    g.set_arrays(X, A, S)
    g.build()
    a = g.arrays()
    wa, wx = orc.probe_adjoint(pts, w, a["X"], a["alpha"], a["sigma"])
    for _ in range(2):
        ga, gx = g.probe_adjoint(pts, w)
        assert rel(ga, wa) < 1e-10 and rel(gx, wx) < 1e-10
    g.close()
