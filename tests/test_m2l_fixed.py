"""The M2L kernel with its plan compiled in (k_m2l_fixed) against the one that reads the plan
(k_m2l_ns), at every order that has one: particles (lattice table), probes (harmonics computed, lists
cut into segments), lists of 1 to a few hundred sources."""
import os
import subprocess

import numpy as np
import pytest

from uvlm_amd import FMMCalculator, make_bodies
from uvlm_amd import workloads as W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fixed_plans_are_the_default_plans(tmp_path):
    exe = str(tmp_path / "m2l_fixed_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "cpp", "m2l_fixed_check.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "6 orders, all match" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("P", [4, 6, 8, 10, 12, 14])
@pytest.mark.parametrize("n,ncrit,theta", [(9, 1, 0.5), (700, 3, 0.3), (6000, 40, 0.5)])
def test_fixed_against_general(monkeypatch, P, n, ncrit, theta):
    """The two differ by the order of the sums alone: some thousand terms an output, 1e-12 of the
    largest result bounds their FP64 rounding with two orders to spare."""
    rng = W.SplitMix64(n + P)
    X = rng.uniform(3 * n).reshape(n, 3) * 2.0 - 1.0
    X[: n // 2] = 0.3 + 0.05 * X[: n // 2]
    A, S = rng.normal(3 * n).reshape(n, 3), np.full(n, 0.01)
    T = np.ascontiguousarray(X[:: max(1, n // 50)] + 0.01)
    out = []
    for slots in (None, "12"):
        if slots:
            monkeypatch.setenv("UVLM_M2L_SLOTS", slots)
        print(f"[m2l] P={P} n={n} ncrit={ncrit} slots={slots}", flush=True)
        g = FMMCalculator(P=P, theta=theta, ncrit=ncrit, precision="fp64")
        g.set_bodies(make_bodies(X, A, S))
        g.build()
        g.calculate()
        t = g.timings()
        s = make_bodies(T, np.zeros_like(T), np.ones(len(T)))
        g.getSensorData(s)
        out.append((t["m2l_slots"], t["n_m2l_pairs"], g.copyBodies2Host()[:, 15:21].copy(), s[:, 15:21].copy()))
        g.close()
    assert out[0][0] in (5, 6, 8) and out[1][0] == 12 and out[0][1] == out[1][1] > 0
    for a, c in zip(out[0][2:], out[1][2:]):
        assert np.isfinite(a).all() and np.abs(a - c).max() <= 1e-12 * np.abs(c).max()


@pytest.mark.gpu
@pytest.mark.parametrize("P", [4, 14])
@pytest.mark.parametrize("n,ncrit", [(40, 1), (900, 70)])
def test_unrolled_orders_against_the_oracle(orc, P, n, ncrit):
    """P2M and L2P with these orders as constants: the parity bar of the other orders, 1e-10."""
    rng = W.SplitMix64(n)
    X = rng.uniform(3 * n).reshape(n, 3) * 2.0 - 1.0
    A, S = rng.normal(3 * n).reshape(n, 3), np.full(n, 0.05)
    ref_b = orc.make_bodies(X, A, S)
    ref = orc.Calculator(P=P, theta=0.4, ncrit=ncrit)
    ref.init(ref_b)
    ref.calculate()
    want = ref.bodies(n)
    print(f"[orders] P={P} n={n}", flush=True)
    g = FMMCalculator(P=P, theta=0.4, ncrit=ncrit)
    g.set_bodies(make_bodies(X, A, S))
    g.build()
    g.calculate()
    got = g.copyBodies2Host()
    assert np.array_equal(got[:, 9:12], want[:, 9:12])
    for sl in (slice(0, 9), slice(15, 21)):
        ok = np.isfinite(want[:, sl])  # a body at its leaf's centre: the reference's L2P is NaN there
        assert np.linalg.norm((got[:, sl] - want[:, sl])[ok]) < 1e-10 * np.linalg.norm(want[:, sl][ok])
    g.close()
