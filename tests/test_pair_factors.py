"""Coefficients of the FP64 pair factors (pair_kernel.hpp) against exact arithmetic on the CPU: the
interpolants of G, G' and G'' on [0, 3] and the far form from x = 3 on, evaluated in double as the
kernels do (Horner), for G(x) = (erf(s) - 2 s e^{-x} / sqrt(pi)) / s^3, x = s^2."""
import math
import os
import re
from decimal import Decimal, getcontext

import numpy as np
import pytest

SRC = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "uvlm_amd", "csrc",
                        "pair_kernel.hpp")).read()
EPS = 2.0 ** -52


def coeffs(name):
    body = re.search(name + r"\[\w+\] = \{(.*?)\};", SRC, re.S).group(1)
    return [float(v) for v in body.split(",")]


def series(x, der):
    """d^der G / dx^der from the power series, in 60 digits (all x used here)."""
    getcontext().prec = 60
    x = Decimal(x)
    pi = Decimal("3.14159265358979323846264338327950288419716939937510582097494459")
    tot, fact = Decimal(0), Decimal(1)
    for i in range(0, 260):
        fact *= i + 1  # (i + 1)!
        if i >= der:
            c = Decimal(2 * (i + 1)) / (Decimal(2 * i + 3) * fact)
            f = math.perm(i, der)
            tot += (-1) ** i * c * f * x ** (i - der)
    return 2 / pi.sqrt() * tot


def horner(c, t):
    r = c[-1]
    for v in c[-2::-1]:
        r = r * t + v
    return r


@pytest.mark.parametrize("name,der", [("c_g64", 0), ("c_gp64", 1), ("c_gpp64", 2)])
def test_near_interpolants(name, der):
    c = coeffs(name)
    for x in [1e-30] + list(np.linspace(0.05, 3.0, 60)):
        want = series(float(x), der)
        # the interpolation error is below 1e-17; Horner in double adds a few roundings of terms no
        # larger than 4 times the value
        assert abs(Decimal(horner(c, float(x) - 1.5)) - want) <= abs(want) * Decimal(8 * EPS)


def test_far_form():
    far, ex = coeffs("c_far64"), coeffs("c_exp64")
    wc = float(re.search(r"FAR64_WC = ([0-9.e-]+)", SRC).group(1))
    wmin = float(re.search(r"FAR64_WMIN = ([0-9.e-]+)", SRC).group(1))
    for x in list(np.linspace(3.0, 12.0, 19)) + [20.0, 30.0, 43.9]:
        x = float(x)
        k = round(-x * 1.4426950408889634)
        r = -x - k * math.log(2.0)
        e = math.ldexp(horner(ex, r), k)
        assert abs(e / math.exp(-x) - 1.0) <= 64 * EPS  # r itself carries the rounding of k ln 2 here
        w = 1.0 / math.sqrt(x)
        p = horner(far, max(w, wmin) - wc)
        two = 2.0 / math.sqrt(math.pi)
        g = 1.0 - e * (two * x * w + p)
        G = g * w ** 3
        Gp = w * w * (two * e - 1.5 * G)
        Gpp = w * w * (-2.5 * Gp - two * e)
        if x <= 30.0:  # the alternating series loses x digits to cancellation: 60 are carried
            for got, der in ((G, 0), (Gp, 1), (Gpp, 2)):
                want = float(series(x, der))
                assert abs(got - want) <= 32 * EPS * abs(want)
