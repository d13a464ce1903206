"""What the framework is timed on: calls a user's program makes, through the public entry points.

A case is one call, or the short run of calls that always go together (upload, build, evaluate,
download), on the particle sets of `uvlm_amd.workloads`: the ring, the random cube, the leapfrogging
rings, the Gaussian blobs with probes, and the 40 x 10 panel wing with its wake.  `kind` names the
call, `set` the particle set, `n` its size; the other entries are the constructor's arguments.

Every pass starts from the same particles, so a pass is the same work each time.  Results of the FP64
path are returned as the library gives them.  The mixed path sums pairs in FP32; its fields are
handed on as a viewer or a statistics pass takes them, in float32.
"""
import math

import numpy as np
import torch

from uvlm_amd import workloads
from uvlm_amd.fmm import BODY_DOUBLES, FMMCalculator, make_bodies
from uvlm_amd.vlm import Wing, design_wing

U_WING = np.array([0.0, 1.0, 0.0])


def listed():
    return [
        # the smallest use: a few hundred particles handed over, stepped and handed back, at the
        # constructor's defaults (P 4, theta 0.3, ncrit 128, FP64).  Latency and launches.
        dict(name="advance_600", kind="advance", set="blobs", n=600, P=4, theta=0.3, ncrit=128, precision="fp64",
             stretching="transposed", dt=0.001),
        # the reference driver's call on the single ring of the benchmark
        dict(name="advance_ring_8k", kind="advance", set="ring", n=8192, P=8, theta=0.5, ncrit=64, precision="fp64",
             stretching="transposed", dt=0.005),
        # one pass of the wing loop: VLM solve against the wake, shedding, wake step
        dict(name="wing_wake_20k", kind="wing", set="wake", n=20000, P=8, theta=0.5, ncrit=64, precision="mixed",
             dt=0.02),
        # a viscous step's rates: classic stretching, reformulated VPM, particle strength exchange
        dict(name="viscous_100k", kind="viscous", set="leapfrog", n=100002, P=6, theta=0.5, ncrit=100,
             precision="fp64", stretching="classic", formulation="rvpm", nu=0.01, dt=0.005),
        # probe velocities from an evaluated particle set
        dict(name="sensors_4k", kind="sensors", set="blobs", n=200003, m=4096, P=8, theta=0.5, ncrit=64,
             precision="fp64"),
        # the direct sum that accuracy checks use: sampled targets against every particle
        dict(name="direct_4k", kind="direct", set="cube", n=200003, m=4096, P=4, theta=0.5, ncrit=64,
             precision="fp64"),
        # the accuracy-qualified setting: high order, small theta, regularised near field
        dict(name="accurate_60k", kind="eval", set="cube", n=60001, P=14, theta=0.3, ncrit=64, precision="mixed",
             stretching="transposed", near=6.0),
        # the random cube of the benchmark
        dict(name="eval_cube_1m", kind="eval", set="cube", n=1 << 20, P=10, theta=0.4, ncrit=64, precision="mixed",
             stretching="transposed", near=0.0),
        # the default precision at scale
        dict(name="eval_rings_1m_fp64", kind="eval", set="leapfrog", n=1 << 20, P=10, theta=0.5, ncrit=96,
             precision="fp64", stretching="transposed", near=0.0),
        # the headline workload at its tuned leaf size
        dict(name="eval_rings_4m", kind="eval", set="leapfrog", n=1 << 22, P=10, theta=0.5, ncrit=192,
             precision="mixed", stretching="transposed", near=0.0),
        # gradient of a probe objective with respect to every particle
        dict(name="probe_adjoint_1m", kind="probe_adjoint", set="blobs", n=1 << 20, m=4096, P=8, theta=0.5, ncrit=64,
             precision="mixed"),
        # vector-Jacobian product of one evaluation, the building block of every step adjoint
        dict(name="eval_vjp_260k", kind="eval_vjp", set="blobs", n=260003, P=8, theta=0.5, ncrit=64,
             precision="mixed", stretching="transposed"),
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm, odd as often as even."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["advance", "advance", "eval", "eval", "eval", "viscous", "sensors", "direct", "probe_adjoint",
                       "eval_vjp", "wing"])
    P = rng.choice([4, 6, 8, 8, 10, 10, 12])
    ncrit = rng.choice([48, 64, 64, 96, 128, 192, 200])
    theta = rng.choice([0.4, 0.5, 0.5])
    precision = rng.choice(["fp64", "mixed"])
    stretching = rng.choice(["transposed", "transposed", "classic"])
    some = rng.choice(["ring", "cube", "leapfrog", "blobs"])
    if kind == "advance":
        return dict(kind=kind, set=some, n=_size(rng, 300, 60000), P=P, theta=theta, ncrit=ncrit, precision="fp64",
                    stretching=stretching, dt=round(rng.uniform(0.0005, 0.005), 5))
    if kind == "eval":
        if rng.random() < 0.25:
            return dict(kind=kind, set="cube", n=_size(rng, 8000, 80000), P=rng.choice([10, 12, 14]), theta=0.3,
                        ncrit=rng.choice([64, 128]), precision=precision, stretching="transposed",
                        near=rng.choice([5.0, 6.0]))
        return dict(kind=kind, set=some, n=_size(rng, 10000, 1000000), P=P, theta=theta, ncrit=ncrit,
                    precision=precision, stretching=stretching, near=0.0)
    if kind == "viscous":
        return dict(kind=kind, set=rng.choice(["ring", "leapfrog", "blobs"]), n=_size(rng, 10000, 150000), P=P,
                    theta=theta, ncrit=ncrit, precision=precision, stretching=stretching,
                    formulation=rng.choice(["cvpm", "rvpm"]), nu=0.01, dt=0.005)
    if kind == "direct":
        return dict(kind=kind, set="cube", n=_size(rng, 2000, 150000), m=_size(rng, 64, 5000), P=4, theta=theta,
                    ncrit=ncrit, precision="fp64")
    if kind in ("sensors", "probe_adjoint"):
        return dict(kind=kind, set="blobs", n=_size(rng, 10000, 300000), m=_size(rng, 64, 8192), P=P, theta=theta,
                    ncrit=ncrit, precision=precision)
    if kind == "eval_vjp":
        return dict(kind=kind, set=some, n=_size(rng, 5000, 300000), P=P, theta=theta, ncrit=ncrit,
                    precision=precision, stretching=stretching)
    return dict(kind="wing", set="wake", n=40 * _size(rng, 25, 1500), P=rng.choice([6, 8]), theta=0.5,
                ncrit=rng.choice([64, 96]), precision=precision, dt=rng.choice([0.01, 0.02]))


def _wake(n, dt, rng):
    """A wake of n particles behind the 40-panel trailing edge: rows of one time step's spacing,
    drifting and rolling up as they age, with the bound circulation's spanwise gradient."""
    rows = -(-n // 40)
    r, k = np.divmod(np.arange(rows * 40), 40)
    x = (k + 0.5) * 0.15
    age = (r + 1) * dt
    s = 2.0 * x / 6.0 - 1.0
    X = np.stack([x - 0.05 * s * age + 0.01 * rng.normal(x.size), 1.0 + age + 0.002 * rng.normal(x.size),
                  -0.09 - 0.1 * (1.0 - s * s) * age + 0.02 * rng.normal(x.size)], 1)
    g = 0.3 * np.sqrt(1.0 - 0.98 * s * s)
    A = np.stack([0.15 * g * 0.05 * rng.normal(x.size), -0.3 * s / np.sqrt(1.0 - 0.98 * s * s) * dt,
                  0.002 * dt * rng.normal(x.size)], 1)
    return X[:n], A[:n], np.full(n, 2.5 * 0.15)


def _particles(case, seed):
    """X, alpha, sigma (float64) of the case's particle set, and its generator."""
    n, kind = case["n"], case["set"]
    if kind == "cube":
        X, A, S, _ = workloads.cube(n=n, seed=seed, n_sample=0)
    elif kind == "blobs":
        X, A, S = workloads.blobs(n=n, seed=seed, n_probe=3, n_check=1)[:3]
    elif kind == "ring":
        X, A, S = workloads.ring(n_stations=-(-n // 128), samples=128, seed=seed)
    elif kind == "leapfrog":
        X, A, S = workloads.leapfrog(n_stations=-(-n // 256), samples=128, seed=seed)
    else:
        X, A, S = _wake(n, case["dt"], workloads.SplitMix64(seed))
    if X.shape[0] > n:  # rings come in whole stations: drop single particles all along them
        keep = np.linspace(0, X.shape[0] - 1, n).astype(np.int64)
        X, A, S = X[keep], A[keep], S[keep]
    return X, A, S


def _points(case, seed, X):
    """m probe or target points among the particles, in no order, and m vectors."""
    rng = workloads.SplitMix64(seed + 77)
    m = case["m"]
    pick = (rng.uniform(m) * X.shape[0]).astype(np.int64)
    return X[pick] + 0.02 * rng.normal(3 * m).reshape(m, 3), rng.normal(3 * m).reshape(m, 3)


def prepare(case, seed):
    kind = case["kind"]
    X, A, S = _particles(case, seed)
    calc = FMMCalculator(P=case["P"], theta=case["theta"], ncrit=case["ncrit"], precision=case["precision"],
                         stretching=case.get("stretching", "transposed"),
                         formulation=case.get("formulation", "cvpm"), scheme="euler")
    st = dict(case=case, calc=calc)
    if kind in ("advance", "wing"):
        # the program keeps its particles on the host and hands them over each pass
        st["bodies"] = make_bodies(X, A, S)
    else:
        calc.set_bodies(make_bodies(X, A, S))
    if kind in ("eval", "viscous"):
        # the program's own result buffer, page-locked as a program that downloads each step has it
        st["rec"] = torch.zeros((case["n"], BODY_DOUBLES), dtype=torch.float64,
                                pin_memory=torch.cuda.is_available())
        if case.get("near", 0.0) > 0.0:
            calc.set_near_field(case["near"])
        if kind == "viscous":
            calc.set_viscosity("pse", case["nu"])
    if kind in ("sensors", "direct", "probe_adjoint"):
        st["pts"], st["vec"] = _points(case, seed, X)
    if kind == "sensors":
        st["probes"] = make_bodies(st["pts"], st["vec"], np.ones(case["m"]))
    if kind in ("sensors", "probe_adjoint", "eval_vjp"):
        calc.build()
    if kind == "sensors":
        calc.calculate()
    if kind == "eval_vjp":
        rng = workloads.SplitMix64(seed + 78)
        st["ubar"], st["abar"] = (rng.normal(3 * case["n"]).reshape(-1, 3) for _ in range(2))
    if kind == "wing":
        st["wing"] = Wing(design_wing(np.deg2rad(5.0), None, span=6.0, chord=1.0, nspan=40, nchord=10))
    calc.sync()
    return st


def _handed_on(case, a):
    """An FP64 path's array as it is; a mixed path's in float32."""
    t = torch.from_numpy(a) if isinstance(a, np.ndarray) else a
    return t if case["precision"] == "fp64" else t.float()


def run(st):
    case, calc = st["case"], st["calc"]
    kind = case["kind"]
    if kind == "advance":
        b = st["bodies"].copy()
        calc.advance(b, case["dt"])
        return {"bodies": b}
    if kind in ("eval", "viscous"):
        calc.build()
        calc.calculate()
        if kind == "viscous":
            calc.viscosity(case["dt"])
        rec = st["rec"]
        calc.copyBodies2Host(rec.numpy())
        if case["precision"] == "fp64":
            return {"bodies": rec}
        return {"J": _handed_on(case, rec[:, 0:9]), "velocity_dadt": _handed_on(case, rec[:, 15:21])}
    if kind == "sensors":
        s = st["probes"].copy()
        calc.getSensorData(s)
        return {"X": s[:, 9:12], "velocity": _handed_on(case, s[:, 15:18])}
    if kind == "direct":
        u, J, d = calc.direct(st["pts"], st["vec"])
        return {"velocity": u, "J": J, "dadt": d}
    if kind == "probe_adjoint":
        ga, gx = calc.probe_adjoint(st["pts"], st["vec"])
        return {"alpha": _handed_on(case, ga), "x": _handed_on(case, gx)}
    if kind == "eval_vjp":
        xb, ab = calc.eval_vjp(st["ubar"], st["abar"])
        return {"x": _handed_on(case, xb), "alpha": _handed_on(case, ab)}
    # the wing loop: its wake as the last pass left it on the host, one step, and the wing back
    calc.set_bodies(st["bodies"])
    gamma, force = st["wing"].step(calc, U_WING, case["dt"])
    wake = calc.copyBodies2Host()
    st["wing"].translate(case["dt"] * U_WING)
    return {"gamma": _handed_on(case, gamma), "force": _handed_on(case, force), "wake": _handed_on(case, wake)}


def _m2l_flops(P):
    """Real operations of one multipole-to-local translation of three components, degrees below P."""
    return 26.0 * sum((j + 1) * (P - j) ** 2 for j in range(P)) + 10.0 * P * P


def work(case):
    """Bytes: the particles in (X, alpha, sigma) and the results out, once.  Operations: 70 for a
    near pair; 10 leaves' worth of near pairs for a particle and 100 translations for a cell of a quarter leaf,
    as the trees of these particle sets have them; every pair of the direct sum."""
    n, P, ncrit, kind = case["n"], case["P"], min(case["ncrit"], case["n"]), case["kind"]
    m = case.get("m", 0)
    near, cells = 70.0 * n * min(10.0 * ncrit, n), n / (0.25 * ncrit)
    far = cells * min(100.0, cells) * _m2l_flops(P) + n * 40.0 * P * P
    if case.get("near", 0.0) > 0.0:  # cores reach past the leaves: a sphere of that many cores of sigma = 2 h
        near = 70.0 * n * min(n, 4.2 * (2.0 * case["near"] + 4.0) ** 3)
    if kind == "direct":
        return {"bytes": 56.0 * n + 168.0 * m, "flops": 70.0 * n * m}
    if kind == "sensors":
        return {"bytes": 56.0 * n + 48.0 * m, "flops": 70.0 * m * min(10.0 * ncrit, n) + 0.25 * m * _m2l_flops(P)}
    if kind == "probe_adjoint":
        return {"bytes": 104.0 * n + 48.0 * m,
                "flops": 70.0 * m * min(10.0 * ncrit, n) + 0.25 * m * _m2l_flops(P) + n * 40.0 * P * P}
    if kind == "eval_vjp":
        return {"bytes": 152.0 * n, "flops": 3.0 * near + 2.0 * far}
    if kind == "viscous":
        return {"bytes": 184.0 * n, "flops": near * 1.5 + far}
    if kind == "wing":
        return {"bytes": 208.0 * n, "flops": 2.0 * (near + far)}
    return {"bytes": 176.0 * n, "flops": near + far}


# ---- 64-bit values by the direct sum, in plain torch ---------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _factors(d, sig):
    """f1 and f2 of the regularised Biot-Savart kernel for separations d [..., 3]."""
    r2 = (d * d).sum(-1)
    hit = r2 == 0.0
    r2 = torch.where(hit, torch.ones_like(r2), r2)
    r = r2.sqrt()
    s = r / (math.sqrt(2.0) * sig)
    t2 = 2.0 / math.sqrt(math.pi) * s * torch.exp(-s * s)
    g = torch.where(hit, torch.zeros_like(r), torch.erf(s) - t2)
    t2 = torch.where(hit, torch.zeros_like(r), t2)
    k = 1.0 / (4.0 * math.pi * r2 * r)
    return g * k, (2.0 * s * s * t2 - 3.0 * g) * k / r2


def _direct(xt, xs, al, sg):
    """u [m, 3] and J [m, 3, 3] at xt of the particles, pair by pair in 64 bits."""
    xt, xs, al, sg = (torch.as_tensor(v, dtype=torch.float64, device=_device()) for v in (xt, xs, al, sg))
    us, Js = [], []
    rows = max(1, 20000000 // xs.shape[0])
    for c in range(0, xt.shape[0], rows):
        d = xt[c:c + rows, None, :] - xs[None]
        f1, f2 = _factors(d, sg)
        w = torch.linalg.cross(d, al.expand_as(d))
        us.append(-(f1[..., None] * w).sum(1))
        J = -torch.matmul((f2[..., None] * w).transpose(1, 2).contiguous(), d.contiguous())
        a = torch.matmul(f1, al)
        z = torch.zeros_like(a[:, 0])
        J = J - torch.stack([z, a[:, 2], -a[:, 1], -a[:, 2], z, a[:, 0], a[:, 1], -a[:, 0], z], 1).reshape(-1, 3, 3)
        Js.append(J)
    return torch.cat(us).cpu().numpy(), torch.cat(Js).cpu().numpy()


def _tree_order(X, ncrit):
    """The order in which the framework returns bodies: octree leaves of at most ncrit bodies by
    their octant digits, the input order inside a leaf."""
    lo, hi = X.min(0), X.max(0)
    c = np.broadcast_to((hi + lo) / 2, X.shape).copy()
    x0 = (hi + lo) / 2
    R = max((x0 - lo).max(), (hi - x0).max()) * 1.00001
    key = np.zeros(X.shape[0], dtype=np.int64)
    for l in range(21):
        up = X > c
        key = key * 8 + up @ np.array([1, 2, 4])
        c += np.where(up, 1.0, -1.0) * (R / (1 << (l + 1)))
    leaf = np.full(X.shape[0], -1, dtype=np.int64)
    for l in range(22):
        part = key >> (3 * (21 - l))
        _, inv, cnt = np.unique(part, return_inverse=True, return_counts=True)
        here = (leaf < 0) & (cnt[inv] <= ncrit)
        leaf[here] = part[here] << (3 * (21 - l))
        if (leaf >= 0).all():
            break
    return np.argsort(leaf, kind="stable")


def exact(case, seed):
    """The direct sum, where the method comes near enough to it to say something (its far field is
    the singular kernel's) and pairs are few enough."""
    kind = case["kind"]
    n, m = case["n"], case.get("m", 0)
    if kind == "direct":
        X, A, S = _particles(case, seed)
        pts, vec = _points(case, seed, X)
        u, J = _direct(pts, X, A, S)
        return {"velocity": u, "J": J.reshape(-1, 9), "dadt": np.einsum("iab,ib->ia", J, vec)}
    if kind == "advance" and (n <= 1000 and case["set"] == "blobs" and case["theta"] <= 0.3) or (
            kind == "eval" and case["near"] > 0.0 and n <= 100000):
        X, A, S = _particles(case, seed)
        o = _tree_order(X, case["ncrit"])
        X, A, S = X[o], A[o], S[o]
        u, J = _direct(X, X, A, S)
        dadt = np.einsum("iab,ib->ia" if case["stretching"] == "classic" else "iba,ib->ia", J, A)
        J = J.reshape(-1, 9)
        if kind == "eval" and case["precision"] == "mixed":
            return {"J": J, "velocity_dadt": np.concatenate([u, dadt], 1)}
        b = make_bodies(X, A, S)
        b[:, 0:9], b[:, 15:18], b[:, 18:21] = J, u, dadt
        if kind == "advance":
            b[:, 9:12] += case["dt"] * u
            b[:, 12:15] += case["dt"] * dadt
        return {"bodies": b}
    return None
