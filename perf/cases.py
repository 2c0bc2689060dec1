"""Performance cases of the ensemble ODE engine: what its users have it do.

A case is one pass through a public entry point (odemi.solve_arrays on device
or host arrays, odemi.solve on an EnsembleProblem, a burst of requests to an
odemi.EnsembleServer) on seeded inputs of the problem families in
odemi.problems, with the distributions that bench.py and the tests use.
`exact` integrates the same equations in FP64 with methods of its own (Taylor
series, extrapolated linearly implicit Euler, closed-form bounces).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ordinarydiffeq.jl_amd"))

import odemi  # noqa: E402
from odemi import problems as P  # noqa: E402

# state sizes of the uneven chain batches: one to eight 16-column tiles, none
# but the largest a multiple of 16, every batch holding each of them
CHAIN_SIZES = (8, 34, 70, 128)
GRAVITY = 9.81
EVERY_STEP = 256   # more than the steps of any trajectory of the ensemble cases


def listed():
    return [
        # the headline workload of bench.py: a parameter sweep of a non-stiff system, final states only
        dict(name="lorenz_fp64_1m", kind="lorenz", n=1048576, precision="fp64", reltol=1e-6, t_lo=1.0, t_hi=10.0),
        # the same sweep on the mixed-precision engine, a batch of odd size
        dict(name="lorenz_mixed_300k", kind="lorenz", n=300007, precision="mixed", reltol=1e-6, t_lo=1.0, t_hi=10.0),
        # a small ensemble at a tight tolerance (the serving and test size): launches and latency count
        dict(name="lorenz_fp64_1k", kind="lorenz", n=1024, precision="fp64", reltol=1e-8, t_lo=1.0, t_hi=1.0),
        # trajectories sampled through the dense output for plotting or fitting
        dict(name="lorenz_saveat_100k", kind="saveat", n=100003, precision="fp64", reltol=1e-6, t_hi=10.0, points=20),
        # numpy in, numpy out: a caller that keeps its ensemble on the host
        dict(name="lorenz_host_200k", kind="host", n=200001, precision="fp64", reltol=1e-6, t_lo=1.0, t_hi=10.0),
        # stiff kinetics, a sweep over rate constants
        dict(name="robertson_fp64_262k", kind="robertson", n=262144, precision="fp64"),
        dict(name="robertson_mixed_20k", kind="robertson", n=20011, precision="mixed"),
        # oscillator chains of uneven size in one call (method of lines, molecular chains)
        dict(name="chain_fp64_96", kind="chain", n=96, precision="fp64", t_hi=0.1),
        dict(name="chain_mixed_1k", kind="chain", n=1025, precision="mixed", t_hi=0.25),
        # event location: bouncing balls with a continuous callback
        dict(name="balls_fp64_500k", kind="balls", n=500009, precision="fp64"),
        # many callers with small ragged ensembles through the continuous-batching server
        dict(name="serving_lorenz_64", kind="serving", n=64, precision="fp64", reltol=1e-6, largest=2048),
        # the EnsembleProblem surface with its defaults (every step saved, one solution object per trajectory)
        dict(name="ensemble_solve_500", kind="ensemble", n=500, precision="fp64", reltol=1e-6, t_hi=2.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lorenz", "lorenz", "saveat", "host", "robertson", "chain", "balls", "serving", "ensemble"])
    c = dict(kind=kind, precision=rng.choice(["fp64", "fp64", "mixed"]))
    if kind in ("lorenz", "host"):
        c.update(n=_log_int(rng, 300, 1000000 if kind == "lorenz" else 300000), reltol=rng.choice([1e-5, 1e-6, 1e-8]),
                 t_lo=1.0, t_hi=round(rng.uniform(1.5, 10.0), 2))
    elif kind == "saveat":
        c.update(n=_log_int(rng, 300, 200000), reltol=rng.choice([1e-5, 1e-6, 1e-7]), t_hi=float(rng.randint(2, 10)),
                 points=rng.randint(3, 25))
    elif kind == "robertson":
        c.update(n=_log_int(rng, 300, 262144))
    elif kind == "chain":
        n = _log_int(rng, 24, 1025)
        if n > 96:
            c["precision"] = "mixed"   # the engine for large batches of large systems
        c.update(n=n, t_hi=round(rng.uniform(0.05, 0.1 if n <= 96 else 0.25), 3))
    elif kind == "balls":
        c.update(n=_log_int(rng, 1000, 500009), precision="fp64")
    elif kind == "serving":
        c.update(n=rng.randint(8, 64), reltol=rng.choice([1e-6, 1e-8]), largest=_log_int(rng, 64, 2048))
    else:
        c.update(n=_log_int(rng, 50, 500), reltol=rng.choice([1e-4, 1e-6]), t_hi=round(rng.uniform(0.5, 2.0), 2),
                 precision="fp64")
    return c


# ---- inputs (numpy, from the seed alone) ----

def _lorenz_inputs(rng, n, t_lo, t_hi):
    """sigma~U[8,12], rho~U[0,28], beta=8/3, u0~U[-1,1]^3, t_end~U[t_lo,t_hi]."""
    p = np.stack([rng.uniform(8.0, 12.0, n), rng.uniform(0.0, 28.0, n), np.full(n, 8.0 / 3.0)])
    u0 = rng.uniform(-1.0, 1.0, (3, n))
    tf = rng.uniform(t_lo, t_hi, n) if t_hi > t_lo else np.full(n, t_hi)
    return u0, p, np.zeros(n), tf


def _inputs(case, seed):
    rng = np.random.Generator(np.random.PCG64([seed, 17]))
    kind, n = case["kind"], case["n"]
    if kind in ("lorenz", "host"):
        return _lorenz_inputs(rng, n, case["t_lo"], case["t_hi"])
    if kind in ("saveat", "ensemble"):
        return _lorenz_inputs(rng, n, case["t_hi"], case["t_hi"])
    if kind == "serving":
        # the sizes belong to the case, their order to the seed
        sizes = np.random.Generator(np.random.PCG64([n, case["largest"]])).integers(1, case["largest"] + 1, n)
        sizes[:2] = 1, case["largest"]
        rng.shuffle(sizes)
        return _lorenz_inputs(rng, int(sizes.sum()), 1.0, 10.0) + (sizes,)
    if kind == "robertson":
        s = np.exp(rng.uniform(math.log(0.5), math.log(2.0), (3, n)))
        p = np.array([0.04, 3e7, 1e4])[:, None] * s
        return np.stack([np.ones(n), np.zeros(n), np.zeros(n)]), p, np.zeros(n), np.full(n, 1e5)
    if kind == "balls":
        u0 = np.stack([rng.uniform(10.0, 50.0, n), rng.uniform(-5.0, 5.0, n)])
        return u0, rng.uniform(0.8, 0.95, (1, n)), np.zeros(n), np.full(n, 10.0)
    nvec = np.resize(np.array(CHAIN_SIZES, dtype=np.int32), n)
    rng.shuffle(nvec)
    p = np.stack([rng.uniform(1.0, 1e4, n), rng.uniform(0.01, 1.0, n), rng.uniform(0.0, 1.0, n)])
    u0 = np.zeros((max(CHAIN_SIZES), n))
    x0 = rng.normal(0.0, 0.1, (max(CHAIN_SIZES) // 2, n))
    inside = np.arange(len(x0))[:, None] < nvec[None, :] // 2
    u0[:len(x0)] = np.where(inside, x0, 0.0)
    return u0, p, np.zeros(n), np.full(n, case["t_hi"]), nvec


def _save_times(case):
    return np.linspace(0.0, case["t_hi"], case["points"] + 1)[1:]


def prepare(case, seed):
    kind = case["kind"]
    data = _inputs(case, seed)
    s = dict(case=case, engine=odemi.EnsembleMI355X(precision=case["precision"]))
    if kind == "serving":
        u0, p, t0, tf, sizes = data
        ends = np.cumsum(sizes)
        s["requests"] = [tuple(np.ascontiguousarray(a[..., e - k:e]) for a in (u0, p, t0, tf))
                         for k, e in zip(sizes, ends)]
        s["server"] = odemi.EnsembleServer(P.LORENZ, 3, 3, odemi.Tsit5(), precision=case["precision"],
                                           reltol=case["reltol"], abstol=case["reltol"], max_slots=1 << 17)
        return s
    if kind == "ensemble":
        u0, p, _, _ = data
        base = odemi.ODEProblem(P.LORENZ, u0[:, 0], (0.0, case["t_hi"]), p[:, 0])
        s["problem"] = odemi.EnsembleProblem(
            base, prob_func=lambda prob, ctx: odemi.remake(prob, u0=u0[:, ctx.sim_id - 1], p=p[:, ctx.sim_id - 1]))
        return s
    if kind == "robertson":
        s.update(fun=P.ROBERTSON, alg=odemi.Rodas5P(), keywords=dict(reltol=1e-6, abstol=1e-10))
    elif kind == "chain":
        s.update(fun=P.CHAIN, alg=odemi.Rodas5P(), keywords=dict(reltol=1e-6, abstol=1e-6, nvec=data[4]))
    elif kind == "balls":
        s.update(fun=P.BALL, alg=odemi.Tsit5(), keywords=dict(reltol=1e-6, abstol=1e-6, callback=P.BALL_BOUNCE))
    else:
        s.update(fun=P.LORENZ, alg=odemi.Tsit5(), keywords=dict(reltol=case["reltol"], abstol=case["reltol"]))
        if kind == "saveat":
            times = _save_times(case)
            s["keywords"].update(saveat=times, max_saves=len(times))
    s["arrays"] = data[:4] if kind == "host" else tuple(torch.as_tensor(a, device="cuda").contiguous()
                                                        for a in data[:4])
    odemi.compile_problem(s["fun"], data[0].shape[0], data[1].shape[0], callback=s["keywords"].get("callback"),
                          algs=("tsit5",) if isinstance(s["alg"], odemi.Tsit5) else ("rodas5p",),
                          ns=sorted(CHAIN_SIZES) if kind == "chain" else None)
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "serving":
        sent = [s["server"].submit(*r) for r in s["requests"]]
        for r in sent:
            if not r.wait(timeout=60):
                raise RuntimeError("a request did not finish")
        return {k: np.concatenate([getattr(r, k) for r in sent], axis=-1) for k in ("u_final", "retcode", "stats")}
    if kind == "ensemble":
        c = s["case"]
        sim = odemi.solve(s["problem"], odemi.Tsit5(), s["engine"], trajectories=c["n"], reltol=c["reltol"],
                          abstol=c["reltol"])
        # the saved steps of every trajectory, as rows padded with zeros
        t, u = np.zeros((c["n"], EVERY_STEP)), np.zeros((c["n"], EVERY_STEP, 3))
        for i, x in enumerate(sim.u):
            t[i, :len(x.t)], u[i, :len(x.t)] = x.t, x.u
        return {"t": t, "u": u, "u_final": np.stack([x.u[-1] for x in sim.u], axis=1),
                "retcode": np.array([int(x.retcode) for x in sim.u]), "stats": sim.arrays["stats"]}
    o = odemi.solve_arrays(s["fun"], s["alg"], *s["arrays"], s["engine"], **s["keywords"])
    names = ["u_final", "t_final", "retcode", "nsaved", "stats"] + (["t_out", "u_out"] if kind == "saveat" else [])
    return {k: o[k] for k in names}


# ---- work: what a pass cannot do without ----

def work(case):
    """Bytes: inputs read and results written once.  Flops: step attempts (the
    engines' mean per trajectory, near enough proportional to the time span)
    times the method's operations (FMA = 2): the right-hand sides, stage sums,
    error norm and controller, for Rodas5P the LU and eight solves too."""
    kind, n = case["kind"], case["n"]
    if kind == "robertson":
        attempts, flops, nbytes = 153.0, 8 * 11 + 27 + 12 + 144 + 525 + 60, 8 * 11 + 8 * 8 + 32
    elif kind == "balls":
        # ~6 attempts and ~185 evaluations of the dense output per ball
        attempts, flops, nbytes = 6.3, 6 + 77 * 2 + 60 + 30 * 48, 8 * 5 + 8 * 6 + 32
    elif kind == "chain":
        attempts = 340.0 * case["t_hi"] + 20.0
        sizes = np.array(CHAIN_SIZES, dtype=float)
        flops = float(np.mean(8 * 5.5 * sizes + 2 * sizes ** 3 / 3 + 16 * sizes ** 2 + 175 * sizes + 60))
        nbytes = 8 * (2 * float(np.mean(sizes)) + 6) + 32
    else:
        t = 0.5 * (case.get("t_lo", case.get("t_hi")) + case["t_hi"]) if kind != "serving" else 5.5
        attempts = 27.0 * t * (1e-6 / case["reltol"]) ** 0.2
        flops, nbytes = 6 * 8 + 77 * 3 + 60, 8 * 8 + 8 * 8 + 32
        if kind == "saveat":
            flops += 14 * 3 * case["points"] / attempts
            nbytes += 32 * case["points"]
        if kind == "serving":
            n = n * case["largest"] / 2
        if kind == "ensemble":
            nbytes += 32 * attempts
    return {"bytes": float(nbytes * n), "flops": float(flops * attempts * n)}


# ---- the same equations in 64 bits, by other methods ----

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lorenz_taylor(u0, p, stops, h=0.025, order=20):
    """States at each of the ascending `stops` (a list of (N,) or scalar times,
    from t = 0) by Taylor series of the given order."""
    dev = _device()
    T = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    sg, rho, beta = T(p[0]), T(p[1]), T(p[2])
    n = u0.shape[1]
    c = torch.zeros((3, order + 1, n), dtype=torch.float64, device=dev)
    c[:, 0] = T(u0)
    t = torch.zeros(n, dtype=torch.float64, device=dev)
    out = []
    for stop in stops:
        stop = torch.broadcast_to(T(stop), (n,))
        for _ in range(int(math.ceil(float((stop - t).max()) / h - 1e-9))):
            step = torch.clamp(stop - t, max=h)
            for k in range(order):
                xz = (c[0, :k + 1] * c[2, :k + 1].flip(0)).sum(0)
                xy = (c[0, :k + 1] * c[1, :k + 1].flip(0)).sum(0)
                c[0, k + 1] = sg * (c[1, k] - c[0, k]) / (k + 1)
                c[1, k + 1] = (rho * c[0, k] - xz - c[1, k]) / (k + 1)
                c[2, k + 1] = (xy - beta * c[2, k]) / (k + 1)
            acc = c[:, order]
            for k in range(order - 1, -1, -1):
                acc = acc * step + c[:, k]
            c[:, 0] = acc
            t = torch.where(step < h, stop, t + step)
        out.append(c[:, 0].cpu().numpy().copy())
    return out


def _chain_taylor(u0, p, t_end, nvec, h=0.004, order=20):
    """Oscillator chains by Taylor series, positions and velocities as (64, N)
    blocks with zeros beyond each chain's end."""
    dev = _device()
    T = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    k, damp, al = T(p[0]), T(p[1]), T(p[2])
    mmax, n = u0.shape[0] // 2, u0.shape[1]
    m = torch.as_tensor(nvec.astype(np.int64) // 2, device=dev)
    inside = (torch.arange(mmax, device=dev)[:, None] < m[None, :]).to(torch.float64)
    x = torch.zeros((order + 1, mmax, n), dtype=torch.float64, device=dev)
    v, sq = torch.zeros_like(x), torch.zeros_like(x)
    x[0] = T(u0[:mmax]) * inside          # every chain starts at rest
    steps = int(math.ceil(t_end / h))
    dt = t_end / steps
    for _ in range(steps):
        for q in range(order):
            sq[q] = (x[:q + 1] * x[:q + 1].flip(0)).sum(0)
            cube = (x[:q + 1] * sq[:q + 1].flip(0)).sum(0)
            s = 2.0 * x[q]
            s[1:] -= x[q, :-1]
            s[:-1] -= x[q, 1:]
            x[q + 1] = v[q] / (q + 1)
            v[q + 1] = (-k * s - damp * v[q] - al * cube) * inside / (q + 1)
        ax, av = x[order], v[order]
        for q in range(order - 1, -1, -1):
            ax, av = ax * dt + x[q], av * dt + v[q]
        x[0], v[0] = ax, av
    xs, vs = x[0].cpu().numpy(), v[0].cpu().numpy()
    out = np.zeros_like(u0)
    for size in set(int(z) for z in nvec):
        j = np.nonzero(nvec == size)[0]
        out[:size // 2, j] = xs[:size // 2, j]
        out[size // 2:size, j] = vs[:size // 2, j]
    return out


def _robertson_extrapolated(p, t_end, ratio=1.06, order=8):
    """Robertson kinetics by the linearly implicit Euler method extrapolated
    over 1..order substeps, time steps growing geometrically (the solution
    varies with log t); 3 x 3 systems by their adjugates."""
    dev = _device()
    k1, k2, k3 = (torch.as_tensor(q, dtype=torch.float64, device=dev) for q in p)
    y = torch.zeros((3, p.shape[1]), dtype=torch.float64, device=dev)
    y[0] = 1.0

    def rhs(a, b, c):
        return -k1 * a + k3 * b * c, k2 * b * b

    grid = [0.0, 1e-6]
    while grid[-1] * ratio < t_end:
        grid.append(grid[-1] * ratio)
    grid.append(t_end)
    for ta, tb in zip(grid[:-1], grid[1:]):
        # I - hJ in the unknowns (d1, d3), d2 = -(d1 + d3) by conservation
        j12, j13, j32 = k3 * y[2], k3 * y[1], 2.0 * k2 * y[1]
        table = []
        for q in range(1, order + 1):
            h = (tb - ta) / q
            m11, m13 = 1.0 + h * (k1 + j12), h * (j12 - j13)
            m31, m33 = h * j32, 1.0 + h * j32
            det = m11 * m33 - m13 * m31
            a, b, c = y[0], y[1], y[2]
            for _ in range(q):
                f1, f3 = rhs(a, b, c)
                d1 = h * (m33 * f1 - m13 * f3) / det
                d3 = h * (m11 * f3 - m31 * f1) / det
                a, b, c = a + d1, b - (d1 + d3), c + d3
            row = [torch.stack((a, b, c))]
            for s in range(1, q):
                row.append(row[s - 1] + (row[s - 1] - table[-1][s - 1]) / (q / (q - s) - 1.0))
            table.append(row)
        y = table[-1][-1]
    return y.cpu().numpy()


def _bounces(u0, p, t_end):
    """Height and velocity of the balls at t_end, bounce by bounce."""
    h, v, e = u0[0].copy(), u0[1].copy(), p[0]
    left = t_end.copy()
    while True:
        fall = (v + np.sqrt(v * v + 2.0 * GRAVITY * h)) / GRAVITY
        hit = fall < left
        if not hit.any():
            break
        v = np.where(hit, -e * (v - GRAVITY * fall), v)
        h = np.where(hit, 0.0, h)
        left = np.where(hit, left - fall, left)
    return np.stack([h + v * left - 0.5 * GRAVITY * left * left, v - GRAVITY * left])


def exact(case, seed):
    kind = case["kind"]
    data = _inputs(case, seed)
    u0, p, tf = data[0], data[1], data[3]
    res = dict(t_final=tf, retcode=None, nsaved=None, stats=None)
    if kind == "robertson":
        u = _robertson_extrapolated(p, 1e5)
    elif kind == "chain":
        u = _chain_taylor(u0, p, case["t_hi"], data[4])
    elif kind == "balls":
        u = _bounces(u0, p, tf)
    elif kind == "saveat":
        times = _save_times(case)
        states = _lorenz_taylor(u0, p, list(times))
        u = states[-1]
        res.update(u_out=np.stack(states), t_out=np.broadcast_to(times[:, None], (len(times), case["n"])).copy())
    else:
        u = _lorenz_taylor(u0, p, [tf])[0]
    if kind == "serving":
        return dict(u_final=u, retcode=None, stats=None)
    if kind == "ensemble":
        return dict(u_final=u, t=None, u=None, retcode=None, stats=None)
    res["u_final"] = u
    return res
