"""The lane kernels' common attempt against the complete rules.

A user stopping time beyond every trajectory's span changes nothing in the
integration, but makes a trajectory irregular for the common attempt, so that
the complete rules make every attempt.  Both ways have to give the same bits:
states, times, return codes, saved points and counters, on batches that mix
ordinary trajectories with ones the common attempt has to leave (spans that
start far from zero, backward or empty or tiny spans, states that are huge, not
finite or blow up) and with options at the edge of its conditions."""
import numpy as np
import pytest

import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu


def _blowup(du, u, p, t):
    du[0] = p[0] * u[0] * u[0]
    du[1] = -u[1] + t
    du[2] = p[1] * u[2]


def _blowup_jac(J, u, p, t):
    for i in range(3):
        for k in range(3):
            J[i, k] = 0.0
    J[0, 0] = 2.0 * p[0] * u[0]
    J[1, 1] = -1.0
    J[2, 2] = p[1]


BLOWUP = odemi.ODEFunction(_blowup, jac=_blowup_jac)


def _batch(fun, N):
    rng = np.random.Generator(np.random.PCG64(91))
    if fun is P.ROBERTSON:
        u0 = np.stack([np.ones(N), np.zeros(N), np.zeros(N)])
        p = np.array([0.04, 3e7, 1e4])[:, None] * np.exp(rng.uniform(-0.7, 0.7, (3, N)))
        t0, tf = np.zeros(N), 10.0 ** rng.uniform(-3, 4, N)
    elif fun is P.LORENZ:
        u0 = rng.uniform(-1.0, 1.0, (3, N))
        p = np.stack([rng.uniform(8.0, 12.0, N), rng.uniform(0.0, 28.0, N), np.full(N, 8.0 / 3.0)])
        t0, tf = np.zeros(N), rng.uniform(0.1, 4.0, N)
    else:
        # the first component blows up at 1 / (p u0): before the end for some
        u0 = rng.uniform(0.2, 2.0, (3, N))
        p = np.stack([rng.uniform(-1.0, 1.0, N), rng.uniform(-3.0, 1.0, N)])
        t0, tf = np.zeros(N), rng.uniform(0.2, 2.0, N)
    k = np.arange(N) % 16
    t0[k == 3] = -5.0                                 # |t0| > |tf|
    t0[k == 5] = tf[k == 5] - 1e-13                   # a span of a few hundred ulp
    t0[k == 6] = tf[k == 6]                           # empty span
    u0[:, k == 8] *= 1e160                            # squares overflow
    u0[0, k == 9] = np.nan
    u0[1, k == 10] = np.inf
    u0[2, k == 11] = 1e-300
    swap = k == 12                                    # backward
    t0[swap], tf[swap] = tf[swap].copy(), t0[swap].copy()
    return u0, p, t0, tf


OPTIONS = {
    "plain": dict(reltol=1e-6, abstol=1e-8),
    "saveat": dict(reltol=1e-5, abstol=1e-7, saveat=np.array([0.05, 0.3, 0.31, 1.7]), max_saves=6),
    "dtmin": dict(reltol=1e-9, abstol=1e-12, dtmin=1e-3),
    "maxiters": dict(reltol=1e-8, abstol=1e-10, maxiters=23),
    "dtmax": dict(reltol=1e-3, abstol=1e-6, dtmax=0.02),
    "user_dt": dict(reltol=1e-4, abstol=1e-6, dt=3.0, saveat=np.array([0.1, 0.6]), max_saves=4),
    "abstol0": dict(reltol=1e-6, abstol=0.0),
    "reltol_half": dict(reltol=0.5, abstol=1e-3),
    "everystep": dict(reltol=1e-4, abstol=1e-6, save_everystep=True, save_start=True, max_saves=64),
}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("alg,fun", [(odemi.Tsit5(), P.LORENZ), (odemi.Tsit5(), BLOWUP),
                                     (odemi.Rodas5P(), P.ROBERTSON), (odemi.Rodas5P(), BLOWUP)],
                         ids=["tsit5-lorenz", "tsit5-blowup", "rodas-robertson", "rodas-blowup"])
@pytest.mark.parametrize("options", list(OPTIONS))
def test_common_attempt_equals_complete_rules(alg, fun, precision, options):
    N = 333
    u0, p, t0, tf = _batch(fun, N)
    kw = dict(OPTIONS[options])
    kw.setdefault("maxiters", 400)   # the lanes that stall end soon
    ea = odemi.EnsembleMI355X(precision=precision)
    print(f"[case] {alg} {options} {precision} N={N}", flush=True)
    a = odemi.solve_arrays(fun, alg, u0, p, t0, tf, ea, **kw)
    b = odemi.solve_arrays(fun, alg, u0, p, t0, tf, ea, tstops=[1e12], **kw)
    for k in ("u_final", "t_final", "retcode", "nsaved", "stats"):
        assert np.array_equal(a[k], b[k], equal_nan=(a[k].dtype.kind == "f")), k
    rows = np.arange(a["t_out"].shape[0])[:, None] < a["nsaved"][None, :]   # what was written
    assert np.array_equal(a["t_out"][rows], b["t_out"][rows])
    assert np.array_equal(np.swapaxes(a["u_out"], 1, 2)[rows], np.swapaxes(b["u_out"], 1, 2)[rows], equal_nan=True)
    assert (a["retcode"] == 1).any()
