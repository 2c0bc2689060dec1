"""Edges of the lane kernels' common attempt against the complete rules: states
that are a negative zero (compared by their bits), and a user dt against the
direction of integration.  A stopping time beyond every span sends each attempt
through the complete rules (see test_gpu_common_attempt.py)."""
import numpy as np
import pytest

import odemi

pytestmark = pytest.mark.gpu


def _growth(du, u, p, t):
    du[0] = -u[0] + t
    du[1] = p[0] * u[1]
    du[2] = p[1] * u[2]


def _growth_jac(J, u, p, t):
    for i in range(3):
        for k in range(3):
            J[i, k] = 0.0
    J[0, 0] = -1.0
    J[1, 1] = p[0]
    J[2, 2] = p[1]


def _pair(du, u, p, t):
    """Rows 0 and 1 of the stage matrix change places, the first pivot is p[1] >
    0; the sign of a zero u[0] shows in u[2]."""
    du[0] = p[0] * u[1]
    du[1] = p[1] * u[0]
    du[2] = -u[2] + 0.1 * np.arctan(1.0 / u[0])


def _pair_jac(J, u, p, t):
    for i in range(3):
        for k in range(3):
            J[i, k] = 0.0
    J[0, 1] = p[0]
    J[1, 0] = p[1]
    J[2, 2] = -1.0


GROWTH = odemi.ODEFunction(_growth, jac=_growth_jac)
PAIR = odemi.ODEFunction(_pair, jac=_pair_jac)
ALGS = pytest.mark.parametrize("alg", [odemi.Tsit5(), odemi.Rodas5P()], ids=["tsit5", "rodas5p"])
PRECISIONS = pytest.mark.parametrize("precision", ["fp64", "mixed"])


def _batch(fun, N):
    rng = np.random.Generator(np.random.PCG64(12))
    u0 = rng.uniform(0.2, 1.0, (3, N))
    if fun is GROWTH:
        # growth rates up to 300: pivots of both signs at the first steps
        p = np.stack([rng.uniform(-5.0, 5.0, N), np.exp(rng.uniform(-2.0, 5.7, N)) * rng.choice([-1.0, 1.0], N)])
    else:
        p = np.stack([rng.uniform(-5.0, 5.0, N), rng.uniform(50.0, 400.0, N)])
        u0[2] *= rng.choice([-9.0, 9.0], N)
    return u0, p, np.zeros(N), rng.uniform(0.05, 1.5, N)


def _zeros(u0):
    k = np.arange(u0.shape[1]) % 8
    u0[1, k == 1] = -0.0
    u0[0, k == 2] = -0.0
    u0[:2, k == 3] = -0.0
    u0[1:, k == 4] = 0.0
    u0[:, k == 5] = -0.0
    u0[2, k == 6] = -5e-324
    u0[0, k == 7] = -1e-290


def _bits(a):
    a = np.where(np.isnan(a), np.nan, a)
    return np.ascontiguousarray(a).view(np.int64)


@ALGS
@PRECISIONS
@pytest.mark.parametrize("fun", [GROWTH, PAIR], ids=["growth", "pair"])
@pytest.mark.parametrize("saveat", [None, [0.02, 0.3, 0.31]], ids=["final", "saveat"])
def test_zero_states_bit_identical(alg, precision, fun, saveat):
    u0, p, t0, tf = _batch(fun, 400)
    _zeros(u0)
    kw = dict(reltol=1e-6, abstol=1e-8, max_saves=4, saveat=saveat, maxiters=2000)
    if fun is PAIR:
        kw.update(dt=0.1, reltol=0.1, abstol=0.1)   # the first stage matrix has p[1] above 1 / (gamma dt)
    ea = odemi.EnsembleMI355X(precision=precision)
    print(f"[case] zero states {alg} {precision} {saveat}", flush=True)
    a = odemi.solve_arrays(fun, alg, u0, p, t0, tf, ea, **kw)
    b = odemi.solve_arrays(fun, alg, u0, p, t0, tf, ea, tstops=[1e12], **kw)
    assert np.array_equal(a["stats"], b["stats"]) and np.array_equal(a["retcode"], b["retcode"])
    assert np.array_equal(_bits(a["u_final"]), _bits(b["u_final"]))
    rows = np.arange(4)[:, None] < a["nsaved"][None, :]
    assert np.array_equal(_bits(np.swapaxes(a["u_out"], 1, 2)[rows]), _bits(np.swapaxes(b["u_out"], 1, 2)[rows]))
    assert (a["retcode"] == 1).mean() > 0.5

@ALGS
@PRECISIONS
@pytest.mark.parametrize("dtmin", [0.0, 1e-3])
def test_user_dt_against_the_direction(alg, precision, dtmin):
    """The complete rules raise a negative dt of a forward solve to max(eps(t),
    dtmin), where it ends (Unstable or DtLessThanMin)."""
    u0, p, t0, tf = _batch(GROWTH, 200)
    t0[::3] = 0.01
    kw = dict(reltol=1e-6, abstol=1e-8, dt=-0.1, dtmin=dtmin, maxiters=500)
    ea = odemi.EnsembleMI355X(precision=precision)
    print(f"[case] negative dt {alg} {precision} dtmin {dtmin}", flush=True)
    a = odemi.solve_arrays(GROWTH, alg, u0, p, t0, tf, ea, **kw)
    b = odemi.solve_arrays(GROWTH, alg, u0, p, t0, tf, ea, tstops=[1e12], **kw)
    outs = [b]
    if precision == "fp64":
        outs.append(odemi.solve_arrays(GROWTH, alg, u0, p, t0, tf, odemi.EnsembleMI355X(engine="plain"), **kw))
    for o in outs:
        assert np.array_equal(a["retcode"], o["retcode"]) and np.array_equal(a["stats"], o["stats"])
        assert np.array_equal(a["u_final"], o["u_final"], equal_nan=True)
        assert np.array_equal(a["t_final"], o["t_final"])
    assert (a["retcode"] != 1).all()
