"""Served trajectories that end in a failure code give the batch engine's
results bit for bit wherever the tick boundaries fall.  After a rejected attempt
a failing trajectory reports that attempt's trial state, so the pool has to keep
it from tick to tick."""
import numpy as np
import pytest

import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu


def _growth(du, u, p, t):
    du[0] = p[0] * u[0] * u[0]      # blows up at 1 / (p u0) for p > 0
    du[1] = p[1] * (u[0] - u[1])
    du[2] = -u[2] + t


def _growth_jac(J, u, p, t):
    for i in range(3):
        for k in range(3):
            J[i, k] = 0.0
    J[0, 0] = 2.0 * p[0] * u[0]
    J[1, 0] = p[1]
    J[1, 1] = -p[1]
    J[2, 2] = -1.0


GROWTH = odemi.ODEFunction(_growth, jac=_growth_jac)


def _batch(fun, N):
    rng = np.random.Generator(np.random.PCG64(7))
    u0 = rng.uniform(0.3, 2.0, (3, N))
    if fun is GROWTH:
        p = np.stack([rng.uniform(-0.5, 2.0, N), rng.uniform(1.0, 30.0, N)])
    else:
        p = np.stack([rng.uniform(8.0, 12.0, N), rng.uniform(0.0, 28.0, N), np.full(N, 8.0 / 3.0)])
    return u0, p, np.zeros(N), rng.uniform(1.0, 4.0, N)


# tick boundaries after every attempt and after every eighth; 32 is a multiple of both
@pytest.mark.parametrize("options", [dict(maxiters=32), dict(dtmin=2e-3), dict(maxiters=20000)],
                         ids=["maxiters", "dtmin", "stall"])
@pytest.mark.parametrize("tick", [1, 8])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("alg,fun", [(odemi.Tsit5(), P.LORENZ), (odemi.Tsit5(), GROWTH), (odemi.Rodas5P(), P.LORENZ),
                                     (odemi.Rodas5P(), GROWTH)],
                         ids=["tsit5-lorenz", "tsit5-growth", "rodas-lorenz", "rodas-growth"])
def test_failed_requests_equal_batch_engine(alg, fun, precision, tick, options):
    N = 300
    u0, p, t0, tf = _batch(fun, N)
    kw = dict(reltol=1e-7, abstol=1e-9, **options)
    print(f"[case] served failures {alg} {precision} tick {tick} {options}", flush=True)
    b = odemi.solve_arrays(fun, alg, u0, p, t0, tf, odemi.EnsembleMI355X(precision=precision), **kw)
    with odemi.EnsembleServer(fun, 3, p.shape[0], alg, precision=precision, tick_attempts=tick, **kw) as srv:
        r = srv.submit(u0, p, t0, tf)
        assert r.wait(timeout=60)
    if options.get("maxiters") == 32 or fun is GROWTH:
        assert (b["retcode"] != 1).any()
    assert np.array_equal(r.retcode, b["retcode"]) and np.array_equal(r.stats, b["stats"])
    assert np.array_equal(r.u_final, b["u_final"], equal_nan=True)
