"""The FP64 workgroup kernels from n = 96 on (eight waves, four with continuous
callbacks) in every engine and with every hook: batch, plain and serving engines,
save times, discrete, continuous and vector callbacks.  Equal to
the CPU restatement bit for bit, or to the batch engine where that is checked."""
import numpy as np
import pytest

import oracle as O
import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu

SIZES = {96: (10, 96), 128: (34, 98, 128)}   # state sizes of a batch padded to the key


def _batch(nmax, N=9, seed=41):
    sizes = SIZES[nmax]
    d = P.chain_ensemble(N=N, seed=seed, m_lo=nmax // 2, m_hi=nmax // 2)
    nv = np.resize(np.array(sizes, dtype=np.int32), N)
    nv[-1] = nmax
    u0 = np.zeros_like(d["u0"])
    for j, n in enumerate(nv):
        u0[:n // 2, j] = d["u0"][:n // 2, j]
    p = d["p"].copy()
    p[0] = np.random.Generator(np.random.PCG64(seed)).uniform(1.0, 100.0, N)   # a few events each
    return u0, p, d["t0"], np.full(N, 0.6), nv


def _wall(itg):
    m = len(itg.u) // 2
    itg.u[m] = -0.5 * itg.u[m]


def _kick(itg):
    m = len(itg.u) // 2
    itg.u[m] = itg.u[m] + itg.p[1]


def _walls(out, u, t, itg):
    out[0] = u[0]
    out[1] = u[1] - 0.02


def _walls_affect(itg, ev):
    m = len(itg.u) // 2
    itg.u[m] = odemi.sym_ifelse(ev[0] == -1, -0.5 * itg.u[m], itg.u[m])


CCB = odemi.ContinuousCallback(lambda u, t, itg: u[0], None, affect_neg=_wall)
DCB = odemi.DiscreteCallback(lambda u, t, itg: odemi.sym_in(t, [0.25, 0.5]), _kick)
VCB = odemi.VectorContinuousCallback(_walls, _walls_affect, 2)
HOOKS = {"none": {}, "continuous": dict(callback=odemi.CallbackSet(CCB, DCB), tstops=[0.25, 0.5]),
         "vector": dict(callback=VCB)}
OPTS = dict(reltol=1e-6, abstol=1e-6)


class _PyCB:
    def __init__(self, cb):
        self.__dict__.update(cb.__dict__)


@pytest.mark.parametrize("nmax,hook", [(96, "continuous"), (128, "none"), (128, "continuous")])
@pytest.mark.parametrize("saves", [dict(save_end=True), dict(saveat=[0.1, 0.45], save_end=True)], ids=["final", "saveat"])
def test_large_chains_equal_restatement(nmax, hook, saves):
    u0, p, t0, tf, nv = _batch(nmax)
    print(f"[case] chain nmax {nmax} wg fp64 {hook} {saves}", flush=True)
    o = odemi.solve_arrays(P.CHAIN, odemi.Rodas5P(), u0, p, t0, tf, nvec=nv, max_saves=256, **saves, **OPTS, **HOOKS[hook])
    py = dict(callbacks=[_PyCB(DCB)] if hook == "continuous" else [], ccallbacks=[_PyCB(CCB)] if hook == "continuous" else [],
              tstops=HOOKS[hook].get("tstops"))
    for j, n in enumerate(nv):
        r = O.solve_builtin(O.PROB_CHAIN, u0[:n, j], p[:, j], (0.0, tf[j]), alg=O.RODAS5P, save_start=False,
                            **saves, **OPTS, **{k: v for k, v in py.items() if v})
        ns = int(o["nsaved"][j])
        assert int(o["retcode"][j]) == r["retcode"] == 1 and ns == r["nsaved"], j
        assert np.array_equal(o["u_final"][:n, j], r["u_final"]), j
        assert np.array_equal(o["t_out"][:ns, j], r["t"]) and np.array_equal(o["u_out"][:ns, :n, j], r["u"]), j
        st = o["stats"][:, j]
        assert (st[0], st[1], st[2], st[6]) == (r["nf"], r["naccept"], r["nreject"], r["ncondition"]), j


@pytest.mark.parametrize("nmax,hook", [(128, "none"), (96, "continuous"), (96, "vector")])
def test_plain_engine_and_server_equal_batch(nmax, hook):
    u0, p, t0, tf, nv = _batch(nmax)
    kw = dict(nvec=nv, save_start=False, save_end=True, max_saves=256, **OPTS, **HOOKS[hook])
    print(f"[case] chain nmax {nmax} plain wg fp64 and server {hook}", flush=True)
    ref = odemi.solve_arrays(P.CHAIN, odemi.Rodas5P(), u0, p, t0, tf, **kw)
    pl = odemi.solve_arrays(P.CHAIN, odemi.Rodas5P(), u0, p, t0, tf, odemi.EnsembleMI355X(engine="plain"), **kw)
    assert (ref["retcode"] == 1).all()
    ts = HOOKS[hook].get("tstops")
    with odemi.EnsembleServer(P.CHAIN, nmax, 3, odemi.Rodas5P(), tick_attempts=5, ns=list(SIZES[nmax]), max_slots=64,
                              max_tstops=2, callback=HOOKS[hook].get("callback"), **OPTS) as srv:
        r = srv.submit(u0, p, t0, tf, nvec=nv, tstops=ts)
        assert r.wait(timeout=100)
    for q in (pl["u_final"], r.u_final):
        for j, n in enumerate(nv):
            assert np.array_equal(q[:n, j], ref["u_final"][:n, j]), j
    assert np.array_equal(pl["stats"], ref["stats"]) and np.array_equal(r.stats, ref["stats"])
    assert np.array_equal(pl["retcode"], ref["retcode"]) and np.array_equal(r.retcode, ref["retcode"])
    if hook in ("continuous", "vector"):
        assert (ref["stats"][6] > 0).all()
