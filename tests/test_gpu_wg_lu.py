"""The blocked FP64 LU and the substitutions of the workgroup Rodas5P kernels
(csrc/kernels/odemi_lu.h) at the edges of their panels (8 columns), tiles (16)
and row slots (64): final states and step counts are those of the CPU
restatement bit for bit, which does the same eliminations element by element."""
import numpy as np
import pytest

import oracle as O
import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu

EDGES = (2, 6, 8, 10, 14, 16, 18, 24, 30, 32, 34, 62, 64, 66, 70, 72, 74, 96, 98, 112, 126, 128)


# scale 1e-130: dividends below the range of the short quotient, so every
# substitution goes through the IEEE divisions (alpha = 0: a linear chain)
@pytest.mark.parametrize("nmax,scale", [(10, 1.0), (18, 1.0), (66, 1.0), (74, 1.0), (128, 1.0), (18, 1e-130)])
def test_lu_edges_bit_identical(nmax, scale):
    sizes = [n for n in EDGES if n <= nmax]
    d = P.chain_ensemble(N=4 * len(sizes), seed=31, m_lo=nmax // 2, m_hi=nmax // 2)
    nvec = np.resize(np.array(sizes, dtype=np.int32), d["u0"].shape[1])
    u0 = np.zeros_like(d["u0"])
    for j, n in enumerate(nvec):
        u0[:n // 2, j] = scale * d["u0"][:n // 2, j]
    p = d["p"].copy()
    if scale != 1.0:
        p[2] = 0.0
    tf = np.full(u0.shape[1], 0.1)
    kw = dict(reltol=1e-6, abstol=1e-6 * scale)
    print(f"[case] chain n {sizes} wg fp64 scale {scale}", flush=True)
    ref = O.ensemble_builtin(O.PROB_CHAIN, u0, p, d["t0"], tf, nvec=nvec, alg=O.RODAS5P, save_start=False, **kw)
    out = odemi.solve_arrays(P.CHAIN, odemi.Rodas5P(), u0, p, d["t0"], tf, nvec=nvec, **kw)
    assert (out["retcode"] == 1).all() and (ref["retcode"] == 1).all()
    assert np.array_equal(out["stats"][1], ref["naccept"]) and np.array_equal(out["stats"][2], ref["nreject"])
    for j, n in enumerate(nvec):
        assert np.array_equal(out["u_final"][:n, j], ref["u_final"][:n, j]), f"n = {n}, trajectory {j}"
