"""The lane kernels choose between the loop with the common attempt and the one
without it per wave, by a sample of the batch.  Each has to give the same bits
for any trajectory: batches that are mostly backward, mostly forward and even,
against the two directions solved apart."""
import numpy as np
import pytest

import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("saveat", [None, [0.05, 0.11, 0.3]], ids=["final", "saveat"])
@pytest.mark.parametrize("every", [2, 5])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("alg", [odemi.Tsit5(), odemi.Rodas5P()], ids=["tsit5", "rodas5p"])
def test_mixed_directions_equal_apart(alg, precision, every, saveat):
    N = 777
    rng = np.random.Generator(np.random.PCG64(23))
    u0 = rng.uniform(-1.0, 1.0, (3, N))
    p = np.stack([rng.uniform(8.0, 12.0, N), rng.uniform(0.0, 28.0, N), np.full(N, 8.0 / 3.0)])
    lo, hi = np.zeros(N), rng.uniform(0.1, 0.4, N)
    kw = dict(reltol=1e-6, abstol=1e-8, saveat=saveat, max_saves=5)
    ea = odemi.EnsembleMI355X(precision=precision)
    print(f"[case] directions {alg} {precision} {every} {saveat}", flush=True)
    odd = np.arange(N) % every != 0
    keys = ("u_final", "t_final", "retcode", "nsaved", "stats")
    for back in (odd, ~odd):
        o = odemi.solve_arrays(P.LORENZ, alg, u0, p, np.where(back, hi, lo), np.where(back, lo, hi), ea, **kw)
        assert (o["retcode"] == 1).all()
        for part, (a, b) in ((back, (hi, lo)), (~back, (lo, hi))):
            r = odemi.solve_arrays(P.LORENZ, alg, u0[:, part], p[:, part], a[part], b[part], ea, **kw)
            for k in keys:
                assert np.array_equal(o[k][..., part], r[k]), k
            rows = np.arange(5)[:, None] < r["nsaved"][None, :]
            assert np.array_equal(o["t_out"][:, part][rows], r["t_out"][rows])
            assert np.array_equal(np.swapaxes(o["u_out"][..., part], 1, 2)[rows], np.swapaxes(r["u_out"], 1, 2)[rows])
