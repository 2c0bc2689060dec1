"""Bursts of requests through the server's staging: more input than the pinned
ring holds (8 MiB), requests just below and above the size that goes through it
(1 MiB), more results than one staging buffer (4 MiB), ragged and single sizes;
with slots for all of them and with few, so that ranges are given back out of
step.  Every result equals the batch engine's, bit for bit."""
import numpy as np
import pytest

import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1 << 19, 40000])
def test_burst_equals_batch_engine(slots):
    sizes = [1, 255, 16383, 256, 257, 16384, 16385, 63] + 12 * [16000, 7] + [20000, 1]
    N = sum(sizes)
    rng = np.random.Generator(np.random.PCG64(77))
    u0 = rng.uniform(-1.0, 1.0, (3, N))
    p = np.stack([rng.uniform(8.0, 12.0, N), rng.uniform(0.0, 28.0, N), np.full(N, 8.0 / 3.0)])
    t0, tf = np.zeros(N), rng.uniform(0.2, 1.0, N)
    kw = dict(reltol=1e-6, abstol=1e-6)
    print(f"[case] serving burst, {len(sizes)} requests, {slots} slots", flush=True)
    ref = odemi.solve_arrays(P.LORENZ, odemi.Tsit5(), u0, p, t0, tf, **kw)
    ends = np.cumsum(sizes)
    with odemi.EnsembleServer(P.LORENZ, 3, 3, odemi.Tsit5(), max_slots=slots, **kw) as srv:
        for again in range(2):
            sent = [srv.submit(u0[:, e - k:e], p[:, e - k:e], t0[e - k:e], tf[e - k:e]) for k, e in zip(sizes, ends)]
            for r in sent:
                assert r.wait(timeout=60)
            for r, k, e in zip(sent, sizes, ends):
                assert np.array_equal(r.u_final, ref["u_final"][:, e - k:e])
                assert np.array_equal(r.retcode, ref["retcode"][e - k:e])
                assert np.array_equal(r.stats, ref["stats"][:, e - k:e])
