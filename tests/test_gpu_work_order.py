"""The longest-first order is left out only where every lane of the launch takes
at most one trajectory: with a launch of fewer lanes than trajectories
(explicit block and blocks_per_cu) sort_by_cost is followed.  The order shows in
the launch count (its queue-order records are unpacked by a launch of their
own); results are the same in any order."""
import numpy as np
import pytest

import odemi
from odemi import problems as P

pytestmark = pytest.mark.gpu


def test_order_follows_the_launch_geometry():
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    N = 200 * cus
    d = P.lorenz_large(N=N)
    args = (P.LORENZ, odemi.Tsit5(), d["u0"], d["p"], d["t0"], d["tf"])
    kw = dict(reltol=d["reltol"], abstol=d["abstol"])
    print(f"[case] work order N={N}", flush=True)
    ref = odemi.solve_arrays(*args, **kw)                                     # a lane each: prep, solve
    few = odemi.solve_arrays(*args, odemi.EnsembleMI355X(block=64, blocks_per_cu=1), **kw)
    off = odemi.solve_arrays(*args, odemi.EnsembleMI355X(block=64, blocks_per_cu=1, sort_by_cost=False), **kw)
    assert (ref["launches"], few["launches"], off["launches"]) == (2, 3, 2)
    for o in (few, off):
        assert np.array_equal(o["u_final"], ref["u_final"]) and np.array_equal(o["stats"], ref["stats"])
