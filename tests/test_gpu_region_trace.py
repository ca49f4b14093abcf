"""Clock stamps of region tasks: taken, first halo loaded, rows stored."""
import numpy as np
import pytest

import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mw", [True, False])
def test_last_stamp_follows_the_stores(dev, mw):
    """One region of 900 rows, each reading the one before: 900 steps of at
    least 50 ns (5 ticks) lie between its first halo (empty) and its last
    store."""
    import torch
    Lp, Li, Lx = W.lap2d_tril(1, 900)
    h = sa.Handle()
    h.set_region_mw(mw)
    h.set_region_cap(1024)
    plan = sa.Plan(*to_dev(Lp, Li, Lx), handle=h)
    assert plan.region_schedule(1) == (1024, 1)
    x = to_dev(W.uniform(3, 0, 900))
    plan.solve(x, executor="regions")
    stamps = torch.zeros(3, dtype=torch.int64, device="cuda")
    h.set_trace(stamps)
    plan.solve(x, executor="regions")
    plan.check()
    h.set_trace(None)
    t = stamps.cpu().numpy()
    assert 0 < t[0] <= t[1] and t[2] - t[1] > 900 * 5, np.diff(t)
