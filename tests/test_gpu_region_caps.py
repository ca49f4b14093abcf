"""Region cap of untuned single right-hand sides on very large plans: 384 rows
for many planes side by side, 1024 for one grid or plane, whose chain of
regions sets the time."""
import numpy as np
import pytest

import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,cap", [("planes", 384), ("plane", 1024), ("grid", 1024),
                                      ("few_planes", 1024)])
def test_cap_of_large_plans(dev, name, cap):
    if name == "plane":
        M = W.lap2d_tril(2100, 2100)
    elif name == "grid":
        M = W.lap3d_tril(165, 165, 165, 6.01, -1.0)
    else:
        w = W.config4(count=512) if name == "planes" else W.config4(count=16, lo=400, hi=700)
        M = (w.Lp, w.meta["global_Li"], w.Lx)
    assert len(M[0]) - 1 > 16 * 1024 * 256
    plan = sa.Plan(*to_dev(*M))
    print(f"[caps] {name} n={len(M[0]) - 1}", flush=True)
    assert plan.region_schedule(1)[0] == cap
