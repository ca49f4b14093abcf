"""The tuner with the row executor among its candidates: timed once, beside the
lanes and tiles of the units (which it does not use), and the lanes that the
plan's transposed solves take are those of the units."""
import re

import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,layout", [(1, "col"), (12, "row"), (40, "col")])
def test_row_executor_is_one_candidate(dev, k, layout):
    Lp, Li, Lx = W.zipf_lower(20000, 1.8, 256, 5000, 61 + k)
    n = len(Lp) - 1
    plan = sa.Plan(*to_dev(Lp, Li, Lx))
    log = plan.tune(k=k, layout=layout).strip().splitlines()
    rows = [x for x in log[:-1] if "rows" in x]
    units = {}
    for x in log[:-1]:
        m = re.match(r"exec=2 lanes=(\d+) tile=(\d+) cap=0 ms=([\d.]+)", x)
        if m:
            assert (m[1], m[2]) not in units
            units[m[1], m[2]] = float(m[3])
    assert len(rows) == 1 and len(units) >= 3, log
    # a long row's lanes matter to the units: they are not one launch
    assert max(units.values()) > 1.2 * min(units.values()), log
    B = W.uniform(62, k, n * k).reshape(k, n)
    X = to_dev(np.ascontiguousarray(B.T) if layout == "row" else B[0] if k == 1 else B)
    plan.solve(X, layout=layout)
    plan.check()
    got = X.cpu().numpy()
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    assert rel_err(got.T if layout == "row" else got.reshape(k, n), want) <= 1e-12


def test_adjoint_keeps_the_lanes_of_the_units(dev):
    Lp, Li, Lx = W.zipf_lower(30000, 1.8, 256, 5000, 63)
    n = len(Lp) - 1
    plan = sa.Plan(*to_dev(Lp, Li, Lx))
    log = plan.tune(k=1).strip().splitlines()
    ms = {}
    for x in log[:-1]:
        m = re.match(r"exec=\d+ lanes=(\d+) .*ms=([\d.]+)", x)
        if m:
            ms[int(m[1])] = min(float(m[2]), ms.get(int(m[1]), 1e9))
    near = [g for g in ms if ms[g] <= 1.04 * min(ms.values())]
    assert "rows" in log[-1] and 2 not in near, log  # otherwise this shows nothing
    x, g = to_dev(W.uniform(64, 0, n)), to_dev(W.uniform(65, 0, n))
    auto, _ = plan.adjoint(x, g)
    plan.check()
    auto = auto.cpu().numpy()
    same = []
    for lanes in ms:
        plan.set_lanes(lanes)
        got, _ = plan.adjoint(x, g, executor="syncfree")
        plan.check()
        if np.array_equal(got.cpu().numpy(), auto):
            same.append(lanes)
    assert set(same) & set(near), (same, near, log)


def test_tuning_holds_no_outgrown_workspace(dev):
    """The graphs of the tuner are gone when it returns, so a wider solve
    replaces the workspace they held (58 MB for 12 columns) by its own (77 MB
    for 16) instead of keeping both."""
    import torch
    Lp, Li, Lx = W.zipf_lower(300000, 1.8, 64, 5000, 66)
    n = len(Lp) - 1
    plan = sa.Plan(*to_dev(Lp, Li, Lx))
    plan.set_lanes(2)
    plan.tune(k=12)
    X = to_dev(W.uniform(67, 0, n * 16).reshape(16, n))
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    plan.solve(X, executor="syncfree")
    plan.check()
    assert before - torch.cuda.mem_get_info()[0] < 40 << 20
