"""The row executor's schedule, built on the device: levels around the 512 rows
a workgroup takes at a time, every class of rows in each of them, every number
of column lanes; and the first solve of a plan, which builds it."""
import time

import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 5, 9, 17, 33, 40, 65, 70, 129, 140, 257, 300]


def levels(sizes, seed=7):
    """Levels of `sizes` rows; a row reads one row of the level before and
    others of all before it, LENGTHS entries in turn."""
    rng = np.random.default_rng(seed)
    Lp, Li, Lx, n, before = [0], [], [], 0, 0
    for s, size in enumerate(sizes):
        for i in range(size):
            c = 0 if s == 0 else min(LENGTHS[(i + s) % len(LENGTHS)], n)
            cols = np.zeros(0, int)
            if c:
                cols = np.unique(np.append(rng.choice(n, c, replace=False),
                                           rng.integers(before, n)))
            v = rng.uniform(-1, 1, len(cols))
            Li += [cols, [n + i]]
            Lx += [v, [1.0 + np.abs(v).sum()]]
            Lp.append(Lp[-1] + len(cols) + 1)
        before, n = n, n + size
    return (np.array(Lp, np.int32), np.concatenate(Li).astype(np.int32), np.concatenate(Lx))


@pytest.mark.parametrize("k,layout", [(1, "col"), (5, "row"), (16, "col"), (32, "row")])
def test_levels_around_a_workgroup(dev, k, layout):
    Lp, Li, Lx = levels([400, 511, 1, 512, 513, 2, 1400, 64, 63])
    n = len(Lp) - 1
    plan = sa.Plan(*to_dev(Lp, Li, Lx))
    assert plan.levels == 9
    plan.set_lanes(2)
    B = W.uniform(71, k, n * k).reshape(k, n)
    X = to_dev(np.ascontiguousarray(B.T) if layout == "row" else B[0] if k == 1 else B)
    print(f"[rows schedule] k={k} {layout}", flush=True)
    plan.solve(X, layout=layout, executor="syncfree")
    plan.check()
    got = X.cpu().numpy()
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    assert rel_err(got.T if layout == "row" else got.reshape(k, n), want) <= 1e-12


def test_first_solve_builds_the_schedule_on_the_device(dev):
    """Zipf matrix of a million rows: a host pass over its rows and the copies
    take 6 to 12 ms, the kernels one."""
    import torch
    M = to_dev(*W.zipf_lower(1_000_000, 1.8, 256, 50000, 2))
    X = torch.zeros(1_000_000, 32, dtype=torch.float64, device="cuda")
    first = []
    for _ in range(3):
        plan = sa.Plan(*M)
        times = []
        for _ in range(4):
            torch.cuda.synchronize()
            t = time.perf_counter()
            plan.solve(X, layout="row", executor="syncfree")
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        first.append(times[0] - min(times))
    assert min(first) < 4e-3, first
