"""Which executor an untuned sync-free solve with several lanes per row takes: the
row executor for long chains of narrow levels, the units for few wide levels
(their order of sums tells, as does a plan whose marks are off, which has the
units only), also where the caller records the solve."""
import time

import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev

pytestmark = pytest.mark.gpu


def two_levels(n, first, length, seed=8):
    """Rows past `first` read about `length` rows before it."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(first, n), length)
    key = np.unique(r * n + rng.integers(0, first, len(r)))
    r, c = np.concatenate([key // n, np.arange(n)]), np.concatenate([key % n, np.arange(n)])
    o = np.lexsort((c, r))
    r, c = r[o], c[o]
    Lp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    v = W.uniform(seed, 0, len(c))
    v[r == c] = 1.0 + length
    return Lp, c.astype(np.int32), v


CASES = {"wide": lambda: two_levels(400_000, 40_000, 16),
         "wide_long": lambda: two_levels(60_000, 6_000, 200),
         "narrow": lambda: W.zipf_lower(20_000, 1.8, 256, 5_000, 9)}


def solved(plan, B, layout):
    X = to_dev(np.ascontiguousarray(B.T) if layout == "row" else B[0] if len(B) == 1 else B)
    plan.solve(X, layout=layout, executor="syncfree")
    plan.check()
    got = X.cpu().numpy()
    return got.T if layout == "row" else got.reshape(B.shape)


@pytest.mark.parametrize("k,layout", [(1, "col"), (8, "row"), (16, "row"), (32, "row"),
                                      (32, "col")])
@pytest.mark.parametrize("name", sorted(CASES))
def test_executor_by_width(dev, name, k, layout):
    M = CASES[name]()
    n = len(M[0]) - 1
    B = W.uniform(81, k, n * k).reshape(k, n)
    units = sa.Handle()
    units.set_marks(False)
    print(f"[rows dispatch] {name} k={k} {layout}", flush=True)
    got = solved(sa.Plan(*to_dev(*M)), B, layout)
    same = np.array_equal(got, solved(sa.Plan(*to_dev(*M), handle=units), B, layout))
    assert same == (name != "narrow")
    assert rel_err(got, oracle.sptrsm_csr(*M, B)) <= 1e-12


@pytest.mark.parametrize("name", ["wide", "narrow"])
def test_recorded_after_another_width(dev, name):
    import torch
    M = CASES[name]()
    n = len(M[0]) - 1
    B = W.uniform(82, 0, n * 12).reshape(12, n)
    want = oracle.sptrsm_csr(*M, B)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for warm, k in ((1, 9), (2, 1), (9, 12), (12, 12)):
            plan = sa.Plan(*to_dev(*M), handle=sa.Handle(stream=stream))
            solved(plan, B[:warm], "row" if warm > 1 else "col")
            X = to_dev(np.ascontiguousarray(B[:k].T))
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=stream):
                plan.solve(X if k > 1 else X.view(-1), layout="row" if k > 1 else "col",
                           executor="syncfree")
            for c in range(3):
                X.copy_(to_dev(np.ascontiguousarray(np.roll(B, c, 0)[:k].T)))
                g.replay()
                plan.check()
                got = X.cpu().numpy().T
                assert rel_err(got, np.roll(want, c, 0)[:k]) <= 1e-12, (warm, k)


def test_wide_levels_are_not_slower_than_the_units(dev):
    """Two levels of long rows, 32 columns: 3.3 ms in tickets of one row, 0.6 on
    the units."""
    import torch
    M = to_dev(*two_levels(300_000, 30_000, 64))
    X = torch.zeros(300_000, 32, dtype=torch.float64, device="cuda")
    best = {}
    for marks in (True, False):
        h = sa.Handle()
        h.set_marks(marks)
        plan = sa.Plan(*M, handle=h)
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            plan.solve(X, layout="row", executor="syncfree")
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        best[marks] = min(t)
    assert best[True] < 1.5 * best[False], best
