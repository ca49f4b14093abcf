"""Forward solves with several lanes per row (the row executor): row lengths
at every edge of its classes (entries per lane, slices per wavefront, rows a
workgroup shares, more than one round of them), every number of column lanes
and a remainder, both layouts and a padded leading dimension, FP64 and FP32,
and replays of a captured solve after the plan's workspace has grown."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 255,
           256, 257, 300, 513, 700]


def matrix(n=4000, seed=4):
    """Rows whose lengths cycle through LENGTHS (as far as columns allow),
    columns from the 900 rows before, dominant diagonals."""
    rng = np.random.default_rng(seed)
    Lp, Li, Lx = [0], [], []
    for i in range(n):
        lo = max(0, i - 900)
        c = min(LENGTHS[(7 * i) % len(LENGTHS)], i - lo)
        cols = np.sort(rng.choice(np.arange(lo, i), c, replace=False)) if c else np.zeros(0, int)
        v = rng.uniform(-1, 1, c)
        Li += [cols, [i]]
        Lx += [v, [1.0 + np.abs(v).sum()]]
        Lp.append(Lp[-1] + c + 1)
    return (np.array(Lp, np.int32), np.concatenate(Li).astype(np.int32), np.concatenate(Lx))


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("k,layout", [(1, "col"), (2, "col"), (8, "row"), (9, "col"), (16, "row"),
                                      (17, "col"), (32, "row"), (32, "col")])
def test_row_classes(dev, k, layout, dtype):
    import torch
    Lp, Li, Lx = matrix()
    n = len(Lp) - 1
    B = W.uniform(17, 0, n * k).reshape(k, n)
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    td = torch.float64 if dtype == "f64" else torch.float32
    dLp, dLi, dLx = to_dev(Lp, Li, Lx)
    plan = sa.Plan(dLp, dLi, dLx.to(td))
    plan.set_lanes(2)
    print(f"[rows] k={k} {layout} {dtype}", flush=True)
    X = to_dev(B if layout == "col" else np.ascontiguousarray(B.T)).to(td)
    plan.solve(X[0] if k == 1 else X, layout=layout, executor="syncfree")
    plan.check()
    got = X.cpu().numpy().astype(np.float64)
    # FP64: the bar of re-associated sums; FP32: 700 products of 2^-24 each on
    # dominant rows, over a chain that they damp
    assert rel_err(got if layout == "col" else got.T, want) <= (1e-12 if dtype == "f64" else 1e-4)


def test_captured_solve_keeps_its_workspace(dev):
    """A graph of a one-column solve, replayed after wider solves on the same
    plan replaced the workspace it was captured with."""
    Lp, Li, Lx = matrix()
    n = len(Lp) - 1
    B = W.uniform(18, 0, n * 32).reshape(32, n)
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    plan = sa.Plan(*to_dev(Lp, Li, Lx))
    plan.set_lanes(2)
    x = to_dev(B[0].copy())
    g = plan.graph(x, executor="syncfree")
    for c in range(3):
        X = to_dev(B.copy())
        plan.solve(X, executor="syncfree")
        plan.check()
        assert rel_err(X.cpu().numpy(), want) <= 1e-12
        x.copy_(to_dev(B[c].copy()))
        g.launch()
        plan.check()
        assert rel_err(x.cpu().numpy(), want[c]) <= 1e-12


def test_solve_captured_by_the_caller_keeps_its_workspace(dev):
    """The same with a capture the caller makes on the handle's stream."""
    import torch
    Lp, Li, Lx = matrix()
    n = len(Lp) - 1
    B = W.uniform(19, 0, n * 32).reshape(32, n)
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        plan = sa.Plan(*to_dev(Lp, Li, Lx), handle=sa.Handle(stream=stream))
        plan.set_lanes(2)
        x = to_dev(B[0].copy())
        plan.solve(x, executor="syncfree")  # builds the schedule
        plan.check()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            plan.solve(x, executor="syncfree")
        for c in range(3):
            X = to_dev(B.copy())
            plan.solve(X, executor="syncfree")
            plan.check()
            assert rel_err(X.cpu().numpy(), want) <= 1e-12
            x.copy_(to_dev(B[c].copy()))
            g.replay()
            plan.check()
            assert rel_err(x.cpu().numpy(), want[c]) <= 1e-12
