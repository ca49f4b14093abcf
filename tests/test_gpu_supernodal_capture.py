"""Supernodal solves recorded by the caller: the temporaries and tags that the
graph reads outlive later, wider solves on the same plan; a wider solve is
refused while recording and leaves the recording whole; and a block whose
temporaries fit no GPU leaves nothing behind for the next solve."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import bitwise_equal, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direction", ["forward", "transposed"])
def test_solve_captured_by_the_caller_keeps_its_temporaries(dev, direction):
    import torch
    sup, nrows, Lp, Li, Lx = W.bcsc_tree(7, 8, 90, 2.0, 5)
    n = int(sup[-1])
    B = W.uniform(41, 0, n * 9).reshape(9, n)
    ref = oracle.sptrsv_csc_block if direction == "forward" else oracle.sptrsv_csc_block_t
    want = [ref(sup, nrows, Lp, Li, Lx, b) for b in B]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        plan = sa.SupernodalPlan(sup, nrows, Lp, Li, handle=sa.Handle(stream=stream))
        solve = plan.solve if direction == "forward" else plan.solve_transposed
        dLx = to_dev(Lx)
        x, X = to_dev(B[0].copy()), to_dev(B.copy())
        solve(dLx, x)
        plan.check()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            with pytest.raises(sa.SymAmdError, match="not prepared before capture"):
                solve(dLx, X)
            solve(dLx, x)
        for c, k in enumerate((3, 9, 5)):  # 3 and 9 replace the temporaries
            X = to_dev(B[:k].copy())
            solve(dLx, X)
            filler = torch.full((1 << 20,), float("nan"), dtype=torch.float64, device="cuda")
            x.copy_(to_dev(B[c].copy()))
            g.replay()
            plan.check()
            assert bitwise_equal(x.cpu().numpy(), want[c])
            for i in range(k):
                assert bitwise_equal(X[i].cpu().numpy(), want[i])
            del filler


def test_solve_after_a_block_that_did_not_fit(dev):
    """A dense triangle of 2000 one-column supernodes has 2 M temporaries per
    column: 20000 columns of them (320 GB) fit no GPU."""
    import torch
    n, k = 2000, 20000
    sup, nrows = np.arange(n + 1, dtype=np.int32), np.arange(n, 0, -1, dtype=np.int32)
    Lp = np.concatenate([[0], np.cumsum(nrows)]).astype(np.int32)
    Li = np.concatenate([np.arange(i, n) for i in range(n)]).astype(np.int32)
    Lx = W.uniform(42, 0, len(Li)) / n
    Lx[Lp[:-1]] = 1.0 + Lx[Lp[:-1]]
    b = W.uniform(43, 0, n)
    plan = sa.SupernodalPlan(sup, nrows, Lp, Li)
    dLx = to_dev(Lx)
    with pytest.raises(sa.SymAmdError, match="temporaries"):
        plan.solve(dLx, torch.zeros(k, n, dtype=torch.float64, device="cuda"))
    x = to_dev(b.copy())
    plan.solve(dLx, x)
    plan.check()
    assert bitwise_equal(x.cpu().numpy(), oracle.sptrsv_csc_block(sup, nrows, Lp, Li, Lx, b))
