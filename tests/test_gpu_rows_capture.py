"""Row executor inside a capture the caller makes on the handle's stream: wider
blocks than any solved before (the schedule and the workspace grow while the
stream is recorded), a plan that has solved nothing yet (refused, the recording
stays whole), and that neither turns the executor off for later solves."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev
from tests.test_gpu_rows import matrix

pytestmark = pytest.mark.gpu


def solved(plan, B, layout="col"):
    X = to_dev(B.copy())
    plan.solve(X, layout=layout, executor="syncfree")
    plan.check()
    return X.cpu().numpy()


@pytest.mark.parametrize("warm", [1, 2, 9])
@pytest.mark.parametrize("k,layout", [(2, "row"), (8, "row"), (12, "row"), (12, "col"),
                                      (32, "row"), (32, "col")])
def test_block_captured_after_another_width(dev, warm, k, layout):
    import torch
    Lp, Li, Lx = matrix(1500)
    n = len(Lp) - 1
    B = W.uniform(51, 0, n * 32).reshape(32, n)
    want = oracle.sptrsm_csr(Lp, Li, Lx, B)
    shape = (lambda A: np.ascontiguousarray(A.T)) if layout == "row" else (lambda A: A)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        plan = sa.Plan(*to_dev(Lp, Li, Lx), handle=sa.Handle(stream=stream))
        plan.set_lanes(32)
        solved(plan, B[:warm] if warm > 1 else B[0])
        X = to_dev(shape(B[:k]).copy())
        print(f"[rows capture] warm={warm} k={k} {layout}", flush=True)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            plan.solve(X, layout=layout, executor="syncfree")
        other = sa.Plan(*to_dev(Lp, Li, Lx), handle=sa.Handle(stream=stream))
        other.set_lanes(32)
        for c in range(3):
            part = np.roll(B, c, axis=0)[:k]
            X.copy_(to_dev(shape(part).copy()))
            g.replay()
            plan.check()
            assert rel_err(shape(X.cpu().numpy()), np.roll(want, c, axis=0)[:k]) <= 1e-12
            # later solves still take the row executor: its order of sums
            for w in (B[0], B[:7], B):
                assert np.array_equal(solved(plan, w), solved(other, w))


def test_first_solve_inside_a_capture(dev):
    import torch
    Lp, Li, Lx = matrix(1500)
    n = len(Lp) - 1
    b = W.uniform(52, 0, n)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        plan = sa.Plan(*to_dev(Lp, Li, Lx), handle=sa.Handle(stream=stream))
        plan.set_lanes(2)
        x, y, X = to_dev(b.copy()), to_dev(b.copy()), to_dev(np.tile(b, (3, 1)))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            for v in (x, X):
                with pytest.raises(sa.SymAmdError, match="not prepared before capture"):
                    plan.solve(v, executor="syncfree")
            y.mul_(2.0)
        g.replay()
        assert np.array_equal(y.cpu().numpy(), 2.0 * b)
        other = sa.Plan(*to_dev(Lp, Li, Lx), handle=sa.Handle(stream=stream))
        other.set_lanes(2)
        got = solved(plan, b)
        assert np.array_equal(got, solved(other, b))
        assert rel_err(got, oracle.sptrsv_csr(Lp, Li, Lx, b)) <= 1e-12
