"""Zero-fill factorizations over the shapes a level set can have: chains (one
row a level, whose packed structure takes no more than the rows need)."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from tests.helpers import bitwise_equal, to_dev
from tests.test_gpu_ic0 import oracle_factor

pytestmark = pytest.mark.gpu


def chain(n):
    """Lower triangle of a tridiagonal SPD matrix."""
    Lp = np.concatenate([[0], 2 * np.arange(1, n + 1) - 1]).astype(np.int32)
    Li = np.repeat(np.arange(n), 2)[1:].astype(np.int32)
    Li[1::2] -= 1
    Lx = np.where(np.arange(2 * n - 1) % 2 == 0, 2.01, -1.0)
    return Lp, Li, Lx


def test_chain_takes_the_memory_of_its_rows(dev):
    """40,000 levels of one row: 28 bytes a row packed (and tags, dependencies
    and pairs, some 80 more), not the 1.8 KB of a full unit."""
    import torch
    Lp, Li, A = chain(40000)
    assert (Li[Lp[1:] - 1] == np.arange(40000)).all()
    plan = sa.Plan(*to_dev(Lp, Li, A))
    a = to_dev(A)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    got, _ = plan.ic0(a, strict=False)
    assert before - torch.cuda.mem_get_info()[0] < 24 << 20
    want = oracle_factor(Lp, Li, A, "left")
    assert bitwise_equal(got.cpu().numpy(), want[0] if isinstance(want, tuple) else want)
