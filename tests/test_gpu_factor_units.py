"""Zero-fill factorizations whose units take both routes of the kernel: units
packed (every row at most 8 entries and 8 update pairs), units read from the
caller's arrays because one row has 9 entries or more pairs, a last unit that
is not full, in place and out of place, and an entry of A that holds the bit
pattern the factor's storage starts with.  Bit-identical to the oracle."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import bitwise_equal, to_dev
from tests.test_gpu_ic0 import oracle_factor

pytestmark = pytest.mark.gpu


def banded(n, half, every, seed):
    """SPD lower triangle: every row holds its `half` left neighbours, each
    `every`-th row two more, so rows of a unit straddle the packed limits."""
    rng = np.random.default_rng(seed)
    Lp, Li, Lx = [0], [], []
    for i in range(n):
        w = half + (2 if every and i % every == 0 else 0)
        cols = np.unique(np.concatenate([np.arange(max(0, i - w), i), [i]]))
        v = rng.uniform(-1, 0, len(cols))
        v[-1] = 40.0
        Li.append(cols)
        Lx.append(v)
        Lp.append(Lp[-1] + len(cols))
    return (np.array(Lp, np.int32), np.concatenate(Li).astype(np.int32), np.concatenate(Lx))


CASES = {"grid": lambda: W.lap3d_tril(9, 7, 11, 6.01, -1.0),
         "two_blocks": lambda: two_blocks(),
         "band3": lambda: banded(300, 3, 0, 1),
         "band4": lambda: banded(300, 4, 0, 2),
         "band6_mixed": lambda: banded(400, 6, 7, 3)}


def two_blocks():
    """A grid beside a band: units of one level hold packed and unpacked rows."""
    Ap, Ai, Ax = W.lap3d_tril(8, 8, 8, 6.01, -1.0)
    Bp, Bi, Bx = banded(200, 9, 3, 4)
    return (np.concatenate([Ap, Ap[-1] + Bp[1:]]), np.concatenate([Ai, Bi + len(Ap) - 1]),
            np.concatenate([Ax, Bx]))


@pytest.mark.parametrize("variant", ["left", "csr"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_ic0_units(dev, name, variant):
    Lp, Li, A = CASES[name]()
    plan = sa.Plan(*to_dev(Lp, Li, A))
    for s in (1.0, 1.5):  # the second factorization reuses the packed units
        want = oracle_factor(Lp, Li, A * s, variant)
        want = want[0] if isinstance(want, tuple) else want
        a = to_dev(A * s)
        got, _ = plan.ic0(a, variant=variant, strict=False)
        assert bitwise_equal(got.cpu().numpy(), want)
        same, _ = plan.ic0(a, variant=variant, out=a, strict=False)
        assert same is a and bitwise_equal(a.cpu().numpy(), want)


@pytest.mark.parametrize("name", sorted(CASES))
def test_ilu0_units(dev, name):
    Lp, Li, A = CASES[name]()
    n = len(Lp) - 1
    # the symmetric pattern, unsymmetric values
    rows = np.repeat(np.arange(n), np.diff(Lp))
    off = Li < rows
    r = np.concatenate([rows, Li[off]])
    c = np.concatenate([Li, rows[off]])
    v = np.concatenate([A, 0.5 * A[off]])
    order = np.lexsort((c, r))
    r, Ai, Ax = r[order], c[order].astype(np.int32), v[order]
    Ap = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    diags = np.flatnonzero(r == Ai).astype(np.int32)
    dAp, dAi, dd = to_dev(Ap, Ai, diags)
    plan = sa.Ilu0Plan(dAp, dAi, dd)
    for s in (1.0, 1.5):
        want, _ = oracle.spilu0_csr(Ap, Ai, Ax * s, diags)
        a = to_dev(Ax * s)
        assert bitwise_equal(plan.factor(a).cpu().numpy(), want)
        plan.factor(a, out=a)
        assert bitwise_equal(a.cpu().numpy(), want)


def test_ilu0_input_with_the_marks_bits(dev):
    """An upper entry of A that no update touches is copied; one holding the
    mark's NaN comes out as a NaN and nothing waits for it."""
    Ap, Ai, Ax, diags = W.grid3d_general(6, 2)
    i = int(np.flatnonzero(np.diff(Ap) > 0)[0])
    p = int(diags[i]) + 1
    Ax = Ax.copy()
    Ax.view(np.uint64)[p] = 0x7FF4D0D0CAFEF00D
    plan = sa.Ilu0Plan(*to_dev(Ap, Ai, diags), handle=sa.Handle(timeout_ms=500))
    got, _ = plan.factor(to_dev(Ax), strict=False)
    want, _ = oracle.spilu0_csr(Ap, Ai, Ax, diags)
    g = got.cpu().numpy()
    assert np.isnan(g[p]) and np.array_equal(np.isnan(g), np.isnan(want))
    ok = ~np.isnan(want)
    assert bitwise_equal(g[ok], want[ok])
