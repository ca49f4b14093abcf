"""Supernodal solves where the workgroup kernels change path: widths around
one wavefront's 64 columns and the column blocks of 8, rows below around the
chunks of 64 and 128, row lists of even and very uneven lengths, every column
tile width, and dividends and diagonals outside the range of the quotients
formed from reciprocals.  Bit-identical to the oracle, both directions."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import bitwise_equal, to_dev

pytestmark = pytest.mark.gpu

WIDTHS = [1, 7, 8, 9, 16, 33, 63, 64, 65, 72, 2, 100, 128, 129, 3, 200, 64, 321, 5, 70]
BELOW = [200, 0, 1, 63, 64, 65, 127, 128, 129, 193, 320, 64, 200, 7, 500, 129, 300, 60, 70, 0]


def build(seed, diag_scale=None):
    """Supernodes of WIDTHS columns with up to BELOW rows below (fewer where
    fewer columns follow), in the generator's storage; the last supernode's
    first row is in every list, so its lists are uneven."""
    rng = np.random.default_rng(seed)
    sup = np.concatenate([[0], np.cumsum(WIDTHS)]).astype(np.int32)
    n, nrows, Lp, Li, Lx = int(sup[-1]), [], [0], [], []
    for i, w in enumerate(WIDTHS):
        e = int(sup[i + 1])
        c = min(BELOW[i], n - e)
        rows = rng.choice(np.arange(e, n), c, replace=False) if c else np.zeros(0, int)
        if c and int(sup[-2]) not in rows and e <= int(sup[-2]):
            rows[0] = int(sup[-2])
        rows = np.concatenate([np.arange(sup[i], e), np.sort(rows)])
        blk = rng.uniform(-1, 1, (w, len(rows))) / len(rows)
        d = 1.0 + rng.uniform(0, 1, w)
        if diag_scale is not None:
            d *= diag_scale[rng.integers(0, len(diag_scale), w)]
        for j in range(w):
            blk[j, :j] = np.nan
            blk[j, j] = d[j]
        nrows.append(len(rows))
        Li.append(np.tile(rows, w))
        Lx.append(blk.ravel())
        Lp.append(Lp[-1] + blk.size)
    return (sup, np.array(nrows, np.int32), np.array(Lp, np.int32),
            np.concatenate(Li).astype(np.int32), np.concatenate(Lx))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 15, 16, 19])
def test_units_and_column_tiles(dev, k):
    sup, nrows, Lp, Li, Lx = build(k)
    n = int(sup[-1])
    B = W.uniform(31, k, k * n).reshape(k, n)
    plan = sa.SupernodalPlan(sup, nrows, Lp, Li)
    dLx = to_dev(Lx)
    print(f"[sn units] k={k} n={n}", flush=True)
    for solve, ref in ((plan.solve, oracle.sptrsv_csc_block),
                       (plan.solve_transposed, oracle.sptrsv_csc_block_t)):
        X = to_dev(B.copy())
        solve(dLx, X if k > 1 else X[0])
        plan.check()
        got = X.cpu().numpy()
        for c in range(k):
            assert bitwise_equal(got[c], ref(sup, nrows, Lp, Li, Lx, B[c])), (solve, c)


@pytest.mark.parametrize("kind", ["zeros", "tiny", "huge", "diagonals"])
def test_quotients_outside_the_reciprocal_range(dev, kind):
    scale = np.array([1.0] * 200 + [2.0 ** -101] + [2.0 ** 110] * 9) if kind == "diagonals" else None
    sup, nrows, Lp, Li, Lx = build(7, scale)
    n, k = int(sup[-1]), 5
    B = W.uniform(33, 0, k * n).reshape(k, n)
    if kind == "zeros":
        B[:, ::3] = 0.0
        B[:, 1::3] = -0.0
        B[0] = -0.0
    elif kind != "diagonals":
        B *= 1e-300 if kind == "tiny" else 1e290
        B[:, ::5] *= 1e-10
    plan = sa.SupernodalPlan(sup, nrows, Lp, Li)
    dLx = to_dev(Lx)
    for solve, ref in ((plan.solve, oracle.sptrsv_csc_block),
                       (plan.solve_transposed, oracle.sptrsv_csc_block_t)):
        with np.errstate(all="ignore"):
            want = [ref(sup, nrows, Lp, Li, Lx, b) for b in B]
        X = to_dev(B.copy())
        solve(dLx, X)
        x1 = to_dev(B[0].copy())
        solve(dLx, x1)
        plan.check()
        got = X.cpu().numpy()
        for c in range(k):
            same = (got[c] == want[c]) & (np.signbit(got[c]) == np.signbit(want[c]))
            assert (same | (np.isnan(got[c]) & np.isnan(want[c]))).all(), (kind, solve, c)
        g1 = x1.cpu().numpy()
        assert ((g1 == want[0]) | (np.isnan(g1) & np.isnan(want[0]))).all()


@pytest.mark.parametrize("k", [1, 2, 5, 17])
def test_long_lists_gathered_ahead_of_wide_tops(dev, k):
    """A tree whose wide tops subtract 15 to 113 temporaries per row: lists
    gathered by the top's own waves, by workgroups in one round and in
    several, at every column tile."""
    sup, nrows, Lp, Li, Lx = W.bcsc_tree(11, 8, 150, 2.0, 4)
    n, w = int(sup[-1]), np.diff(sup)
    cnt = np.zeros(n, int)
    for i in range(len(w)):
        cnt[Li[Lp[i] + w[i]:Lp[i] + nrows[i]]] += 1
    longest = np.maximum.reduceat(cnt, sup[:-1])[w > 64]
    assert longest.min() <= 48 and longest.max() > 64 and ((longest > 48) & (longest <= 64)).any()
    B = W.uniform(35, 0, k * n).reshape(k, n)
    plan = sa.SupernodalPlan(sup, nrows, Lp, Li)
    X = to_dev(B.copy())
    print(f"[sn lists] k={k} n={n}", flush=True)
    plan.solve(to_dev(Lx), X if k > 1 else X[0])
    plan.check()
    got = X.cpu().numpy()
    for c in range(k):
        assert bitwise_equal(got[c], oracle.sptrsv_csc_block(sup, nrows, Lp, Li, Lx, B[c])), c


@pytest.mark.parametrize("k", [16, 33])
def test_chains_of_narrow_supernodes(dev, k):
    """One supernode after another: tiles of one column run side by side, and a
    block takes no longer than its columns' chain (in tiles of four, 1.9 times
    as long as one column)."""
    import torch
    m, w = 300, 40
    sup = (np.arange(m + 1) * w).astype(np.int32)
    n = m * w
    nrows = np.full(m, 2 * w, np.int32)
    nrows[-1] = w
    Lp = np.concatenate([[0], np.cumsum(nrows * w)]).astype(np.int32)
    Li = np.concatenate([np.tile(np.arange(i * w, i * w + nrows[i]), w) for i in range(m)])
    rng = np.random.default_rng(5)
    Lx = rng.uniform(-1, 1, len(Li)) / (2 * w)
    for i in range(m):
        Lx[Lp[i] + np.arange(w) * (nrows[i] + 1)] = 1.5
    plan = sa.SupernodalPlan(sup, nrows, Lp, Li.astype(np.int32))
    dLx = to_dev(Lx)
    B = W.uniform(36, 0, k * n).reshape(k, n)

    def best(X):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ms = []
        for _ in range(6):
            X.zero_()
            X.add_(1.0)
            e[0].record()
            plan.solve(dLx, X)
            e[1].record()
            e[1].synchronize()
            ms.append(e[0].elapsed_time(e[1]))
        return min(ms)

    X = to_dev(B.copy())
    plan.solve(dLx, X)
    plan.check()
    got = X.cpu().numpy()
    for c in range(k):
        assert bitwise_equal(got[c], oracle.sptrsv_csc_block(sup, nrows, Lp, Li, Lx, B[c])), c
    assert best(X) < 1.5 * best(X[0])
