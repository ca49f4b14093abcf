"""Region schedules of grids whose sides are no powers of two: the regions are
boxes (their number and the longest chain of regions say so), and the CPU
emulation of the region kernel reproduces the serial solve bit for bit, forward
and transposed.  Patterns that only look like a grid keep the general
clustering and solve the same way."""
import numpy as np
import pytest

import oracle
from sympiler_amd import workloads as W
from tests.helpers import bitwise_equal
from tests.region_emul import _records, emulate, schedule_host


def depth(sch):
    d = []
    for r in _records(sch):
        d.append(1 + max((d[int(w) & ((1 << 26) - 1)] for w in r["deps"]), default=0))
    return max(d)


def check(Lp, Li, Lx, cap, band=4):
    n = len(Lp) - 1
    b = W.uniform(9, 0, n)
    sch = schedule_host(Lp, Li, Lx, cap, band)
    assert bitwise_equal(emulate(sch, n, b), oracle.sptrsv_csr(Lp, Li, Lx, b))
    sch_t = schedule_host(Lp, Li, Lx, cap, band, transposed=True)
    Cp, Ci, Cx, _ = oracle.csr_to_csc(Lp, Li, Lx)
    assert bitwise_equal(emulate(sch_t, n, b), oracle.ltsolve(Cp, Ci, Cx, b))
    return sch, sch_t


@pytest.mark.parametrize("grid,cap,boxes,chain", [((13, 11, 17), 512, 2 * 2 * 2, 4),
                                                  ((19, 9, 7), 64, None, None),
                                                  ((3, 29, 5), 128, None, None),
                                                  ((2, 2, 41), 32, None, None)])
def test_odd_grids_are_cut_into_boxes(grid, cap, boxes, chain):
    Lp, Li, A = W.lap3d_tril(*grid, 6.01, -1.0)
    for sch in check(Lp, Li, A, cap):
        if boxes:
            assert (sch["R"], depth(sch)) == (boxes, chain)


@pytest.mark.parametrize("nx,ny,cap", [(37, 23, 128), (101, 7, 512), (2, 90, 64)])
def test_planes(nx, ny, cap):
    check(*W.lap2d_tril(nx, ny), cap)


def test_uneven_batch_of_planes():
    w = W.config4(count=9, lo=5, hi=31, seed=11)
    check(w.Lp, w.meta["global_Li"], w.Lx, 128)


def without(Lp, Li, Lx, keep):
    rows = np.repeat(np.arange(len(Lp) - 1), np.diff(Lp))[keep]
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=len(Lp) - 1))])
    return ptr.astype(np.int32), Li[keep], Lx[keep]


@pytest.mark.parametrize("kind", ["holes", "wrapped", "diagonal", "ragged", "line", "mixed"])
def test_patterns_beside_the_grid(kind):
    """holes: entries missing from a grid; wrapped: a line's end joined to the
    next line; diagonal: a fourth offset; ragged: rows that fill no last
    plane; line: one offset; mixed: a grid followed by a line."""
    Lp, Li, Lx = W.lap3d_tril(11, 9, 7, 6.01, -1.0)
    n = len(Lp) - 1
    if kind == "holes":
        rng = np.random.default_rng(3)
        keep = rng.random(len(Li)) < 0.7
        keep[Lp[1:] - 1] = True
        Lp, Li, Lx = without(Lp, Li, Lx, keep)
    elif kind == "ragged":
        n -= 40
        Lp, Li, Lx = Lp[:n + 1], Li[:Lp[n]], Lx[:Lp[n]]
    elif kind == "line":
        Lp, Li, Lx = W.lap2d_tril(1, 700)
    elif kind == "mixed":
        Mp, Mi, Mx = W.lap2d_tril(1, 300)
        Lp, Li, Lx = (np.concatenate([Lp, Lp[-1] + Mp[1:]]), np.concatenate([Li, Mi + n]),
                      np.concatenate([Lx, Mx]))
    else:
        rows = [list(zip(Li[Lp[i]:Lp[i + 1]], Lx[Lp[i]:Lp[i + 1]])) for i in range(n)]
        for i in range(12, n):
            if kind == "wrapped" and i % 11 == 0:
                rows[i].append((i - 1, -0.5))
            elif kind == "diagonal" and i % 11:
                rows[i].append((i - 12, -0.5))
        rows = [sorted(dict(r).items()) for r in rows]
        Lp = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
        Li = np.array([c for r in rows for c, _ in r])
        Lx = np.array([v for r in rows for _, v in r])
    check(Lp.astype(np.int32), Li.astype(np.int32), Lx.astype(np.float64), 128)


@pytest.mark.parametrize("nx,ny,boxes,chain", [(1500, 500, (47, 16), 62), (700, 700, (22, 22), 43),
                                               (100, 100, (3, 4), 6)])
def test_boxes_of_planes_for_one_column(nx, ny, boxes, chain):
    """Long chains take boxes as square as they come (1500 x 500 was cut into
    36 x 21 of 42 x 24 points, 0.87 ms against 0.77), short ones the fewest."""
    sch = schedule_host(*W.lap2d_tril(nx, ny), 1024, 4)
    assert sch["R"] == boxes[0] * boxes[1] and depth(sch) == chain


@pytest.mark.parametrize("grid,regions", [((37, 37), 3), ((24, 24), 2), ((10, 10, 10), 2),
                                          ((42, 42), 4), ((9, 13, 17), 8)])
def test_few_boxes_against_the_matching(grid, regions):
    """Small grids and blocks of right-hand sides: the matching's regions where
    their chain is clearly shorter (37 x 37 in 3 regions instead of 4 boxes, 24 x
    24 and 10^3 in uneven ones), boxes elsewhere."""
    M = W.lap2d_tril(*grid) if len(grid) == 2 else W.lap3d_tril(*grid, 6.01, -1.0)
    sch, _ = check(*M, 512, 255)
    rows = sorted(len(r["rows"]) for r in _records(sch))
    assert sch["R"] == regions
    if regions == 2:
        levels = sum(len(r["slices"]) - 1 for r in _records(sch))
        assert rows[0] < rows[1] or levels < 2 * 22, (rows, levels)  # boxes: 22 each


@pytest.mark.parametrize("grid,cap", [((13, 11, 17), 512), ((19, 9, 7), 64), ((3, 29, 5), 128),
                                      ((2, 2, 41), 32), ((37, 23, 1), 128), ((101, 7, 1), 512),
                                      ((2, 90, 1), 64)])
@pytest.mark.parametrize("transposed", [False, True])
def test_every_region_is_a_box(grid, cap, transposed):
    nx, ny, nz = grid
    M = W.lap3d_tril(*grid, 6.01, -1.0) if nz > 1 else W.lap2d_tril(nx, ny)
    sch = schedule_host(*M, cap, 4, transposed=transposed)
    seen = 0
    for r in _records(sch):
        i = np.asarray(r["rows"], np.int64)
        sides = [len(np.unique(c)) for c in (i % nx, i // nx % ny, i // (nx * ny))]
        spans = [np.ptp(c) + 1 for c in (i % nx, i // nx % ny, i // (nx * ny))]
        assert sides == spans and np.prod(sides) == len(i) <= cap
        seen += len(i)
    assert seen == nx * ny * nz
