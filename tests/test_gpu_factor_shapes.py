"""Zero-fill factorizations over the shapes a level set can have: chains (one
row a level, whose packed structure takes no more than the rows need), and
levels of more units than the card has CUs, with packed and unpacked units; and
the units' tags, which in-place factorizations without room for a copy of A
wait for (with the marked protocol off, as here, all do)."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import bitwise_equal, to_dev
from tests.test_gpu_factor_units import banded
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
    for _ in range(2):  # the second one packs the units
        got, _ = plan.ic0(a, strict=False)
    assert before - torch.cuda.mem_get_info()[0] < 24 << 20
    want = oracle_factor(Lp, Li, A, "left")
    assert bitwise_equal(got.cpu().numpy(), want[0] if isinstance(want, tuple) else want)


def colours(g, stencil):
    """Lower triangle of a grid's Laplacian, rows ordered by colour: two levels
    (stencil 7, red and black) or eight (27)."""
    i = np.arange(g ** 3)
    x, y, z = i % g, i // g % g, i // (g * g)
    r, c = [], []
    for d in range(1, 14):
        dz, rem = divmod(d + 4, 9)
        dy, dx = rem // 3 - 1, rem % 3 - 1
        if stencil == 7 and abs(dx) + abs(dy) + abs(dz) != 1:
            continue
        ok = (x + dx >= 0) & (x + dx < g) & (y + dy >= 0) & (y + dy < g) & (z + dz < g)
        r.append(i[ok])
        c.append((i + dx + g * (dy + g * dz))[ok])
    r, c = np.concatenate(r), np.concatenate(c)
    colour = (x + y + z) % 2 if stencil == 7 else x % 2 + 2 * (y % 2) + 4 * (z % 2)
    new = np.empty(g ** 3, int)
    new[np.argsort(colour, kind="stable")] = i
    lo, hi = np.minimum(new[r], new[c]), np.maximum(new[r], new[c])
    rows, cols = np.concatenate([hi, i]), np.concatenate([lo, i])
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    Lp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=g ** 3))]).astype(np.int32)
    v = np.full(len(cols), -1.0)
    v[rows == cols] = stencil - 1 + 0.01
    return Lp, cols.astype(np.int32), v


@pytest.mark.parametrize("stencil,levels", [(7, 2), (27, 8)])
def test_levels_wider_than_the_card(dev, stencil, levels):
    Lp, Li, A = colours(48, stencil)
    plan = sa.Plan(*to_dev(Lp, Li, A))
    assert plan.levels == levels
    want = oracle_factor(Lp, Li, A, "left")
    want = want[0] if isinstance(want, tuple) else want
    a = to_dev(A)
    got, _ = plan.ic0(a, strict=False)
    assert bitwise_equal(got.cpu().numpy(), want)
    plan.ic0(a, out=a, strict=False)
    assert bitwise_equal(a.cpu().numpy(), want)


def test_wide_levels_use_the_whole_card(dev):
    """Red-black 96^3: 6,912 units a level, which one wavefront per CU takes 27
    rounds for; limiting the waves to that makes it slower."""
    import torch
    Lp, Li, A = colours(96, 7)
    a = to_dev(A)
    out = torch.empty_like(a)

    def best(waves):
        h = sa.Handle()
        h.set_max_waves(waves)
        plan = sa.Plan(*to_dev(Lp, Li, A), handle=h)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ms = []
        for _ in range(8):
            e[0].record()
            plan.ic0(a, out=out, strict=False)
            e[1].record()
            e[1].synchronize()
            ms.append(e[0].elapsed_time(e[1]))
        return min(ms)

    assert best(0) < 0.8 * best(256)


@pytest.mark.parametrize("tickets", [False, True])
@pytest.mark.parametrize("name", ["red_black", "colours", "chain", "band"])
def test_tagged_units_need_no_copy(dev, name, tickets):
    import torch
    Lp, Li, A = {"red_black": lambda: colours(40, 7), "colours": lambda: colours(24, 27),
                 "chain": lambda: chain(3000), "band": lambda: banded(3000, 6, 7, 3)}[name]()
    n = len(Lp) - 1
    h = sa.Handle(timeout_ms=2000)
    h.set_marks(False)
    h.set_tickets(tickets)
    print(f"[tagged] {name} n={n}", flush=True)
    plan = sa.Plan(*to_dev(Lp, Li, A), handle=h)
    for variant in ("left", "csr"):
        want = oracle_factor(Lp, Li, A, variant)
        want = want[0] if isinstance(want, tuple) else want
        a = to_dev(A)
        got, _ = plan.ic0(a, variant=variant, strict=False)
        assert bitwise_equal(got.cpu().numpy(), want)
        plan.ic0(a, variant=variant, out=a, strict=False)
        assert bitwise_equal(a.cpu().numpy(), want)


def test_tagged_factor_in_place_takes_no_workspace(dev):
    """3.5 M entries: a copy of A takes 28 MB."""
    import torch
    Lp, Li, A = colours(96, 7)
    h = sa.Handle()
    h.set_marks(False)
    plan = sa.Plan(*to_dev(Lp, Li, A), handle=h)
    a = to_dev(A)
    for _ in range(2):  # the second one packs the units
        want, _ = plan.ic0(a, strict=False)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    plan.ic0(a, out=a, strict=False)
    assert before - torch.cuda.mem_get_info()[0] < 8 << 20
    assert torch.equal(a, want)


def test_tagged_ilu0_with_the_marks_bits(dev):
    """An entry of A that holds the mark's NaN, and one that no update touches:
    no unit waits for it."""
    Ap, Ai, Ax, diags = W.grid3d_general(6, 2)
    p = int(diags[np.flatnonzero(np.diff(Ap) > 0)[0]]) + 1
    for bad in (False, True):
        A = Ax.copy()
        if bad:
            A.view(np.uint64)[p] = 0x7FF4D0D0CAFEF00D
        h = sa.Handle(timeout_ms=500)
        h.set_marks(False)
        plan = sa.Ilu0Plan(*to_dev(Ap, Ai, diags), handle=h)
        a = to_dev(A)
        plan.factor(a, out=a, strict=False)
        want, _ = oracle.spilu0_csr(Ap, Ai, A, diags)
        g, ok = a.cpu().numpy(), ~np.isnan(want)
        assert np.array_equal(np.isnan(g), ~ok) and bitwise_equal(g[ok], want[ok])


def test_first_factorization_packs_nothing(dev):
    """64^3: the packed units (13 MB) are built by the second factorization; the
    first gives the same factor without them."""
    import torch
    Lp, Li, A = W.lap3d_tril(64, 64, 64, 6.01, -1.0)
    warm = sa.Plan(*to_dev(Lp, Li, A))
    a = to_dev(A)
    out = torch.empty_like(a)
    warm.ic0(a, out=out)
    torch.cuda.synchronize()
    plan = sa.Plan(*to_dev(Lp, Li, A))
    taken = []
    for _ in range(3):
        before = torch.cuda.mem_get_info()[0]
        plan.ic0(a, out=out)
        taken.append(before - torch.cuda.mem_get_info()[0])
        want = out.clone() if len(taken) == 1 else want
        assert torch.equal(out, want)
    assert taken[1] > 8 << 20 and taken[2] < 2 << 20, taken
