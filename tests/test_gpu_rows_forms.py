"""Row executor: the forms a right-hand side comes in.  Padded leading
dimensions in both layouts (the padding stays as it was), column-major blocks
solved in place, more columns than one tile, and infinities and NaN beside
rows that read nothing."""
import numpy as np
import pytest

import oracle
import sympiler_amd as sa
from sympiler_amd import workloads as W
from tests.helpers import rel_err, to_dev
from tests.test_gpu_rows import matrix

pytestmark = pytest.mark.gpu


def rows_plan(M, **kw):
    plan = sa.Plan(*to_dev(*M), **kw)
    plan.set_lanes(2)
    return plan


@pytest.mark.parametrize("direct", [False, True])
@pytest.mark.parametrize("k", [2, 13, 32])
@pytest.mark.parametrize("layout", ["col", "row"])
def test_padded_leading_dimension(dev, layout, k, direct):
    import torch
    M = matrix(2000)
    n = len(M[0]) - 1
    B = W.uniform(91, k, n * k).reshape(k, n)
    h = sa.Handle()
    h.set_colmajor_direct(direct)
    plan = rows_plan(M, handle=h)
    shape = (k, n + 5) if layout == "col" else (n, k + 3)
    full = torch.full(shape, 7.25, dtype=torch.float64, device="cuda")
    X = full[:, :n] if layout == "col" else full[:, :k]
    X.copy_(to_dev(B if layout == "col" else np.ascontiguousarray(B.T)))
    print(f"[rows forms] {layout} k={k} direct={direct}", flush=True)
    # the Python entry takes contiguous blocks; the C one a leading dimension
    sa._check(sa.lib().symamd_solve(h._h, plan._p, sa._ptr(full), k, full.stride(0),
                                    sa.COL_MAJOR if layout == "col" else sa.ROW_MAJOR,
                                    sa.EXEC["syncfree"]))
    plan.check()
    got = full.cpu().numpy()
    inner, pad = np.split(got, [n if layout == "col" else k], axis=1)
    assert (pad == 7.25).all()
    assert rel_err(inner if layout == "col" else inner.T, oracle.sptrsm_csr(*M, B)) <= 1e-12


@pytest.mark.parametrize("k,layout", [(33, "row"), (70, "col")])
def test_several_column_tiles(dev, k, layout):
    M = W.zipf_lower(20000, 1.8, 256, 5000, 93)
    n = len(M[0]) - 1
    plan = sa.Plan(*to_dev(*M))
    assert "rows" in plan.tune(k=k, layout=layout).strip().splitlines()[-1]
    B = W.uniform(94, k, n * k).reshape(k, n)
    X = to_dev(B if layout == "col" else np.ascontiguousarray(B.T))
    plan.solve(X, layout=layout)
    plan.check()
    got = X.cpu().numpy()
    assert rel_err(got if layout == "col" else got.T, oracle.sptrsm_csr(*M, B)) <= 1e-12


@pytest.mark.parametrize("k", [1, 4, 16, 32])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_infinities_and_nan_beside_empty_rows(dev, bad, k):
    """Row 0 and every 27th read nothing; a bad value in one of them reaches the
    rows that read it, and no other."""
    M = matrix(2000)
    n = len(M[0]) - 1
    empty = np.flatnonzero(np.diff(M[0]) == 1)
    B = W.uniform(95, k, n * k).reshape(k, n)
    B[:, empty[3]] = bad
    B[-1, empty[-1]] = bad
    B[:, n - 5] = bad
    with np.errstate(all="ignore"):
        want = oracle.sptrsm_csr(*M, B)
    plan = rows_plan(M)
    X = to_dev(np.ascontiguousarray(B.T))
    if k == 1:
        plan.solve(X.view(-1), executor="syncfree")
    else:
        plan.solve(X, layout="row", executor="syncfree")
    plan.check()
    got = X.cpu().numpy().T
    fin = np.isfinite(want)
    assert (~fin).any() and fin[:, :empty[3]].all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert rel_err(got[fin], want[fin]) <= 1e-12
