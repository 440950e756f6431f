"""CSR kernels that stream the contiguous entries of a block's rows (fa_spmv,
fa_dirichlet_*): empty rows, rows longer than a block's chunk, one row, rows
around the block's count, boundary rows without entries or diagonal.  The oracle
is dense FP64 on the CPU; a row's sum of m products differs by m units in the
last place of the sum of their magnitudes at most."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp
import torch

import fealpy_amd as fa
from fealpy_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _matrix(n, mean, seed, long_row=0):
    g = np.random.default_rng(seed)
    counts = np.minimum(g.poisson(mean, n), n)
    counts[g.random(n) < 0.2 * (n > 1)] = 0
    if long_row:
        counts[n // 2] = min(long_row, n)
    cols = [np.sort(g.choice(n, c, replace=False)) for c in counts]
    crow = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    col = np.concatenate(cols).astype(np.int32) if counts.sum() else np.zeros(0, np.int32)
    return crow, col, g.standard_normal(len(col))


SHAPES = [(1, 5, 0), (3, 2, 0), (64, 4, 0), (257, 7, 0), (300, 16, 0), (700, 40, 650), (6000, 9, 5000), (500, 120, 0)]


@pytest.mark.parametrize("n,mean,long_row", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_spmv(n, mean, long_row, dtype):
    crow, col, val = _matrix(n, mean, n + mean, long_row)
    v = torch.as_tensor(val, dtype=dtype)
    x = torch.as_tensor(np.random.default_rng(1).standard_normal(n), dtype=dtype)
    A = fa.CSRTensor(torch.as_tensor(crow, device=DEV), torch.as_tensor(col, device=DEV), v.to(DEV), (n, n))
    S = sp.csr_matrix((v.double().numpy(), col, crow), shape=(n, n))
    ref, size = S @ x.double().numpy(), abs(S) @ np.abs(x.double().numpy())
    eps = 2.2e-16 if dtype == torch.float64 else 1.2e-7
    bound = eps * (np.diff(crow) + 2) * size
    assert np.all(np.abs((A @ x.to(DEV)).cpu().double().numpy() - ref) <= bound)


@pytest.mark.parametrize("n,mean,long_row", SHAPES)
def test_dirichlet_forms(n, mean, long_row):
    crow, col, val = _matrix(n, mean, n + mean, long_row)
    g = np.random.default_rng(2)
    bd = g.random(n) < 0.3
    uh, f = np.where(bd, g.standard_normal(n), 0.0), g.standard_normal(n)
    L = nat.lib()
    d = lambda a: torch.as_tensor(a, device=DEV)              # noqa: E731
    dc, dj, dv, db, du, df = d(crow), d(col), d(val), d(bd.astype(np.uint8)), d(uh), d(f)
    p = nat.ptr
    nptr = torch.empty(n + 1, dtype=torch.int32, device=DEV)
    ws = nat.workspace(L.fa_dirichlet_work_bytes(n), DEV)
    nnz = ctypes.c_int64(0)
    nat.check(L.fa_dirichlet_count(n, p(dc), p(dj), p(db), p(nptr), ctypes.byref(nnz), p(ws), ws.numel(), nat.stream()))
    nidx = torch.full((nnz.value,), -1, dtype=torch.int32, device=DEV)
    nval, nval2 = (torch.full((nnz.value,), 7.0, dtype=torch.float64, device=DEV) for _ in range(2))
    out, out2, out3 = (torch.empty(n, dtype=torch.float64, device=DEV) for _ in range(3))
    nat.check(L.fa_dirichlet_fill(0, 0, n, p(dc), p(dj), p(dv), p(db), p(nptr), p(nidx), p(nval), nat.stream()))
    nat.check(L.fa_dirichlet_apply(0, n, p(dc), p(dj), p(dv), p(db), p(nptr), p(nval2), p(du), p(df), p(out),
                                   nat.stream()))
    nat.check(L.fa_dirichlet_rhs(0, n, p(dc), p(dj), p(dv), p(db), p(du), p(df), p(out2), nat.stream()))
    kept = dv.clone()                                          # in place
    nat.check(L.fa_dirichlet_apply_keep(0, n, p(dc), p(dj), p(kept), p(db), p(kept), p(du), p(df), p(out3),
                                        nat.stream()))
    rows = np.repeat(np.arange(n), np.diff(crow))
    keep = ~bd[rows] & ~bd[col]
    r = np.concatenate([rows[keep], np.flatnonzero(bd)])
    c = np.concatenate([col[keep], np.flatnonzero(bd)])
    v = np.concatenate([val[keep], np.ones(bd.sum())])
    order = np.lexsort((c, r))
    assert np.array_equal(nptr.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]))
    assert np.array_equal(nidx.cpu().numpy(), c[order]) and np.array_equal(nval.cpu().numpy(), v[order])
    assert torch.equal(nval, nval2) and torch.equal(out, out2) and torch.equal(out, out3)
    assert np.array_equal(kept.cpu().numpy(), np.where(bd[rows], rows == col, np.where(bd[col], 0.0, val)))
    S = sp.csr_matrix((val, col, crow), shape=(n, n))
    ref = np.where(bd, uh, f - S @ uh)
    bound = 2.2e-16 * (np.diff(crow) + 3) * (abs(S) @ np.abs(uh) + np.abs(f) + np.abs(uh))
    assert np.all(np.abs(out.cpu().numpy() - ref) <= bound)


@pytest.mark.parametrize("mean,long_row", [(7, 0), (40, 0), (9, 5000)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_row_sums_lose_nothing(mean, long_row, dtype):
    """FP32 products and sums are exact but for the result's rounding; FP64 ones but for each product's and the result's,
    whatever the row's length (positive terms, so that their size is the result's)."""
    n = 6000
    crow, col, val = _matrix(n, mean, n + mean, long_row)
    v, x = (torch.as_tensor(np.abs(a), dtype=dtype) for a in (val, np.random.default_rng(1).standard_normal(n)))
    ptr = [torch.as_tensor(a, device=DEV) for a in (crow, col)]
    A = fa.CSRTensor(*ptr, v.to(DEV), (n, n))
    terms = v.numpy().astype(np.longdouble) * x.numpy()[col].astype(np.longdouble)
    ref = np.zeros(n, np.longdouble)
    np.add.at(ref, np.repeat(np.arange(n), np.diff(crow)), terms)
    half = 2.0 ** -53 if dtype == torch.float64 else 2.0 ** -24
    bound = half * (2.01 if dtype == torch.float64 else 1.01) * ref
    assert np.all(np.abs((A @ x.to(DEV)).cpu().numpy().astype(np.longdouble) - ref) <= bound)
    if dtype == torch.float64:                    # the right-hand side's A uh: one rounding more, of f - A uh
        out = torch.empty(n, dtype=dtype, device=DEV)
        zero, bd = torch.zeros(n, dtype=dtype, device=DEV), torch.zeros(n, dtype=torch.uint8, device=DEV)
        p, xd, vd = nat.ptr, x.to(DEV), v.to(DEV)
        nat.check(nat.lib().fa_dirichlet_rhs(0, n, p(ptr[0]), p(ptr[1]), p(vd), p(bd), p(xd), p(zero), p(out),
                                             nat.stream()))
        assert np.all(np.abs(out.cpu().numpy().astype(np.longdouble) + ref) <= bound)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("terms,expected", [([np.inf, 1.0, 2.0], np.inf), ([1.0, -np.inf, 3.0], -np.inf),
                                            ([np.inf, -np.inf, 1.0], np.nan), ([1.0, np.nan, 2.0], np.nan)])
def test_infinite_terms(terms, expected, dtype):
    """Row 1 of three holds the terms; its neighbours stay as they are."""
    crow = torch.tensor([0, 1, 4, 5], dtype=torch.int32, device=DEV)
    col = torch.tensor([0, 0, 1, 2, 2], dtype=torch.int32, device=DEV)
    val = torch.tensor([2.0, *terms, 3.0], dtype=dtype, device=DEV)
    y = (fa.CSRTensor(crow, col, val, (3, 3)) @ torch.ones(3, dtype=dtype, device=DEV)).cpu().numpy()
    np.testing.assert_array_equal(y, np.array([2.0, expected, 3.0]))
