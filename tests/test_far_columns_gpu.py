"""Matrices whose columns are spread over all rows: the solvers choose between
the resident launch and the launches per iteration by what other workgroups'
rows cost, so Ellpack slots (which may take either) are about as fast as
SlicedEllpack ones (always launch by launch) where the resident launch is the
slower, and faster where it is not."""
import time

import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S
from test_grid_cg_gpu import _band

pytestmark = pytest.mark.gpu


def _random(n, k, rng):
    """k columns per row, uniform, the diagonal among them; strictly dominant."""
    c = rng.integers(0, n, (n, k))
    c[:, 0] = np.arange(n)
    c.sort(1)
    keep = np.ones((n, k), bool)
    keep[:, 1:] = c[:, 1:] != c[:, :-1]
    v = np.where(c == np.arange(n)[:, None], 1.0 * k, 0.1 * rng.standard_normal((n, k)))
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, c[keep].astype(np.int32), v[keep]


def _seconds(s, A, b):
    s.setMatrix(A)
    s.setConvergenceResidue(1e-300)
    s.setMaxIterations(200)
    x = torch.zeros_like(b)
    best = np.inf
    for _ in range(3):
        torch.cuda.synchronize()
        t = time.perf_counter()
        s.solve(b, x.zero_())
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best, s.getIterations(), x


def _compare(make, n, csr, inner=None):
    b = torch.from_numpy(np.random.default_rng(1).standard_normal(n)).cuda()
    t, x = [], []
    for fmt, param in ((tnl.ELLPACK, 0), (tnl.SLICED_ELLPACK, 32)):
        A = tnl.SparseMatrix.from_csr(n, n, *csr, fmt=fmt, param=param)
        s = make()
        if inner is not None:
            s.setInnerMatrix(tnl.SparseMatrix(n, n, A.segments, A.values.to(inner), A.column_indexes))
        got = _seconds(s, A, b)
        t.append(got[0] / got[1])
        x.append(got[2])
    assert float((x[0] - x[1]).norm()) <= 1e-6 * float(x[1].norm())
    print(f"{make.__name__} n {n}: Ellpack {t[0] * 1e6:.1f}, SlicedEllpack {t[1] * 1e6:.1f} us per iteration", flush=True)
    return t[0] / t[1]


@pytest.mark.parametrize("n,k", [(1000000, 12), (1 << 20, 4), (400000, 16)])
def test_random_columns_cg(n, k):
    assert _compare(S.CG, n, _random(n, k, np.random.default_rng(n))) <= 1.2


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_random_columns_reliable(dtype):
    n = 1000000
    assert _compare(S.ReliableMixedCG, n, _random(n, 12, np.random.default_rng(n)), dtype) <= 1.2


def test_random_columns_bicgstab():
    n = 1000000
    assert _compare(S.BICGStab, n, _random(n, 20, np.random.default_rng(n))) <= 1.05


@pytest.mark.parametrize("n,k", [(131072, 16), (150000, 4)])
def test_few_random_columns_stay_resident(n, k):
    assert _compare(S.CG, n, _random(n, k, np.random.default_rng(n))) <= 0.95


@pytest.mark.parametrize("n", [131073, 1 << 20])
def test_near_columns_stay_resident(n):
    assert _compare(S.CG, n, _band(n, 3, np.random.default_rng(n))) <= 0.95


@pytest.mark.parametrize("solver", ["CG", "ReliableMixedCG"])
def test_far_stencil_runs_on_row_masks(monkeypatch, solver):
    """Few pairs, but far ones: below 2^20 rows the masks take such a matrix too."""
    n = 1000003
    i = np.arange(n)
    offs = [-300000, -250000, -200000, -150000, -100000, -50000, -20000]
    cols = np.stack([i + o for o in offs + [0] + [-o for o in reversed(offs)]], 1)
    keep = (cols >= 0) & (cols < n)
    vals = np.where(cols == i[:, None], 15.0, -1.0)
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    A = tnl.SparseMatrix.from_csr(n, n, off, cols[keep].astype(np.int32), vals[keep], fmt=tnl.ELLPACK)
    b = torch.from_numpy(np.random.default_rng(3).standard_normal(n)).cuda()
    got = []
    for codes in ("1", "0"):
        monkeypatch.setenv("TNLMI_COLUMN_CODES", codes)
        s = getattr(S, solver)()
        if solver == "ReliableMixedCG":
            s.setInnerMatrix(tnl.SparseMatrix(n, n, A.segments, A.values.float(), A.column_indexes))
        else:
            s.setPreconditioner(S.Diagonal(A))
        s.setMatrix(A)
        s.setConvergenceResidue(1e-10)
        x = torch.full_like(b, 0.5)
        assert s.solve(b, x)
        assert S.true_residual(A, x, b) <= 1e-9
        got.append((s.getIterations(), x))
    assert abs(got[0][0] - got[1][0]) <= 1
    assert float((got[0][1] - got[1][1]).norm()) <= 1e-8 * float(got[1][1].norm())


def test_next_workgroups_columns_stay_resident():
    n = 1 << 20
    rng = np.random.default_rng(n)
    off, cols, vals = _random(n, 8, rng)
    row = np.repeat(np.arange(n), np.diff(off))
    diagonal = cols == row
    cols = np.where(diagonal, row, np.clip(row + rng.integers(-3000, 3001, len(cols)), 0, n - 1)).astype(np.int32)
    cols = np.where(~diagonal & (cols == row), (row + 7) % n, cols).astype(np.int32)
    assert _compare(S.CG, n, (off, cols, vals)) <= 0.95
