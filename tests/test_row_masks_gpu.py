"""CG on row masks (large matrices of few distinct (column - row, value) pairs):
the iterations of the stored matrix, for 1-byte and 2-byte masks, a diagonal
that varies or not, and matrices that the masks must refuse."""
import time

import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S

pytestmark = pytest.mark.gpu


def _stencil(nx, ny, coefficient, swap=False):
    """A 5-point diffusion matrix: coefficient(ix, iy) per cell, faces by the cell's mean."""
    n = nx * ny
    i = np.arange(n)
    x, y = i % nx, i // nx
    c = coefficient(x, y)
    right, up = np.where(x < nx - 1, c + c[np.minimum(i + 1, n - 1)], 0), np.where(y < ny - 1, c + c[np.minimum(i + nx, n - 1)], 0)
    left, down = np.where(x > 0, right[np.maximum(i - 1, 0)], 0), np.where(y > 0, up[np.maximum(i - nx, 0)], 0)
    cols = np.stack([i - nx, i - 1, i, i + 1, i + nx], 1)
    vals = np.stack([-down, -left, left + right + up + down + c, -right, -up], 1)
    keep = np.stack([y > 0, x > 0, x >= 0, x < nx - 1, y < ny - 1], 1)
    if swap:  # the last two entries of every row the other way round
        cols, vals, keep = cols[:, [0, 1, 2, 4, 3]], vals[:, [0, 1, 2, 4, 3]], keep[:, [0, 1, 2, 4, 3]]
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


CASES = {
    "laplace_odd": (1031, 1021, lambda x, y: np.ones(len(x)), False),       # the corner and edge diagonals differ
    "two_materials": (1100, 1000, lambda x, y: np.where(x < 500, 1.0, 3.0), False),
    "refused_order": (1030, 1024, lambda x, y: np.ones(len(x)), True),
    "refused_values": (1030, 1024, lambda x, y: 1.0 + (x + 3 * y) % 50, False),
}


@pytest.mark.parametrize("fmt", ["CSR", "Ellpack", "SlicedEllpack"])
@pytest.mark.parametrize("name", CASES)
def test_same_iterations(monkeypatch, name, fmt):
    nx, ny, coefficient, swap = CASES[name]
    off, cols, vals = _stencil(nx, ny, coefficient, swap)
    n = len(off) - 1
    f, param = {"CSR": (tnl.CSR, 0), "Ellpack": (tnl.ELLPACK, 0), "SlicedEllpack": (tnl.SLICED_ELLPACK, 32)}[fmt]
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=f, param=param)
    b = torch.from_numpy(np.random.default_rng(8).standard_normal(n)).cuda()
    for pre in (True, False):
        got = []
        for codes in ("1", "0"):
            monkeypatch.setenv("TNLMI_COLUMN_CODES", codes)
            s = S.CG()
            s.setMatrix(A)
            if pre:
                s.setPreconditioner(S.Diagonal(A))
            s.setConvergenceResidue(1e-9)
            s.setMaxIterations(60)
            x = torch.full_like(b, 0.25)
            s.solve(b, x)
            got.append((s.getIterations(), s.getResidue(), x))
        assert got[0][0] == got[1][0]
        # the partial sums are grouped differently: rounding only
        assert abs(got[0][1] - got[1][1]) <= 1e-9 * got[1][1]
        assert float((got[0][2] - got[1][2]).norm()) <= 1e-12 * float(got[1][2].norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_reliable_updates(dtype):
    off, cols, vals = _stencil(1031, 1021, lambda x, y: np.ones(len(x)))
    n = len(off) - 1
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals)
    b = torch.from_numpy(np.random.default_rng(9).standard_normal(n)).cuda()
    s = S.ReliableMixedCG()
    s.setMatrix(A)
    s.setInnerMatrix(tnl.SparseMatrix(n, n, A.segments, A.values.to(dtype), A.column_indexes))
    s.setConvergenceResidue(1e-10)
    x = torch.zeros_like(b)
    assert s.solve(b, x)
    assert S.true_residual(A, x, b) <= 1e-10
    t = S.TrueResidualCG(column_codes=True)
    t.setMatrix(A)
    t.setPreconditioner(S.Diagonal(A))
    t.setConvergenceResidue(1e-10)
    y = torch.zeros_like(b)
    assert t.solve(b, y) and S.true_residual(A, y, b) <= 1e-10


def test_pairs_of_signed_zero_and_nan():
    """Values are compared bit by bit: a -0.0 and a NaN entry keep their own pairs."""
    n = (1 << 20) + 5
    off = np.arange(n + 1, dtype=np.int32)
    vals = np.ones(n)
    vals[7] = -0.0
    A = tnl.SparseMatrix.from_csr(n, n, off, np.arange(n, dtype=np.int32), vals, fmt=tnl.ELLPACK)
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    s = S.CG()
    s.setMatrix(A)
    s.setMaxIterations(3)
    x = torch.zeros_like(b)
    s.solve(b, x)
    assert bool(torch.isfinite(x).all())
    vals[7] = np.nan
    A = tnl.SparseMatrix.from_csr(n, n, off, np.arange(n, dtype=np.int32), vals, fmt=tnl.ELLPACK)
    s.setMatrix(A)
    x.zero_()
    assert not s.solve(b, x)


def _seconds(A, b, limit):
    s = S.CG()
    s.setMatrix(A)
    s.setConvergenceResidue(1e-30)
    s.setMaxIterations(limit)
    x = torch.zeros_like(b)
    best = np.inf
    for _ in range(4):
        torch.cuda.synchronize()
        t = time.perf_counter()
        s.solve(b, x.zero_())
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("kind", ["all_differ", "last_row"])
def test_refusal_is_cheap(monkeypatch, kind):
    """A matrix of many pairs is refused within the time of a few iterations (0.2 ms
    each here), wherever its pairs begin to differ."""
    nx, ny = 2048, 1024
    coefficient = (lambda x, y: 1.0 + (x * 7919 + y * 104729) % 100003 / 1e5) if kind == "all_differ" else \
        (lambda x, y: np.where(x + nx * y > nx * ny - 40, 2.0 + x / nx, 1.0))
    off, cols, vals = _stencil(nx, ny, coefficient)
    n = nx * ny
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=tnl.ELLPACK)
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    t = {}
    for codes in ("1", "0"):
        monkeypatch.setenv("TNLMI_COLUMN_CODES", codes)
        t[codes] = _seconds(A, b, 20)
    print(kind, t, flush=True)
    assert t["1"] <= t["0"] + 1e-3


def test_short_solves_of_small_matrices_pay_nothing(monkeypatch):
    """A few iterations on 300^2 rows: as without masks (0.3 ms; looking for the pairs
    took 0.14 ms more).  The bound is half of that."""
    off, cols, vals = _stencil(300, 300, lambda x, y: np.ones(len(x)))
    n = 90000
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=tnl.SLICED_ELLPACK, param=32)
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    t = {"1": np.inf, "0": np.inf}
    for codes in ("1", "0", "1", "0", "1", "0"):
        monkeypatch.setenv("TNLMI_COLUMN_CODES", codes)
        t[codes] = min(t[codes], _seconds(A, b, 5))
    print(t, flush=True)
    assert t["1"] <= t["0"] + 7e-5
