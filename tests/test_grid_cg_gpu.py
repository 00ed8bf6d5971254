"""CG iterations in one resident launch (Ellpack slots of at most 2^20 rows): the
same iterations as launch by launch (the SlicedEllpack matrix), at the edges of
its shapes -- rows per thread and workgroup, entries held in registers."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S

pytestmark = pytest.mark.gpu


def _band(n, half, rng):
    """A symmetric diagonally dominant matrix with entries at +-1, +-7, +-3*7, ... (half of them)."""
    shifts = [s for s in [1, 7, 40, 300][:half] if s < n]
    i = np.arange(n)
    w = {s: -rng.random(n) for s in shifts}
    cols, vals, keep = [], [], []
    for s in reversed(shifts):
        cols.append(i - s), vals.append(np.concatenate([np.zeros(s), w[s][:-s]])), keep.append(i >= s)
    diag = len(cols)
    cols.append(i), vals.append(np.zeros(n)), keep.append(i >= 0)
    for s in shifts:
        cols.append(i + s), vals.append(w[s]), keep.append(i < n - s)
    cols, vals, keep = np.stack(cols, 1), np.stack(vals, 1), np.stack(keep, 1)
    vals[:, diag] = np.where(keep, np.abs(vals), 0).sum(1) + 0.1 + rng.random(n)
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


def _solve(A, pre, b, limit, tol=1e-10):
    s = S.CG()
    s.setMatrix(A)
    if pre:
        s.setPreconditioner(S.Diagonal(A))
    s.setConvergenceResidue(tol)
    s.setMaxIterations(limit)
    x = torch.zeros_like(b)
    ok = s.solve(b, x)
    return ok, s.getIterations(), s.getResidue(), x


@pytest.mark.parametrize("n,half", [(1, 1), (2, 1), (255, 3), (256, 4), (257, 2), (5000, 4), (65536, 3), (65537, 3),
                                    (131073, 3), (131073, 4), (262145, 2), (524289, 2), (1 << 20, 2),
                                    ((1 << 20) + 1, 2)])
@pytest.mark.parametrize("pre", [False, True], ids=["none", "diagonal"])
def test_iterations_match_launch_by_launch(n, half, pre):
    rng = np.random.default_rng(n + half)
    off, cols, vals = _band(n, half, rng)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    ell = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=tnl.ELLPACK)
    ref = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=tnl.SLICED_ELLPACK, param=32)
    for limit in (7, 400):
        got, want = _solve(ell, pre, b, limit), _solve(ref, pre, b, limit)
        assert got[0] == want[0] and abs(got[1] - want[1]) <= (1 if limit > 7 else 0)
        if got[1] == want[1]:
            # sums in another order: rounding, grown over the iterations
            assert abs(got[2] - want[2]) <= 1e-6 * max(want[2], 1e-10)
        assert float((got[3] - want[3]).norm()) <= 1e-9 * float(want[3].norm())
        again = _solve(ell, pre, b, limit)
        assert again[1:3] == got[1:3] and torch.equal(again[3], got[3])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,half", [(300, 2), (70001, 3), (300000, 4), (600000, 2)])
def test_reliable_updates(n, half, dtype):
    rng = np.random.default_rng(n)
    off, cols, vals = _band(n, half, rng)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals)
    s = S.ReliableMixedCG()
    s.setMatrix(A)
    s.setInnerMatrix(tnl.SparseMatrix(n, n, A.segments, A.values.to(dtype), A.column_indexes))
    s.setConvergenceResidue(1e-10)
    s.setMaxIterations(5000)
    x = torch.zeros_like(b)
    assert s.solve(b, x)
    assert S.true_residual(A, x, b) <= 1e-10


def test_zero_curvature_and_exact_start():
    """(p, Ap) = 0 ends the solve as in the launches; a start at the solution needs no iteration."""
    n = 512
    off = np.arange(n + 1, dtype=np.int32)
    A = tnl.SparseMatrix.from_csr(n, n, off, np.arange(n, dtype=np.int32), np.zeros(n), fmt=tnl.ELLPACK)
    ref = tnl.SparseMatrix.from_csr(n, n, off, np.arange(n, dtype=np.int32), np.zeros(n), fmt=tnl.SLICED_ELLPACK, param=32)
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    assert _solve(A, False, b, 50)[1:3] == _solve(ref, False, b, 50)[1:3]
    A = tnl.SparseMatrix.from_csr(n, n, off, np.arange(n, dtype=np.int32), np.ones(n), fmt=tnl.ELLPACK)
    s = S.CG()
    s.setMatrix(A)
    x = b.clone()
    assert s.solve(b, x) and torch.equal(x, b)
