"""BiCGStab and GMRES with their iterations in one resident launch (Ellpack
slots of at most 2^20 rows): the same answers as launch by launch (the
SlicedEllpack matrix), at the edges of rows per thread and workgroup, of the
width held in registers and of the restart length."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S

pytestmark = pytest.mark.gpu


def _matrix(n, half, rng):
    """Diagonally dominant and nonsymmetric, 2 half + 1 entries in the inner rows."""
    shifts = [s for s in [1, 7, 40, 300, 1000][:half] if s < n]
    i = np.arange(n)
    offs = [-s for s in reversed(shifts)] + [0] + shifts
    cols = np.stack([i + o for o in offs], 1)
    keep = (cols >= 0) & (cols < n)
    vals = rng.standard_normal((n, len(offs)))
    vals[:, len(shifts)] = np.where(keep, np.abs(vals), 0).sum(1) * 1.05 + 0.2
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


def _run(make, n, csr, fmt, param, pre, b, x0):
    A = tnl.SparseMatrix.from_csr(n, n, *csr, fmt=fmt, param=param)
    s = make()
    s.setMatrix(A)
    if pre:
        s.setPreconditioner(S.Diagonal(A))
    x = x0.clone()
    ok = s.solve(b, x)
    return ok, s.getIterations(), s.getResidue(), x, A


def _both(make, n, half, pre, start=False):
    rng = np.random.default_rng(3 * n + half)
    csr = _matrix(n, half, rng)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    x0 = torch.full_like(b, 0.5) if start else torch.zeros_like(b)
    got = _run(make, n, csr, tnl.ELLPACK, 0, pre, b, x0)
    again = _run(make, n, csr, tnl.CSR, 0, pre, b, x0)  # (a copy of the same slots)
    want = _run(make, n, csr, tnl.SLICED_ELLPACK, 32, pre, b, x0)
    return got, again, want, b


SIZES = [(1, 1), (255, 3), (257, 4), (65536, 3), (65537, 2), (131073, 3), (262145, 2), (524289, 2), (1 << 20, 2),
         ((1 << 20) + 1, 1)]


@pytest.mark.parametrize("n,half", SIZES)
@pytest.mark.parametrize("pre", [False, True], ids=["none", "diagonal"])
def test_bicgstab(n, half, pre):
    def make():
        s = S.BICGStab()
        s.setConvergenceResidue(1e-9)
        s.setMaxIterations(300)
        return s
    got, again, want, b = _both(make, n, half, pre, start=True)
    assert got[0] == want[0] and abs(got[1] - want[1]) <= 1
    if want[0]:
        assert S.true_residual(got[4], got[3], b) <= 1e-7
        assert float((got[3] - want[3]).norm()) <= 1e-6 * float(want[3].norm())
    assert abs(got[1] - again[1]) <= 1  # (the first residual: CSR and Ellpack products round differently)


@pytest.mark.parametrize("variant", ["CGS", "CGSR", "MGS", "MGSR"])
@pytest.mark.parametrize("n,half,restart", [(1, 1, 5), (300, 4, 10), (70000, 3, 31), (131073, 2, 17), (300000, 2, 8),
                                            (600000, 2, 16), (1 << 20, 2, 9), ((1 << 20) + 1, 1, 9)])
def test_gmres(variant, n, half, restart):
    for limit, pre in ((restart * 2 + 3, True), (400, False)):
        def make():
            s = S.GMRES()
            s.setup(variant, restart, restart)
            s.setConvergenceResidue(1e-9)
            s.setMaxIterations(limit)
            return s
        got, again, want, b = _both(make, n, half, pre)
        assert got[0] == want[0] and abs(got[1] - want[1]) <= (0 if limit < 400 else 1)
        assert float((got[3] - want[3]).norm()) <= 1e-7 * float(want[3].norm())
        assert abs(got[1] - again[1]) <= 1  # (the first residual: CSR and Ellpack products round differently)


def test_gmres_adaptive_restart_and_limits():
    def make():
        s = S.GMRES()
        s.setup("MGSR", 4, 12, 2, 4)
        s.setConvergenceResidue(1e-10)
        s.setMaxIterations(500)
        s.setMinIterations(30)
        return s
    got, _, want, _ = _both(make, 5000, 3, True)
    assert got[0] and want[0] and abs(got[1] - want[1]) <= 1 and got[1] >= 30
    assert float((got[3] - want[3]).norm()) <= 1e-8 * float(want[3].norm())


def test_zero_pivot_and_nan():
    """A zero matrix (a zero on the Hessenberg diagonal) fails as launch by launch; NaN ends a solve."""
    n = 700
    zero = (np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.zeros(n))
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    x0 = torch.zeros_like(b)

    def gmres():
        s = S.GMRES()
        s.setMaxIterations(40)
        return s

    def bicgstab():
        s = S.BICGStab()
        s.setMaxIterations(40)
        return s
    for make in (gmres, bicgstab):
        ends = []
        for vals in (zero[2], np.where(np.arange(n) == 9, np.nan, 1.0)):
            for fmt, param in ((tnl.ELLPACK, 0), (tnl.SLICED_ELLPACK, 32)):
                try:
                    ends.append(_run(make, n, (zero[0], zero[1], vals), fmt, param, False, b, x0)[:2])
                except tnl.TnlmiError as e:
                    ends.append(str(e))
        assert ends[0] == ends[1] and ends[2] == ends[3]
