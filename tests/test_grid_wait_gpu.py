"""Resident solves whose workgroups give up waiting for each other go on launch
by launch and end with the same answer, wherever the wait was given up: the
limit is set so short that every kernel gives up, or some of its sums do."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S
from test_grid_cg_gpu import _band

pytestmark = pytest.mark.gpu


def _cg():
    return S.CG()


def _gmres(variant):
    s = S.GMRES()
    s.setup(variant, 12, 12)
    return s


SOLVERS = {"CG": _cg, "CGS": lambda: _gmres("CGS"), "CGSR": lambda: _gmres("CGSR"), "MGSR": lambda: _gmres("MGSR"),
           "BICGStab": S.BICGStab}


def _solve(make, A, b):
    s = make()
    s.setMatrix(A)
    s.setPreconditioner(S.Diagonal(A))
    s.setConvergenceResidue(1e-10)
    s.setMaxIterations(2000)
    x = torch.zeros_like(b)
    return s.solve(b, x), s.getIterations(), x


@pytest.mark.parametrize("name", SOLVERS)
@pytest.mark.parametrize("n", [3000, 70000, 300000])
def test_given_up_solves_end_right(monkeypatch, name, n):
    rng = np.random.default_rng(n)
    A = tnl.SparseMatrix.from_csr(n, n, *_band(n, 3, rng), fmt=tnl.ELLPACK)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    make = SOLVERS[name]
    ok, its, want = _solve(make, A, b)
    assert ok
    for wait in (0, 2, 3, 4, 6, 10, 20):
        monkeypatch.setenv("TNLMI_GRID_WAIT_US", str(wait))
        ok, more, x = _solve(make, A, b)
        print(name, n, wait, its, more, flush=True)
        assert ok
        assert S.true_residual(A, x, b) <= 1e-9
        assert float((x - want).norm()) <= 1e-8 * float(want.norm())
        if wait == 0:  # nothing was done in the resident launch: the launches' own sums
            assert abs(more - its) <= 1 and not torch.equal(x, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [3000, 300000])
def test_given_up_reliable_updates(monkeypatch, n, dtype):
    rng = np.random.default_rng(n)
    A = tnl.SparseMatrix.from_csr(n, n, *_band(n, 3, rng))
    inner = tnl.SparseMatrix(n, n, A.segments, A.values.to(dtype), A.column_indexes)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    for wait in (0, 3, 6, 20):
        monkeypatch.setenv("TNLMI_GRID_WAIT_US", str(wait))
        s = S.ReliableMixedCG()
        s.setMatrix(A)
        s.setInnerMatrix(inner)
        s.setConvergenceResidue(1e-10)
        s.setMaxIterations(5000)
        x = torch.zeros_like(b)
        assert s.solve(b, x)
        assert S.true_residual(A, x, b) <= 1e-10
