"""The ILU(0) triangular solves as a pipeline of row strips: the oracle's solve
within rounding, and the level-by-level solves' bits, at the edges of strips,
steps and the LDS windows."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import solvers as S

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _grid(nx, ny, nz, rng):
    n = nx * ny * nz
    i = np.arange(n)
    x, y, z = i % nx, i // nx % ny, i // (nx * ny)
    cols = np.stack([i - nx * ny, i - nx, i - 1, i, i + 1, i + nx, i + nx * ny], 1)
    keep = np.stack([z > 0, y > 0, x > 0, x >= 0, x < nx - 1, y < ny - 1, z < nz - 1], 1)
    vals = np.where(cols == i[:, None], 7.0, -1.0) + 0.2 * rng.random((n, 7))
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


def _scattered(n, rng):
    """Up to three entries on each side of the diagonal, anywhere: dependencies
    many steps back and in any earlier strip."""
    rows = []
    for r in range(n):
        lo = rng.choice(r, size=min(r, 3), replace=False) if r else np.zeros(0, np.int64)
        hi = r + 1 + rng.choice(n - 1 - r, size=min(n - 1 - r, 3), replace=False) if r < n - 1 else np.zeros(0, np.int64)
        rows.append(np.sort(np.concatenate([lo, [r], hi])).astype(np.int32))
    off = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    cols = np.concatenate(rows)
    row = np.repeat(np.arange(n), np.diff(off))
    return off, cols, np.where(cols == row, 9.0, rng.standard_normal(len(cols)))


def _far(width, lines, rng):
    """Three entries on each side of the diagonal, all about `width` rows away:
    with lines of more rows than a strip keeps in LDS, every one is an import."""
    n = width * lines
    i = np.arange(n)
    shifts = [-width - 1, -width, -width + 1, 0, width - 1, width, width + 1]
    cols = np.stack([i + s for s in shifts], 1)
    keep = (cols >= 0) & (cols < n)
    vals = np.where(cols == i[:, None], 9.0, rng.standard_normal((n, 7)))
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


def _scattered_band(n, low, high, rng):
    """Up to three entries on each side of the diagonal, low to high rows away."""
    i = np.arange(n)
    d = np.sort(rng.integers(low, high, (n, 6)), 1)
    cols = np.sort(np.concatenate([i[:, None] - d[:, :3], i[:, None], i[:, None] + d[:, 3:]], 1), 1)
    keep = (cols >= 0) & (cols < n)
    keep[:, 1:] &= cols[:, 1:] != cols[:, :-1]
    vals = np.where(cols == i[:, None], 9.0, rng.standard_normal((n, 7)))
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return off, cols[keep].astype(np.int32), vals[keep]


CASES = {
    "rows127": lambda g: _grid(127, 1, 1, g), "rows128": lambda g: _grid(128, 1, 1, g),
    "line64": lambda g: _grid(64, 64, 1, g), "line65": lambda g: _grid(65, 130, 1, g),
    "thin": lambda g: _grid(700, 9, 1, g), "tall": lambda g: _grid(9, 700, 1, g),
    "plane": lambda g: _grid(17, 19, 23, g), "cube": lambda g: _grid(40, 40, 40, g),
    "scattered": lambda g: _scattered(2500, g), "scattered_strips": lambda g: _scattered(12000, g),
    "far_one_strip": lambda g: _far(5000, 3, g), "far_strips": lambda g: _far(6000, 20, g),
    "band_strips": lambda g: _scattered_band(60000, 200, 300, g),
    "band_full": lambda g: _scattered_band(100000, 64, 800, g), "band_full_small": lambda g: _scattered_band(20000, 128, 640, g),
}
# the strips of either factor (test_tri_strips_plan.py checks the plans): none, one or more than one
STRIPS = {name: (1, 1) if name in ("line64", "thin", "scattered")
          else (0, 0) if name in ("rows127", "scattered_strips", "far_one_strip", "far_strips")
          else (1, 256) if name.startswith("band_full") else (2, 256) for name in CASES}
FULL_RING = ("band_full", "band_full_small")  # one factor has almost three imports per row in two groups of steps


@pytest.mark.parametrize("name", CASES)
def test_strip_solve_matches_oracle_and_levels(orc, monkeypatch, name):
    rng = np.random.default_rng(61)
    off, cols, vals = CASES[name](rng)
    n = len(off) - 1
    b = rng.standard_normal(n)
    b[rng.integers(0, n, n // 3)] = 0.0  # zero quotients take the division
    L, U = orc.ilu0(off, cols, vals)
    want = orc.ilu0_solve(L, U, b)
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals)
    P = S.ILU0(A)
    x = torch.full((n,), 5.0, dtype=torch.float64, device="cuda")
    got = [P.solve(dev(b), x).cpu().numpy() for _ in range(3)]
    np.testing.assert_allclose(got[0], want, rtol=1e-12, atol=1e-13 * np.abs(want).max())
    np.testing.assert_array_equal(got[0], got[1])
    np.testing.assert_array_equal(got[0], got[2])
    inplace = dev(b)
    np.testing.assert_array_equal(P.solve(inplace, inplace).cpu().numpy(), got[0])
    monkeypatch.setenv("TNLMI_ILU_FLOW", "0")
    levels = S.ILU0(A).solve(dev(b), x).cpu().numpy()
    np.testing.assert_array_equal(got[0], levels)


@pytest.mark.parametrize("scale", [1e-300, 1e-135, 1e135, 1e300])
def test_strip_solve_pivots_at_the_ends_of_the_range(monkeypatch, scale):
    """Pivots and quotients for which the corrected reciprocal is not used, an
    infinite and a NaN entry, and a right-hand side that holds the solve's own
    mark of an unsolved value: as the level solves."""
    rng = np.random.default_rng(62)
    off, cols, vals = _grid(70, 70, 1, rng)
    n = len(off) - 1
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals * scale)
    b = rng.standard_normal(n)
    special = b.copy()
    special[n // 2], special[n // 3] = np.inf, np.nan
    special[:1] = np.array([0x7FF4DEAD5EED0001], np.uint64).view(np.float64)
    for rhs in (b, special):
        monkeypatch.setenv("TNLMI_ILU_FLOW", "1")
        got = S.ILU0(A).solve(dev(rhs), torch.zeros(n, dtype=torch.float64, device="cuda")).cpu().numpy()
        monkeypatch.setenv("TNLMI_ILU_FLOW", "0")
        want = S.ILU0(A).solve(dev(rhs), torch.zeros(n, dtype=torch.float64, device="cuda")).cpu().numpy()
        np.testing.assert_array_equal(got, want)


def test_strip_solve_in_a_graph():
    """A captured apply, replayed with other right-hand sides and eager applies between: the
    counter of the started strips is cleared in the graph."""
    rng = np.random.default_rng(63)
    off, cols, vals = _grid(65, 130, 1, rng)
    n = len(off) - 1
    P = S.ILU0(tnl.SparseMatrix.from_csr(n, n, off, cols, vals))
    b, x = dev(rng.standard_normal(n)), torch.zeros(n, dtype=torch.float64, device="cuda")
    P.solve(b, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        P.solve(b, x)
    for _ in range(4):
        b.copy_(dev(rng.standard_normal(n)))
        x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = x.clone()
        want = P.solve(b, torch.zeros_like(x))
        torch.cuda.synchronize()
        assert torch.equal(got, want)
