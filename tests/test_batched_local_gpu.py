"""The batched solve from LDS and registers, at the edges of its shapes (rows per
thread and workgroup, slots per row) and beyond them (the general kernel)."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl
from tnl_amd import batched as B

pytestmark = pytest.mark.gpu


def _system(n, half, rng):
    """A diagonally dominant symmetric matrix with 2 half + 1 entries in the inner rows (half 0: a diagonal)."""
    shifts = [s for s in [1, 5, 37, 200][:half] if s < n]
    i = np.arange(n)
    w = {s: -rng.random(n) for s in shifts}
    offs = [-s for s in reversed(shifts)] + [0] + shifts
    cols = np.stack([i + o for o in offs], 1)
    keep = (cols >= 0) & (cols < n)
    vals = np.stack([np.concatenate([np.zeros(-o), w[-o][:o]]) if o < 0 else w[o] if o > 0 else np.zeros(n)
                     for o in offs], 1)
    vals[:, len(shifts)] = np.where(keep, np.abs(vals), 0).sum(1) + 0.05 + rng.random(n)
    return keep.sum(1), cols[keep], vals[keep]


def _batch(sizes, half, rng):
    lens, cols, vals, at = [], [], [], 0
    for n in sizes:
        ln, c, v = _system(n, half, rng)
        lens.append(ln), cols.append(c + at), vals.append(v)
        at += n
    off = np.concatenate([[0], np.cumsum(np.concatenate(lens))]).astype(np.int32)
    return off, np.concatenate(cols).astype(np.int32), np.concatenate(vals), np.concatenate([[0], np.cumsum(sizes)])


@pytest.mark.parametrize("fmt,param", [(tnl.CSR, 0), (tnl.SLICED_ELLPACK, 32)])
@pytest.mark.parametrize("sizes,half", [
    ([1, 2, 3, 64, 65], 1), ([511, 512, 513, 2047, 2048], 2), ([2049, 7, 4096], 3), ([4097, 1000, 8192], 2),
    ([8193, 16384, 5], 2), ([16384, 300], 3), ([16385, 300], 2), ([700, 900], 4), ([600, 0, 40], 0)])
def test_sizes(orc, fmt, param, sizes, half):
    rng = np.random.default_rng(sum(sizes) + half)
    off, cols, vals, sys_rows = _batch(sizes, half, rng)
    n = int(sys_rows[-1])
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=fmt, param=param)
    b = rng.standard_normal(n)
    if len(sizes) > 1:
        b[sys_rows[1]:sys_rows[2]] = 0.0  # a system that is solved by x = 0
    bc = B.BatchedCG(A, sys_rows)
    x = torch.full((n,), 0.3, dtype=torch.float64, device="cuda")
    its, res = bc.solve(torch.from_numpy(b).cuda(), x, 1e-10, use_graph=False)
    xs, its = x.cpu().numpy(), its.cpu().numpy()
    for k, rows in enumerate(sizes):
        r0, r1 = int(sys_rows[k]), int(sys_rows[k + 1])
        if not rows:
            continue
        o, c, v = off[r0:r1 + 1] - off[r0], cols[off[r0]:off[r1]] - r0, vals[off[r0]:off[r1]]
        if not b[r0:r1].any():
            assert not xs[r0:r1].any() and its[k] == 0
            continue
        xo, so = orc.cg(o, c, v, b[r0:r1], precond=1, tol=1e-10, x0=np.full(rows, 0.3))
        assert so.converged and abs(int(its[k]) - so.iterations) <= 1
        np.testing.assert_allclose(xs[r0:r1], xo, rtol=1e-7, atol=1e-9)
    again = torch.full_like(x, 0.3)
    bc.solve(torch.from_numpy(b).cuda(), again, 1e-10, use_graph=True)
    torch.cuda.synchronize()
    assert torch.equal(again, x)


def test_values_written_between_solves():
    """The slots are laid out by every solve: values changed in place are the next solve's."""
    rng = np.random.default_rng(2)
    off, cols, vals, sys_rows = _batch([900, 40, 3000], 2, rng)
    n = int(sys_rows[-1])
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals)
    b = torch.from_numpy(rng.standard_normal(n)).cuda()
    bc = B.BatchedCG(A, sys_rows)
    x = torch.zeros_like(b)
    for scale in (1.0, 3.0, 0.25):
        A.values.copy_(torch.from_numpy(vals * scale))
        for graph in (False, True):
            x.zero_()
            bc.solve(b, x, 1e-11, use_graph=graph)
            y = torch.zeros_like(b)
            A.vectorProduct(x, y)
            assert float((y - b).norm()) <= 1e-8 * float(b.norm())


def test_nan_and_iteration_limit():
    rng = np.random.default_rng(3)
    off, cols, vals, sys_rows = _batch([300, 300, 300], 1, rng)
    vals[off[310]] = np.nan
    n = int(sys_rows[-1])
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals)
    bc = B.BatchedCG(A, sys_rows)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    its, res = bc.solve(b, x, 1e-10, use_graph=False)
    assert bool(torch.isnan(res[1])) and float(res[0]) < 1e-10 and float(res[2]) < 1e-10
    x.zero_()
    its, res = bc.solve(b, x, 1e-10, max_iterations=3, use_graph=False)
    assert int(its[0]) == 4 and int(its[2]) == 4  # (the reference counts the refused iteration)


def test_autotune_times_what_it_shapes(monkeypatch):
    """Where the shapes leave the FP64 solve alone the mixed one is timed."""
    rng = np.random.default_rng(4)
    mixed = []
    solve = B.BatchedCG.solve
    monkeypatch.setattr(B.BatchedCG, "solve", lambda self, *a, **kw: (mixed.append(kw["mixed"]), solve(self, *a, **kw))[1])
    for half, sizes, want in ((2, [900, 40], True), (4, [900, 40], False), (1, [16385], False)):
        off, cols, vals, sys_rows = _batch(sizes, half, rng)
        mixed.clear()
        B.autotune(off, cols, vals, sys_rows, candidates=[(tnl.CSR, 0)], blocks=[256], lanes=[1, 4], cache=False)
        assert set(mixed) == {want}
