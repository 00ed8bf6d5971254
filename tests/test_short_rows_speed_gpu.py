"""Products with very short rows in the padded formats: about as fast as the CSR
product of the same matrix."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl

pytestmark = pytest.mark.gpu


def _us(n, k, fmt, param, organization):
    i = np.arange(n)
    cols = i[:, None] + np.arange(k)
    keep = cols < n
    off = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    vals = np.ones(off[-1], np.float32)
    A = tnl.SparseMatrix.from_csr(n, n, off, cols[keep].astype(np.int32), vals, fmt=fmt, param=param,
                                  organization=organization)
    x = torch.ones(n, dtype=torch.float32, device="cuda")
    y = torch.zeros_like(x)
    best = np.inf
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(40):
            A.vectorProduct(x, y)
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 40 * 1e3)
    return best


@pytest.mark.parametrize("fmt,param", [(tnl.ELLPACK, 0), (tnl.SLICED_ELLPACK, 32)])
def test_one_slot(fmt, param):
    """2,000,000 rows: CSR 8.4 us, Ellpack 8.0, 32-row slices 9.2; as a batch of 8
    slots for the one 9.5 and 12.0.  The bound lies halfway between 9.2 and 12.0 (the
    caches hold these matrices; with 4,000,000 rows slices take 1.28 of CSR's time)."""
    n = 2000000
    csr, padded = _us(n, 1, tnl.CSR, 0, tnl.COLUMN_MAJOR), _us(n, 1, fmt, param, tnl.COLUMN_MAJOR)
    print(f"{tnl.FORMAT_NAMES[fmt]}: {padded:.1f} us, CSR {csr:.1f} us", flush=True)
    assert padded <= 1.25 * csr


@pytest.mark.parametrize("k", [1, 3])
def test_short_chunks(k):
    """Row-major chunks of few slots take what column-major ones do (10 us for 1 slot, 14
    for 3); through tiles of 16 slots they took 51 and 59."""
    n = 2000000
    rm, cm = (_us(n, k, tnl.CHUNKED_ELLPACK, 0, o) for o in (tnl.ROW_MAJOR, tnl.COLUMN_MAJOR))
    print(f"row-major {rm:.1f} us, column-major {cm:.1f} us", flush=True)
    assert rm <= 2 * cm


@pytest.mark.parametrize("widths", [(9, 10), (10,), (10, 11), (11,), (1,) * 600 + (40,) * 300, (3,) * 900 + (17,) * 2])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_chunk_sizes_around_the_choice(dtype, widths):
    """Matrices whose chunks are all short, all long, and both."""
    rng = np.random.default_rng(len(widths))
    n = 1500
    size = np.array([widths[r % len(widths)] for r in range(n)])
    off = np.concatenate([[0], np.cumsum(size)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in size]).astype(np.int32)
    vals, x = rng.standard_normal(off[-1]).astype(dtype), rng.standard_normal(n).astype(dtype)
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=tnl.CHUNKED_ELLPACK, organization=tnl.ROW_MAJOR)
    y = torch.full((n,), np.nan, dtype=torch.from_numpy(x).dtype, device="cuda")
    A.vectorProduct(torch.from_numpy(x).cuda(), y)
    terms = vals.astype(np.float64) * x[cols]
    want, mass = np.add.reduceat(terms, off[:-1]), np.add.reduceat(np.abs(terms), off[:-1])
    # one rounding per product and at most one per addition
    assert (np.abs(y.cpu().numpy() - want) <= (size + 1) * np.finfo(dtype).eps * mass).all()
