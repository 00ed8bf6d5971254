"""Products of the padded formats with rows around the batch of slots that a lane loads together."""
import numpy as np
import pytest
import torch

import tnl_amd as tnl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("organization", [tnl.COLUMN_MAJOR, tnl.ROW_MAJOR])
@pytest.mark.parametrize("fmt,param", [(tnl.ELLPACK, 0), (tnl.SLICED_ELLPACK, 32), (tnl.SLICED_ELLPACK, 1),
                                       (tnl.BIELLPACK, 32), (tnl.CHUNKED_ELLPACK, 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("widths", [(1,), (7,), (8,), (9,), (15, 16, 17), (0, 1, 7, 8, 9, 24, 25, 63)])
def test_row_lengths(organization, fmt, param, dtype, widths):
    rng = np.random.default_rng(sum(widths))
    n = 333
    size = np.array([widths[r % len(widths)] for r in range(n)])
    off = np.concatenate([[0], np.cumsum(size)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in size]).astype(np.int32)
    vals, x = rng.standard_normal(off[-1]).astype(dtype), rng.standard_normal(n).astype(dtype)
    A = tnl.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=fmt, param=param,
                                  organization=organization)
    y = torch.full((n,), np.nan, dtype=torch.from_numpy(x).dtype, device="cuda")
    A.vectorProduct(torch.from_numpy(x).cuda(), y)
    want, mass = np.zeros(n), np.zeros(n)
    for r in range(n):
        s = slice(off[r], off[r + 1])
        terms = vals[s].astype(np.float64) * x[cols[s]]
        want[r], mass[r] = terms.sum(), np.abs(terms).sum()
    # one rounding per product and at most one per addition
    assert (np.abs(y.cpu().numpy() - want) <= (size + 1) * np.finfo(dtype).eps * mass).all()
    if organization == tnl.COLUMN_MAJOR and fmt in (tnl.ELLPACK, tnl.SLICED_ELLPACK):  # the host's order: products rounded, added left to right
        host = np.zeros(n, dtype)
        for r in range(n):
            for k in range(off[r], off[r + 1]):
                host[r] = host[r] + vals[k] * x[cols[k]]
        assert np.array_equal(y.cpu().numpy(), host)
