"""Batched CG over many independent SPD systems (tnlmi_batched_cg_*), the
seeded variable-coefficient diffusion batch, and the autotuner that picks the
segment format, slice size, workgroup size and rows per wavefront of the
persistent kernel."""
import ctypes
import json
import os
import time

import numpy as np

from . import _lib
from . import SparseMatrix, _stream, _ptr, CSR, ELLPACK, SLICED_ELLPACK, FORMAT_NAMES


def diffusion_batch(nsys, smin=16, smax=128, seed=0):
    """The batch as one block-diagonal CSR matrix: (sides, offsets, columns,
    values, sys_rows) with sys_rows[k] .. sys_rows[k+1] the rows of system k."""
    L = _lib.lib()
    sides = np.zeros(nsys, np.int32)
    rows, nnz = ctypes.c_int64(), ctypes.c_int64()
    L.tnlmi_gen_batched_diffusion(nsys, smin, smax, seed, _ptr(sides), ctypes.byref(rows), ctypes.byref(nnz), None,
                                  None, None)
    off = np.zeros(rows.value + 1, np.int32)
    col = np.zeros(nnz.value, np.int32)
    val = np.zeros(nnz.value, np.float64)
    L.tnlmi_gen_batched_diffusion(nsys, smin, smax, seed, _ptr(sides), ctypes.byref(rows), ctypes.byref(nnz),
                                  _ptr(off), _ptr(col), _ptr(val))
    sys_rows = np.zeros(nsys + 1, np.int64)
    sys_rows[1:] = np.cumsum(sides.astype(np.int64) ** 2)
    return sides, off, col, val, sys_rows


class BatchedCG:
    """One persistent launch solving every diagonal block of A (FP64 values).
    lanes_per_row (1, 2, 4, 8): the lanes that sum one row, so a wavefront
    covers 64 / lanes_per_row rows.  Both shapes are those of the general
    kernel; systems of at most 16,384 rows with at most 8 slots per row are
    solved from LDS and registers by workgroups of the library's choice."""

    def __init__(self, A, sys_rows, A_lo=None, block_size=512, lanes_per_row=1, stream=None):
        self.sys_rows = np.ascontiguousarray(sys_rows, np.int64)
        self.nsys = len(self.sys_rows) - 1
        self.A, self.A_lo = A, A_lo
        h = ctypes.c_void_p()
        _lib.check(_lib.lib().tnlmi_batched_cg_create(ctypes.byref(A._m), ctypes.byref(A_lo._m) if A_lo else None,
                                                      _ptr(self.sys_rows), self.nsys, block_size, lanes_per_row,
                                                      _stream(stream), ctypes.byref(h)))
        self.handle = h
        import torch
        self.iters = torch.zeros(self.nsys, dtype=torch.int64, device="cuda")
        self.res = torch.zeros(self.nsys, dtype=torch.float64, device="cuda")

    def __del__(self):
        h = getattr(self, "handle", None)
        try:
            if h is not None and h.value and _lib._lib is not None:
                _lib.lib().tnlmi_batched_cg_destroy(h)
        except (AttributeError, TypeError):
            pass
        self.handle = None

    def solve(self, b, x, tolerance=1e-10, max_iterations=100_000, mixed=False, inner_tolerance=1e-4,
              use_graph=True, stream=None):
        """Asynchronous; returns the per-system (iterations, residues) device tensors."""
        _lib.check(_lib.lib().tnlmi_batched_cg_solve(self.handle, int(mixed), ctypes.c_void_p(b.data_ptr()),
                                                     ctypes.c_void_p(x.data_ptr()), tolerance, max_iterations,
                                                     inner_tolerance, ctypes.c_void_p(self.iters.data_ptr()),
                                                     ctypes.c_void_p(self.res.data_ptr()), int(use_graph),
                                                     _stream(stream)))
        return self.iters, self.res


CANDIDATES = [(CSR, 0), (SLICED_ELLPACK, 32), (SLICED_ELLPACK, 64), (ELLPACK, 0)]
BLOCKS = [256, 512, 1024]
LANES = [1, 2, 4]  # lanes per row: 64, 32 or 16 rows per wavefront


def _cache_path():
    return os.environ.get("TNL_AMD_AUTOTUNE_CACHE",
                          os.path.join(os.path.expanduser("~"), ".cache", "tnl_amd", "autotune.json"))


def _device_name():
    import torch
    p = torch.cuda.get_device_properties(0)
    return f"{p.name}:{getattr(p, 'gcnArchName', '')}"


# The FP64 kernel from LDS and registers takes a batch whose systems all have at
# most LOCAL_ROWS rows and LOCAL_SLOTS slots per row (kLocalMost and kLocalWidth of
# csrc/batched.hip).
LOCAL_ROWS, LOCAL_SLOTS = 16384, 8


def _sample(off, cols, vals, sys_rows, k):
    """The first k systems as a batch of their own, and whether the FP64 solve of the
    whole batch runs in the kernel from LDS and registers.  If it does not though
    that of the first k would, the first system beyond its limits is added."""
    rows_of = np.diff(sys_rows)
    wide = np.flatnonzero(np.diff(off) > LOCAL_SLOTS)
    beyond = np.flatnonzero(rows_of > LOCAL_ROWS)
    first = [int(beyond[0])] if len(beyond) else []
    if len(wide):
        first.append(int(np.searchsorted(sys_rows, wide[0], side="right")) - 1)
    rows = int(sys_rows[k])
    o, c, v, s = off[: rows + 1], cols[: int(off[rows])], vals[: int(off[rows])], sys_rows[: k + 1]
    if first and min(first) >= k:
        r0, r1 = int(sys_rows[min(first)]), int(sys_rows[min(first) + 1])
        e0, e1 = int(off[r0]), int(off[r1])
        extra = cols[e0:e1]
        o = np.concatenate([o, off[r0 + 1 : r1 + 1] - e0 + o[-1]]).astype(off.dtype)
        c = np.concatenate([c, np.where(extra >= 0, extra - r0 + rows, extra)]).astype(cols.dtype)
        v = np.concatenate([v, vals[e0:e1]])
        s = np.append(s, rows + r1 - r0)
    return o, c, v, s, not first


def autotune(off, cols, vals, sys_rows, sample=256, candidates=CANDIDATES, blocks=BLOCKS, lanes=LANES,
             tolerance=1e-10, cache=True, log=None):
    """Times every (format, slice size, workgroup size, rows per wavefront)
    candidate on the first `sample` systems and returns the fastest as a dict.
    The FP64 solve is timed, or the mixed one where the FP64 solve of the batch
    runs in a kernel of its own, which no candidate shapes.  Results are cached in a JSON file
    keyed by the batch's shape, the solve timed, the device, the candidate lists and the
    tolerance."""
    import torch
    nsys = len(sys_rows) - 1
    k = min(sample, nsys)
    o, c, v, rows_k, mixed = _sample(*(a.cpu().numpy() if hasattr(a, "cpu") else np.asarray(a)
                                       for a in (off, cols, vals, sys_rows)), k)
    key = (f"batched_cg:solve={'mixed' if mixed else 'fp64'}:local={LOCAL_ROWS}x{LOCAL_SLOTS}:nsys={nsys}:rows={int(sys_rows[-1])}:nnz={int(off[-1])}:sample={sample}"
           f":device={_device_name()}:candidates={sorted((int(f), int(p)) for f, p in candidates)}"
           f":blocks={sorted(int(b) for b in blocks)}:lanes={sorted(int(t) for t in lanes)}"
           f":tolerance={float(tolerance)!r}")
    path = _cache_path()
    if cache and os.path.exists(path):
        with open(path) as f:
            db = json.load(f)
        if key in db:
            return db[key]
    rows = int(rows_k[-1])
    b = torch.ones(rows, dtype=torch.float64, device="cuda")
    x = torch.zeros(rows, dtype=torch.float64, device="cuda")
    trials = []
    for fmt, param in candidates:
        A = SparseMatrix.from_csr(rows, rows, o, c, v, fmt=fmt, param=param)
        A_lo = SparseMatrix(A.rows, A.columns, A.segments, A.values.float(), A.column_indexes) if mixed else None
        for bs in blocks:
            for lpr in lanes:
                bc = BatchedCG(A, rows_k, A_lo, block_size=bs, lanes_per_row=lpr)
                x.zero_()
                bc.solve(b, x, tolerance, mixed=mixed, use_graph=False)
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                for _ in range(2):
                    x.zero_()
                    bc.solve(b, x, tolerance, mixed=mixed, use_graph=False)
                torch.cuda.synchronize()
                t = (time.perf_counter() - t0) / 2
                trials.append(dict(format=FORMAT_NAMES[fmt], format_id=fmt, param=param, block=bs, lanes_per_row=lpr,
                                   rows_per_wavefront=64 // lpr, seconds=t))
                if log:
                    log(f"autotune {FORMAT_NAMES[fmt]}{param or ''} block {bs} lanes/row {lpr}: {t * 1e3:.2f} ms")
        del A, A_lo
    best = min(trials, key=lambda d: d["seconds"])
    result = dict(best, trials=trials)
    if cache:
        db = {}
        if os.path.exists(path):
            with open(path) as f:
                db = json.load(f)
        db[key] = result
        os.makedirs(os.path.dirname(path), exist_ok=True)
        with open(path, "w") as f:
            json.dump(db, f, indent=1)
    return result
