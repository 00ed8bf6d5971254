"""CPU checks of the strip solves.  The host's plans of the strip solves (ILU(0) factors): every factor that
tests/test_tri_strips_gpu.py solves is planned as it is meant to be, and the
imports that the solving wave can wait for fit the LDS ring that holds them."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import test_tri_strips_gpu as gpu_cases
from test_barrier_loops import CSRC, HIPCC, ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(ROOT, "tnl_amd", "libtnlmi.so")


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if not os.path.exists(HIPCC) or not os.path.exists(LIB):
        pytest.skip("hipcc or the library is missing")
    so = str(tmp_path_factory.mktemp("plan") / "strips_plan.so")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-O1", "-std=c++17", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, os.path.join(HERE, "strips_plan.cpp"), "-o", so,
                    "-L" + os.path.dirname(LIB), "-ltnlmi", "-Wl,-rpath," + os.path.dirname(LIB)],
                   check=True, capture_output=True)
    lib = ctypes.CDLL(so)
    lib.strips_plan.argtypes = [ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_double,
                                ctypes.c_void_p]
    return lib


def _factor(off, cols, upper):
    """(ptr, col) of a factor's pattern in solve order, the upper rows reversed with the pivot first."""
    n = len(off) - 1
    row = np.repeat(np.arange(n), np.diff(off))
    keep = cols >= row if upper else cols < row
    r, c = row[keep], cols[keep]
    order = np.lexsort((c, n - 1 - r if upper else r))
    count = np.bincount(n - 1 - r if upper else r, minlength=n)
    return np.concatenate([[0], np.cumsum(count)]).astype(np.int32), c[order].astype(np.int32)


def _levels_us(ptr, col, upper):
    """What the solves by levels are expected to take, as ilu0_build counts it."""
    n = len(ptr) - 1
    level = np.zeros(n, np.int64)
    for t in range(n):
        for g in range(ptr[t] + (1 if upper else 0), ptr[t + 1]):
            level[t] = max(level[t], level[n - 1 - col[g] if upper else col[g]] + 1)
    us, narrow = 0.0, False
    for width in np.bincount(level):
        if width > 2048:
            us += 5.0
        else:
            us += 0.65 if narrow else 10.65
        narrow = width <= 2048
    return us


def _plan(planner, off, cols, upper):
    ptr, col = _factor(off, cols, upper)
    strips = ctypes.c_int32()
    most = planner.strips_plan(len(ptr) - 1, ptr.ctypes.data, col.ctypes.data, int(upper),
                               _levels_us(ptr.tolist(), col.tolist(), upper), ctypes.byref(strips))
    return strips.value, most


@pytest.mark.parametrize("name", gpu_cases.CASES)
def test_cases_are_planned_as_meant(planner, name):
    off, cols, _ = gpu_cases.CASES[name](np.random.default_rng(61))
    full = 0
    for upper in (False, True):
        strips, most = _plan(planner, off, cols, upper)
        low, high = gpu_cases.STRIPS[name]
        assert low <= strips <= high
        full = max(full, most)
        # the solving wave waits for a group's imports before it has published the
        # group before as used: both must be in the ring at a time
        assert most <= planner.strips_imports()
    if name in gpu_cases.FULL_RING:
        assert full > 1100  # (two groups of three imports per row: 1,152)


@pytest.mark.parametrize("width,lines", [(5000, 3), (6000, 20), (300, 400)])
def test_any_plan_fits_the_ring(planner, width, lines):
    """The strips at their fullest, whether or not another solve is expected to be faster."""
    off, cols, _ = gpu_cases._far(width, lines, np.random.default_rng(1))
    for upper in (False, True):
        ptr, col = _factor(off, cols, upper)
        strips = ctypes.c_int32()
        most = planner.strips_plan(len(ptr) - 1, ptr.ctypes.data, col.ctypes.data, int(upper), 1e9, ctypes.byref(strips))
        assert strips.value > 0 and most <= planner.strips_imports()
        assert width < 1000 or most == 1152


def test_no_strips_that_wait_too_long(planner):
    """Eight chains of rows: 8 rows a step, strip after strip.  The last strip would wait
    for all steps, longer than a wait may last by default."""
    n = 17000000
    row = np.arange(n, dtype=np.int64)
    ptr = np.maximum(np.arange(n + 1) - 8, 0).astype(np.int32)
    col = (row[8:] - 8).astype(np.int32)
    strips = ctypes.c_int32(-1)
    planner.strips_plan(n, ptr.ctypes.data, col.ctypes.data, 0, 1e9, ctypes.byref(strips))
    assert strips.value == 0
    m = 800000  # (the same, shorter)
    planner.strips_plan(m, ptr.ctypes.data, col.ctypes.data, 0, 1e9, ctypes.byref(strips))
    assert strips.value > 0


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_strips_are_taken_in_the_order_of_starting(tmp_path):
    """A strip waits for earlier ones, and workgroups need not start in the order of
    their numbers (each XCD starts its own): every solve kernel takes its strip
    from a counter, by an atomic that returns the value before."""
    out = tmp_path / "tri_strips.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "--cuda-device-only", "-S",
                    "-o", str(out), os.path.join(CSRC, "tri_strips.hip")], check=True, capture_output=True)
    kernels = re.findall(r"^(_Z\w*10tri_stripsI\w*):(.*?)s_endpgm", out.read_text(), re.M | re.S)
    assert len(kernels) == 4
    for name, body in kernels:
        first = body.index("s_barrier")
        assert re.search(r"global_atomic_add v\d+, .* sc0", body[:first]), name
