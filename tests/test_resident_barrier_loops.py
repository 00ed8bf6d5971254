"""The solvers that stay resident for many iterations loop around workgroup
barriers: every such loop's exit is a scalar branch in the built assembly."""
import os
import subprocess

import pytest

import barrier_loops
from test_barrier_loops import CSRC, HIPCC, ROOT


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("src", ["krylov_resident.hip", "tri_strips.hip", "krylov_ns.hip", "spmv.hip"])
def test_uniform_barrier_loops(tmp_path, src):
    out = tmp_path / (src + ".s")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "--cuda-device-only", "-S",
           "-o", str(out), os.path.join(CSRC, src)]
    subprocess.run(cmd, check=True, capture_output=True)
    assert barrier_loops.scan(out.read_text()) == []
