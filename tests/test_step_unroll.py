"""The step kernel compiles with every value of its unroll macro, small ones
among them: no product is left with rounds of no blocks, which would not end
(a static assertion in spmv_rounds)."""
import os
import subprocess

import pytest

from mprgp_amd import build


@pytest.mark.parametrize("unroll", [1, 2, 3, 4])
def test_step_kernel_compiles(unroll):
    r = subprocess.run([build.HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "--cuda-device-only",
                        f"-DMPRGP_STEP_UNROLL={unroll}", "-I", os.path.join(build.HERE, "..", "include"),
                        os.path.join(build.CSRC, "mprgp_kernels.hip")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
