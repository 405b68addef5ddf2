"""The documented compile-time options of the kernels: every translation unit
that shares them compiles with each (front end only, no GPU needed)."""
import os
import subprocess

import pytest

from hyperelasticsolver_amd import build

SOURCES = [s for s in build.SOURCES if s != "hes_noalloc.hip"]  # it moves no values between lanes


@pytest.mark.parametrize("source", SOURCES)
def test_lane_shifts_by_the_lds_crossbar(source):
    flags = [f for f in build.HIPCC_FLAGS if f != "-shared"]
    r = subprocess.run([build.hipcc(), *flags, "-DHES_DPP_SHIFT=0", "-fsyntax-only",
                        os.path.join(build.CSRC, source)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
