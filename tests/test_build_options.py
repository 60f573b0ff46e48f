"""Build options that the kernels cannot serve end the build."""
import os
import subprocess

import pytest

from anerend_amd import build


@pytest.mark.parametrize("define", ["ANE_TRACE_STACK=12", "ANE_TRACE_BLOCK=192"])
def test_ring_sizes_other_than_powers_of_two_do_not_build(define):
    """The traversal's stack ring wraps by a mask: at 12 entries levels would share one."""
    res = subprocess.run([build.hipcc(), "--offload-arch=gfx950", "-std=c++17", "--cuda-device-only", "-fsyntax-only",
                          "-D" + define, os.path.join(build.CSRC, "trace.hip")], capture_output=True, text=True)
    assert res.returncode != 0 and "powers of two" in res.stderr
