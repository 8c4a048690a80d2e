"""Workgroup size of the Canuto producer (csrc/turb_shape.h): four waves on
the 0.1 degree grid and a quarter of it, which one wave made 10% and 6%
slower, one wave on the blocks that it was taken for.  CPU only."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "licom3-hip_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs the host compiler")
@pytest.mark.parametrize("nx,ny,lanes", [(3600, 2302, 256), (1800, 1151, 256), (1400, 900, 64), (900, 576, 64),
                                         (360, 218, 64), (128, 96, 64), (1, 1, 64)])
def test_turb_lanes(nx, ny, lanes):
    src = f'#include "turb_shape.h"\nstatic_assert(licom::turb_lanes((size_t){nx + 4} * {ny + 4}) == {lanes}, "");\n'
    r = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", CSRC, "-x", "c++", "-"], input=src, text=True,
                       capture_output=True, timeout=60)
    assert r.returncode == 0, r.stderr
