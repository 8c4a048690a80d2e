"""The column solve's convadj (csrc/tracer_convect.h) on the host, under
AddressSanitizer and UndefinedBehaviorSanitizer, bit for bit against the
oracle (oracle/convect_driver.cpp, built by `make -C oracle convect`): random
columns of 2 to 64 levels with mixed regions at the surface, at the bottom
and several to a column, every array of exactly the extent that the routine
may touch.  CPU only."""
import os
import shutil
import subprocess

import pytest

ORACLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle")


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("gcc") is None, reason="needs the host compilers")
def test_convadj_of_the_column_solve_stays_in_bounds_and_equals_the_oracle():
    b = subprocess.run(["make", "-C", ORACLE, "convect"], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stdout[-2000:] + b.stderr[-2000:]
    r = subprocess.run([os.path.join(ORACLE, "_san", "convect_driver")], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="halt_on_error=1:verify_asan_link_order=0",
                                UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1"))
    out = r.stdout + r.stderr
    assert r.returncode == 0 and out.startswith("ok "), out[-4000:]
