"""GPU parity of the Canuto producer on both sides of the line between its
workgroup sizes, at column counts that leave the last workgroup part empty:
the checks of test_gpu_turb.py."""
import pytest

import licom_synth as ls
from test_gpu_turb import announce, check, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1599, 976), (1603, 981)], ids=["64 lanes", "256 lanes"])
def test_turb_either_side_of_the_workgroup_line(nx, ny, need_gpu):
    announce(f"turb {nx}x{ny}x5")
    c = ls.make_case("C3", nx=nx, ny=ny, km=5, seed=6)
    cols = c.imt * c.jmt
    assert cols % 256 and (cols < 3 << 19) == (nx == 1599)
    out, ref, _ = run_both(ls.make_turb_case(c, seed=6))
    check(out, ref, f"turb {nx}x{ny}")
