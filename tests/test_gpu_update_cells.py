"""GPU parity of k_flags / k_update where their cell runs can go wrong, bit for
bit against the oracle: row lengths below, at and above a wave's 124 cells,
odd rows (every other row starts on an odd cell of a lane's pair), two rows of
ocean, two and three levels (no level between the first and the last), and a
plane wide enough that a workgroup walks whole columns."""
import numpy as np
import pytest

import licom_synth as ls
from test_gpu_parity import announce, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hmix", [2, 4], ids=["del2", "del4"])
@pytest.mark.parametrize("nx,ny,km", [(4, 2, 2), (5, 4, 3), (8, 6, 4), (27, 9, 5), (119, 6, 4), (120, 5, 7), (121, 7, 3),
                                      (225, 16, 55), (701, 383, 3)])
def test_update_cells_bitwise(nx, ny, km, hmix, need_gpu):
    announce(f"k_flags / k_update {nx}x{ny}x{km} del{hmix}")
    over = dict(dlat=0.2, nx=nx, ny=ny, km=km, seed=31 + nx, depth_min=-3000.0, depth_max=5000.0, sigma=1.5)
    if hmix == 4:
        over.update(hmix=4, ah=-1.0e10)
    case = ls.make_case("C1", **over)
    case.name = f"{nx}x{ny}x{km} del{hmix}"
    assert np.any(case.grid["kmt"] > 0)
    run_pair(case, 2, tol=1e-10)
