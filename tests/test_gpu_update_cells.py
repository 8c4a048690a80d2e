"""GPU parity of k_flags / k_update where their cell runs can go wrong, bit for
bit against the oracle: row lengths below, at and above a wave's 124 cells,
odd rows (every other row starts on an odd cell of a lane's pair), two rows of
ocean, two and three levels (no level between the first and the last), and a
plane wide enough that a workgroup walks whole columns."""
import numpy as np
import pytest

import licom_ensemble as le
import licom_synth as ls
import licom_tracer as lt
from test_gpu_mixed import FLAGS, errors
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


@pytest.mark.parametrize("hmix", [2, 4], ids=["del2", "del4"])
@pytest.mark.parametrize("nx,ny,km", [(4, 2, 2), (8, 6, 4), (118, 6, 4), (120, 5, 7), (122, 7, 3), (226, 16, 55),
                                      (702, 383, 3)])
def test_mixed_update_cells(nx, ny, km, hmix, need_gpu):
    """k_flags_mx / k_update_mx at the same edges, one step against the FP64
    path (the one-step bound of test_gpu_mixed.py), and the batched kernels
    (del2 and del4 members, fewer workgroups than items) bit for bit."""
    announce(f"k_flags_mx / k_update_mx {nx}x{ny}x{km} del{hmix}")
    over = dict(dlat=0.2, nx=nx, ny=ny, km=km, seed=31 + nx, depth_min=-3000.0, depth_max=5000.0, sigma=1.5)
    if hmix == 4:
        over.update(hmix=4, ah=-1.0e10)
    case = ls.make_case("C1", **over)
    ref, got, one, other = (lt.TracerModel(case, precision=p) for p in ("fp64", "mixed", "mixed", "mixed"))
    ref.tracer(0, FLAGS)
    got.tracer(0, FLAGS)
    a, b = got.host_state(), ref.host_state()
    dT, dS = errors(case, a["at"], b["at"])
    print(f"max|dT| {dT:.3e} K, max|dS| {dS:.3e} psu", flush=True)
    assert dT <= 1e-6 and dS <= 1e-6
    ens = le.Ensemble([one, other], march_grid=11)
    ens.step(1)
    ens.sync()
    for m in (one, other):
        c = m.host_state()
        assert all(np.array_equal(a[k], c[k]) for k in ("at", "atb", "ws"))
        assert all(np.array_equal(got.host_diag()[k], m.host_diag()[k]) for k in ("ax", "ay", "az", "dz", "penetrate"))
    ens.close()
    for m in (ref, got, one, other):
        m.close()
