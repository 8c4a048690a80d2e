"""GPU parity: the HIP library against the CPU oracle on the same seeded
inputs.  The FP64 drop-in is built with -ffp-contract=off, as is the oracle,
so results are compared bit for bit (+0 == -0); the stated tolerances of the
path (1e-12 relative per step, 1e-10 after 10 steps) are checked as well.

Each test prints the case it runs before touching the GPU."""
import sys

import numpy as np
import pytest

import licom_synth as ls
import licom_tracer as lt
import orc
from helpers import inner, mismatch, rel_err, report

pytestmark = pytest.mark.gpu

STATE_OUT = ("at", "atb", "ws", "utf", "vtf", "h0f", "akt")
DIAG_OUT = ("ax", "ay", "az", "dz", "tend", "dt_diff", "dt_conv", "penetrate")


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def forcing_case(case, seed=7):
    rng = np.random.default_rng(seed)
    j, i = case.jmt, case.imt
    f = case.forcing
    f["swv"] = rng.uniform(0, 200, (j, i))
    f["nswv"] = rng.uniform(-150, 50, (j, i))
    f["sst"] = rng.uniform(5, 25, (j, i))
    f["seaice"] = rng.uniform(0, 0.3, (j, i))
    f["sss"] = rng.uniform(-2e-3, 1e-3, (j, i))
    f["fresh"] = rng.uniform(-1e-5, 1e-5, (j, i))
    case.params["gamma"] = 1.0 / (30.0 * 86400.0)
    return case


def compare(model, oracle_state, oracle_diag, tag, exact=True, tol=1e-12):
    gs = model.host_state()
    gd = model.host_diag()
    msgs, bad = [], []
    for k in STATE_OUT:
        a, b = gs[k], oracle_state[k]
        if k == "ws":    # interface 0 is an input; 1..km-1 computed on [1,jmt-1)x[1,imt-1)
            a, b = a[1:-1, 1:-1, 1:-1], b[1:-1, 1:-1, 1:-1]
        n, e = mismatch(a, b), rel_err(a, b)
        msgs.append(report(k, a, b))
        if (exact and n) or e > tol:
            bad.append(k)
    for k in DIAG_OUT:
        a, b = inner(gd[k]), inner(oracle_diag[k])
        n, e = mismatch(a, b), rel_err(a, b)
        msgs.append(report(k, a, b))
        if (exact and n) or e > tol:
            bad.append(k)
    a, b = gd["net"], oracle_diag["net"]
    kmt = model.case.grid["kmt"]
    a, b = a[:, kmt > 0], b[:, kmt > 0]
    if mismatch(a, b) and rel_err(a, b) > tol:
        bad.append("net")
    print(f"[{tag}] " + "; ".join(msgs), flush=True)
    assert not bad, f"{tag}: mismatch in {bad}"


def run_pair(case, steps, flags=lt.LICOM_STEP_SIDE_EFFECTS | lt.LICOM_STEP_CONVADJ, exact=True,
             tol=1e-12):
    o = orc.Oracle(case)
    st = case.copy_state()
    od = orc.Oracle.new_diag(case)
    m = lt.TracerModel(case)
    for s in range(steps):
        o.step(st, od, convadj=int(bool(flags & lt.LICOM_STEP_CONVADJ)))
        m.tracer(s, flags)
    compare(m, st, od, f"{case.name} x{steps}", exact=exact, tol=tol)
    m.close()


@pytest.mark.parametrize("name,over", [
    ("C1", {}),
    ("C1-land", dict(depth_min=-3000.0, depth_max=5000.0, sigma=1.5, seed=11)),
    ("C1-del4", dict(hmix=4, ah=-1.0e10)),
])
def test_one_step_bitwise(name, over, need_gpu):
    announce(f"one step {name} {over}")
    case = ls.make_case("C1", **over)
    case.name = name
    run_pair(case, 1)


def test_ten_steps_c1_bitwise(need_gpu):
    announce("ten steps C1")
    run_pair(ls.make_case("C1"), 10, tol=1e-10)


def test_ten_steps_c2_bitwise(need_gpu):
    announce("ten steps C2")
    run_pair(ls.make_case("C2"), 10, tol=1e-10)


def test_staged_kernels_match_oracle(need_gpu):
    """The one-kernel-per-stage cross-check path gives the same bits."""
    announce("staged path C1-land del4 x3")
    case = ls.make_case("C1", depth_min=-3000.0, sigma=1.5, seed=11, hmix=4, ah=-1.0e10)
    case.name = "C1-staged"
    run_pair(case, 3, flags=lt.LICOM_STEP_SIDE_EFFECTS | lt.LICOM_STEP_CONVADJ | lt.LICOM_STEP_STAGED,
             tol=1e-10)


def test_forcing_restore_sssnorm(need_gpu):
    """Non-zero surface forcing (FRC_CORE fluxes, SSSNORM) and restoring.
    The SSSNORM sum runs in a different order on the device (compensated
    tree vs the host's plain loop), so this case is checked to 1e-12."""
    announce("forcing + restore C1")
    case = forcing_case(ls.make_case("C1", depth_min=-2000.0, sigma=2.0, seed=5))
    case.params["boundary_restore"] = 1
    case.forcing["restore"] = case.state["at"] + 0.5
    case.name = "C1-forcing"
    run_pair(case, 1, exact=False, tol=1e-12)


def test_tracer_without_convadj_and_convadj_alone(need_gpu):
    """tracer_ alone, then convadj_ as a separate entry (the GPU driver's
    ii==0 cadence)."""
    announce("tracer then convadj C1")
    case = ls.make_case("C1")
    o = orc.Oracle(case)
    st = case.copy_state()
    od = orc.Oracle.new_diag(case)
    o.step(st, od, convadj=0)
    o.convadj(st, od)
    m = lt.TracerModel(case)
    m.tracer(0, lt.LICOM_STEP_SIDE_EFFECTS)
    m.convadj()
    compare(m, st, od, "C1 tracer+convadj")
    m.close()


def test_derived_masks_and_coefficients_bitwise(need_gpu):
    """kmt/kmu bit-exact and every derived coefficient identical."""
    announce("derived grid C1-land, del2 and del4")
    for hmix, ah in ((2, 1e3), (4, -1e10)):
        case = ls.make_case("C1", depth_min=-3000.0, sigma=1.5, seed=11, hmix=hmix, ah=ah)
        o = orc.Oracle(case)
        m = lt.TracerModel(case, diagnostics=False)
        d = m.derived()
        assert np.array_equal(d["kmt"], o.kmt)
        assert np.array_equal(d["kmu"], o.d["kmu"])
        for k in ("tarea_r", "ohbt", "ohbu", "dtn", "dts", "dte", "dtw", "ahf", "dzp", "odzp", "odzt"):
            assert np.array_equal(d[k], o.d[k]), k
        assert d["area_t"] == o.area_t
        m.close()


def test_wide_grid_bitwise(need_gpu):
    """520 columns: the solve takes one 128-column row per workgroup (the
    launch used for the 0.1 deg grid) and a row holds more than four of the
    update's 124-cell runs; two steps with del4, bit for bit."""
    announce("two steps 520x24x12 del4 (wide-grid launch shapes)")
    case = ls.make_case("C1", nx=520, ny=24, km=12, seed=21, hmix=4, ah=-1.0e10)
    case.name = "C1-wide"
    run_pair(case, 2)


def test_full_size_content_and_masks(need_gpu):
    """At the 0.1 deg workload size (3600x2302x55, del4, dt=600 s, no surface
    forcing): kmt as exported is the generator's bit for bit, and the T and S
    contents sum(dzp*tarea*vit*at) are conserved over two steps with convadj
    to 1e-11 relative (FP64 roundoff of 455.8 M cells; the oracle's own pin
    of the same property holds to 1e-13 with exact summation)."""
    import torch
    announce("full size 3600x2302x55: content conservation over 2 steps")
    case = ls.make_case("C3")
    kmt = case.grid["kmt"]
    tarea = case.grid["tarea"]
    m = lt.TracerModel(case, diagnostics=False)
    case.state = None
    d = m.derived()
    assert np.array_equal(d["kmt"], kmt)
    dev = m.state["at"].device
    km = case.km
    vit = torch.arange(km, device=dev)[:, None, None] < torch.from_numpy(kmt).to(dev)[None]
    w = (torch.from_numpy(d["dzp"]).to(dev)[:, None, None] * torch.from_numpy(tarea).to(dev)[None]
         * vit)[:, 2:-2, 2:-2]
    del vit

    def content():
        m.sync()
        return [float((w * m.state["at"][n, :, 2:-2, 2:-2]).sum()) for n in range(2)]

    before = content()
    flags = lt.LICOM_STEP_SIDE_EFFECTS | lt.LICOM_STEP_CONVADJ
    for s in range(2):
        m.tracer(s, flags)
    after = content()
    rel = [abs(a - b) / abs(b) for a, b in zip(after, before)]
    print(f"[full size] T content {before[0]:.6e} -> {after[0]:.6e} (rel {rel[0]:.2e}), "
          f"S content {before[1]:.6e} -> {after[1]:.6e} (rel {rel[1]:.2e})", flush=True)
    m.close()
    del w, m
    torch.cuda.empty_cache()
    assert rel[0] <= 1e-11 and rel[1] <= 1e-11
