"""FP64 step on odd row lengths and on arrays that are only 8-byte aligned,
which take the fused kernels like every other layout: the three advection
schemes with surface forcing, restoring, icesnow and convadj, the VTL_SCRATCH
forms, and the limiter flags cell for cell, against the oracle (bit for bit,
but for the SSSNORM sum, whose order differs) and a numpy restatement of the
tspas predictor.  The forms that refuse such layouts still do."""
import ctypes

import numpy as np
import pytest

import licom_synth as ls
import licom_tracer as lt
import orc
from helpers import inner, mismatch, plant_cold
from test_gpu_parity import announce, compare, forcing_case

pytestmark = pytest.mark.gpu

SIDE, CONV, ICE, VTL = (lt.LICOM_STEP_SIDE_EFFECTS, lt.LICOM_STEP_CONVADJ, lt.LICOM_STEP_ICESNOW,
                        lt.LICOM_STEP_VTL_SCRATCH)
# odd rows with odd and even row counts, one chunk of two levels, several
# chunks, and a width just over a wave's 124 cells
SHAPES = [(61, 37, 2), (63, 40, 13), (121, 22, 30)]


def build(nx, ny, km, adv, hmix, seed=51, sssnorm=0):
    over = dict(hmix=4, ah=-1.0e10) if hmix == 4 else {}
    case = ls.make_case("C1", nx=nx, ny=ny, km=km, seed=seed, depth_min=-3000.0, depth_max=5000.0, sigma=1.5,
                        t_noise=0.6, s_noise=0.2, **over)
    forcing_case(case)
    plant_cold(case, case.state, seed)
    case.params.update(adv=adv, nss=3, boundary_restore=1, sssnorm=sssnorm)
    case.forcing["restore"] = case.state["at"] + 0.5
    case.name = f"{nx}x{ny}x{km} adv={adv} del{hmix}"
    return case


def oracle_steps(case, steps):
    """tracer_, icesnow_, convadj_ (stepon.cpp:69-75)."""
    o = orc.Oracle(case)
    st, od, q = case.copy_state(), orc.Oracle.new_diag(case), np.zeros((case.jmt, case.imt))
    froze = mixed = 0
    for _ in range(steps):
        o.step(st, od, convadj=0)
        o.icesnow(st, q, reset=True)
        before = st["at"].copy()
        o.convadj(st, od)
        froze += int(np.count_nonzero(q))
        mixed += int((st["at"] != before).any(axis=(0, 1)).sum())
    print(f"{froze} columns froze, {mixed} mixed", flush=True)
    assert froze > 0 and mixed > 0
    return st, od, q


@pytest.mark.parametrize("hmix", [2, 4], ids=["del2", "del4"])
@pytest.mark.parametrize("adv", [ls.ADV_CENTERED, ls.ADV_FLUX, ls.ADV_TSPAS], ids=["centered", "flux", "tspas"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_odd_widths_forced_with_icesnow_bitwise(shape, adv, hmix, need_gpu):
    case = build(*shape, adv, hmix)
    announce(f"odd width, forced, icesnow: {case.name}")
    st, od, q = oracle_steps(case, 2)
    m = lt.TracerModel(case)
    for s in range(2):
        m.tracer(s, SIDE | CONV | ICE)
    assert mismatch(m.licomqice.cpu().numpy(), q) == 0
    compare(m, st, od, case.name, exact=True, tol=1e-10)
    m.close()


def test_odd_width_with_sssnorm(need_gpu):
    case = build(63, 40, 13, ls.ADV_TSPAS, 4, sssnorm=1)
    announce(f"odd width, SSSNORM: {case.name}")
    st, od, q = oracle_steps(case, 1)
    m = lt.TracerModel(case)
    m.tracer(0, SIDE | CONV | ICE)
    compare(m, st, od, case.name, exact=False, tol=1e-12)
    m.close()


@pytest.mark.parametrize("ice", [False, True], ids=["split", "staged by icesnow"])
def test_odd_width_vtl_scratch(ice, need_gpu):
    case = build(63, 40, 13, ls.ADV_TSPAS, 2)
    announce(f"odd width, VTL_SCRATCH, icesnow {ice}: {case.name}")
    o = orc.Oracle(case)
    st, od, q = case.copy_state(), orc.Oracle.new_diag(case), np.zeros((case.jmt, case.imt))
    o.step(st, od, convadj=0)
    vtl = st["at"][1].copy()          # tracer_'s S (tracer.cpp:1891)
    if ice:
        o.icesnow(st, q, reset=True)
    o.convadj(st, od)
    assert (st["at"][1] != vtl).any()
    m = lt.TracerModel(case)
    m.tracer(0, SIDE | CONV | VTL | (ICE if ice else 0))
    compare(m, st, od, f"vtl {case.name}", exact=True)
    assert mismatch(m.host_state()["vtl"], vtl) == 0
    m.close()


def misalign(m):
    """Every 3-D array of the model one double off a 16-byte boundary."""
    def off(t):
        v = m.torch.zeros(t.numel() + 2, dtype=t.dtype, device=t.device)[1:1 + t.numel()].view(t.shape)
        v.copy_(t)
        assert v.data_ptr() % 16 == 8
        return v
    for d in (m.state, m.diag):
        for k, t in d.items():
            if t.dim() >= 3:
                d[k] = off(t)
    m.restore = off(m.restore)


@pytest.mark.parametrize("adv", [ls.ADV_CENTERED, ls.ADV_TSPAS], ids=["centered", "tspas"])
@pytest.mark.parametrize("nx", [63, 64])
def test_arrays_off_16_byte_alignment_bitwise(nx, adv, need_gpu):
    case = build(nx, 40, 13, adv, 4)
    announce(f"arrays off 16-byte alignment: {case.name}")
    st, od, q = oracle_steps(case, 2)
    m = lt.TracerModel(case)
    misalign(m)
    for s in range(2):
        m.tracer(s, SIDE | CONV | ICE)
    assert mismatch(m.licomqice.cpu().numpy(), q) == 0
    compare(m, st, od, f"misaligned {case.name}", exact=True, tol=1e-10)
    m.close()


def limiter_flags(case, ws):
    """tspas limiter flags of the physical cells (tracer.cpp:311-545) from the
    state before the step and the step's vertical velocity."""
    o = orc.Oracle(case)
    p, g, d, km = case.params, case.grid, o.d, case.km
    S = case.state
    oncc, dts = p["oncc"], p["dts"]
    uw, vs = o.faces(ls.ADV_TSPAS, 0.5 * (S["utf"] * oncc) + 0.5 * S["utl"], 0.5 * (S["vtf"] * oncc) + 0.5 * S["vtl"])
    C, E, W, N, So = ((slice(2, -2), slice(2, -2)), (slice(2, -2), slice(3, -1)), (slice(2, -2), slice(1, -3)),
                      (slice(1, -3), slice(2, -2)), (slice(3, -1), slice(2, -2)))
    tr, kmt = d["tarea_r"][C], g["kmt"]
    dx, dy = g["htw"] * g["hun"], g["hts"] * g["hue"]
    out = np.zeros((2, km, case.jmt - 4, case.imt - 4), np.uint8)
    for n in range(2):
        for k in range(km):
            T, oz, ot = S["at"][n], d["odzp"][k], d["odzt"][k]
            Tc, Te, Tw, Tn, Ts = (T[k][s] for s in (C, E, W, N, So))
            Ue, Uw, Vs, Vn = uw[k][E], uw[k][C], vs[k][C], vs[k][N]
            x0 = (Te + Tc) * Ue * tr - (Tc + Tw) * Uw * tr
            y0 = ((Ts + Tc) * Vs - (Tc + Tn) * Vn) * tr
            c1, c2 = -Tc * (Ue - Uw) * tr * 2.0, -Tc * (Vs - Vn) * tr * 2.0
            xy1 = -dts * (Te - Tc) * 2.0 * tr * Ue * Ue / dx[E]
            xy2 = dts * (Tc - Tw) * 2.0 * tr * Uw * Uw / dx[C]
            xy3 = -dts * (Ts - Tc) * 2.0 * tr * Vs * Vs / dy[C]
            xy4 = dts * (Tc - Tn) * 2.0 * tr * Vn * Vn / dy[N]
            Wk, zb1, zb2 = ws[k][C], 0.0, 0.0
            if k > 0:
                Tu = T[k - 1][C]
                zb1 = -0.5 * oz * Wk * Wk * ot * (Tu - Tc) * dts
            if k < km - 1:
                Td, Wb = T[k + 1][C], ws[k + 1][C]
                zb2 = 0.5 * oz * Wb * Wb * d["odzt"][k + 1] * (Tc - Td) * dts
            if k == 0:
                za, zc = -0.5 * oz * Wb * (Td + Tc), oz * Tc * Wb
            elif k == km - 1:
                za, zc = 0.5 * oz * Wk * (Tc + Tu), -oz * Tc * Wk
            else:
                za = 0.5 * oz * Wk * (Tc + Tu) - 0.5 * oz * Wb * (Tc + Td)
                zc = -oz * Tc * (Wk - Wb)
            a00 = Tc + (-(x0 + xy1 + xy2 + c1) + -(y0 + xy3 + xy4 + c2) + -(zb1 + zb2 + za + zc)) * dts
            near = [(Tc, kmt[C] > k)] + [(v, kmt[s] > k) for v, s in ((Tn, N), (Ts, So), (Tw, W), (Te, E))]
            near += [(Tu, kmt[C] > k - 1)] if k > 0 else []
            near += [(Td, kmt[C] > k + 1)] if k < km - 1 else []
            hi = np.max([np.where(wet, v, -1.0e10) for v, wet in near], axis=0)
            lo = np.min([np.where(wet, v, 1.0e10) for v, wet in near], axis=0)
            out[n, k] = (a00 > hi) | (a00 < lo)
    return out


@pytest.mark.parametrize("shape", SHAPES + [(64, 37, 13)], ids=str)
def test_limiter_flags_cell_for_cell(shape, need_gpu):
    case = build(*shape, ls.ADV_TSPAS, 4)
    announce(f"limiter flags: {case.name}")
    m = lt.TracerModel(case)
    m.limiter_flags()
    m.tracer(0, SIDE | CONV)
    got = inner(m.flags.cpu().numpy())
    want = limiter_flags(case, m.host_state()["ws"])
    print(f"{int(want.sum())} of {want.size} cells limited, {mismatch(got, want)} differ", flush=True)
    assert 0 < want.sum() < want.size and mismatch(got, want) == 0
    m.close()


@pytest.mark.parametrize("nx,shift", [(63, 0), (64, 1)], ids=["odd width", "off alignment"])
def test_forms_that_refuse_these_layouts_still_do(nx, shift, need_gpu):
    case = build(nx, 40, 13, ls.ADV_TSPAS, 2)
    announce(f"refused layouts: {case.name} shift {shift}")
    m = lt.TracerModel(case)
    if shift:
        misalign(m)
    F, D = m._fields(), m._diag()
    with pytest.raises(lt.LicomError, match="even imt"):
        lt.check(lt.lib().licom_tracer_step_noalloc(m.ctx, ctypes.byref(F), ctypes.byref(D), SIDE), "noalloc")
    m.close()
    m = lt.TracerModel(case, precision="mixed")
    if shift:
        for k in ("at", "atb"):
            m.state[k] = m.torch.zeros(m.state[k].numel() + 2, dtype=m.state[k].dtype, device=m.device)[
                1:1 + m.state[k].numel()].view(m.state[k].shape).copy_(m.state[k])
    with pytest.raises(lt.LicomError, match="even imt"):
        m.step()
    m.close()
