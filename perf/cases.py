"""Workloads of the tracer framework, for timing and for checking its outputs.

A case is a dict of plain values; ``kind`` names the entry point it goes
through:

* ``step``     one FP64 model step, ``TracerModel.step`` (tracer_ + convadj_),
               with the options a model run sets: del2 or del4 mixing, the three
               advection schemes, surface forcing with restoring and the
               freshwater normalisation, icesnow_, diagnostics on or off
* ``mixed``    the same step in the mixed-precision form
* ``ensemble`` four steps of a batch of mixed-precision members of uneven sizes
               (``Ensemble.step``), the chunk a serving loop launches at a time
* ``readyt``, ``readyc``, ``turb``, ``barotr``, ``bclinc``  the other parts of a
               model step: density and pressure terms; shear, AKMU and momentum
               tendencies; the Canuto mixing coefficients; four barotropic
               subcycles; a leapfrog baroclinic momentum step

``exact`` restates each of them in plain torch, in 64 bits.  Grids are the
regional 0.5 degree, global 1 degree and 0.1 degree ones of
``licom_synth.WORKLOADS`` or blocks of them, of 30 or 55 levels; a block of a
domain that is cut over several GPUs has any width, odd ones included.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "licom3-hip_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import licom_barotr  # noqa: E402
import licom_bclinc  # noqa: E402
import licom_ensemble  # noqa: E402
import licom_readyc  # noqa: E402
import licom_readyt  # noqa: E402
import licom_synth as ls  # noqa: E402
import licom_tracer as lt  # noqa: E402
import licom_turb  # noqa: E402

DEV = "cuda:0"
F64 = dict(dtype=torch.float64, device=DEV)
DIAG3 = ("ax", "ay", "az", "dz", "tend", "dt_diff", "dt_conv")


def _c(name, kind, nx, ny, km, grid, **more):
    return dict(name=name, kind=kind, nx=nx, ny=ny, km=km, grid=grid, **more)


def listed():
    return [
        # the regional 0.5 degree domain on one GPU: a step of a few hundred microseconds
        _c("step_regional", "step", 128, 96, 30, "C1", hmix=2, adv=2, forced=False, ice=False, diag=True),
        # a block of the 0.1 degree domain cut over 16 x 16 GPUs: an odd width, biharmonic mixing
        _c("step_block_odd", "step", 225, 145, 55, "C3", hmix=4, adv=2, forced=False, ice=False, diag=True),
        # the 1 degree global domain with its surface forcing, restoring and sea ice
        _c("step_global_forced", "step", 360, 218, 30, "C2", hmix=2, adv=2, forced=True, ice=True, diag=True),
        # a quarter of the 0.1 degree domain, every diagnostic on: the largest call
        _c("step_tenth", "step", 1800, 1151, 55, "C3", hmix=4, adv=2, forced=False, ice=False, diag=True),
        # one small request of the serving loop, alone on its GPU
        _c("mixed_request", "mixed", 96, 64, 55, "C1", hmix=2, adv=2, forced=False, ice=False, diag=True),
        # a quarter of the 0.1 degree domain in the mixed-precision form
        _c("mixed_tenth", "mixed", 1800, 1151, 55, "C3", hmix=4, adv=2, forced=False, ice=False, diag=True),
        # members of uneven sizes advanced as one batch
        _c("ensemble", "ensemble", 360, 218, 55, "C1", members=16, shapes=4999),
        # the rest of a model step, on blocks of a cut 0.1 degree or on the 1 degree domain
        _c("readyt_block", "readyt", 900, 576, 55, "C3"),
        _c("readyc_block", "readyc", 900, 576, 55, "C3", hmix=4),
        _c("turb_global", "turb", 360, 218, 30, "C2"),
        _c("barotr_block", "barotr", 1800, 1151, 30, "C3", hmix=4),
        _c("bclinc_block", "bclinc", 360, 231, 55, "C3"),
    ]


def draw(rng):
    kind = rng.choice(("step", "step", "mixed", "ensemble", "readyt", "readyc", "turb", "barotr", "bclinc"))
    km = rng.choice((30, 55, rng.randint(20, 60)))
    if kind == "ensemble":
        return dict(kind=kind, nx=360, ny=218, km=55, grid="C1", members=rng.randint(2, 16), shapes=rng.randint(1, 1 << 20))
    nx = int(round(math.exp(rng.uniform(math.log(90), math.log(1800 if kind in ("step", "mixed") else 1200)))))
    ny = int(round(math.exp(rng.uniform(math.log(60), math.log(1100 if kind in ("step", "mixed") else 700)))))
    grid = rng.choice(("C1", "C3"))
    case = dict(kind=kind, nx=nx, ny=ny, km=km, grid=grid)
    if kind == "mixed":
        case["nx"] += nx % 2                     # the mixed form takes even widths only
    if kind in ("step", "mixed"):
        case.update(hmix=rng.choice((2, 4)), adv=2, forced=rng.random() < 0.5, ice=rng.random() < 0.5,
                    diag=rng.random() < 0.75)
        if kind == "step" and rng.random() < 0.25:
            case["adv"] = rng.choice((0, 1))
    if kind in ("readyc", "barotr"):
        case["hmix"] = rng.choice((2, 4))
    return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *s):
    return torch.randn(s, generator=g, **F64)


def _rand(g, *s):
    return torch.rand(s, generator=g, **F64)


def _smooth(g, ny, nx, scale=12):
    """A smooth field of zero mean and unit deviation with features of `scale` cells."""
    a = _randn(g, 1, 1, ny // scale + 3, nx // scale + 3)
    a = torch.nn.functional.interpolate(a, size=(ny, nx), mode="bicubic", align_corners=True)[0, 0]
    return (a - a.mean()) / a.std()


def _halo(a):
    """Cyclic ghost columns and zero ghost rows, as the model's halo update leaves them."""
    a[..., 0:2] = a[..., -4:-2]
    a[..., -2:] = a[..., 2:4]
    a[..., 0:2, :] = 0
    a[..., -2:, :] = 0
    return a


def _block(case, seed):
    """The grid of a case: metrics of the generator, bathymetry of its own (an ocean with land, shelves and deep basins)."""
    nx, ny, km = case["nx"], case["ny"], case["km"]
    spec = dict(ls.WORKLOADS[case["grid"]], nx=nx, ny=ny, km=km, seed=seed, sigma=0.0)
    if case["grid"] == "C1":
        spec["lat_north"] = 54.0
    if case["grid"] == "C1" and 54.0 - spec["dlat"] * (ny + 2) < -75.0:
        spec.update(lat_mode=1, dlon=0.5)
    cfg = ls.make_cfg(**spec)
    imt, jmt = nx + 4, ny + 4
    grid = {f: np.zeros((jmt, imt)) for f in ("htw", "hts", "hun", "hue", "tarea", "dxu", "dyu", "au0", "aus", "auw", "ausw")}
    grid.update(kmt=np.zeros((jmt, imt), np.int32), zkp=np.zeros(km + 1), pen=np.zeros(km - 1), to=np.zeros(km),
                so=np.zeros(km), eosc=np.zeros((9, km)), lat_t=np.zeros(jmt))
    s = ls.SynthGrid()
    for f, _ in ls.SynthGrid._fields_:
        if f != "imt_global":
            setattr(s, f, ls.iptr(grid[f]) if f == "kmt" else ls.dptr(grid[f]))
    if ls.lib().licom_synth_make_grid(ctypes.byref(cfg), ctypes.byref(s)) != 0:
        raise ValueError("no grid for %r" % (case,))
    depth = 2800.0 + 2200.0 * _smooth(_gen(seed), ny, nx)
    floor = torch.from_numpy(-grid["zkp"][1:]).to(DEV)
    kmt = torch.zeros((jmt, imt), dtype=torch.int32, device=DEV)
    kmt[2:-2, 2:-2] = (floor[:, None, None] <= depth[None]).sum(0).to(torch.int32) * (depth >= 200.0)
    grid["kmt"] = _halo(kmt).cpu().numpy()
    params = ls.default_params(case.get("hmix", 2), -1.0e10 if case.get("hmix", 2) == 4 else 1.0e3, spec["dts"])
    if case["grid"] == "C1" and case.get("hmix") == 4:
        params["ah"] = -1.0e13
    params["adv"] = case.get("adv", 2)
    if case.get("forced"):
        params.update(gamma=1.0 / (30.0 * 86400.0), boundary_restore=1)
    return ls.Case(name=case["grid"], nx=nx, ny=ny, km=km, imt=imt, jmt=jmt, imt_global=s.imt_global, grid=grid,
                   state={}, forcing={}, params=params)


def _depth(block):
    z = block.grid["zkp"]
    return torch.from_numpy(-0.5 * (z[:-1] + z[1:])).to(DEV)[:, None, None]


def _wet(block, n):
    return (torch.arange(block.km, device=DEV)[:, None, None] < torch.as_tensor(n, device=DEV)[None]).to(torch.float64)


def _kmu(kmt):
    m = np.minimum
    out = np.zeros_like(kmt)
    out[:-1, 1:] = m(m(kmt[:-1, :-1], kmt[:-1, 1:]), m(kmt[1:, :-1], kmt[1:, 1:]))
    out[:, 0:2], out[:, -2:] = out[:, -4:-2].copy(), out[:, 2:4].copy()
    out[0:2], out[-2:] = 0, 0
    return out


def _flow(block, g, viv):
    """Velocities of a smooth streamfunction, 0.5 m/s at most, decaying with depth."""
    psi = _smooth(g, block.jmt + 1, block.imt + 1, 20)
    u, v = psi[1:, :-1] - psi[:-1, :-1], psi[:-1, 1:] - psi[:-1, :-1]
    top = 0.5 / float(torch.sqrt(u * u + v * v).max())
    e = torch.exp(-_depth(block) / 1000.0) * top
    return _halo(u[None] * e * viv), _halo(-v[None] * e * viv)


def _tracers(block, g, t_pert=0.0):
    km, jmt, imt = block.km, block.jmt, block.imt
    d = _depth(block)
    clat = torch.from_numpy(np.cos(np.deg2rad(block.grid["lat_t"]))).to(DEV)[None, :, None]
    vit = _wet(block, block.grid["kmt"])
    at = torch.empty((2, km, jmt, imt), **F64)
    at[0] = (2.0 + 25.0 * torch.exp(-d / 700.0) * clat + (0.05 + t_pert) * _randn(g, km, jmt, imt)) * vit
    at[1] = (34.7 + 0.6 * torch.exp(-d / 500.0) + 0.02 * _randn(g, km, jmt, imt) - 35.0) * 1.0e-3 * vit
    _halo(at)
    atb = torch.zeros((2, km + 1, jmt, imt), **F64)
    atb[:, 1:] = at
    return at, atb, vit


def _ocean(case, block, seed, t_pert=0.0):
    """State and forcing of a tracer step."""
    g = _gen(seed + 1)
    km, jmt, imt = block.km, block.jmt, block.imt
    at, atb, vit = _tracers(block, g, t_pert)
    akt = torch.exp(math.log(1.0e-5) + _rand(g, 2, km, jmt, imt) * math.log(1.0e3)) * vit
    akt[:, -1] = 0.0
    _halo(akt)
    u, v = _flow(block, g, _wet(block, _kmu(block.grid["kmt"])))
    wet = vit[0]
    st = dict(at=at, atb=atb, akt=akt, utf=2.0 * u, vtf=2.0 * v, utl=u, vtl=v, ws=torch.zeros((km + 1, jmt, imt), **F64),
              h0f=_halo(0.3 * _randn(g, jmt, imt) * wet), h0l=_halo(0.3 * _randn(g, jmt, imt) * wet))
    if case.get("ice"):                          # polar surface cells at the freezing point
        at[0, 0] = torch.where(_rand(g, jmt, imt) < 0.02, -1.8 - _rand(g, jmt, imt), at[0, 0]) * wet
        _halo(at)
        atb[:, 1:] = at
    fo = {k: torch.zeros((jmt, imt), **F64) for k in lt.FORCING_KEYS}
    restore = None
    if case.get("forced"):
        fo = dict(swv=150.0 * _rand(g, jmt, imt), nswv=-150.0 * _rand(g, jmt, imt), sst=at[0, 0] + 0.5 * _randn(g, jmt, imt),
                  seaice=_rand(g, jmt, imt) * (_rand(g, jmt, imt) < 0.1), sss=at[1, 0] + 1.0e-4 * _randn(g, jmt, imt),
                  fresh=1.0e-5 * _randn(g, jmt, imt))
        restore = at + torch.tensor([0.3, 3.0e-4], **F64)[:, None, None, None] * _randn(g, 2, km, jmt, imt)
    return st, fo, restore


def _turb_case(block, seed):
    return ls.make_turb_case_device(block, torch, torch.device(DEV), seed=seed, tables=_tables())


_TABLES = {}


def _tables():
    """The closure's lookup tables: constants that do not depend on the seed."""
    if not _TABLES:
        _TABLES.update(ls.turb_tables())
    return _TABLES


def _readyt_inputs(case, seed):
    block = _block(case, seed)
    g = _gen(seed + 2)
    km, jmt, imt = block.km, block.jmt, block.imt
    grid = ls.readyt_grid(block, seed=seed)
    at, atb, vit = _tracers(block, g)
    viv = _wet(block, grid["kmu"])
    u, v = _flow(block, g, viv)
    atb = atb + 0.01 * _randn(g, *atb.shape)
    s2 = (jmt, imt)
    f = dict(vit=vit, viv=viv, at=at, atb=atb, h0=0.3 * _randn(g, *s2), u=1.01 * u, v=0.99 * v, psa=5.0 * _randn(g, *s2),
             swv=3.0e-5 * _rand(g, *s2), nswv=-4.0e-5 * _rand(g, *s2), h0l=0.3 * _randn(g, *s2), h0f=0.3 * _randn(g, *s2),
             utl=u.clone(), vtl=v.clone(), utf=u, vtf=v)
    return block, grid, f


def _readyc_inputs(case, seed):
    block = _block(case, seed)
    g = _gen(seed + 3)
    km, jmt, imt = block.km, block.jmt, block.imt
    s2, s3 = (jmt, imt), (km, jmt, imt)
    rg = ls.readyt_grid(block, seed=seed)
    grid = ls.readyc_grid(block, rg, seed=seed)
    mg = ls.readyc_mgrid(block, rg, del4=case["hmix"] == 4, seed=seed)
    _scale_viscosity(mg, block)
    viv = _wet(block, rg["kmu"])
    u, v = _flow(block, g, viv)
    up, vp = (u + 0.02 * _randn(g, *s3)) * viv, (v + 0.02 * _randn(g, *s3)) * viv
    f = dict(vit=_wet(block, block.grid["kmt"]), viv=viv, up=up, vp=vp, h0=0.3 * _randn(g, *s2), h0bf=0.3 * _randn(g, *s2),
             rict=1.0e-5 * _rand(g, km - 1, *s2), ric=1.0e-5 * _rand(g, km - 1, *s2))
    akmt = torch.exp(math.log(1.0e-5) + _rand(g, *s3) * math.log(1.0e3)) * f["vit"]
    mf = dict(u=up * (1.0 + 0.05 * _randn(g, *s3)), v=vp * (1.0 + 0.05 * _randn(g, *s3)), su=0.1 * _randn(g, *s2),
              sv=0.1 * _randn(g, *s2))
    ws0 = 1.0e-6 * _randn(g, *s2)
    return block, grid, mg, f, akmt, mf, ws0


def _scale_viscosity(g, block):
    """A viscosity for the block's own spacing, with a factor near one."""
    dx = float(block.grid["dxu"].min())
    g["amf"] = np.clip(g["amf"], 0.5, 1.0)
    g["am"] = -5.0e-6 * dx ** 4 if g["del4"] else 1.0e-4 * dx * dx


def _barotr_inputs(case, seed):
    block = _block(case, seed)
    g = _gen(seed + 4)
    s2 = (block.jmt, block.imt)
    rg = ls.readyt_grid(block, seed=seed)
    del4 = case["hmix"] == 4
    dx = float(block.grid["dxu"].min())
    grid = ls.barotr_grid(block, rg, del4=del4, dtb=min(20.0, dx / 400.0), seed=seed)
    _scale_viscosity(grid, block)
    grid["ahf"] = np.clip(grid["ahf"], 0.5, 1.0)
    grid["ah"] = -5.0e-5 * dx ** 4 if del4 else 1.0e-4 * dx * dx
    vit, viv = _wet(block, block.grid["kmt"])[0].contiguous(), _wet(block, grid["kmu"])[0].contiguous()
    sm = lambda a: a * _smooth(g, *s2)  # noqa: E731
    h0p, ubp, vbp = sm(0.3) * vit, sm(0.05) * viv, sm(0.05) * viv
    f = dict(vit=vit, viv=viv, dzph=(3000.0 + sm(200.0)) * viv, dlub=sm(1.0e-7), dlvb=sm(1.0e-7), wgp=0.9 + 0.1 * _rand(g, *s2),
             pax=sm(1.0e-8), pay=sm(1.0e-8), pxb=sm(1.0e-8), pyb=sm(1.0e-8), whx=sm(1.0e-8), why=sm(1.0e-8),
             h0=(h0p + 0.01 * _randn(g, *s2)) * vit, h0p=h0p, ub=ubp.clone(), vb=vbp.clone(), ubp=ubp, vbp=vbp,
             h0f=sm(0.3), h0bf=sm(0.3), work=torch.zeros(s2, **F64), wka=torch.zeros((6,) + s2, **F64))
    for k in BAROTR_OUT[:-1]:
        _halo(f[k])
    return block, grid, f


def _bclinc_inputs(case, seed):
    block = _block(case, seed)
    g = _gen(seed + 5)
    km, jmt, imt = block.km, block.jmt, block.imt
    s2, s3 = (jmt, imt), (km, jmt, imt)
    rg = ls.readyt_grid(block, seed=seed)
    grid = ls.bclinc_grid(block, rg, dtc=60.0, seed=seed)
    vit, viv = _wet(block, block.grid["kmt"]), _wet(block, grid["kmu"])
    u, v = _flow(block, g, viv)
    f = dict(vit=vit, viv=viv, gg=(2.0e-3 * _randn(g, *s3) - 1.0e-2) * vit,
             akmu=torch.exp(math.log(1.0e-4) + _rand(g, *s3) * math.log(500.0)) * viv, su=0.1 * _randn(g, *s2),
             sv=0.1 * _randn(g, *s2), psa=1.0e3 + 5.0 * _randn(g, *s2), h0bl=0.3 * _randn(g, *s2), ub=0.05 * _randn(g, *s2),
             vb=0.05 * _randn(g, *s2), h0bf=1.2 * _randn(g, *s2), u=u, v=v, up=u * (1.0 + 0.02 * _randn(g, *s3)),
             vp=v * (1.0 + 0.02 * _randn(g, *s3)), dlu=1.0e-6 * _randn(g, *s3) * viv, dlv=1.0e-6 * _randn(g, *s3) * viv,
             wka=torch.zeros(s3, **F64), utf=0.1 * _randn(g, *s3), vtf=0.1 * _randn(g, *s3),
             sbcx=torch.zeros(s2, **F64), sbcy=torch.zeros(s2, **F64), bbcx=torch.zeros(s2, **F64), bbcy=torch.zeros(s2, **F64))
    return block, grid, f


class _Exchange:
    """The caller's halo update between the barotropic stages, on one block: cyclic columns, closed rows."""

    def __init__(self, fields, jmt, imt):
        at = torch.arange(jmt * imt, device=DEV).view(jmt, imt)
        src = _halo(at.clone() + 1) - 1
        ghost = (_box(at, 2, -2, 2, -2) == 0) & ((src != at) | (src < 0))
        self.to, self.frm = at[ghost], src[ghost].clamp(min=0)
        self.keep = (src[ghost] >= 0).to(torch.float64)
        self.flat = dict(work=fields["work"].view(1, -1), wka=fields["wka"].view(6, -1)[2:4])

    def __call__(self, names):
        for k in names:
            a = self.flat[k]
            a.index_copy_(1, self.to, a.index_select(1, self.frm) * self.keep)


# ------------------------------------------------------- the framework's calls
def _member_cases(case):
    r = random.Random(case["shapes"])
    out = []
    for _ in range(case["members"]):
        nx, ny = r.choice(licom_ensemble.DOMAINS)
        out.append(dict(kind="mixed", nx=nx, ny=ny, km=r.choice(licom_ensemble.LEVELS),
                        grid="C2" if (nx, ny) == (360, 218) else "C1", hmix=2, adv=2))
    return out


def _model(case, seed, t_pert=0.0):
    precision = "fp64" if case["kind"] == "step" else "mixed"
    block = _block(case, seed)
    m = lt.TracerModel(block, device=DEV, diagnostics=case.get("diag", True), precision=precision)
    st, m.forcing, m.restore = _ocean(case, block, seed, t_pert)
    m.state = {k: v.to(torch.float32) if precision == "mixed" and k in m.MIXED_F32 else v for k, v in st.items()}
    return m


def _step_outputs(m):
    out = {k: m.state[k] for k in ("at", "atb", "akt", "ws", "utf", "vtf", "h0f")}
    out.update(m.diag or {})
    out["licomqice"] = m.licomqice
    return out


MEMBER_STATE = ("at", "atb", "akt", "utf", "vtf", "utl", "vtl", "ws")
MEMBER_OUT = ("at", "atb", "ws")


def _together(models):
    """The members' fields as parts of one array for each field, as a program that keeps an ensemble would hold them."""
    flat = {}
    for where, names in (("state", MEMBER_STATE), ("diag", DIAG3)):
        for k in names:
            parts = [getattr(m, where)[k] for m in models]
            size = [-(-p.numel() // 64) * 64 for p in parts]
            flat[k] = torch.zeros(sum(size), dtype=parts[0].dtype, device=DEV)
            at = 0
            for m, p, n in zip(models, parts, size):
                view = flat[k][at:at + p.numel()].view(p.shape)
                view.copy_(p)
                getattr(m, where)[k] = view
                at += n
    return flat


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "mixed"):
        flags = lt.LICOM_STEP_SIDE_EFFECTS | lt.LICOM_STEP_CONVADJ | (lt.LICOM_STEP_ICESNOW if case["ice"] else 0)
        return dict(kind=kind, model=_model(case, seed), flags=flags)
    if kind == "ensemble":
        models = [_model(c, seed + 17 * n, t_pert=0.1) for n, c in enumerate(_member_cases(case))]
        flat = _together(models)
        torch.cuda.synchronize()
        return dict(kind=kind, models=models, flat=flat, ensemble=licom_ensemble.Ensemble(models))
    if kind == "readyt":
        block, grid, f = _readyt_inputs(case, seed)
        return dict(kind=kind, call=licom_readyt.Readyt(block.imt, block.jmt, block.km, grid, f, device=DEV))
    if kind == "readyc":
        block, grid, mg, f, akmt, mf, ws0 = _readyc_inputs(case, seed)
        call = licom_readyc.Readyc(block.imt, block.jmt, block.km, grid, f, device=DEV)
        call.momentum_grid(mg)
        akmu = torch.zeros_like(akmt)
        mf = call.momentum_fields(dict(mf, up=f["up"], vp=f["vp"], h0=f["h0"], vit=f["vit"], viv=f["viv"], akmu=akmu))
        mf["ws"][0] = ws0
        return dict(kind=kind, call=call, akmt=akmt, akmu=akmu, mf=mf)
    if kind == "turb":
        return dict(kind=kind, call=licom_turb.TurbProducer(_turb_case(_block(case, seed), seed), device=DEV))
    if kind == "barotr":
        block, grid, f = _barotr_inputs(case, seed)
        call = licom_barotr.Barotr(block.imt, block.jmt, grid, f, device=DEV)
        return dict(kind=kind, call=call, halo=_Exchange(call.fields, block.jmt, block.imt))
    block, grid, f = _bclinc_inputs(case, seed)
    return dict(kind=kind, call=licom_bclinc.Bclinc(block.imt, block.jmt, block.km, grid, f, device=DEV))


BCLINC_OUT = ("u", "v", "up", "vp", "dlu", "dlv", "wka", "utf", "vtf", "h0bf", "sbcx", "sbcy", "bbcx", "bbcy")
BAROTR_OUT = ("h0", "h0p", "ub", "vb", "ubp", "vbp", "h0f", "h0bf", "work")


def run(state):
    kind = state["kind"]
    if kind in ("step", "mixed"):
        state["model"].step(state["flags"])
        return _step_outputs(state["model"])
    if kind == "ensemble":
        state["ensemble"].step(4)
        return {k: state["flat"][k] for k in MEMBER_OUT + DIAG3}
    call = state["call"]
    if kind == "readyt":
        call.readyt(1)
        return {k: call.fields[k] for k in licom_readyt.SHIFTED + licom_readyt.OUTPUTS}
    if kind == "readyc":
        call.shear()
        call.akmu(state["akmt"], out=state["akmu"])
        call.momentum(state["mf"])
        out = {k: call.fields[k] for k in licom_readyc.OUTPUTS}
        out.update(akmu=state["akmu"], **{"m_" + k: state["mf"][k] for k in licom_readyc.MOUTPUTS})
        return out
    if kind == "turb":
        call.run()
        return dict(call.outputs)
    if kind == "barotr":
        call.run(4, state["halo"])
        return {k: call.fields[k] for k in BAROTR_OUT}
    call.step(2)
    return {k: call.fields[k] for k in BCLINC_OUT}


# -------------------------------------------------------------- cost, tolerance
def work(case):
    """Bytes: every field that a call reads and every field that it writes, once.  Flops: the additions, products
    and divisions that the formulas of one cell spell out."""
    kind = case["kind"]
    if kind == "ensemble":
        parts = [work(c) for c in _member_cases(case)]
        return {k: 4 * sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n2 = (case["nx"] + 4) * (case["ny"] + 4)
    n3 = n2 * case["km"]
    diag = 15 if case.get("diag", True) else 0
    if kind == "step":
        # at, atb, akt, utf, vtf, utl, vtl read; at, atb, ws, utf, vtf written
        return {"bytes": n3 * 8 * (10 + 7 + diag + (2 if case.get("forced") else 0)), "flops": n3 * 480}
    if kind == "mixed":
        return {"bytes": n3 * (8 * 8 + 4 * (6 + 3 + diag) + (16 if case.get("forced") else 0)), "flops": n3 * 480}
    if kind == "readyt":
        return {"bytes": n3 * 8 * (10 + 16) + (n3 - n2) * 8 * 5, "flops": n3 * 260}
    if kind == "readyc":
        return {"bytes": n3 * 8 * (4 + 7 + 1 + 1 + 2 + 4) + (n3 - n2) * 8 * 3, "flops": n3 * 330}
    if kind == "turb":
        return {"bytes": n3 * 8 * (8 + 7), "flops": n3 * 400}
    if kind == "barotr":
        return {"bytes": n2 * 8 * (20 + 35 + 11), "flops": n2 * 4 * 300}
    return {"bytes": n3 * 8 * (12 + 9), "flops": n3 * 160}


def tolerance(case):
    kind = case["kind"]
    # four times what `exact` differs by, and more where a flipped limiter decision sets it
    if kind == "mixed":
        return {"rel": 5.0e-6, "max": 0.02}
    if kind == "ensemble":                       # four steps
        return {"rel": 1.3e-4, "max": 0.1}
    if kind == "turb":                           # differences of nearly equal terms in a few cells
        return {"rel": 1.4e-6, "max": 6.0e-4}
    if case.get("forced"):                       # the global freshwater sum
        return {"rel": 1.0e-12, "max": 4.0e-12}
    # the FP64 calls keep the order of every operation: a run continued on another build gives the same bits
    return "exact"


# ------------------------------------------------ the same results in plain torch
def _e(x):
    return torch.roll(x, -1, -1)


def _w(x):
    return torch.roll(x, 1, -1)


def _s(x):
    return torch.roll(x, -1, -2)


def _n(x):
    return torch.roll(x, 1, -2)


def _up(x):
    """The level above, 0 above the first."""
    return torch.cat([torch.zeros_like(x[:1]), x[:-1]])


def _down(x):
    """The level below, 0 below the last."""
    return torch.cat([x[1:], torch.zeros_like(x[:1])])


def _box(like, j0, j1, i0, i1):
    """1 on rows j0..j1-1 and columns i0..i1-1 of the last two axes, where negative ends count from the far side."""
    jmt, imt = like.shape[-2:]
    m = torch.zeros((jmt, imt), **F64)
    m[j0:jmt + j1, i0:imt + i1] = 1.0
    return m


def _dev(a):
    return torch.as_tensor(a, device=DEV) if a.dtype == np.int32 else torch.from_numpy(np.ascontiguousarray(a, np.float64)).to(DEV)


def _lev(a):
    return _dev(np.asarray(a, np.float64))[:, None, None]


class _Grid:
    """The masks and coefficients a tracer step derives from its grid."""

    def __init__(self, block):
        g, p = block.grid, block.params
        self.kmt, self.p, self.km = _dev(g["kmt"]), p, block.km
        for k in ("htw", "hts", "hun", "hue", "tarea", "dxu", "dyu", "au0", "aus", "auw", "ausw"):
            setattr(self, k, _dev(g[k]))
        self.kmu = _dev(_kmu(g["kmt"]))
        self.vit, self.viv = _wet(block, self.kmt), _wet(block, self.kmu)
        zkp = g["zkp"]
        dzp, zkt = zkp[:-1] - zkp[1:], 0.5 * (zkp[:-1] + zkp[1:])
        self.dz, self.oz = [float(x) for x in dzp], [float(1.0 / x) for x in dzp]
        self.ot = [float(2.0 / dzp[0])] + [float(1.0 / (a - b)) for a, b in zip(zkt[:-1], zkt[1:])]
        self.dzp, self.odzp, self.odzt = _lev(dzp), _lev(1.0 / dzp), _lev(self.ot)
        self.pen = [float(x) for x in g["pen"]]
        self.to, self.so, self.eosc = _dev(g["to"]), _dev(g["so"]), _dev(g["eosc"])
        inv = lambda h: torch.where(h > 0, 1.0 / h.clamp(min=1e-300), torch.zeros_like(h))  # noqa: E731
        self.ohbt, self.ohbu = inv((self.vit * self.dzp).sum(0)), inv((self.viv * self.dzp).sum(0))
        tr = self.tr = 1.0 / self.tarea
        dxg = 2.0 * 6371000.0 * math.pi / block.imt_global
        first = lambda a, ax: torch.cat([torch.zeros_like(a.narrow(ax, 0, 1)), a.narrow(ax, 0, a.shape[ax] - 1)], ax)  # noqa: E731
        last = lambda a, ax: torch.cat([a.narrow(ax, 1, a.shape[ax] - 1), torch.zeros_like(a.narrow(ax, 0, 1))], ax)  # noqa: E731
        if p["hmix"] == 4:
            self.ahf = (self.tarea / dxg ** 2) ** 1.5
            a, b = self.hts / self.hue, self.htw / self.hun
        else:
            self.ahf = torch.sqrt(self.tarea) / dxg
            a = self.hts / self.hue * 0.5 * (self.ahf + last(self.ahf, 0))
            b = self.htw / self.hun * 0.5 * (self.ahf + first(self.ahf, 1))
        self.dts, self.dtn, self.dtw, self.dte = a * tr, first(a, 0) * tr, b * tr, last(b, 1) * tr
        self.inner, self.ring = _box(self.vit, 2, -2, 2, -2), _box(self.vit, 1, -1, 1, -1)
        self.area = float((self.tarea * self.inner * (self.kmt > 0)).sum())

    def lap(self, x):
        """The masked 5-point operator of a 3-D field."""
        v = self.vit
        cn, cs, ce, cw = self.dtn * _n(v), self.dts * _s(v), self.dte * _e(v), self.dtw * _w(v)
        return (cn * _n(x) + cs * _s(x) + ce * _e(x) + cw * _w(x) - (cn + cs + ce + cw) * x) * v * self.ring

    def dens(self, k, t, s):
        c = self.eosc[:, k] if isinstance(k, int) else self.eosc[:, k].reshape((9,) + tuple(k.shape))
        return ((c[0] + (c[3] + c[6] * s) * s + (c[2] + c[7] * s + c[5] * t) * t) * t + (c[1] + (c[4] + c[8] * s) * s) * s)


def _tspas(G, dts, T, U, V, W):
    """The two-step shape-preserving scheme: (x, y, z) advective tendencies on rows and columns 1..-2."""
    tr, oz, ot = G.tr, G.odzp, G.odzt
    Te, Tw, Ts, Tn, Tu, Td = _e(T), _w(T), _s(T), _n(T), _up(T), _down(T)
    Ue, Vn = _e(U), _n(V)
    Wk = W.clone()
    Wk[0] = 0.0                                   # no vertical flux through the surface in this form
    Wb, otb = _down(Wk), _down(ot)
    cx, cy = G.htw * G.hun, G.hts * G.hue
    x = [(Te + T) * Ue * tr - (T + Tw) * U * tr, -T * (Ue - U) * tr * 2.0]
    y = [((Ts + T) * V - (T + Tn) * Vn) * tr, -T * (V - Vn) * tr * 2.0]
    z = [0.5 * oz * Wk * (T + Tu) - 0.5 * oz * Wb * (T + Td), -oz * T * (Wk - Wb)]
    lw = [-dts * (Te - T) * 2.0 * tr * Ue * Ue / _e(cx), dts * (T - Tw) * 2.0 * tr * U * U / cx,
          -dts * (Ts - T) * 2.0 * tr * V * V / cy, dts * (T - Tn) * 2.0 * tr * Vn * Vn / _n(cy),
          -0.5 * oz * Wk * Wk * ot * (Tu - T) * dts, 0.5 * oz * Wb * Wb * otb * (T - Td) * dts]
    at00 = T - (x[0] + x[1] + lw[0] + lw[1] + y[0] + y[1] + lw[2] + lw[3] + z[0] + z[1] + lw[4] + lw[5]) * dts
    v = G.vit
    hi, lo = T * v + (1.0 - v) * -1.0e10, T * v + (1.0 - v) * 1.0e10
    edge = torch.full_like(T[:1], 1.0e10)
    most, least = hi, lo
    for f in (_e, _w, _s, _n):
        most, least = torch.maximum(most, f(hi)), torch.minimum(least, f(lo))
    most = torch.maximum(most, torch.cat([-edge, hi[:-1]]))
    most = torch.maximum(most, torch.cat([hi[1:], -edge]))
    least = torch.minimum(least, torch.cat([edge, lo[:-1]]))
    least = torch.minimum(least, torch.cat([lo[1:], edge]))
    fl = ((at00 > most) | (at00 < least)) & (G.ring > 0)
    del most, least, hi, lo, at00
    jmt, imt = G.kmt.shape
    i, j = torch.arange(imt, device=DEV)[None, :], torch.arange(jmt, device=DEV)[:, None]
    ends = torch.zeros((G.km, 1, 1), dtype=torch.bool, device=DEV)
    ends[0], ends[-1] = True, True
    inside = (i <= imt - 3, i >= 2, j <= jmt - 3, j >= 2)
    up = [torch.where(ends, fl | (f(fl) & b), (fl | f(fl)) & b) for f, b in zip((_e, _w, _s, _n), inside)]
    up += [fl | _up(fl), fl | _down(fl)]
    lim = [-(Te - T) * Ue.abs() * tr, (T - Tw) * U.abs() * tr, -(Ts - T) * V.abs() * tr, (T - Tn) * Vn.abs() * tr,
           -0.5 * Wk.abs() * oz * (Tu - T), 0.5 * Wb.abs() * oz * (T - Td)]
    f = [torch.where(c, a, b) for c, a, b in zip(up, lim, lw)]
    return -(x[0] + x[1] + f[0] + f[1]), -(y[0] + y[1] + f[2] + f[3]), -(z[0] + z[1] + f[4] + f[5])


def _plain_advection(G, adv, nss, T, U, V, W):
    """The centered (0) and flux (1) schemes: the tendency and, for centered, its x, y and z parts over nss."""
    Te, Tw, Ts, Tn, Tu, Td = _e(T), _w(T), _s(T), _n(T), _up(T), _down(T)
    Ue, Vn, Wk = _e(U), _n(V), W.clone()
    Wk[0] = 0.0
    Wb = _down(Wk)
    if adv == 0:
        x, y = (-U * (T - Tw) - Ue * (Te - T)) * G.tr, (-V * (Ts - T) - Vn * (T - Tn)) * G.tr
        z = -0.5 * G.odzp * (Wk * (Tu - T) + Wb * (T - Td))
        return x + y + z, x / nss, y / nss, z / nss
    a = (-U * (T + Tw) + Ue * (Te + T) - Vn * (T + Tn) + V * (Ts + T)) * G.tr
    a = a - G.odzp * 0.5 * (Wb * (T + Td) - Wk * (Tu + T))
    return a, None, None, None


def _exact_step(block, st, fo, restore, ice, out):
    """One tracer step: st and the diagnostics of `out` are updated in place."""
    G, p = _Grid(block), block.params
    km, dts, v = block.km, p["dts"], None
    v = G.vit
    st["h0f"] = st["h0f"] * p["onbc"]
    h = 0.5 * st["h0f"] + 0.5 * st["h0l"]
    st["utf"], st["vtf"] = st["utf"] * p["oncc"], st["vtf"] * p["oncc"]
    wkd, wkb = 0.5 * st["utf"] + 0.5 * st["utl"], 0.5 * st["vtf"] + 0.5 * st["vtl"]
    ubox = _box(v, 0, -1, 1, 0)
    hu = (G.au0 * h + G.aus * _s(h) + G.auw * _w(h) + G.ausw * _s(_w(h))) * ubox
    uk, vk = (1.0 + hu * G.ohbu) * wkd * ubox, (1.0 + hu * G.ohbu) * wkb * ubox
    div = 0.5 * ((_e(uk) + _e(_n(uk))) * _e(G.htw) - (uk + _n(uk)) * G.htw + (_e(vk) + vk) * G.hts
                 - (_e(_n(vk)) + _n(vk)) * _n(G.hts)) * G.tr * v * _box(v, 1, 0, 0, -1)
    del uk, vk
    col = -(G.dzp * div * v).sum(0)
    scale = 1.0 / (1.0 + h * G.ohbt)
    w = [st["ws"][0]]
    for k in range(1, km):
        w.append(v[k] * (w[-1] + G.dz[k - 1] * (col * G.ohbt + div[k - 1])))
    ws = st["ws"].clone()
    for k in range(1, km):
        ws[k] = torch.where(G.ring > 0, w[k] * scale, ws[k])
    st["ws"] = ws
    del div, w
    if p["adv"] == 1:
        V, U = (wkb * G.dxu + _e(wkb * G.dxu)) * 0.25, (_n(wkd * G.dyu) + wkd * G.dyu) * 0.25
    else:
        V, U = (wkb + _e(wkb)) * G.hts * 0.25, (_n(wkd) + wkd) * G.htw * 0.25
    V, U = V * _box(v, 0, 0, 1, -1), U * _box(v, 1, -1, 0, 0)
    del wkd, wkb
    W, wet = ws[:km], G.kmt > 0
    for n in range(2):
        T, B = st["at"][n], st["atb"][n][1:]
        if p["adv"] == 2:
            x, y, z = _tspas(G, dts, T, U, V, W)
            adv = x + y + z
            d3 = dict(ax=x, ay=y, az=z)
        else:
            adv, x, y, z = _plain_advection(G, p["adv"], p["nss"], T, U, V, W)
            d3 = {} if x is None else dict(ax=out["ax"][n] + x, ay=out["ay"][n] + y, az=out["az"][n] + z)
        if n == 0 or p["hmix"] == 2:
            st["akt"][n][0] = torch.where((G.ring > 0) & (st["akt"][n][0] < p["dwndmix"]), p["dwndmix"], st["akt"][n][0])
        akt = st["akt"][n]
        mix = G.ahf * G.lap(B) if p["hmix"] == 4 else B
        tf = (adv * v + p["ah"] * G.lap(mix)) * G.inner
        del adv, mix, x, y, z
        if n == 0:
            pen = torch.zeros_like(T)
            flux = [fo["swv"] * G.pen[k] * v[k + 1] for k in range(km - 1)]     # through the bottom of level k
            for k in range(km):
                a = flux[k - 1] if k else 0.0
                b = flux[k] if k < km - 1 else 0.0
                pen[k] = (a - b) * G.oz[k] * G.inner
            out["penetrate"] = pen
            tf = tf + pen
        below = _down(v) * akt * (B - _down(B)) * _down(G.odzt)                  # diffusive flux through the bottom
        dz = G.odzp * (_up(below) - below) * 0.5
        tf = tf + dz * G.inner
        d3["dz"] = dz
        if n == 1:
            sb = B[0]
            stf = fo["fresh"] * 34.7 * p["od0"] / 1000.0 + p["gamma"] * (fo["sss"] - sb) * fo["seaice"] / G.oz[0] \
                + p["gamma"] * 30.0 / 365.0 / 4.0 * 50.0 * (fo["sss"] - sb) / G.oz[0] * (1.0 - fo["seaice"])
        else:
            stf = (fo["swv"] + fo["nswv"]) * p["od0cp"] + fo["seaice"] * p["gamma"] * (fo["sst"] - B[0]) / G.oz[0]
        net = torch.where(wet, stf * G.oz[0], torch.zeros_like(stf))
        out["net"][n] = net
        stf = torch.where(wet, stf, h)            # land keeps the surface height averaged into this field
        tf[0] = tf[0] + 0.5 * net
        if n == 1 and p["sssnorm"]:
            err = -(G.tarea * net * v[0] * G.inner).sum() / G.area
            out["fw_norm2"][0] = err
            tf[0] = tf[0] + err * v[0]
        if p["boundary_restore"] and restore is not None:
            add = v * (restore[n] - B) * (1.0 / (15.0 * 86400.0))
            add[0] = 0.0
            tf = tf + add * G.inner
        ori = (T + dts * tf) * G.inner
        # the implicit half of the vertical diffusion
        e = f = torch.zeros_like(h)
        es, fs = [None] * km, [None] * km
        for k in range(km - 1, -1, -1):
            act, bot = k < G.kmt, k == G.kmt - 1
            a = akt[k - 1] * G.ot[k] * G.oz[k] * dts * 0.5 if k else torch.full_like(h, G.oz[0] * dts * 0.5)
            c = akt[k] * G.ot[k + 1] * G.oz[k] * dts * 0.5 if k < km - 1 else torch.zeros_like(h)
            b = torch.where(bot, 1.0 + a, 1.0 + c + (a if k else 0.0))
            g0 = 1.0 / (b - torch.where(bot, 0.0 * c, c) * e)
            e, f = torch.where(act, a * g0, 0.0 * h), torch.where(act, (ori[k] + torch.where(bot, 0.0 * c, c) * f) * g0, 0.0 * h)
            es[k], fs[k] = e, f
        new, x = torch.zeros_like(T), None
        for k in range(km):
            x = es[k] * (stf if k == 0 else x) + fs[k]
            new[k] = torch.where(k < G.kmt, x, ori[k]) * G.inner
        del es, fs
        d3["dt_diff"] = (new - ori) / dts * v
        d3["dt_diff"][0] = d3["dt_diff"][0] - stf * 0.5 * G.oz[0]
        _halo(new)
        d3["tend"] = (new - T) / dts * v
        for k, a in d3.items():
            out[k][n] = a * G.inner
        st["at"][n] = new
        st["atb"][n][1:] = new
    if ice:
        T, S = st["at"][0], st["at"][1]
        cold = torch.where((T[0] < -1.8) & wet, -1.8 - T[0], torch.zeros_like(h))
        out["licomqice"][:] = cold
        S[0] += cold * (34.7 - 4.0) * 3996.0 / 3.337e5 * 0.001
        T.clamp_(min=-1.8)
    _exact_convadj(G, st["at"])
    for n in range(2):
        dc = (st["at"][n] - st["atb"][n][1:]) / dts * v * G.inner
        out["dt_conv"][n] = dc
        out["tend"][n] += dc
        st["atb"][n][1:] = st["at"][n]


def _exact_convadj(G, at):
    """Convective adjustment of every column: statically unstable neighbours are mixed until the column is stable."""
    km, M = G.km, G.kmt.numel()
    ts = at.view(2, km, M)
    kcon = G.kmt.reshape(M).long()
    lev = torch.arange(km, device=DEV)
    unstable = torch.zeros((km, M), dtype=torch.bool, device=DEV)      # [k]: level k-1 is denser than level k, at level k
    for k in range(1, km):
        rho = [G.dens(k, ts[0, m] - G.to[k], ts[1, m] - G.so[k]) for m in (k - 1, k)]
        unstable[k] = (rho[0] > rho[1]) & (k < kcon)
    cols = unstable.any(0).nonzero()[:, 0]
    if not cols.numel():
        return
    x, uns, kc = ts[:, :, cols].permute(0, 2, 1).contiguous(), unstable[:, cols].t().contiguous(), kcon[cols]
    dz = G.dzp[:, 0, 0]
    sel = torch.arange(cols.numel(), device=DEV)
    a = torch.where(uns, lev, km).min(1)[0]                             # 1-based first level of the mixed part
    b = a + 1

    def rho(n, k, l):                                                    # density of level l (0-based) at level k's reference
        return G.dens(k, x[0, n, l] - G.to[k], x[1, n, l] - G.so[k])

    def mix(n):
        inside = (lev >= a[n, None] - 1) & (lev < b[n, None])
        wgt = torch.where(inside, dz, torch.zeros_like(dz))
        for m in range(2):
            y = x[m, n]
            x[m, n] = torch.where(inside, ((y * wgt).sum(1) / wgt.sum(1))[:, None], y)

    mix(sel)
    while sel.numel():
        n = sel
        can = b[n] < kc[n]
        kb = torch.where(can, b[n], b[n] - 1)
        grow = can & (rho(n, kb, b[n] - 1) > rho(n, kb, kb))
        can = (a[n] > 1) & ~grow
        ka = (a[n] - 1).clamp(min=0)
        rise = can & (rho(n, ka, (a[n] - 2).clamp(min=0)) > rho(n, ka, ka))
        b[n] += grow.long()
        a[n] -= rise.long()
        moved = grow | rise
        still = n[~moved]                                                # these parts are done: on to the next one below
        later = uns[still] & (lev > b[still, None]) & (lev < kc[still, None])
        more = later.any(1)
        nxt = torch.where(later, lev, km).min(1)[0]
        again = still[more]
        a[again], b[again] = nxt[more], nxt[more] + 1
        sel = torch.cat([n[moved], again])
        if sel.numel():
            mix(sel)
    ts[:, :, cols] = x.permute(0, 2, 1)


def _exact_tracer(case, seed, steps=1, t_pert=0.0):
    block = _block(case, seed)
    st, fo, restore = _ocean(case, block, seed, t_pert)
    if case["kind"] == "mixed":
        st = {k: a.float().double() if k in lt.TracerModel.MIXED_F32 else a for k, a in st.items()}
    km, jmt, imt = block.km, block.jmt, block.imt
    out = {k: torch.zeros((2, km, jmt, imt), **F64) for k in DIAG3}
    out.update(penetrate=torch.zeros((km, jmt, imt), **F64), net=torch.zeros((2, jmt, imt), **F64),
               fw_norm2=torch.zeros(1, **F64), licomqice=torch.zeros((jmt, imt), **F64))
    for _ in range(steps):
        _exact_step(block, st, fo, restore, case.get("ice"), out)
    got = {k: st[k] for k in ("at", "atb", "akt", "ws", "utf", "vtf", "h0f")}
    got.update(out if case.get("diag", True) else {"licomqice": out["licomqice"]})
    return got


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "mixed"):
        return _exact_tracer(case, seed)
    if kind == "ensemble":
        flat = {k: [] for k in MEMBER_OUT + DIAG3}
        for n, c in enumerate(_member_cases(case)):
            got = _exact_tracer(c, seed + 17 * n, steps=4, t_pert=0.1)
            for k in flat:
                x = got[k].reshape(-1)
                flat[k].append(torch.nn.functional.pad(x, (0, -x.numel() % 64)))
        return {k: torch.cat(x) for k, x in flat.items()}
    return {"readyt": _exact_readyt, "readyc": _exact_readyc, "turb": _exact_turb, "barotr": _exact_barotr,
            "bclinc": _exact_bclinc}[kind](case, seed)


def _grad(a, g):
    """x and y gradients at U points of a T field."""
    sw = _s(_w(a))
    return g["dxur"] * 0.5 * (_s(a) - _w(a) - sw + a), g["dyur"] * 0.5 * (_s(a) - _w(a) + sw - a)


def _to_u(a, g):
    return g["au0"] * a + g["aus"] * _s(a) + g["auw"] * _w(a) + g["ausw"] * _s(_w(a))


def _fluxdiv(u, v, g):
    return 0.5 * ((_e(u) + _e(_n(u))) * _e(g["htw"]) - (u + _n(u)) * g["htw"] + (_e(v) + v) * g["hts"]
                  - (_e(_n(v)) + _n(v)) * _n(g["hts"]))


def _on_device(grid):
    return {k: _dev(a) if isinstance(a, np.ndarray) else a for k, a in grid.items()}


def _eos(c, k, t, s):
    c = c[:, k]
    return (c[0] + (c[3] + c[6] * s) * s + (c[2] + c[7] * s + c[5] * t) * t) * t + (c[1] + (c[4] + c[8] * s) * s) * s


def _exact_readyt(case, seed):
    block, grid, f = _readyt_inputs(case, seed)
    g, km, grav, od0 = _on_device(grid), block.km, 9.806, grid["od0"]
    vit, viv = f["vit"], f["viv"]
    (T, S), (Tb, Sb) = f["at"], f["atb"][:, 1:]
    ubox = _box(vit, 0, -1, 1, 0)
    dz, oz, zk = ([float(x) for x in grid[k]] for k in ("dzp", "odzt", "zkt"))
    o = dict(h0l=f["h0f"], h0f=f["h0"], utl=f["utf"], vtl=f["vtf"], utf=f["u"], vtf=f["v"], rit=torch.zeros_like(T[1:]),
             akt=torch.zeros_like(f["at"]))
    tu, su = _to_u(Tb, g), _to_u(Sb, g)
    ric, rict = torch.zeros_like(T[1:]), torch.zeros_like(T[1:])
    rho = torch.empty_like(T)
    for k in range(km):
        rho[k] = _eos(g["eosc"], k, T[k] - g["to"][k], S[k] - g["so"][k])
        if k:
            for out, mask, t, s in ((ric, viv, tu, su), (rict, vit, Tb, Sb)):
                d = [_eos(g["eosc"], k, t[m] - g["to"][k], s[m] - g["so"][k]) for m in (k - 1, k)]
                out[k - 1] = mask[k] * od0 * grav * (d[1] - d[0]) * oz[k] * ubox
    po = g["po"][:, None, None]
    pden = torch.where(vit > 0, 1000.0 + po + rho, torch.zeros_like(rho))
    gg = -od0 * grav * pden * vit
    pp, ppa, ppb, ppc = (torch.empty_like(T) for _ in range(4))
    pp[0], ppa[0], ppb[0], ppc[0] = 0.5 * dz[0] * gg[0] * vit[0], f["psa"] * vit[0], T[0] * vit[0], S[0] * vit[0]
    for k in range(1, km):
        pp[k] = vit[k] * (pp[k - 1] + 0.5 * (gg[k] * dz[k] + gg[k - 1] * dz[k - 1]))
        ppa[k] = vit[k] * (ppa[k - 1] + gg[k - 1] * dz[k - 1])
        r = dz[k - 1] / (dz[k - 1] + dz[k])
        ppb[k], ppc[k] = vit[k] * (T[k - 1] - (T[k - 1] - T[k]) * r), vit[k] * (S[k - 1] - (S[k - 1] - S[k]) * r)
    t, s, m = ppb, ppc * 1000.0, -ppa / od0 / 10000.0 * vit
    beta = (0.785567e-3 - 0.301985e-5 * t + 0.555579e-7 * t ** 2 - 0.415613e-9 * t ** 3
            + s * (-0.356603e-6 + 0.788212e-8 * t + 0.408195e-10 * m - 0.602281e-15 * m ** 2) + s ** 2 * 0.515032e-8
            + m * (-0.121555e-7 + 0.192867e-9 * t - 0.2131127e-11 * t ** 2) + m ** 2 * (0.176621e-12 - 0.175379e-14 * t)
            + m ** 3 * 0.12155e-17) * vit
    alpha = (0.665157e-1 + 0.170907e-1 * t - 0.203814e-3 * t ** 2 + 0.298357e-5 * t ** 3 - 0.255019e-7 * t ** 4
             + s * (0.378110e-2 - 0.846960e-4 * t - 0.164759e-6 * m - 0.251520e-11 * m ** 2) - s ** 2 * 0.678662e-5
             + m * (0.380374e-4 - 0.933746e-6 * t + 0.791325e-8 * t ** 2) + 0.512857e-12 * m ** 2 * t ** 2
             - 0.302285e-13 * m ** 3) * beta * vit
    cols = _box(vit, 0, 0, 1, -1)
    alpha, beta = alpha * cols, beta * cols
    dT, dS = T[:-1] - T[1:], S[:-1] - S[1:]
    od = g["odzt"][1:, None, None]
    ms = vit[1:] * grav * (dT * alpha[1:] + 1000.0 * dS * beta[1:]) * od * cols
    dt = vit[1:] / ((dT + 1.0e-25) * alpha[1:]) * 1000.0 * dS * beta[1:]
    dt = torch.where((cols > 0).expand_as(dt), dt, torch.zeros_like(dt))
    buoy = vit[0] * alpha[0] * grav * grid["od0cp"]
    gg = -od0 * grav * torch.where(vit > 0, rho, pden - po - 1000.0) * vit
    dlu, dlv = _grad(pp, g)
    wet = _wet(block, g["kmu"]) * ubox
    dlu, dlv = dlu * wet, dlv * wet
    dzp = g["dzp"][:, None, None]
    px, py = ((dzp * g["ohbu"] * a * viv).sum(0) for a in (dlu, dlv))
    a = gg * g["ohbt"] * dzp
    dlu[0], dlu[1] = a.sum(0), (a * g["zkt"][:, None, None]).sum(0)
    dlv[0], dlv[1] = (dlu[0] + dlu[1] * g["ohbt"]) / grav, dlu[1] * g["ohbt"] * g["ohbt"]
    wgp, wrk = _to_u(dlv[0], g) * ubox, _to_u(dlv[1], g) * ubox
    w1, w2 = _grad(f["psa"], g)
    wet0 = (g["kmu"] >= 1) * ubox
    o.update(dlu=dlu, dlv=dlv, pdensity=pden, gg=gg, pp=pp, ppa=ppa, ppb=ppb, ppc=ppc, alpha=alpha, beta=beta, ric=ric, rict=rict,
             ricdttms=ms, ricdt=dt, buoytur=buoy * f["nswv"], buoysol=buoy * f["swv"], pxb=px, pyb=py, wgp=wgp, work=wrk,
             whx=g["hbx"] * wrk * viv[0], why=g["hby"] * wrk * viv[0], work1=w1 * wet0, work2=w2 * wet0,
             pax=-od0 * w1 * wet0, pay=-od0 * w2 * wet0)
    return o


def _lap_u(a, b, g):
    """The momentum Laplacian of (a, b): its rotation terms enter with the other sign for the second component."""
    du = lambda x: (g["duc"] + g["dum"]) * x + g["dun"] * _n(x) + g["dus"] * _s(x) + g["due"] * _e(x) + g["duw"] * _w(x)  # noqa: E731
    dm = lambda x: g["dmc"] * x + g["dmn"] * _n(x) + g["dms"] * _s(x) + g["dme"] * _e(x) + g["dmw"] * _w(x)  # noqa: E731
    return du(a) + dm(b), du(b) - dm(a)


def _viscosity(u, v, g, vit, viv, region, del4):
    """am times the momentum Laplacian, or the Laplacian of the flow-scaled Laplacian."""
    if not del4:
        a, b = _lap_u(u, v, g)
        return g["am"] * a * region * viv, g["am"] * b * region * viv
    div = _fluxdiv(u, v, g) * g["tarea_r"] * vit * _box(u, 1, 0, 0, -1)
    vd, ud = v * g["dyu"], u * g["dxu"]
    curl = 0.5 * (vd + _n(vd) - _w(vd) - _n(_w(vd)) - ud - _w(ud) + _n(ud) + _n(_w(ud))) * vit * _box(u, 1, 0, 1, 0)
    ubox = _box(u, 0, -1, 1, 0)
    q = sum(c * c for a in (div, curl) for c in _grad(a, g)) * viv * ubox
    side = torch.sqrt(1.0 / g["uarea_r"])
    am_f = (torch.sqrt(q) * side ** 5 * 45.0 / (g["am"] * g["amf"]).abs()).clamp(1.0, 40.0)
    a, b = _lap_u(u, v, g)
    wide = viv * _box(u, g["jb"] - 2, g["je"] + 1 - u.shape[-2], g["ib"] - 2, g["ie"] + 1 - u.shape[-1])
    a, b = _lap_u(am_f * g["amf"] * a * wide, am_f * g["amf"] * b * wide, g)
    return g["am"] * a * region * viv, g["am"] * b * region * viv


def _exact_readyc(case, seed):
    block, grid, mg, f, akmt, mf, ws0 = _readyc_inputs(case, seed)
    c, g, km = _on_device(grid), dict(_on_device(mg), **_on_device(grid)), block.km
    vit, viv, up, vp = f["vit"], f["viv"], f["up"], f["vp"]
    z3 = torch.zeros_like(up)
    tbox, ubox, ring = _box(up, 1, 0, 0, -1), _box(up, 0, -1, 1, 0), _box(up, 1, -1, 1, -1)
    ot = _lev(grid["odzt"])

    def to_t(a):
        return c["at0"] * a + c["atn"] * _n(a) + c["ate"] * _e(a) + c["atne"] * _n(_e(a))

    den = to_t(viv) + 1.0e-25
    w12, w13 = (vit * to_t(a * viv) / den * tbox for a in (up, vp))
    s2t, s2u, riu = z3.clone(), z3.clone(), z3.clone()
    r1, r2 = (w * vit - _down(w * vit) for w in (w12, w13))
    s2t[:-1] = (vit[1:] * (r1 * r1 + r2 * r2)[:-1] * ot[1:] * ot[1:]) * tbox
    rit = vit[1:] * f["rict"] / (s2t[:-1] + 1.0e-25) * tbox
    r1, r2 = up - _down(up), vp - _down(vp)
    r1[-1], r2[-1] = 0.0, 0.0
    s2u[:-1] = viv[1:] * (r1 * r1 + r2 * r2)[:-1] * ot[1:] * ot[1:]
    riu[1:] = viv[1:] * f["ric"] / (s2u[:-1] + 1.0e-25)
    akmu = _to_u(akmt, c) * ubox * _down(viv)
    o = dict(h0bl=f["h0bf"], h0bf=f["h0"], wp12=w12, wp13=w13, riv1=r1, riv2=r2, s2t=s2t, rit=rit, s2u=s2u, riu=riu, akmu=akmu)
    # momentum tendencies
    u, v, h = mf["u"], mf["v"], f["h0"]
    dz, od = [float(x) for x in mg["dzp"]], _lev(mg["odzp"])
    sc = (1.0 + _to_u(h, c) * ubox * g["ohbu"]) * ubox
    div = _fluxdiv(u * sc, v * sc, g) * g["tarea_r"] * _wet(block, g["kmt"]) * tbox
    col = -(_lev(mg["dzp"]) * div * vit).sum(0)
    w = [ws0]
    for k in range(1, km):
        w.append(vit[k] * (w[-1] + dz[k - 1] * (col * g["ohbt"] + div[k - 1])))
    over = 1.0 / (1.0 + h * g["ohbt"])
    ws = torch.stack([ws0] + [x * over * ring for x in w[1:]])
    wu = _to_u(ws, c) * ubox
    uw, vs = (_w(u) + u) * 0.25 * _w(g["hue"]) * ubox, (v + _s(v)) * 0.25 * _s(g["hun"]) * ubox
    wu[0] = 0.0
    adv = []
    for a in (u, v):
        x = (-uw * (a - _w(a)) - _e(uw) * (_e(a) - a) - vs * (_s(a) - a) - _n(vs) * (a - _n(a))) * g["uarea_r"]
        adv.append((x - 0.5 * od * (wu * (_up(a) - a) + _down(wu) * (a - _down(a)))) * ring)
    region = _box(up, mg["jb"] - 1, mg["je"] - block.jmt, mg["ib"] - 1, mg["ie"] - block.imt)
    vis = _viscosity(up, vp, g, _wet(block, g["kmt"]), _wet(block, g["kmu"]), region, case["hmix"] == 4)
    dl = [a + b * ring for a, b in zip(adv, vis)]
    wka = g["c0f"] * torch.sqrt(up * up + vp * vp)
    bot = (g["kmu"].long() - 1)
    at = lambda a: torch.gather(a, 0, bot.clamp(min=0)[None])[0]  # noqa: E731
    ub, vb, sn, cag, sag = at(up), at(vp), g["snlat"], g["cag"], g["sag"]
    wetu = (bot >= 0) * ring
    drag = g["c0f"] * torch.sqrt(ub * ub + vb * vb)
    sb = [a * g["od0"] * wetu for a in (mf["su"], mf["sv"])]
    bb = [drag * (ub * cag + sn * vb * sag) * wetu, drag * (vb * cag - sn * ub * sag) * wetu]
    mean = [(_lev(mg["dzp"]) * g["ohbu"] * a * viv).sum(0) + (s - b) * g["ohbu"] * ring for a, s, b in zip(dl, sb, bb)]
    turned = (up * cag + sn * vp * sag, vp * cag - sn * up * sag)
    dry = 1.0 - _down(viv)
    for n, (a, top) in enumerate(((up, mf["su"]), (vp, mf["sv"]))):
        low = akmu * 0.5 * (a - _down(a)) * _down(ot) * _down(viv) + dry * wka * 0.5 * turned[n]
        high = _up(low)
        high[0] = top * g["od0"] * 0.5
        dl[n] = dl[n] + od * (high - low) * ring
    o.update(m_ws=ws, m_dlu=dl[0], m_dlv=dl[1], m_wka=wka, m_dlub=mean[0], m_dlvb=mean[1], m_sbcx=sb[0], m_sbcy=sb[1],
             m_bbcx=bb[0], m_bbcy=bb[1])
    return o


def _exact_barotr(case, seed):
    block, grid, f = _barotr_inputs(case, seed)
    g = _on_device(grid)
    z = torch.zeros_like(f["h0"])
    jmt, imt = z.shape
    ubox, tbox, inner = _box(z, 0, -1, 1, 0), _box(z, 1, 0, 0, -1), _box(z, 2, -2, 2, -2)
    wt, wu, dtb, del4 = (g["kmt"] > 0).double(), (g["kmu"] > 0).double(), grid["dtb"], case["hmix"] == 4
    region = _box(z, grid["jb"] - 1, grid["je"] - jmt, grid["ib"] - 1, grid["ie"] - imt)
    wide = _box(z, grid["jb"] - 2, grid["je"] + 1 - jmt, grid["ib"] - 2, grid["ie"] + 1 - imt)

    def lap_t(x):
        cs = [g[k] * (g["kmt" + s] > 0) for k, s in (("dtn", "n"), ("dts", "s"), ("dte", "e"), ("dtw", "w"))]
        return (sum(a * s(x) for a, s in zip(cs, (_n, _s, _e, _w))) - sum(cs) * x) * wt

    gbox = inner if del4 else _box(z, 2, 0, 1, -1)
    for nc in range(4):
        hu = _to_u(f["h0"], g) * ubox
        tx, ty = (f[k] * (f["dzph"] + hu) * tbox for k in ("ub", "vb"))
        work = _fluxdiv(tx, ty, g) * g["tarea_r"] * f["vit"] * -0.25 * wt * inner
        work = _halo(torch.where(inner > 0, work, hu))
        h0 = f["h0p"] + work * dtb
        vx, vy = _viscosity(f["ubp"], f["vbp"], g, wt, wu if del4 else f["viv"] * wu, region, del4)
        gx, gy = (a * wu * ubox for a in _grad(h0, g))
        gs = (f["wgp"] - 1.0) * 9.806
        work = _to_u(h0, g) * ubox
        ax = f["viv"] * (vx + gs * gx + f["dlub"] - g["fcor"] * f["vbp"] + f["pax"] + f["pxb"] - work * f["whx"])
        ay = f["viv"] * (vy + gs * gy + f["dlvb"] + g["fcor"] * f["ubp"] + f["pay"] + f["pyb"] - work * f["why"])
        wx, wy = _halo((g["ebea"] * ax - g["ebeb"] * ay) * inner), _halo((g["ebea"] * ay + g["ebeb"] * ax) * inner)
        f["ub"], f["vb"] = f["ubp"] + wx * dtb, f["vbp"] + wy * dtb
        tx, ty = (f[k] * (f["dzph"] + work) for k in ("ub", "vb"))
        if del4:
            # the transport of the last column is what the viscosity's vorticity pass left there
            vd, ud = f["vbp"] * g["dyu"], f["ubp"] * g["dxu"]
            curl = 0.5 * (vd + _n(vd) - _w(vd) - _n(_w(vd)) - ud - _w(ud) + _n(ud) + _n(_w(ud))) * wt * _box(z, 1, 0, 1, 0)
            tx = torch.where(tbox > 0, tx, curl)
        else:
            last = gbox * (vx + gs * gx)
            tx = torch.where(tbox > 0, tx, last)
        ty = torch.where(tbox > 0, ty, (gbox * (vy + gs * gy)) if not del4 else z)
        div = _fluxdiv(tx, ty, g) * g["tarea_r"] * wt
        mix = z
        if (nc + 1) % 4 == 0:
            x = g["ahf"] * lap_t(f["h0p"]) * wide * tbox if del4 else f["h0p"]
            mix = g["ah"] * lap_t(x) * region
        work = _halo(torch.where(tbox > 0, (mix - div) * f["vit"], work))
        h0 = f["h0p"] + work * dtb
        f.update(h0p=h0, h0=h0, ubp=f["ub"], vbp=f["vb"], h0f=f["h0f"] + h0, h0bf=f["h0bf"] + h0, work=work)
    return {k: f[k] for k in BAROTR_OUT}


def _exact_bclinc(case, seed):
    block, grid, f = _bclinc_inputs(case, seed)
    g, km = _on_device(grid), block.km
    vit, viv, gg = f["vit"], f["viv"], f["gg"]
    z2 = torch.zeros_like(f["su"])
    ubox, inner, ring = _box(z2, 0, -1, 1, 0), _box(z2, 2, -2, 2, -2), _box(z2, 1, -1, 1, -1)
    dz, dzp, dt = [float(x) for x in grid["dzp"]], _lev(grid["dzp"]), grid["dtc2"]
    bot = g["kmu"].long() - 1
    at = lambda a: torch.gather(a, 0, bot.clamp(min=0)[None])[0]  # noqa: E731
    wet2 = (bot >= 0) * ring
    ub, vb = at(f["up"]), at(f["vp"])
    drag = g["c0f"] * torch.sqrt(ub * ub + vb * vb)
    sb = [f[k] * g["od0"] * wet2 for k in ("su", "sv")]
    bb = [drag * (ub * g["cag"] + g["snlat"] * vb * g["sag"]) * wet2, drag * (vb * g["cag"] - g["snlat"] * ub * g["sag"]) * wet2]
    h0bf = f["h0bf"] * g["onbb"]
    work = 0.5 * h0bf + 0.5 * f["h0bl"]
    p = [(f["psa"] * g["od0"] + work * 9.806) * vit[0]]
    for k in range(km):
        p.append(p[-1] - gg[k] * dz[k] * vit[k])
    w1 = torch.stack([0.5 * (a + b) for a, b in zip(p[:-1], p[1:])])
    w2 = (1.0 + g["ohbt"] * _lev(grid["zkt"])) * work * vit
    (x1, y1), (x2, y2) = _grad(w1, g), _grad(w2, g)
    ggu = 0.25 * (gg + _w(gg) + _s(gg) + _s(_w(gg)))
    wet = _wet(block, g["kmu"])
    gx = g["fcor"] * f["vp"] + (x1 - ggu * x2) * wet - f["dlu"]
    gy = -g["fcor"] * f["up"] + (y1 - ggu * y2) * wet - f["dlv"]
    dlv = torch.where(ubox > 0, -(g["epla"] * gy + g["eplb"] * gx) * viv, f["dlv"])
    dlu = torch.where(ubox > 0, -(g["epla"] * gx - g["eplb"] * gy) * viv, f["dlu"])
    od, ot = [float(x) for x in grid["odzp"]], [float(x) for x in grid["odzt"]]

    def solve(x, sbc, bbc):
        x = x.clone()
        e = ff = z2
        es, fs = [None] * km, [None] * km
        for k in range(km - 1, -1, -1):
            act, last = k <= bot, k == bot
            a = f["akmu"][k - 1] * ot[k] * od[k] * dt * 0.5 if k else torch.full_like(z2, od[0] * dt * 0.5)
            c = f["akmu"][k] * ot[k + 1] * od[k] * dt * 0.5 if k < km - 1 else z2
            c = torch.where(last, z2, c)
            b = torch.where(last, 1.0 + a, 1.0 + c + (a if k else 0.0))
            d = x[k] - torch.where(last, bbc * od[k] * dt * 0.5, z2)
            g0 = 1.0 / (b - c * e)
            e, ff = torch.where(act, a * g0, z2), torch.where(act, (d + c * ff) * g0, z2)
            es[k], fs[k] = e, ff
        y = sbc
        for k in range(km):
            y = (es[k] * y + fs[k]) * viv[k]
            x[k] = torch.where((k <= bot) & (inner > 0), y, x[k])
        return x

    def mean(x):
        return (dzp * g["ohbu"] * x * viv).sum(0)

    # v, then u with the new v; the depth mean is replaced by the barotropic velocity
    w = torch.where(inner > 0, f["vp"] + dlv * dt, w2)
    w = solve(w, sb[1], bb[1])
    w = (w - mean(w) + f["vb"]) * viv
    vp, v = grid["afc2"] * f["v"] + grid["afc1"] * (f["vp"] + w), w
    w = torch.where(inner > 0, f["up"] + dlu * dt, w)
    w = solve(w, sb[0], bb[0])
    x = (w - mean(w) + f["ub"]) * viv
    up = grid["afc2"] * f["u"] + grid["afc1"] * (f["up"] + x)
    return dict(u=x, v=v, up=up, vp=vp, dlu=dlu, dlv=dlv, wka=w, utf=f["utf"] + x, vtf=f["vtf"] + v, h0bf=h0bf, sbcx=sb[0],
                sbcy=sb[1], bbcx=bb[0], bbcy=bb[1])


class _Canuto:
    """The closure's tables on the device and their interpolation, for vectors of columns."""

    def __init__(self, t):
        self.t = {k: torch.from_numpy(np.ascontiguousarray(a)).to(DEV) if isinstance(a, np.ndarray) else a for k, a in t.items()}
        self.mt, self.mt0, self.nth = ls.TURB_MT, ls.TURB_MT0, ls.TURB_NTH

    def cell(self, xt, x):
        """The two table points around x, the one nearer zero first; both the end point beyond the table."""
        lo = torch.searchsorted(xt, x, right=True).clamp(1, 2 * self.mt) - 1     # xt[lo] <= x < xt[lo + 1]
        neg = x < 0.0
        on = xt[lo] == x
        below = torch.where(on & neg, lo - 1, lo).clamp(min=0)
        l0, l1 = torch.where(neg, below + 1, lo), torch.where(neg, below, lo + 1)
        end = x.abs() >= xt[-1]
        tip = torch.where(neg, 0, 2 * self.mt)
        return torch.where(end, tip, l0), torch.where(end, tip, l1)

    def line(self, x):
        t = self.t
        xt = t["and2on2a1"]
        x = torch.minimum(torch.maximum(x, xt[0]), xt[-1])
        a, b = self.cell(xt, x)
        span, d = xt[b] - xt[a], x - xt[a]
        span = torch.where(a == b, torch.ones_like(span), span)
        return [t[k][a] + (t[k][b] - t[k][a]) / span * d for k in ("amtaun2a1", "sma1", "sha1", "ssa1")]

    def plane(self, ri, rd):
        t = self.t
        rb = t["rib"]
        lo, hi = rb[0], rb[-1]
        big = torch.maximum(ri.abs() , rd.abs())
        far = (big > hi)
        ri2, rd2 = torch.where(far, hi * ri / big, ri), torch.where(far, hi * rd / big, rd)
        d0, d1 = self.cell(rb, rd2)
        most = torch.minimum(rb[self.mt + t["irimax"][d0].long()], rb[self.mt + t["irimax"][d1].long()])
        r0, r1 = self.cell(rb, ri2)
        sd, sr = rb[d1] - rb[d0], rb[r1] - rb[r0]
        flat = d0 == d1
        sd, sr = torch.where(flat, torch.ones_like(sd), sd), torch.where(r0 == r1, torch.ones_like(sr), sr)
        out = []
        for k in ("slq2b", "smb", "shb", "ssb"):
            f = t[k]
            f0 = f[d0, r0]
            val = f0 + torch.where(flat, 0.0 * f0, (f[d0, r1] - f0) / sr) * (ri2 - rb[r0]) \
                + torch.where(flat, 0.0 * f0, (f[d1, r0] - f0) / sd) * (rd2 - rb[d0])
            out.append(torch.where(ri2 > most, 0.0 * val, val))
        return ri2, rd2, out


def _exact_turb(case, seed):
    block = _block(case, seed)
    tc = _turb_case(block, seed)
    C, f, km = _Canuto(tc.tables), tc.fields, block.km
    t, b1 = C.t, tc.tables["b1"]
    jmt, imt = block.jmt, block.imt
    kmt = _dev(tc.grid["kmt"]).long()
    cols = ((_box(f["vit"], 1, -1, 1, -1) > 0) & (f["vit"][0] > 0.5)).reshape(-1).nonzero()[:, 0]
    q = {k: a.reshape(-1, jmt * imt)[:, cols] for k, a in f.items()}
    n, cor = kmt.reshape(-1)[cols] - 1, _dev(tc.grid["fcort"]).reshape(-1)[cols]
    dz, zkp = tc.grid["dzp"], tc.grid["zkp"]
    zero = torch.zeros(cols.numel(), **F64)
    z, tt, ri, rid, s2, an2, rh = ([] for _ in range(7))
    for k in range(km - 1):
        a = (k < n).double()
        r = float(dz[k] / (dz[k] + dz[k + 1]))
        z.append(-a * float(zkp[k + 1]) * 100.0)
        tt.append(a * (q["at"][k] - (q["at"][k] - q["at"][k + 1]) * r))
        for out, key in ((ri, "rit"), (rid, "ricdttms"), (s2, "s2t"), (an2, "rict")):
            out.append(a * q[key][k])
        rh.append(a * (q["pdensity"][k] + (q["pdensity"][k + 1] - q["pdensity"][k]) * r) * 1.0e-3)
    z, tt, ri, rid, s2, an2, rh = (torch.stack(a) for a in (z, tt, ri, rid, s2, an2, rh))
    # mixed layer: where the temperature first differs by 0.1 from the first level's
    k = torch.arange(km - 1, device=DEV)[:, None]
    off = ((tt - tt[0]).abs() > 0.1) & (k < n)
    first = torch.where(off, k, km).min(0)[0]
    at = lambda a, i: torch.gather(a, 0, i.clamp(0, km - 2)[None])[0]  # noqa: E731
    tk, tm, zk, zm = at(tt, first), at(tt, first - 1), at(z, first), at(z, first - 1)
    tl = tt[0] - torch.where(tt[0] - tk >= 0, 0.1, -0.1)
    mld = torch.where(first < km, zk + (zm - zk) * (tl - tk) / (tm - tk + 1.0e-20), at(z, n - 1))
    mld = torch.where(n > 0, mld, 0.0 * mld)      # a column of one level has no interface
    al0 = 0.17 * mld
    buoy = (q["buoytur"][0] + q["buoysol"][0]) * q["vit"][0] * 1.0e4
    quarter, dth = math.atan(1.0), tc.tables["deltheta_r"]
    f30, an0 = 4.0 * quarter / 43082.0, 5.24e-3
    den = f30 * math.acosh(an0 / f30)
    ak = [torch.zeros((km, cols.numel()), **F64) for _ in range(3)]
    alive = torch.ones_like(zero, dtype=torch.bool)
    below = ~alive
    an = zero
    fmx, wnd = tc.params["dfricmx"] * 1.0e4, tc.params["dwndmix"] * 1.0e4
    for k in range(km - 1):
        act = alive & (k < n)
        if not bool(act.any()):
            break
        r, rd, N2, sh2 = ri[k], rid[k], an2[k], s2[k]
        an = torch.where(N2 >= 0, torch.sqrt(N2.clamp(min=0)), an)
        small = an < cor.abs()
        x = (rd / (r + 1.0e-25) * N2) / (N2 + 1.0e-25)
        pure = N2 < float(tc.tables["rib"][0]) * sh2
        amt, *l3 = C.line(torch.nan_to_num(x))
        ri1, rid1, (p0, *p3) = C.plane(r, rd)
        ri1 = torch.where(pure, r, ri1)
        slq2 = torch.where(pure, -amt / (b1 * b1 * r + 1.0e-25), p0)
        sm, sh, ss = (torch.where(pure, a, b) for a, b in zip(l3, p3))
        alive = alive & ~(act & ~pure & (slq2 < 0))
        below = below | (act & ~pure & (slq2 == 0))
        upper = (~below | small | ((ri1 < 0) & (k <= 1))) & (slq2 > 0)
        epsy = torch.where(slq2 == 0, zero, -buoy / (1.0 / (b1 * b1 * slq2) - 0.5 * sm))
        use = (epsy >= 0) & upper
        akz = 0.4 * z[k]
        al2 = (akz * al0 / (al0 + akz)) ** 2
        lim = ~below & ~use & (ri1 > 0) & (slq2 * ri1 > 0.281)
        al2 = torch.where(lim, al2 * 0.281 / (slq2 * ri1), al2)
        slq2 = torch.where(lim, 0.281 / (ri1 + 1.0e-20), slq2)
        lat = torch.where(small, zero, cor.abs() * torch.acosh((an / cor.abs().clamp(min=1e-300)).clamp(min=1.0)) / den)
        lat = torch.where(cor.abs() == 0, zero, lat).clamp(min=7.0e-2)
        eps2 = torch.where(N2 < 0, 0.288 + zero, 0.288 * lat)
        # background mixing on the polar grid
        a, c = (r + rd) / 2.0, (r - rd) / 2.0
        ra = torch.sqrt(a * a + c * c)
        th = torch.where(a == 0, torch.where(c == 0, quarter, 2.0 * quarter), torch.atan(c / torch.where(a == 0, 1.0, a)))
        th = torch.where(th < -quarter, th + 4.0 * quarter, th)
        i0 = ((th + quarter) / dth).long() - C.nth
        i1 = i0 + 1
        rp, rn = tc.tables["theta_rcrp"], tc.tables["theta_rcrn"]
        ca = (i0 * dth <= rp) & (th > rp)
        cb = ~ca & (i1 * dth >= rn) & (th < rn)
        th = torch.where(ca, i1 * dth, torch.where(cb, i0 * dth, th))
        i0, i1 = torch.where(ca, i0 + 1, torch.where(cb, i0 - 1, i0)), torch.where(ca, i1 + 1, torch.where(cb, i1 - 1, i1))
        out = (i1 > 3 * C.nth) | (i0 < -C.nth)
        j0, j1 = (C.nth + i0).clamp(0, 4 * C.nth), (C.nth + i1).clamp(0, 4 * C.nth)
        wgt = (th - torch.where(ca, (i1 - 1) * dth, i0 * dth)) / dth
        pick = lambda key: t[key][j0] + wgt * (t[key][j1] - t[key][j0])  # noqa: E731
        br = pick("back_ra_r")
        glt = ((th <= rp) | (th >= rn)) & (br > ra)
        br = torch.where(glt, ra, br)
        out = out | (br < 0)
        bt, bc = torch.cos(th) * br, torch.sin(th) * br
        bri, _, bp = C.plane(bt + bc, bt - bc)
        bri = torch.where(glt, bri, bt + bc)
        bk = [torch.where(glt, p, pick(key)) for p, key in zip(bp, ("slq2_r1", "sm_r1", "sh_r1", "ss_r1"))]
        pos = r > 0
        out = out | (bk[0] < 0)
        alive = alive & ~(act & pos & out)
        bri = torch.where(pos, bri, zero)
        sb = [torch.where(pos & (ri1 > 0), v, zero) for v in bk[1:]]
        tb = 0.5 * b1 * b1 * bri * torch.where(pos, bk[0], zero) * eps2
        back = [tb * v for v in sb]
        bad = (sb[0] < 0) | (sb[1] < 0) | (sb[2] < 0) | (back[0] < 0) | (back[1] < 0) | (back[2] < 0)
        bad = bad | (pos & ((back[0] == 0) | (back[1] == 0)))
        alive = alive & ~(act & bad)
        # the mixing time or length scale
        deep = below & ~(ri1 >= 0) & (k >= 2)
        tmp = torch.where(below & (ri1 >= 0), 0.5 * b1 * b1 * ri1 * slq2 * eps2, zero)
        if k >= 2:
            kd = min(k + 1, km - 2)
            lastl = n - 1 == k
            gap = torch.where(lastl, z[k] - z[k - 1], z[kd] - z[k - 1])
            d1 = torch.where(lastl, rh[k] - rh[k - 1], rh[kd] - rh[k - 1])
            d2 = torch.where(lastl, rh[k] - 2.0 * rh[k - 1] + rh[k - 2], rh[kd] - 2.0 * rh[k] + rh[k - 1])
            al = 0.17 * ((d1 / gap) / (4.0 * d2 / (gap * gap))).abs()
            al = 0.4 * z[k] * al / (al + 0.4 * z[k])
            al2 = torch.where(deep, al * al, al2)
        s2k = sh2.clamp(min=1.0e-14)
        root = 0.5 * b1 * al2 * torch.sqrt(s2k / (slq2 + 1.0e-40))
        other = ~pure & ~(below & (ri1 >= 0))
        tmp = torch.where(other, torch.where(use & ~deep, 0.5 * epsy / (s2k + 1.0e-40), root), tmp)
        tmp = torch.where(pure, 0.5 * b1 * b1 * al2 * torch.sqrt(-N2 / amt), tmp)
        ok = act & alive
        for m, (s, v) in enumerate(zip((sm, sh, ss), back)):
            ak[m][k] = torch.where(ok, (tmp * s + v).clamp(max=fmx), zero)
    for m in range(3):
        ak[m][0] = torch.where(alive & (n > 0), ak[m][0].clamp(min=wnd), ak[m][0])
    tide = torch.zeros((km, cols.numel()), **F64)
    lev = torch.arange(km - 1, device=DEV)[:, None] < n
    v = 1.0e-6 + 0.20 * 0.33 * q["wave_dis"][0] * q["fz_tide"][:-1] / (q["rict"][:km - 1].clamp(min=1.0e-8) * (rh * 1000.0))
    v = torch.where(lev, v.clamp(max=1.0e-2), torch.full_like(v, 1.0))
    v = torch.flip(torch.cummin(torch.flip(v, (0,)), 0)[0], (0,))
    tide[:-1] = torch.where(lev, v, torch.zeros_like(v))
    ncc = tc.params["ncc"]

    def whole(a):
        full = torch.zeros((a.shape[0], jmt * imt), **F64)
        full[:, cols] = a
        return full.view(a.shape[0], jmt, imt)

    keep = torch.zeros((km, cols.numel()), **F64)
    keep[:-1] = 1.0
    seen = torch.zeros((km, cols.numel()), **F64)
    seen[:-1] = lev.double()
    pad = lambda a: torch.cat([a, torch.zeros_like(a[:1])])  # noqa: E731
    return dict(akmt=whole((ak[0] * 1.0e-4 + tide * 5.0) * keep),
                akt=torch.stack([whole((ak[m] * 1.0e-4 + tide) / ncc * keep) for m in (1, 2)]), ak_tide=whole(tide),
                amld=whole(mld[None] * 1.0e-2)[0], richardson=whole(q["rict"][:km] * seen), fztidal=whole(q["fz_tide"][:km] * seen),
                wp3_tidal=whole(pad(rh) * seen))
