// tracer_fused.hip -- production path of the FP64 tracer step on gfx950.
//
// Five 3-D passes per step instead of the reference's ~21 launches per
// tracer (plus the 2-D surface, SSSNORM and halo kernels that the staged
// path in tracer_kernels.hip shares):
//
//   k_prelude_col<KM>  a 64x4 block of columns marches k: face velocities
//                  u_wface/v_sface (advection_tracer_1_0), the divergence of
//                  the barotropic-corrected velocity (upwell_2,
//                  operators_div) and the continuity w (upwell_3/4), the
//                  divergence profile held in registers.
//   k_flags        tspas predictor and limiter flag of every cell (one byte)
//   k_update       limited fluxes, horizontal mixing, shortwave and explicit
//                  vertical diffusion.  Writes the explicit update (tracer_8's
//                  vtl) and the advective / vertical-diffusion diagnostics.
//   k_solve<KM>    two lanes per column (T and S): the implicit vertical
//                  diffusion (invtrit) with checkpointed elimination
//                  coefficients in registers, tracer_9's tendencies, and a
//                  streaming stability check of convadj; statically unstable
//                  columns are then mixed in place exactly as convadj_cu does.
//   k_side3/k_side2  the in-place side effects on utf, vtf, h0f and akt.
//
// Arithmetic is shared with the per-stage kernels through tracer_device.h,
// so both paths give identical bits.
#include <hip/hip_runtime.h>

#include "tracer_cells.h"
#include "tracer_device.h"
#include "tracer_internal.h"
#include "tracer_solve.h"

namespace licom {
namespace {

constexpr int KMAXF = LICOM_MAX_KM;

// ------------------------------------------------------------- prelude
// One-pass prelude: a 64x4 block of columns marches k.  Each level's wkd /
// wkb window (the block plus its east column and north row, 65 x 5) is
// staged in LDS from registers loaded a level ahead, so every velocity value
// is read from HBM once; the metrics and the barotropic factors
// (1 + work_u*ohbu, upwell_2) are loaded once per column; the divergence
// profile stays in registers for the column sum and the continuity recursion
// of upwell_3/4 (tracer.cpp:1029-1080).
template <int KM, bool FLUX>
__global__ __launch_bounds__(256) void k_prelude_col(KGrid g, KPar p, const double *__restrict__ utf,
                                                     const double *__restrict__ utl,
                                                     const double *__restrict__ vtf,
                                                     const double *__restrict__ vtl,
                                                     const double *__restrict__ work_u,
                                                     const double *__restrict__ stf_pre,
                                                     double *__restrict__ ws, double *__restrict__ uw,
                                                     double *__restrict__ vs, XcdGrid xg) {
    constexpr int WX = 65, WN = 5 * WX;
    __shared__ double sD[2][WN], sBv[2][WN];
    // dzp from LDS: a global load inside the level loop would carry a vmcnt
    // wait that also waits for the level's stores and the next level's loads
    __shared__ double sDZ[KMAXF];
    int bx, by;
    if (!xcd_block(xg, bx, by)) return;
    const int t = threadIdx.x, tx = t % 64, ty = t / 64;
    const int i0 = bx * 64, j0 = by * 4;
    const int i = i0 + tx, j = j0 + ty;
    const int imt = g.imt, jmt = g.jmt, km = g.km;
    for (int r = t; r < km; r += 256) sDZ[r] = g.dzp[r];
    const size_t n2 = (size_t)imt * jmt;
    const double oncc = p.oncc;
    // this lane's window elements: e = t and e = t + 256
    size_t wq[2];
    bool wv[2], wok[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = t + 256 * u, wr = e / WX, wc = e - wr * WX;
        const int jj = j0 - 1 + wr, ii = i0 + wc;
        wv[u] = e < WN;
        wok[u] = wv[u] && jj >= 0 && jj < jmt && ii < imt;
        wq[u] = wok[u] ? (size_t)jj * imt + ii : 0;
    }
    // window loads and the face-velocity stores go through plane buffers
    // (masked lanes read 0 / drop their store without a branch)
    uint32_t wo[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) wo[u] = buf_off(wok[u], wq[u], 8);
    const size_t pb = n2 * sizeof(double);
    double f_ut[2], f_ul[2], f_vt[2], f_vl[2];
    auto fetch = [&](int k) {
        const size_t o = (size_t)k * n2;
        const auto r_ut = plane_rsrc(utf + o, pb), r_ul = plane_rsrc(utl + o, pb);
        const auto r_vt = plane_rsrc(vtf + o, pb), r_vl = plane_rsrc(vtl + o, pb);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f_ut[u] = buf_load(r_ut, wo[u], 0.0);
            f_ul[u] = buf_load(r_ul, wo[u], 0.0);
            f_vt[u] = buf_load(r_vt, wo[u], 0.0);
            f_vl[u] = buf_load(r_vl, wo[u], 0.0);
        }
    };
    fetch(0);
    const bool in = i < imt && j < jmt;
    const size_t q = in ? (size_t)j * imt + i : 0;
    const bool do_u = in && j >= 1 && j < jmt - 1;
    const bool do_v = in && i >= 1 && i < imt - 1;
    const bool do_w = do_u && do_v;
    const double htw_c = in ? g.htw[q] : 0.0, hts_c = in ? g.hts[q] : 0.0;
    // flux faces (tracer.cpp:106-117): U-cell widths at (j-1,i), (j,i) and
    // (j,i), (j,i+1)
    double dyu_n = 0.0, dyu_c = 0.0, dxu_c = 0.0, dxu_e = 0.0;
    if constexpr (FLUX) {
        if (do_u) {
            dyu_n = g.dyu[q - imt];
            dyu_c = g.dyu[q];
        }
        if (do_v) {
            dxu_c = g.dxu[q];
            dxu_e = g.dxu[q + 1];
        }
    }
    double fc = 0, fe = 0, fn = 0, fne = 0, htw_e = 0, hts_n = 0, tr = 0;
    double ohbt = 0, stfp = 0, prev = 0;
    int kmt = 0;
    if (do_w) {
        ohbt = g.ohbt[q];
        stfp = stf_pre[q];
        prev = ws[q];
        const size_t qe = q + 1, qn = q - imt, qne = q - imt + 1;
        fc = 1.0 + work_u[q] * g.ohbu[q];
        fe = 1.0 + work_u[qe] * g.ohbu[qe];
        fn = 1.0 + work_u[qn] * g.ohbu[qn];
        fne = 1.0 + work_u[qne] * g.ohbu[qne];
        htw_e = g.htw[qe];
        hts_n = g.hts[qn];
        tr = g.tarea_r[q];
        kmt = g.kmt[q];
    }
    const uint32_t ou = buf_off(do_u, q, 8), ov = buf_off(do_v, q, 8);
    // everything loaded so far completes here, so that no wait for it stays
    // inside the level loop
    wait_all_vmem();
    const int w0 = (ty + 1) * WX + tx;
    double wka[KM];
    double w = 0.0;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        wka[k] = 0.0;
        if (k < km) {
            const int b = k & 1;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (wv[u]) {
                    sD[b][t + 256 * u] = dev::wk(f_ut[u], f_ul[u], oncc);
                    sBv[b][t + 256 * u] = dev::wk(f_vt[u], f_vl[u], oncc);
                }
            }
            if (k + 1 < km) fetch(k + 1);
            __syncthreads();
            const double dc = sD[b][w0], bc = sBv[b][w0];
            if constexpr (FLUX) {
                buf_store(plane_rsrc(uw + (size_t)k * n2, pb), ou, (sD[b][w0 - WX] * dyu_n + dc * dyu_c) * 0.25);
                buf_store(plane_rsrc(vs + (size_t)k * n2, pb), ov, (bc * dxu_c + sBv[b][w0 + 1] * dxu_e) * 0.25);
            } else {
                buf_store(plane_rsrc(uw + (size_t)k * n2, pb), ou, (sD[b][w0 - WX] + dc) * htw_c * 0.25);
                buf_store(plane_rsrc(vs + (size_t)k * n2, pb), ov, (bc + sBv[b][w0 + 1]) * hts_c * 0.25);
            }
            if (do_w && k <= kmt - 1) {
                const double de = sD[b][w0 + 1], dn = sD[b][w0 - WX], dne = sD[b][w0 - WX + 1];
                const double be = sBv[b][w0 + 1], bn = sBv[b][w0 - WX], bne = sBv[b][w0 - WX + 1];
                // operators_div (tracer.cpp:995-1003) on uk,vk of upwell_2
                const double d = 0.5 *
                                 ((fe * de + fne * dne) * htw_e - (fc * dc + fn * dn) * htw_c +
                                  (fe * be + fc * bc) * hts_c - (fne * bne + fn * bn) * hts_n) *
                                 tr;
                wka[k] = d;
                w = w - sDZ[k] * d * 1.0;
            }
        }
    }
    if (!do_w) return;
    // upwell_3 / upwell_4 (tracer.cpp:1045-1079)
    const double sc = 1.0 / (1.0 + stfp * ohbt);
#pragma unroll
    for (int k = 1; k < KM; ++k) {
        if (k < km) {
            const double cur = (k < kmt ? 1.0 : 0.0) * (prev + sDZ[k - 1] * (w * ohbt + wka[k - 1]));
            ws[(size_t)k * n2 + q] = cur * sc;
            prev = cur;
        }
    }
}

// --------------------------------------------------- limiter flags and update
// Replaces a march of 16 x 12 tiles whose planes a fourth wave staged in LDS
// (two barriers a level, two workgroups per CU: bound by the latency of its
// level loop, 7.03 ms at 1800 x 1151 x 55, 71 us at 128 x 96 x 30; now 6.5 ms
// and 32 us, k_flags bound by its ~200 FP64 instructions a cell and k_update
// by its 11 + 8 planes of HBM traffic, 4.2 TB/s; at 3600 x 2302 x 55 it
// was 26.5 ms and is 24.8).  Neither kernel carries anything from one
// level to the next but values it has already loaded, so a column is cut into
// chunks of levels and every (chunk, run of cells, tracer) is a workgroup of
// its own.  Runs of cells and chunks: tracer_cells.h.

// tspas predictor and limiter flag (advection_tracer_2, tracer.cpp:311-545),
// one byte per cell, of every cell off the outermost rows and columns (the
// outermost columns get bytes that nothing reads).
__global__ __launch_bounds__(256, 4) void k_flags(KGrid g, double dts, const double *__restrict__ at,
                                                  const double *__restrict__ uw, const double *__restrict__ vs,
                                                  const double *__restrict__ ws, uint8_t *__restrict__ flags,
                                                  const double *__restrict__ odzp, const double *__restrict__ odzt,
                                                  FlatGrid fg) {
    int n, blk, k0;
    const int item = xcd_item((int)blockIdx.x, fg.per);
    if (item >= fg.total) return;
    flat_item(fg, item, n, blk, k0);
    const int imt = g.imt, km = g.km, n2 = imt * g.jmt, lane = (int)threadIdx.x & 63;
    const int p = lane_cell(fg, blk);
    const int pc = clamp_cell(p, n2), pn = clamp_cell(p - imt, n2), ps = clamp_cell(p + imt, n2);
    uint32_t bc = 8u * (uint32_t)pc, bn = 8u * (uint32_t)pn, bs = 8u * (uint32_t)ps;
    const bool own = lane >= 1 && lane <= 62;
    const bool own0 = own && p < fg.last, own1 = own && p + 1 < fg.last;
    const double *T = at + (size_t)n * n2 * km;
    uint8_t *F = flags + (size_t)n * n2 * km;
    const Faces fc = load_faces(g, pc, pn);
    int kc[4], kn[2], ks[2];     // wet levels: cells -1..2, and the rows beside
    kc[1] = g.kmt[pc];
    kc[2] = g.kmt[pc + 1];
    kc[0] = dpp<kFromPrev>(kc[2]);
    kc[3] = dpp<kFromNext>(kc[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        kn[e] = g.kmt[pn + e];
        ks[e] = g.kmt[ps + e];
    }
    const int k1 = min(k0 + fg.kc, km);
    const size_t o0 = (size_t)k0 * n2;
    D2 Tu{}, Tc = ld2(T + o0, bc), Wk = ld2(ws + o0, bc);
    if (k0 > 0) Tu = ld2(T + o0 - n2, bc);
    march_levels(k0, k1, km, [&](auto pos, int K) {
        constexpr bool top = pos == 0, bot = pos == 2;
        const double oz = odzp[K], ot = odzt[K], ot1 = bot ? 0.0 : odzt[K + 1];
        const size_t o = (size_t)K * n2;
        fresh(bc);
        fresh(bn);
        fresh(bs);
        const D2 Tn = ld2(T + o, bn), Ts = ld2(T + o, bs);
        const D2 U = ld2(uw + o, bc), Vs = ld2(vs + o, bc), Vn = ld2(vs + o, bn);
        D2 Td{}, Wb{};
        if constexpr (!bot) {
            Td = ld2(T + o + n2, bc);
            Wb = ld2(ws + o + n2, bc);
        }
        const D2 Tw = west(Tc), Te = east(Tc), Ue = east(U);
        uint32_t fl = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const double tc = Tc.v[e];
            dev::PTerms t;
            dev::pterms(tc, Te.v[e], Tw.v[e], Ts.v[e], Tn.v[e], Tu.v[e], Td.v[e], Ue.v[e], U.v[e], Vs.v[e], Vn.v[e],
                        Wk.v[e], Wb.v[e], fc.tr[e], fc.dx[e + 1], fc.dx[e], fc.ds[e], fc.dn[e], top ? 0 : 1, bot ? 2 : 3, oz, ot, ot1, dts, t);
            const double a00 = dev::predictor(t, tc, dts);
            // 7-point bounds with land masked to -+1e10 (tracer.cpp:416-545)
            const double lo = -1.0e10, hi = 1.0e10;
            const int kz = kc[e + 1];
            double mx = kz > K ? tc : lo, mn = kz > K ? tc : hi;
            auto bound = [&](bool wet, double v) {
                mx = fmax(mx, wet ? v : lo);
                mn = fmin(mn, wet ? v : hi);
            };
            bound(kn[e] > K, Tn.v[e]);
            bound(ks[e] > K, Ts.v[e]);
            bound(kc[e] > K, Tw.v[e]);
            bound(kc[e + 2] > K, Te.v[e]);
            if constexpr (!top) bound(kz > K - 1, Tu.v[e]);
            if constexpr (!bot) bound(kz > K + 1, Td.v[e]);
            fl |= (uint32_t)(a00 > mx || a00 < mn) << (8 * e);
        }
        const uint32_t fc8 = bc >> 3;
        if (own1) *reinterpret_cast<licom_u16 *>(F + o + fc8) = (uint16_t)fl;
        else if (own0) F[o + fc8] = (uint8_t)fl;
        Tu = Tc;
        Tc = Td;
        Wk = Wb;
    });
}

// del2 stencil of a lane's two cells in one row (DTN..DTW).
struct Del2 {
    D2 dn, ds, de, dw;
};
// cc * X + sum of the wet neighbours' terms (tracer.cpp:1165-1180, 1249-1286)
__device__ __forceinline__ double del2(const Del2 &m, uint32_t wet, int e, uint32_t k, double Xc, double Xn, double Xs,
                                       double Xe, double Xw) {
    double h = 0.0, cc = 0.0;
    if (k < (wet & 255u)) { h += m.dn.v[e] * Xn; cc -= m.dn.v[e]; }
    if (k < (wet >> 8 & 255u)) { h += m.ds.v[e] * Xs; cc -= m.ds.v[e]; }
    if (k < (wet >> 16 & 255u)) { h += m.de.v[e] * Xe; cc -= m.de.v[e]; }
    if (k < (wet >> 24)) { h += m.dw.v[e] * Xw; cc -= m.dw.v[e]; }
    return cc * Xc + h;
}

struct UpdateArgs {
    const double *stf_n, *err_norm2, *swv, *restore;
    double *ax, *ay, *az, *dz, *pen;
    uint8_t *flags_out;   // the limiter flag of every physical cell, or NULL
};

// Limited fluxes, horizontal mixing, shortwave and explicit vertical
// diffusion of every interior cell: tracer_8's explicit update (ori) and the
// ax/ay/az/dz/penetrate diagnostics.  The biharmonic operator's first pass is
// formed again for the rows on both sides of the lane's own (two more loads
// of atb a level, where its 16 bytes a cell would be written and read back).
// Waves per SIMD: del4 two (its 19 slots of metrics leave LDS for two
// workgroups).  del2 three, with 16 registers a lane spilled; at two nothing
// spills and it takes as long (4.78 against 4.81 ms at 1800 x 1151 x 55, 112
// against 114 us at 360 x 218 x 30, 21 us both at 128 x 96 x 30).
template <int ADV, bool DEL4>
__global__ __launch_bounds__(256, DEL4 ? 2 : 3) void k_update(KGrid g, KPar p, const double *__restrict__ at,
                                                   const double *__restrict__ atb, const double *__restrict__ akt,
                                                   const double *__restrict__ uw, const double *__restrict__ vs,
                                                   const double *__restrict__ ws, const uint8_t *__restrict__ flags,
                                                   double *__restrict__ ori, const double *__restrict__ odzp,
                                                   const double *__restrict__ odzt, const double *__restrict__ penk,
                                                   UpdateArgs a, FlatGrid fg) {
    constexpr bool tspas = ADV == LICOM_ADV_TSPAS;
    int n, blk, k0;
    const int item = xcd_item((int)blockIdx.x, fg.per);
    if (item >= fg.total) return;
    flat_item(fg, item, n, blk, k0);
    const int imt = g.imt, jmt = g.jmt, km = g.km, n2 = imt * jmt, lane = (int)threadIdx.x & 63;
    const size_t n3 = (size_t)n2 * km;
    const int pl = lane_cell(fg, blk);
    const int pc = clamp_cell(pl, n2), pn = clamp_cell(pl - imt, n2), ps = clamp_cell(pl + imt, n2);
    uint32_t bc = 8u * (uint32_t)pc, bn = 8u * (uint32_t)pn, bs = 8u * (uint32_t)ps;
    bool own[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int c = pl + e, i = c % imt;
        own[e] = lane >= 1 && lane <= 62 && c < fg.last && i >= 2 && i < imt - 2;
    }

    const double *T = at + n * n3;
    const double *TB = atb + n * (n3 + n2) + n2;     // level k at plane k
    const double *A = akt + n * n3;
    const uint8_t *F = flags + n * n3;
    const double dts = p.dts;
    int kmt[2];
    double sw[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        kmt[e] = g.kmt[pc + e];
        sw[e] = (n == 0 && a.swv) ? a.swv[pc + e] : 0.0;
    }
    const bool rest = p.boundary_restore == 1 && a.restore != nullptr;
    const double lamda = 1.0 / (15.0 * 86400.0);
    const double aidif = 0.5;

    // The lane's metrics wait in LDS and are read anew at each level: in
    // registers they would leave too few for the level's loads and waves.
    // del4 adds the stencils of the rows on both sides (outer rows bN, bS).
    __shared__ licom_d2a sM[DEL4 ? 19 : 8][256];
    auto keep = [&](int slot, double x, double y) { sM[slot][threadIdx.x] = licom_d2a{x, y}; };
    auto get = [&](int slot) {
        const licom_d2a x = sM[slot][threadIdx.x];
        return D2{{x.x, x.y}};
    };
    {
        const Faces fc = load_faces(g, pc, pn);
        keep(0, fc.tr[0], fc.tr[1]);
        keep(1, fc.dx[0], fc.dx[1]);
        keep(2, fc.ds[0], fc.ds[1]);
        keep(3, fc.dn[0], fc.dn[1]);
    }
    uint32_t wet[3][2];
    uint32_t bN = 0, bS = 0;
    load_wet(g, pc, pn, ps, wet[0]);
    if constexpr (DEL4) {
        const int pN = clamp_cell(pl - 2 * imt, n2), pS = clamp_cell(pl + 2 * imt, n2);
        load_wet(g, pn, pN, pc, wet[1]);
        load_wet(g, ps, pc, pS, wet[2]);
        bN = 8u * (uint32_t)pN;
        bS = 8u * (uint32_t)pS;
    }
    {
        const double *co[5] = {g.dtn, g.dts, g.dte, g.dtw, g.ahf};
#pragma unroll
        for (int r = 0; r < (DEL4 ? 3 : 1); ++r)
#pragma unroll
            for (int c = 0; c < (DEL4 ? 5 : 4); ++c) {
                const int cell = r == 0 ? pc : (r == 1 ? pn : ps);
                keep(4 + r * 5 + c, co[c][cell], co[c][cell + 1]);
            }
    }
    auto stencil = [&](int r) { return Del2{get(4 + r * 5), get(5 + r * 5), get(6 + r * 5), get(7 + r * 5)}; };

    const int k1 = min(k0 + fg.kc, km);
    const size_t o0 = (size_t)k0 * n2;
    D2 Tu{}, Bu{}, Au{}, Tc = ld2(T + o0, bc), Bc = ld2(TB + o0, bc), Wk = ld2(ws + o0, bc);
    uint32_t fu = 0, f0 = 0;
    if constexpr (tspas) f0 = ldf2(F + o0, (uint32_t)pc);
    if (k0 > 0) {
        Tu = ld2(T + o0 - n2, bc);
        Bu = ld2(TB + o0 - n2, bc);
        Au = ld2(A + o0 - n2, bc);
#pragma unroll
        for (int e = 0; e < 2; ++e) Au.v[e] = dev::floor_akt(Au.v[e], k0 - 1, n, p.hmix, p.dwndmix);
        if constexpr (tspas) fu = ldf2(F + o0 - n2, (uint32_t)pc);
    }

    march_levels(k0, k1, km, [&](auto pos, int k) {
        constexpr bool top = pos == 0, bot = pos == 2;
        // the shared expressions tell first, inner and last levels apart
        constexpr int kp = top ? 0 : 1, kq = bot ? 2 : 3;
        const double oz = odzp[k], ot = odzt[k], ot1 = bot ? 0.0 : odzt[k + 1];
        const double pe = bot ? 0.0 : penk[k], peu = top ? 0.0 : penk[k - 1];
        const size_t o = (size_t)k * n2, on = n * n3 + o;
        fresh(bc);
        fresh(bn);
        fresh(bs);
        if constexpr (DEL4) {
            fresh(bN);
            fresh(bS);
        }
        const D2 Tn = ld2(T + o, bn), Ts = ld2(T + o, bs);
        const D2 Bn = ld2(TB + o, bn), Bs = ld2(TB + o, bs);
        const D2 U = ld2(uw + o, bc), Vs = ld2(vs + o, bc), Vn = ld2(vs + o, bn);
        D2 Ac = ld2(A + o, bc), Td{}, Wb{}, Bd{}, BN{}, BS{}, Rk{};
        uint32_t fd = 0, fn = 0, fs = 0;
        if constexpr (DEL4) {
            BN = ld2(TB + o, bN);
            BS = ld2(TB + o, bS);
        }
        if constexpr (tspas) {
            fn = ldf2(F + o, bn >> 3);
            fs = ldf2(F + o, bs >> 3);
        }
        if constexpr (!bot) {
            Td = ld2(T + o + n2, bc);
            Bd = ld2(TB + o + n2, bc);
            Wb = ld2(ws + o + n2, bc);
            if constexpr (tspas) fd = ldf2(F + o + n2, bc >> 3);
        }
        const bool rk = !top && rest;
        if (rk) Rk = ld2(a.restore + on, bc);
        const D2 Tw = west(Tc), Te = east(Tc), Bw = west(Bc), Be = east(Bc), Ue = east(U);
        // horizontal mixing (tracer_del4_2 / tracer_4)
        double hm[2];
        asm volatile("" ::: "memory");
        const Del2 M = stencil(0);
        if constexpr (DEL4) {
            const D2 Nw = west(Bn), Ne = east(Bn), Sw = west(Bs), Se = east(Bs);
            D2 dc, dn, ds;
            {
                const Del2 R = stencil(1);
                const D2 ahf = get(13);
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    dn.v[e] = ahf.v[e] * del2(R, wet[1][e], e, k, Bn.v[e], BN.v[e], Bc.v[e], Ne.v[e], Nw.v[e]);
            }
            {
                const Del2 R = stencil(2);
                const D2 ahf = get(18);
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    ds.v[e] = ahf.v[e] * del2(R, wet[2][e], e, k, Bs.v[e], Bc.v[e], BS.v[e], Se.v[e], Sw.v[e]);
            }
            const D2 ahf = get(8);
#pragma unroll
            for (int e = 0; e < 2; ++e)
                dc.v[e] = ahf.v[e] * del2(M, wet[0][e], e, k, Bc.v[e], Bn.v[e], Bs.v[e], Be.v[e], Bw.v[e]);
            const D2 dw = west(dc), de = east(dc);
#pragma unroll
            for (int e = 0; e < 2; ++e) hm[e] = del2(M, wet[0][e], e, k, dc.v[e], dn.v[e], ds.v[e], de.v[e], dw.v[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) hm[e] = del2(M, wet[0][e], e, k, Bc.v[e], Bn.v[e], Bs.v[e], Be.v[e], Bw.v[e]);
        }
        // limiter flags of the cells to the west and east
        const uint32_t fw = ((uint32_t)dpp<kFromPrev>((int)f0) >> 8) | (f0 << 8);
        const uint32_t fe = (f0 >> 8) | ((uint32_t)dpp<kFromNext>((int)f0) << 8);
        const D2 mtr = get(0), mdx = get(1), mds = get(2), mdn = get(3);
        const double mde[2] = {mdx.v[1], dppd<kFromNext>(mdx.v[0])};
        double xx[2], yy[2], zz[2], dzv[2], pv[2], out[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const double tc = Tc.v[e], wk = Wk.v[e], wb = Wb.v[e], tr = mtr.v[e];
            const double vk = k < kmt[e] ? 1.0 : 0.0;
            double tf;
            if constexpr (!tspas) {
                // advection_tracer_1 (tracer.cpp:120-289); the centered form
                // accumulates its diagnostics (the caller's ax/ay/az carry the
                // sum over the diagnostic period)
                const dev::CFAdv cf = dev::adv_cf(ADV, tc, Te.v[e], Tw.v[e], Ts.v[e], Tn.v[e], Tu.v[e], Td.v[e],
                                                  Ue.v[e], U.v[e], Vs.v[e], Vn.v[e], wk, wb, tr, kp, kq, oz);
                const double nss = (double)p.nss;
                xx[e] = cf.hx / nss;
                yy[e] = cf.hy / nss;
                zz[e] = cf.vz / nss;
                tf = cf.adv * vk;
            } else {
                const bool lim = (f0 >> (8 * e)) & 1u;
                dev::PTerms t;
                dev::pterms(tc, Te.v[e], Tw.v[e], Ts.v[e], Tn.v[e], Tu.v[e], Td.v[e], Ue.v[e], U.v[e], Vs.v[e],
                            Vn.v[e], wk, wb, tr, mde[e], mdx.v[e], mds.v[e], mdn.v[e], kp, kq, oz, ot, ot1, dts, t);
                // a face is upwind where a cell beside it is limited
                // (tracer.cpp:574-658; every face of an interior cell passes
                // the reference's index tests)
                auto up = [&](uint32_t f) { return lim || ((f >> (8 * e)) & 1u); };
                const double xy1 = up(fe) ? dev::up_xy1(Te.v[e], tc, Ue.v[e], tr) : t.xy1;
                const double xy2 = up(fw) ? dev::up_xy2(tc, Tw.v[e], U.v[e], tr) : t.xy2;
                const double xy3 = up(fs) ? dev::up_xy1(Ts.v[e], tc, Vs.v[e], tr) : t.xy3;
                const double xy4 = up(fn) ? dev::up_xy2(tc, Tn.v[e], Vn.v[e], tr) : t.xy4;
                double zb1 = 0.0, zb2 = 0.0;
                if constexpr (!top) zb1 = up(fu) ? dev::up_zb1(Tu.v[e], tc, wk, oz) : t.zb1;
                if constexpr (!bot) zb2 = up(fd) ? dev::up_zb2(tc, Td.v[e], wb, oz) : t.zb2;
                xx[e] = -(t.x0 + xy1 + xy2 + t.c1);
                yy[e] = -(t.y0 + xy3 + xy4 + t.c2);
                zz[e] = -(t.za + zb1 + zb2 + t.zc);
                tf = (xx[e] + yy[e] + zz[e]) * vk;
            }
            tf += p.ah * hm[e];
            // shortwave penetration (T) and explicit vertical diffusion
            // (tracer_5, boundary levels as its k==0 thread applies them)
            const double v1 = (!bot && k + 1 < kmt[e]) ? 1.0 : 0.0;
            {
                double ts;
                if constexpr (top) {
                    const double wt1 = sw[e] * pe * (1 < kmt[e] ? 1.0 : 0.0);
                    ts = tf - oz * wt1;
                    pv[e] = -wt1 * oz;
                } else if constexpr (bot) {
                    const double wt2 = sw[e] * peu * vk;
                    ts = tf + oz * wt2;
                    pv[e] = wt2 * oz;
                } else {
                    const double wt1 = sw[e] * peu * vk;
                    const double wt2 = sw[e] * pe * v1;
                    ts = tf + (wt1 - wt2) * oz;
                    pv[e] = (wt1 - wt2) * oz;
                }
                tf = n == 0 ? ts : tf;
            }
            Ac.v[e] = dev::floor_akt(Ac.v[e], k, n, p.hmix, p.dwndmix);
            const double b = Bc.v[e];
            if constexpr (top) {
                const double wt1 = Ac.v[e] * (b - Bd.v[e]) * ot1 * v1;
                tf = tf - oz * wt1 * 0.5;
                dzv[e] = -oz * wt1 * 0.5;
            } else if constexpr (bot) {
                const double wt2 = Au.v[e] * (Bu.v[e] - b) * ot * vk;
                tf = tf + oz * wt2 * (1.0 - aidif);
                dzv[e] = oz * wt2 * 0.5;
            } else {
                const double wt1 = Au.v[e] * (Bu.v[e] - b) * ot * vk;
                const double wt2 = Ac.v[e] * (b - Bd.v[e]) * ot1 * v1;
                tf = tf + oz * (wt1 - wt2) * 0.5;
                dzv[e] = oz * (wt1 - wt2) * 0.5;
            }
            // surface fluxes (tracer_5 n=1, tracer_6) and restoring (tracer_7)
            if constexpr (top) {
                const double stf = a.stf_n[(size_t)n * n2 + pc + e];
                if (n == 1) {
                    if (kmt[e] > 0) tf = tf + stf * (1.0 - aidif) * oz;
                    if (p.sssnorm) tf = tf + a.err_norm2[0] * vk;
                } else if (kmt[e] > 0) {
                    tf = tf + stf * oz * 0.5;
                }
            }
            if (rk) tf = tf + vk * (Rk.v[e] - b) * lamda;
            // tracer_8: the explicit update entering the implicit solve
            out[e] = tc + dts * tf;
        }
        if constexpr (ADV == LICOM_ADV_CENTERED) {
            auto add = [&](double *d, double sign, const double (&x)[2]) {
                const D2 y = ld2(d + on, bc);
                const double s[2] = {y.v[0] + sign * x[0], y.v[1] + sign * x[1]};
                st2(d + on, bc, s, own[0], own[1]);
            };
            if (a.ax) add(a.ax, 1.0, xx);
            if (a.ay) add(a.ay, 1.0, yy);
            if (a.az) add(a.az, -1.0, zz);
        } else if constexpr (tspas) {
            if (a.ax) st2(a.ax + on, bc, xx, own[0], own[1]);
            if (a.ay) st2(a.ay + on, bc, yy, own[0], own[1]);
            if (a.az) st2(a.az + on, bc, zz, own[0], own[1]);
        }
        if (n == 0 && a.pen) st2(a.pen + o, bc, pv, own[0], own[1]);
        if (a.dz) st2(a.dz + on, bc, dzv, own[0], own[1]);
        if (a.flags_out) {
            if (own[0]) a.flags_out[on + (bc >> 3)] = (uint8_t)(f0 & 1u);
            if (own[1]) a.flags_out[on + (bc >> 3) + 1] = (uint8_t)(f0 >> 8);
        }
        st2(ori + on, bc, out, own[0], own[1]);
        Tu = Tc;
        Tc = Td;
        Bu = Bc;
        Bc = Bd;
        Au = Ac;
        Wk = Wb;
        fu = f0;
        f0 = fd;
    });
}

template <int ADV>
void launch_update(licom_ctx *ctx, const licom_fields *f, const licom_diag *d, const Scratch &s) {
    const KGrid &g = ctx->g;
    hipStream_t st = ctx->stream;
    if constexpr (ADV == LICOM_ADV_TSPAS) {
        Timer t(ctx, "k_flags");
        const FlatGrid fg = flat_grid(g.imt, (g.jmt - 1) * g.imt, g.km);
        k_flags<<<8 * fg.per, 256, 0, st>>>(g, ctx->kp.dts, f->at, s.uw, s.vs, f->ws, s.flags, g.odzp, g.odzt, fg);
    }
    Timer t(ctx, "k_update");
    UpdateArgs a{};
    a.stf_n = s.stf_n;
    a.err_norm2 = s.err_norm2;
    a.swv = f->swv;
    a.restore = f->restore;
    a.ax = d ? d->ax : nullptr;
    a.ay = d ? d->ay : nullptr;
    a.az = d ? d->az : nullptr;
    a.dz = d ? d->dz : nullptr;
    a.pen = d ? d->penetrate : nullptr;
    a.flags_out = ctx->flags_out;
    const FlatGrid fg = update_grid(g.imt, g.jmt, g.km);
    auto kern = ctx->kp.hmix == LICOM_HMIX_DEL4 ? k_update<ADV, true> : k_update<ADV, false>;
    kern<<<8 * fg.per, 256, 0, st>>>(g, ctx->kp, f->at, f->atb, f->akt, s.uw, s.vs, f->ws, s.flags, s.ori, g.odzp,
                                     g.odzt, g.pen, a, fg);
}

// Side effects of tracer_1_0 / tracer_1 / tracer_del4_2 (tracer.cpp:1088,
// 1107-1108, 1187, 1315): utf, vtf *= oncc over the whole 3-D arrays (one
// or two elements per lane, a pure streaming pass), then h0f *= onbc and the
// AKT surface floor written back on the 2-D plane.
template <typename V>
__global__ __launch_bounds__(256) void k_side3(V *__restrict__ utf, V *__restrict__ vtf, size_t n,
                                               double oncc) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    V a = utf[t], b = vtf[t];
    if constexpr (sizeof(V) == 16) {
        a.x *= oncc; a.y *= oncc;
        b.x *= oncc; b.y *= oncc;
    } else {
        a *= oncc;
        b *= oncc;
    }
    utf[t] = a;
    vtf[t] = b;
}

__global__ __launch_bounds__(256) void k_side2(KGrid g, KPar p, double *h0f, double *akt) {
    const size_t n2 = (size_t)g.imt * g.jmt, n3 = n2 * g.km;
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n2) return;
    h0f[t] = h0f[t] * p.onbc;
    const int j = (int)(t / g.imt), i = (int)(t % g.imt);
    if (i >= 1 && i < g.imt - 1 && j >= 1 && j < g.jmt - 1)
        for (int n = 0; n < 2; ++n)
            akt[n * n3 + t] = dev::floor_akt(akt[n * n3 + t], 0, n, p.hmix, p.dwndmix);
}

void launch_side(licom_ctx *ctx, const licom_fields *f) {
    const KGrid &g = ctx->g;
    hipStream_t st = ctx->stream;
    Timer t(ctx, "k_side");
    const size_t n3 = ctx->n3;
    const bool vec = ((reinterpret_cast<uintptr_t>(f->utf) | reinterpret_cast<uintptr_t>(f->vtf)) & 15) == 0 &&
                     n3 % 2 == 0;
    if (vec) {
        const size_t n = n3 / 2;
        k_side3<double2><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(
            reinterpret_cast<double2 *>(f->utf), reinterpret_cast<double2 *>(f->vtf), n, ctx->kp.oncc);
    } else {
        k_side3<double><<<(unsigned)((n3 + 255) / 256), 256, 0, st>>>(f->utf, f->vtf, n3, ctx->kp.oncc);
    }
    k_side2<<<(unsigned)((ctx->n2 + 255) / 256), 256, 0, st>>>(g, ctx->kp, f->h0f, f->akt);
}

template <int KM>
void launch_prelude_solve(licom_ctx *ctx, const licom_fields *f, const licom_diag *d, int flags,
                          bool prelude, const Scratch &s) {
    const KGrid &g = ctx->g;
    const KPar &p = ctx->kp;
    hipStream_t st = ctx->stream;
    if (prelude) {
        Timer t(ctx, "k_prelude");
        const XcdGrid xg = xcd_grid((g.imt + 63) / 64, (g.jmt + 3) / 4);
        if (p.adv == LICOM_ADV_FLUX)
            k_prelude_col<KM, true><<<xcd_blocks(xg), 256, 0, st>>>(g, p, f->utf, f->utl, f->vtf, f->vtl,
                                                                    s.work_u, s.stf_pre, f->ws, s.uw, s.vs, xg);
        else
            k_prelude_col<KM, false><<<xcd_blocks(xg), 256, 0, st>>>(g, p, f->utf, f->utl, f->vtf, f->vtl,
                                                                     s.work_u, s.stf_pre, f->ws, s.uw, s.vs, xg);
    } else {
        Timer t(ctx, "k_solve");
        const dim3 gr = solve_grid(g.imt, g.jmt, ctx->solve_shape);
        if (flags & LICOM_STEP_ICESNOW)
            k_solve_ice<KM, double, double><<<gr, 256, 0, st>>>(g, p, flags, f->at, f->atb, f->akt, s.ori, s.stf_n,
                                                  d ? d->tend : nullptr, d ? d->dt_diff : nullptr,
                                                  d ? d->dt_conv : nullptr, s.mix_count, ctx->solve_shape,
                                                  ctx->qice);
        else
            k_solve<KM, double, double><<<gr, 256, 0, st>>>(g, p, flags, f->at, f->atb, f->akt, s.ori, s.stf_n,
                                              d ? d->tend : nullptr, d ? d->dt_diff : nullptr,
                                              d ? d->dt_conv : nullptr, s.mix_count, ctx->solve_shape);
    }
}

void launch_column(licom_ctx *ctx, const licom_fields *f, const licom_diag *d, int flags,
                   bool prelude, const Scratch &s) {
    switch (ctx->km) {
        case 30: launch_prelude_solve<30>(ctx, f, d, flags, prelude, s); break;
        case 55: launch_prelude_solve<55>(ctx, f, d, flags, prelude, s); break;
        default: launch_prelude_solve<KMAXF>(ctx, f, d, flags, prelude, s); break;
    }
}

}  // namespace

int launch_step_fused(licom_ctx *ctx, const licom_fields *f, const licom_diag *d, int flags,
                      const Scratch &s) {
    if (int rc = launch_surface(ctx, f, d, s)) return rc;
    launch_column(ctx, f, d, flags, true, s);
    switch (ctx->kp.adv) {
        case LICOM_ADV_CENTERED: launch_update<LICOM_ADV_CENTERED>(ctx, f, d, s); break;
        case LICOM_ADV_FLUX: launch_update<LICOM_ADV_FLUX>(ctx, f, d, s); break;
        default: launch_update<LICOM_ADV_TSPAS>(ctx, f, d, s); break;
    }
    launch_column(ctx, f, d, flags, false, s);
    if (flags & LICOM_STEP_SIDE_EFFECTS) launch_side(ctx, f);
    return launch_halo(ctx, f, flags);
}

}  // namespace licom
