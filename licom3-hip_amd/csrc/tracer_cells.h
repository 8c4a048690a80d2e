// tracer_cells.h -- the FP64 and the mixed limiter-flag and update kernels'
// split of a plane: runs of two cells a lane, chunks of levels.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tracer_internal.h"

namespace licom {
namespace {

// Each lane takes two consecutive cells of the plane, whatever the row
// length, and neighbours along i come from the lanes beside it (DPP): the
// vector cache handles a 16-byte access of a wave in the same 16 cycles as an
// 8-byte one, and with one cell per lane (and so e and w loads of their own)
// its access rate, not HBM, bounded the kernels.  A wave's first and last
// lane only feed their neighbours: 124 of its 128 cells are its own.
constexpr int kWaveCells = 124;

struct FlatGrid {
    int first, last;  // cells [first, last) of the plane
    int nch, kc;      // chunks of a column, levels per chunk
    int total, per;   // workgroups, and workgroups per XCD
    bool apart;       // all of one tracer before the other (update_grid)
};

// Whole columns, where those give the 256 CUs four workgroups each (smaller
// chunks read the levels around them again: at 1800 x 1151 x 55 chunks of 55,
// 28, 14 and 7 levels took 6.65, 6.69, 6.79 and 7.16 ms for both FP64 kernels,
// their tracers side by side), and otherwise as many chunks as that takes
// (want: its share of the 1024 workgroups), of two levels at least.  A plane
// has five rows or more, so it is never without cells.
inline FlatGrid flat_grid(int first, int last, int km, int want = 1024) {
    const int nb = (last - first + 4 * kWaveCells - 1) / (4 * kWaveCells);
    int nch = std::max((want + 2 * nb - 1) / (2 * nb), 1);
    const int kc = std::max((km + nch - 1) / nch, 2);
    nch = (km + kc - 1) / kc;
    const int total = 2 * nb * nch;
    return FlatGrid{first, last, nch, kc, total, (total + 7) / 8, false};
}

// The update's grid.  Where its plane fills the chip with whole columns, all
// workgroups of T come before those of S: side by side, the two tracers have
// twice as many planes open at a time, which costs more there than the face
// velocities and metrics that they could share (k_update_mx at 3600 x 2302 x 55
// 15.8 -> 14.6 ms, with which the mixed step takes 42.1 ms and not 43.2; at
// 1800 x 1151 x 55 3.64 -> 3.57; k_update 19.0 -> 18.2 and 5.10 -> 4.96; at
// 600 x 440 x 55 either way the same).  On small planes, which the L2s hold, it
// is the other way round (k_update_mx at 96 x 64 x 55: 13.4 us side by side, 14.4
// apart; k_update at 128 x 96 x 30: 21.3, 23), and for the flags on every plane
// (k_flags_mx at 3600 x 2302 x 55: 4.46, 4.68 ms).
inline FlatGrid update_grid(int imt, int jmt, int km, int want = 1024) {
    FlatGrid f = flat_grid(2 * imt, (jmt - 2) * imt, km, want);
    f.apart = f.total / f.nch >= 1024;
    return f;
}

// Block -> (tracer, chunk, block of the plane): the two tracers of one place
// (unless they are kept apart), then its chunks, run next to each other, and
// the hardware's round-robin deal of blocks to the eight XCDs is undone, so
// that each XCD's L2 sees a run of neighbouring blocks, whose rows and face
// velocities they share.
__device__ __forceinline__ int xcd_item(int b, int per) { return (b & 7) * per + (b >> 3); }
__device__ __forceinline__ void flat_item(const FlatGrid &f, int L, int &n, int &blk, int &k0) {
    const int half = f.total >> 1;
    n = f.apart ? L >= half : L & 1;
    const int h = f.apart ? L - n * half : L >> 1;
    blk = h / f.nch;
    k0 = (h - blk * f.nch) * f.kc;
}

// First of this lane's two cells; it may lie outside the plane for lanes
// that own none of their cells.
__device__ __forceinline__ int lane_cell(const FlatGrid &f, int blk) {
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    return f.first + (blk * 4 + wave) * kWaveCells + 2 * (lane - 1);
}

// Two cells of a plane at byte offset `off`: the plane's address is the same
// in every lane, so an access needs one 32-bit address register.
struct D2 {
    double v[2];
};
typedef double licom_d2 __attribute__((ext_vector_type(2), aligned(8)));
typedef double licom_d2a __attribute__((ext_vector_type(2)));
typedef uint16_t licom_u16 __attribute__((aligned(1)));
__device__ __forceinline__ D2 ld2(const double *plane, uint32_t off) {
    const licom_d2 x = *reinterpret_cast<const licom_d2 *>(reinterpret_cast<const char *>(plane) + off);
    return D2{{x.x, x.y}};
}
__device__ __forceinline__ uint32_t ldf2(const uint8_t *plane, uint32_t off) {
    return *reinterpret_cast<const licom_u16 *>(plane + off);
}
// Stores of the cells that a0 and a1 mark.  Non-temporal: on a large grid
// nothing reads them again before the caches have turned over (k_update 5.22 ->
// 5.02 ms at 1800 x 1151 x 55).  On a small one k_solve reads ori, one of them,
// from the caches; with ori alone stored plainly k_update takes 22.6 us in
// place of 21.3 at 128 x 96 x 30, 121 in place of 113 at 360 x 218 x 30, and the
// solve the same to 2 us, so ori goes the same way.
__device__ __forceinline__ void st2(double *plane, uint32_t off, const double (&x)[2], bool a0, bool a1) {
    char *p = reinterpret_cast<char *>(plane) + off;
    if (a0 && a1) {
        __builtin_nontemporal_store(licom_d2{x[0], x[1]}, reinterpret_cast<licom_d2 *>(p));
    } else if (a0 || a1) {
        *reinterpret_cast<double *>(p + (a0 ? 0 : 8)) = a0 ? x[0] : x[1];
    }
}

// Value of the lane before / after this one (DPP wave shift).
template <int CTRL>
__device__ __forceinline__ int dpp(int x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double dppd(double x) {
    const licom_v2i v = __builtin_bit_cast(licom_v2i, x);
    return __builtin_bit_cast(double, licom_v2i{dpp<CTRL>(v.x), dpp<CTRL>(v.y)});
}
constexpr int kFromPrev = 0x138, kFromNext = 0x130;   // wave_shr:1, wave_shl:1

// West and east neighbours of a lane's two cells.
__device__ __forceinline__ D2 west(const D2 &x) { return D2{{dppd<kFromPrev>(x.v[1]), x.v[0]}}; }
__device__ __forceinline__ D2 east(const D2 &x) { return D2{{x.v[1], dppd<kFromNext>(x.v[0])}}; }

// Runs level(position, k) for the levels [k0, k1): position 0 is the surface
// level, 2 the deepest and 1 any other, compiled apart so that the middle
// levels are one run of instructions without branches.
template <class F>
__device__ __forceinline__ void march_levels(int k0, int k1, int km, F &&level) {
    int k = k0;
    if (k == 0) level(std::integral_constant<int, 0>{}, k++);
    for (const int e = min(k1, km - 1); k < e; ++k) level(std::integral_constant<int, 1>{}, k);
    if (k < k1) level(std::integral_constant<int, 2>{}, k);
}

// First of the lane's cells, or of those some rows away, kept inside the
// plane.  What is read for a cell in columns 1..imt-2 is never clamped; a lane
// that owns the last cell of row jmt-2 (k_flags with an odd cell count) has the
// row below clamped, and the flag it stores there is one that nothing reads.
__device__ __forceinline__ int clamp_cell(int p, int n2) { return min(max(p, 0), n2 - 2); }

// Keeps the compiler from forming plane + offset once per array outside the
// level loop: 20 64-bit lane addresses, which spill, in place of scalar plane
// addresses and one shared offset.
__device__ __forceinline__ void fresh(uint32_t &off) { asm("" : "+v"(off)); }

// Face products of the tspas terms: htw*hun at the west faces of the two
// cells and of the one after them, hts*hue at their south and north faces.
struct Faces {
    double dx[3], ds[2], dn[2], tr[2];
};
__device__ __forceinline__ Faces load_faces(const KGrid &g, int pc, int pn) {
    Faces f;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        f.tr[e] = g.tarea_r[pc + e];
        f.dx[e] = g.htw[pc + e] * g.hun[pc + e];
        f.ds[e] = g.hts[pc + e] * g.hue[pc + e];
        f.dn[e] = g.hts[pn + e] * g.hue[pn + e];
    }
    f.dx[2] = dppd<kFromNext>(f.dx[0]);
    return f;
}

// For each of a lane's two cells, a byte each (n, s, e, w from the low end),
// the number of levels at which it and that neighbour are both wet.
__device__ __forceinline__ void load_wet(const KGrid &g, int pc, int pn, int ps, uint32_t (&wet)[2]) {
    const int a = g.kmt[pc], b = g.kmt[pc + 1];
    const int w = dpp<kFromPrev>(b), z = dpp<kFromNext>(a);
    const int kz[2] = {a, b}, kw[2] = {w, a}, ke[2] = {b, z};
#pragma unroll
    for (int e = 0; e < 2; ++e)
        wet[e] = (uint32_t)min(kz[e], g.kmt[pn + e]) | (uint32_t)min(kz[e], g.kmt[ps + e]) << 8 |
                 (uint32_t)min(kz[e], ke[e]) << 16 | (uint32_t)min(kz[e], kw[e]) << 24;
}

}  // namespace
}  // namespace licom
