// tracer_convect.h -- convadj of one column, as the column solve runs it.
// On its own, so that it also compiles for the host, where a test runs its two
// lanes as threads, with bounds checks.
#pragma once
#include <hip/hip_runtime.h>

#include "tracer_device.h"

namespace licom {
namespace {

// convadj_cu (convadj.cpp:52-256) for one column, driven by the mask of
// statically unstable interfaces found with the unmixed densities (bit k:
// rholo(k-1) > rhoup(k)).  Every density the reference reads after mixing
// starts is either recomputed by it or belongs to a level that mixing has not
// touched, so the mask plus on-demand recomputation reproduces its decisions.
// The two lanes of a column run this together: each holds its own tracer's
// column X (the state just written, stride n2), the T lane forms the mixed
// region's density and the S lane the tested level's, and they swap values
// with __shfl_xor over 32 lanes.  Every step is a link of a serial chain, so
// what it waits for is kept short: both ends of the region are tested in one
// step (the lower one decides first), their values are loaded a step ahead,
// and the coefficients (C, to, so, dzp) come from LDS (solve of 128 x 96 x 30
// 58 -> 50 us, 225 x 145 x 55 121 -> 103 us, 360 x 218 x 30 with icesnow, half
// of whose columns mix, 427 -> 377 us).  Returns the mixed level range in
// lo/hi.
__device__ __noinline__ void convect_sparse(const double *C, const double *to, const double *so,
                                            const double *dzp, int km, int kcon, uint64_t mask,
                                            int n, double *X, size_t n2, int &lo, int &hi) {
    lo = km;
    hi = -1;
    int lcon = __ffsll((unsigned long long)mask) - 1;
    auto at = [&](int k) { return X[(size_t)min(max(k, 0), kcon - 1) * n2]; };
    // the mixed region's density and v's, both at level k
    auto both = [&](int k, double mix, double v, double &rmix, double &rv) {
        const double got = __shfl_xor(n == 0 ? v : mix, 32);
        const double mine = dev::dens(C, km, k, (n == 0 ? mix : got) - to[k], (n == 0 ? got : v) - so[k]);
        const double other = __shfl_xor(mine, 32);
        rmix = n == 0 ? mine : other;
        rv = n == 0 ? other : mine;
    };
    for (;;) {   // CONV_1
        int lcona = lcon, lconb = lcon + 1;
        const double x0 = at(lcona - 1), x1 = at(lconb - 1);
        // the levels below and above the region, and those after them
        double vb = at(lconb), nb = at(lconb + 1), va = at(lcona - 2), na = at(lcona - 3);
        double dztsum = dzp[lcona - 1] + dzp[lconb - 1];
        double trasum = x0 * dzp[lcona - 1] + x1 * dzp[lconb - 1];
        double tramix = trasum / dztsum;
        for (;;) {   // CONV_2
            const bool can_b = lconb != kcon, can_a = lcona > 1;
            const int kb = can_b ? lconb : lconb - 1;
            double rmix, rv;
            both(kb, tramix, vb, rmix, rv);
            const bool down = can_b && rmix > rv;
            both(lcona - 1, tramix, va, rmix, rv);
            const bool up = can_a && rv > rmix;
            if (down) {
                dztsum = dztsum + dzp[lconb];
                trasum = trasum + vb * dzp[lconb];
                lconb = lconb + 1;
                vb = nb;
                nb = at(lconb + 1);
            } else if (up) {
                dztsum = dztsum + dzp[lcona - 2];
                trasum = trasum + va * dzp[lcona - 2];
                lcona = lcona - 1;
                va = na;
                na = at(lcona - 3);
            } else {
                break;
            }
            tramix = trasum / dztsum;
        }
        for (int l = lcona - 1; l < lconb; ++l) X[(size_t)l * n2] = tramix;
        lo = min(lo, lcona - 1);
        hi = max(hi, lconb - 1);
        if (lconb == kcon) return;
        // CONV_3: next unstable interface below the mixed region
        const uint64_t below = lconb >= 63 ? 0ull : (mask & ~((2ull << lconb) - 1ull));
        if (below == 0) return;
        lcon = __ffsll((unsigned long long)below) - 1;
    }
}

}  // namespace
}  // namespace licom
