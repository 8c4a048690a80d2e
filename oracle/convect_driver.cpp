// convect_driver.cpp -- csrc/tracer_convect.h on the host, under
// AddressSanitizer and UndefinedBehaviorSanitizer, against orc_convadj (test
// infrastructure only: tests/test_convect_host.py builds it with `make -C
// oracle convect`).  The two lanes of a column run as two threads; every array
// the routine is given has exactly the extent that it may touch, so an index
// outside a column, a table or the wet levels stops the run, as does a swap
// that only one lane makes.  Columns of 2 to 64 levels, with any number of
// unstable interfaces.
#include <hip/hip_runtime.h>

#include <cstring>
#include <random>

#include "licom_synth.h"
#include "oracle.h"
#include "tracer_convect.h"

namespace {

struct Levels {   // per-level tables of a grid of km levels, no slack behind them
    std::vector<double> to, so, eosc, dzp;
};

Levels levels(int km) {
    licom_synth_cfg cfg;
    licom_synth_defaults(&cfg);
    cfg.nx = 8;
    cfg.ny = 4;
    cfg.km = km;
    cfg.lat_mode = 0;
    cfg.dlon = cfg.dlat = 0.5;
    cfg.lat_north = 54.0;
    const size_t n2 = 12 * 8;
    std::vector<double> a[11], zkp(km + 1), pen(km - 1), lat(8);
    for (auto &v : a) v.assign(n2, 0.0);
    std::vector<int32_t> kmt(n2);
    Levels L;
    L.to.resize(km);
    L.so.resize(km);
    L.eosc.resize((size_t)9 * km);
    licom_synth_grid g{kmt.data(), zkp.data(), pen.data(), a[0].data(), a[1].data(), a[2].data(), a[3].data(),
                       a[4].data(), a[5].data(), a[6].data(), a[7].data(), a[8].data(), a[9].data(), a[10].data(),
                       L.to.data(), L.so.data(), L.eosc.data(), lat.data(), 0};
    if (licom_synth_make_grid(&cfg, &g) != 0) std::exit(3);
    for (int k = 0; k < km; ++k) L.dzp.push_back(zkp[k] - zkp[k + 1]);
    return L;
}

}  // namespace

int main() {
    std::mt19937_64 rng(5);
    auto uniform = [&](double lo, double hi) { return std::uniform_real_distribution<double>(lo, hi)(rng); };
    long columns = 0, top = 0, bottom = 0, regions = 0;
    for (int km : {2, 3, 4, 7, 30, 55, 63, 64}) {
        const Levels L = levels(km);
        const double *C = L.eosc.data();
        for (int rep = 0; rep < 400; ++rep) {
            const int kcon = rep < 3 * km ? 2 + rep % (km - 1) : 2 + (int)(rng() % (unsigned)(km - 1));
            // a stable profile, reversed over random stretches or shaken throughout
            std::vector<double> x[2];
            const double shake = rep % 4 == 0 ? uniform(0.0, 6.0) : 0.0;
            for (int k = 0; k < kcon; ++k) {
                x[0].push_back(2.0 + 20.0 * std::exp(-4.0 * k / km) + uniform(-shake, shake));
                x[1].push_back(1.0e-3 * (-0.3 + 0.6 * k / km + uniform(-0.02, 0.02)));
            }
            for (int s = (int)(rng() % 4); s > 0; --s) {
                const int a = (int)(rng() % (unsigned)kcon), b = (int)(rng() % (unsigned)kcon);
                std::reverse(x[0].begin() + std::min(a, b), x[0].begin() + std::max(a, b) + 1);
            }
            if (rep % 5 == 0) x[0].front() -= 15.0;
            if (rep % 5 == 1) x[0].back() += 15.0;
            uint64_t mask = 0;   // as the solve finds it
            for (int k = 1; k < kcon; ++k) {
                const double up = licom::dev::dens(C, km, k, x[0][k] - L.to[k], x[1][k] - L.so[k]);
                const double lo = licom::dev::dens(C, km, k, x[0][k - 1] - L.to[k], x[1][k - 1] - L.so[k]);
                if (lo > up) mask |= 1ull << k;
            }
            if (mask == 0) continue;

            const size_t stride = 1 + rng() % 3;
            std::vector<double> col[2];
            for (int n = 0; n < 2; ++n) {
                col[n].assign((kcon - 1) * stride + 1, -7.0);
                for (int k = 0; k < kcon; ++k) col[n][k * stride] = x[n][k];
            }
            LanePair pair;
            int lo[2], hi[2];
            auto lane = [&](int n) {
                lane_pair = &pair;
                lane_id = n;
                licom::convect_sparse(C, L.to.data(), L.so.data(), L.dzp.data(), km, kcon, mask, n, col[n].data(),
                                      stride, lo[n], hi[n]);
                pair.done[n].store(true);
            };
            std::thread other(lane, 1);
            lane(0);
            other.join();

            // the oracle, on a grid of this one column
            orc_grid g;
            std::memset(&g, 0, sizeof g);
            g.imt = g.jmt = 1;
            g.km = km;
            int32_t kmt = kcon;
            std::vector<double> at(2 * km, 0.0), atb(2 * (km + 1), 0.0), vit(km, 1.0), to = L.to, so = L.so, e = L.eosc,
                dzp = L.dzp;
            for (int n = 0; n < 2; ++n) std::copy(x[n].begin(), x[n].end(), at.begin() + n * km);
            g.kmt = &kmt;
            g.to = to.data();
            g.so = so.data();
            g.eosc = e.data();
            g.dzp = dzp.data();
            g.vit = vit.data();
            orc_params p;
            std::memset(&p, 0, sizeof p);
            p.dts = 1.0;
            orc_fields f;
            std::memset(&f, 0, sizeof f);
            f.at = at.data();
            f.atb = atb.data();
            orc_diag d;
            std::memset(&d, 0, sizeof d);
            orc_convadj(&g, &p, &f, &d);

            bool ok = lo[0] == lo[1] && hi[0] == hi[1] && lo[0] >= 0 && lo[0] < hi[0] && hi[0] < kcon;
            for (int n = 0; n < 2 && ok; ++n)
                for (size_t r = 0; r < col[n].size(); ++r) {
                    const int k = (int)(r / stride);
                    if (r % stride != 0) {
                        ok = ok && col[n][r] == -7.0;
                    } else {
                        ok = ok && std::memcmp(&col[n][r], &at[n * km + k], 8) == 0;
                        ok = ok && ((k >= lo[0] && k <= hi[0]) || col[n][r] == x[n][k]);
                    }
                }
            if (!ok) {
                std::printf("differs: km %d kcon %d mask %llx lo %d hi %d\n", km, kcon, (unsigned long long)mask, lo[0],
                            hi[0]);
                return 1;
            }
            ++columns;
            top += lo[0] == 0;
            bottom += hi[0] == kcon - 1;
            for (int k = lo[0]; k < hi[0]; ++k)
                if (col[0][k * stride] == x[0][k] && col[1][k * stride] == x[1][k]) {
                    ++regions;   // a level between two mixed regions
                    break;
                }
        }
    }
    std::printf("ok %ld columns, %ld mixed from the surface, %ld to the bottom, %ld in several regions\n", columns, top,
                bottom, regions);
    return columns > 1000 && top > 100 && bottom > 100 && regions > 100 ? 0 : 2;
}
