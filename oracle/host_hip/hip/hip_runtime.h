// hip_runtime.h -- the few HIP names that csrc/tracer_device.h and
// csrc/tracer_convect.h use, for a host compiler (test infrastructure only;
// found before ROCm's header by oracle/Makefile's `convect` target).  A lane
// is a thread: __shfl_xor swaps a value with the other lane of its pair.
#pragma once
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

struct LanePair {
    double slot[2][2] = {};            // [parity of the swap][lane]
    std::atomic<long> swaps[2] = {};   // swaps begun by each lane
    std::atomic<bool> done[2] = {};
};
inline thread_local LanePair *lane_pair = nullptr;
inline thread_local int lane_id = 0;

inline double __shfl_xor(double v, int) {
    LanePair &p = *lane_pair;
    const long mine = p.swaps[lane_id].load() + 1;
    p.slot[mine & 1][lane_id] = v;
    p.swaps[lane_id].store(mine);
    while (p.swaps[lane_id ^ 1].load() < mine) {
        if (p.done[lane_id ^ 1].load() && p.swaps[lane_id ^ 1].load() < mine) {
            std::fprintf(stderr, "a lane swaps with one that has left\n");
            std::abort();
        }
        std::this_thread::yield();
    }
    // the other lane cannot write this slot again before this lane begins its
    // swap after next
    return p.slot[mine & 1][lane_id ^ 1];
}
inline int __ffsll(unsigned long long x) { return __builtin_ffsll((long long)x); }
using std::max;
using std::min;

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __noinline__
