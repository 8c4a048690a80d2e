// turb_shape.h -- workgroup size of the Canuto producer (turb.hip).
#pragma once
#include <cstddef>

namespace licom {

// Lanes of a workgroup for a block of `columns` columns: one wave on small
// blocks, so that the CUs' shares differ by a wave and not by four; four waves
// on large ones (a CU's eight waves then work on two places of every plane and
// not on eight; handing neighbouring one-wave workgroups to one XCD instead
// made no difference).  Which is faster in between depends on the bathymetry.
// One wave / four waves, ms; "even": nearly all columns 46 of 55 (22 of 30)
// levels deep, "rough": depths spread over all levels, so that a workgroup
// waits for its deepest wave:
//                   even            rough
//  128 x  96 x 30   0.242 / 0.272   0.307 / 0.358
//  360 x 218 x 30   0.335 / 0.354   0.475 / 0.515
//  360 x 231 x 55   0.732 / 0.774   1.02  / 1.10
//  600 x 400 x 55   1.575 / 1.567   2.26  / 2.30
// 1200 x 700 x 55   5.13  / 4.98    6.90  / 7.26
// 1400 x 900 x 55   7.68  / 7.45   10.06  / 10.63
// 1800 x 1151 x 55  12.78 / 12.08  16.6   / 17.2
// 3600 x 2302 x 55  52.0  / 47.3   65.1   / 65.3
// The line lies where one wave's loss on even depths passes its gain on rough
// ones.
constexpr int turb_lanes(size_t columns) { return columns < (size_t(3) << 19) ? 64 : 256; }

}  // namespace licom
