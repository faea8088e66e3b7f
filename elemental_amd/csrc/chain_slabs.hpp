// How many 16-column slabs of right-hand sides one launch of the triangular
// solves takes (solve_chain.hip).
#pragma once

#include <algorithm>

namespace elemamd {

// helpers: helper workgroups a slab; cus: compute units of the device.
//
// Speed: as many as leave every workgroup a CU of its own, at least 8.  More
// than that and the helpers of one slab keep the chains of others waiting: n =
// 8192, 256 columns 1.28 ms in two launches, 2.2 to 7.8 in one.  Fewer, and
// small factors pay for launches: n = 512, 400 columns 155 us with 8, 60 with
// all 25.
//
// Progress: a chain holds a CU while it waits for helpers, which are dispatched
// behind all chains of the launch.  So launches that run at the same time must
// leave CUs to the helpers: with four hardware queues a process (HIP's
// default) an eighth of the CUs each fills half the device at most.  (n = 512,
// 1024 columns: 98 us with all 64 slabs in a launch, 102 with 32.)  Without
// helpers nothing waits for another workgroup.
inline int chain_slabs(int helpers, int cus) {
    if (helpers <= 0) return std::max(1, cus);
    return std::min(std::max(8, cus / (1 + helpers)), std::max(1, cus / 8));
}

}  // namespace elemamd
