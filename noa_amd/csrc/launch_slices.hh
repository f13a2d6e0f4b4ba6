// Launches of any number of workgroups. HIP takes fewer than 2^32 work items
// along x (gridDim.x * blockDim.x), which 256-lane workgroups reach at 2^24 of
// them, long before the 2^31 - 1 that a grid dimension holds.
#pragma once

#include <algorithm>
#include <cstdint>

namespace noa_hip {

// Calls launch(first, count) for consecutive ranges of the `workgroups` of
// `lanes` work items each, every range within one launch; stops at the first
// non-zero return value and returns it.
template <class Launch>
int launch_slices(int64_t workgroups, int lanes, Launch&& launch) {
    const int64_t most = int64_t(0xffffffff) / lanes;
    for (int64_t first = 0; first < workgroups; first += most)
        if (int rc = launch(first, uint32_t(std::min(most, workgroups - first)))) return rc;
    return 0;
}

}  // namespace noa_hip
