// Index arithmetic of the PUMAS table search (pumas_table.hip), compiled by
// hipcc for the kernels and by a host compiler for its test.
#pragma once

#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define NOA_SEARCH_HD __host__ __device__ __forceinline__
#else
#define NOA_SEARCH_HD inline
#endif

namespace noa_hip {
namespace pumas {

// The cell of the nodes t[0..n-1] that holds x (t[0] <= x < t[n - 1]), or 0 for
// NaN: four parts a step, so that three loads are in flight. A lane whose
// point the table does not serve (`in` false) gets 0 as well, whatever the
// nodes: where they are all zero, as the first element's search sees them, any
// x that is not below them would run past the last cell.
NOA_SEARCH_HD int cell(const float* t, int n, float x, bool in) {
    if (!in) x = -INFINITY;
    const int last = n - 1;
    int i = 0;
    for (int d = last; d > 1;) {
        d = (d + 3) / 4;
        const int ia = i + d < last ? i + d : last;
        const int ib = i + 2 * d < last ? i + 2 * d : last;
        const int ic = i + 3 * d < last ? i + 3 * d : last;
        const float a = t[ia], b = t[ib], c = t[ic];
        i += d * (int(x >= a) + int(x >= b) + int(x >= c));
    }
    return i;
}

// The nodes of the first `levels` levels of a decision tree of 31 nodes, which
// are numbered by level, as a mask. (The lane beside a tree's 31 asks for one
// level more than there are.)
NOA_SEARCH_HD constexpr uint32_t tree_levels(int levels) {
    return (uint32_t(1) << ((1 << (levels < 5 ? levels : 5)) - 1)) - 1;
}

}  // namespace pumas
}  // namespace noa_hip
