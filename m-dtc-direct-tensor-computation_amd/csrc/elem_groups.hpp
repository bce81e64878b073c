// elem_groups.hpp -- the work list of the HEX20 element pass.
#pragma once

#include <cstdint>
#include <vector>

#include <hip/hip_runtime.h>

namespace dtc {

// Workgroups of k20_elem with em elements each: (domain group, first element, elements of the
// group, its first one in ye20): as many as the groups need.  (A grid of the largest group's
// workgroups times the groups had 142,911 for 3,442 with one 27^3 domain beside 200 of 6^3,
// 404 -> 305 ms in FP64, and bounded the groups by the grid's y limit.)
inline std::vector<int4> elem_groups(const std::vector<int64_t>& ebase, int em) {
    std::vector<int4> w;
    for (size_t g = 0; g + 1 < ebase.size(); ++g) {
        const int64_t ne = ebase[g + 1] - ebase[g];
        for (int64_t e = 0; e < ne; e += em) w.push_back(make_int4((int)g, (int)e, (int)ne, (int)ebase[g]));
    }
    return w;
}

}  // namespace dtc
