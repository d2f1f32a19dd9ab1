// Runs of points with equal normals in a patch point set.
#pragma once

#include <algorithm>
#include <cstddef>

namespace beep {

// The shortest run of consecutive points with the same normal (x, y, z, nx,
// ny, nz, w per point) within a patch, over the first patches of a set of n:
// the points of a planar triangle share theirs.  A normal with a NaN (a
// triangle without area) equals none, its own included, so its point is a run
// of one.
inline int shortest_normal_run(int n, const int* ptr, const double* pts) {
    int run = 0x7fffffff;
    for (int p = 0; p < std::min(n, 64); ++p)
        for (int a = ptr[p], k; a < ptr[p + 1]; a = k) {
            const double* first = pts + 7 * size_t(a) + 3;
            for (k = a + 1; k < ptr[p + 1] && std::equal(first, first + 3, pts + 7 * size_t(k) + 3); ++k) {}
            run = std::min(run, k - a);
        }
    return run;
}

}  // namespace beep
