// CPU check of shortest_normal_run (point_runs.hpp): prints the shortest run
// of five point sets, one per line.
#include <cmath>
#include <cstdio>
#include <vector>

#include "point_runs.hpp"

// three patches of 24 points, two triangles of 12 each; `bad` points get a
// NaN in their normal
static int run(int gs, std::vector<int> bad) {
    const int n = 3, m = 24;
    std::vector<int> ptr(n + 1);
    std::vector<double> pts(size_t(7) * n * m);
    for (int p = 0; p <= n; ++p) ptr[p] = p * m;
    for (int k = 0; k < n * m; ++k) pts[7 * k + 3] = k / gs;
    for (int k : bad) pts[7 * k + 4] = std::nan("");
    return beep::shortest_normal_run(n, ptr.data(), pts.data());
}

int main() {
    std::printf("%d %d %d %d %d\n", run(12, {}), run(24, {}), run(12, {0}), run(12, {17}),
                run(12, {48, 49, 50, 71}));
}
