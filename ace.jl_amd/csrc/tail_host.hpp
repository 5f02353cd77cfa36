// Host-side (CPU): tail tiles of a product-DAG launch.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace acehost {

// Tail tiles for the automatic parts choice.  The grid runs in rounds of ncu
// workgroups of equal length d.  Giving the last n tiles P + 1 parts fills the
// partial last round with shorter workgroups of length dh (segment kernel:
// 1/(P + 1) of the tile's work plus 8 % for re-staging and thinner task lists,
// measured 0.200 ms per workgroup with 4 parts against 0.246 ms with 3 at 100k
// environments).  The makespan of a greedy dispatch of such workgroups onto
// ncu units is flat over a range of n; take the middle of that range.  Units
// of equal load take their workgroups together, so a makespan is a few steps
// (a heap of the units, one workgroup after another, took 1 to 2.5 ms at the
// first call of each tile count; 20,011 order-4 environments take 0.47 ms).
inline int64_t choose_tail(int64_t ntile, int P, int ncu, double d, double dh) {
    auto makespan = [&](int64_t nhi) {
        // the P-part workgroups: full rounds, then r units busy one more
        const int64_t w = (ntile - nhi) * P, f = w / ncu, r = w % ncu;
        const double t0 = (double)f * d, t1 = (double)(f + 1) * d;
        double end = r > 0 ? t1 : t0;
        // the others, to whichever of the two groups of units is free first
        int64_t n0 = 0, n1 = 0;
        for (int64_t left = nhi * (P + 1); left > 0;) {
            const double s0 = t0 + (double)n0 * dh, s1 = t1 + (double)n1 * dh;
            const bool first = r == 0 || s0 <= s1;
            left -= first ? ncu - r : r;
            ++(first ? n0 : n1);
            end = std::max(end, (first ? s0 : s1) + dh);
        }
        return end;
    };
    const int64_t nmax = std::min<int64_t>(ntile, ncu);
    std::vector<double> ms((size_t)nmax + 1);
    double best = 1e300;
    for (int64_t n = 0; n <= nmax; ++n) {
        ms[(size_t)n] = makespan(n);
        best = std::min(best, ms[(size_t)n]);
    }
    std::vector<int64_t> ties;
    for (int64_t n = 0; n <= nmax; ++n)
        if (ms[(size_t)n] <= best * (1.0 + 1e-9)) ties.push_back(n);
    return ties[ties.size() / 2];
}

}  // namespace acehost
