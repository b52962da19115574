// Host-side partition of the batch's work lists (plain C++ on HIP's vector
// types, so that it can be checked on the CPU).
//
// A list holds (solve, tile) items in solve order, each with an estimated
// cost.  It is split into 8 contiguous chunks of about equal cost, one per
// XCD; workgroup b of an XCD's G8 workgroups takes positions b, b + G8,
// b + 2 G8, ... of its chunk, so the workgroups of an XCD sweep a solve's
// neighbouring tiles together and share their halos in that XCD's L2.
#pragma once
#include <algorithm>
#include <cstdint>
#include <numeric>
#include <vector>

#include <hip/hip_runtime.h>

namespace dgmi {

// cut[0..parts]: `parts` contiguous ranges of [0, n) of about equal cost
inline void cost_cuts(const double* cost, int n, int parts, int* cut) {
    cut[0] = 0;
    for (int k = 1; k <= parts; k++) cut[k] = n;
    const double total = std::accumulate(cost, cost + n, 0.0);
    double run = 0;
    int x = 1;
    for (int i = 0; i < n && x < parts; i++) {
        run += cost[i];
        while (x < parts && run >= total * x / parts) cut[x++] = i + 1;
    }
}

// A list appended to out in its 8 XCD chunks; bounds[0..8] = the chunks'
// start positions in out and the end of the last.
inline void xcd_chunks(const std::vector<int2>& items, const std::vector<double>& cost, std::vector<int2>& out,
                       int* bounds) {
    int cut[9];
    cost_cuts(cost.data(), (int)items.size(), 8, cut);
    const int base = (int)out.size();
    for (int k = 0; k <= 8; k++) bounds[k] = base + cut[k];
    out.insert(out.end(), items.begin(), items.end());
}

// Whether a batch whose launch form is not set runs FP64 stages per kernel
// class, by the lane and tile classes present and the triangles in them.  A
// launch of its own class holds more wavefronts, and each further launch of a
// stage costs about 8 us a step.  One launch / per class, us per step: one
// class is always faster (advection lanes 2,682 triangles 46 / 41, Euler tiles
// 273,568 577 / 433); two with tiles among them cross between 27,000 and
// 200,000 (advection and Euler tiles 27,370 79 / 83, 144,688 250 / 207; Euler
// lanes and tiles 55,930 141 / 144, 273,568 392 / 364); both lane classes or all
// four near 400,000 to 520,000 (273,568 217 / 220 and 311 / 356, 510,380
// 365 / 304 and 524 / 522, 909,414 625 / 489 and 947 / 813).
inline int64_t per_class_line(int lane_classes, int tile_classes) {
    const int n = lane_classes + tile_classes;
    if (n <= 1) return 0;
    return n == 2 && tile_classes > 0 ? 65536 : 524288;
}
// `running`: solves of an earlier list run in form `now`, which is kept within
// an eighth of the line (a server's solves come and go around it, and each
// change of form captures the step again)
inline bool take_per_class(int lane_classes, int tile_classes, int64_t elems, bool running, bool now) {
    const int64_t line = per_class_line(lane_classes, tile_classes);
    return elems >= (!running ? line : now ? line - line / 8 : line + line / 8);
}

}  // namespace dgmi
