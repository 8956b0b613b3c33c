// resident_window.cpp -- block and LDS shapes of the on-chip solvers (host
// side, plain C++; the kernels that use them are in cg_resident.hip).
#include "resident_window.h"

#include <algorithm>

#include "slot_layout.h"

namespace tflows {

namespace {

constexpr int kLanes = 64;             // lanes of a wavefront: the posts it polls at once
constexpr int kXcds = 8;
// One block up to this many rows: its synchronisations are block barriers
// (CG, us an iteration, one block / several of 1024 rows: 1,331 rows 3.1 / 4.8,
// 2,744 3.9 / 5.2, 4,096 4.7 / 5.2).
constexpr int kResOneBlockRows = 4096;
// Else blocks of at least this many (2048: 5.0 -> 5.7 at 4,913 rows, 9.0 -> 9.9
// at 175,616; 512: 5.0 -> 5.1 and 9.0 -> 8.2), up to twice as many where that
// keeps to the 64 blocks that synchronise in one step (64 / more blocks: 85,184
// rows 7.4 / 8.6, 97,336 7.4 / 7.9, 125,000 7.6 / 9.1, locality order 7.5 / 8.7;
// at 216,000 rows in 64 blocks 9.0 -> 10.4).
constexpr int kResMinRows = 1024;

}  // namespace

ResidentShape resident_shape(int n, int rows_per_thread, int cus) {
    ResidentShape r;
    if (n <= 0 || cus <= 0) return r;
    int grid = 1;
    if (n > kResOneBlockRows) {
        grid = std::min(cus, (n + kResMinRows - 1) / kResMinRows);
        if (grid > kLanes && n <= kLanes * 2 * kResMinRows) grid = kLanes;
        if (grid >= kXcds) grid = grid / kXcds * kXcds;
    }
    const int64_t rows = (((int64_t)n + grid - 1) / grid + kSliceRows - 1) / kSliceRows * kSliceRows;
    if (rows > (int64_t)rows_per_thread * kResThreads) return r;
    r.grid = grid;
    r.rows = (int)rows;
    return r;
}

// values of LDS: own rows and halo (the reads of the threads past the
// block's rows stay inside), and D
template <typename T>
static size_t window_elems(const ResidentShape& sh, int lo, int hi, int nfar) {
    const int R = window_kernel_rows((sh.rows + kResThreads - 1) / kResThreads);
    return (size_t)lo + hi + (size_t)nfar * sh.rows + (size_t)R * kResThreads * (window_d_in_lds<T>(R) ? 2 : 1);
}

template <typename T>
bool window_shape(const ResidentShape& sh, const std::vector<int>& offsets, WindowShape& w) {
    w = WindowShape{};
    if ((int)offsets.size() > window_slots<T>()) return false;
    for (int d : offsets) {
        const int64_t ad = d < 0 ? -(int64_t)d : d;
        if (ad < sh.rows) w.lo = std::max(w.lo, halo_rows((int)ad));
        else if (w.nfar < kMaxFar) w.far[w.nfar++] = d;
        else return false;
    }
    w.farbase = 2 * w.lo + sh.rows;
    for (int d : offsets) {
        w.disp[w.nslots] = d;
        for (int f = 0; f < w.nfar; ++f)
            if (w.far[f] == d) w.disp[w.nslots] = w.farbase + f * sh.rows - w.lo;
        w.offset[w.nslots++] = d;
    }
    w.lds = sizeof(T) * window_elems<T>(sh, w.lo, w.lo, w.nfar);
    return w.lds <= kResLdsBytes;
}
template <typename T>
bool window_shape(const ResidentShape& sh, const std::vector<int>& deps, int n, WindowShape& w) {
    w = WindowShape{};
    size_t most = window_elems<T>(sh, 0, 0, 0);
    for (int b = 0; b < sh.grid && sh.grid > 1 && (int64_t)b * sh.rows < n; ++b)
        most = std::max(most, window_elems<T>(sh, halo_rows(b * sh.rows - deps[2 * b]),
                                              halo_rows(deps[2 * b + 1] + 1 - (b + 1) * sh.rows), 0));
    w.lds = sizeof(T) * most;
    return w.lds <= kResLdsBytes;
}
template bool window_shape<double>(const ResidentShape&, const std::vector<int>&, WindowShape&);
template bool window_shape<float>(const ResidentShape&, const std::vector<int>&, WindowShape&);
template bool window_shape<double>(const ResidentShape&, const std::vector<int>&, int, WindowShape&);
template bool window_shape<float>(const ResidentShape&, const std::vector<int>&, int, WindowShape&);

}  // namespace tflows
