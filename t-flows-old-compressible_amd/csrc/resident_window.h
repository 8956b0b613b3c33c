// resident_window.h -- how the on-chip solvers (cg_resident.hip) split a
// system into blocks and which rows of other blocks each keeps in LDS (plain
// C++: the kernels and their host check share it; constexpr functions are
// device functions, too).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace tflows {

constexpr int kResThreads = 512;      // threads of a block
constexpr size_t kResLdsBytes = 160 * 1024 - 16 * 1024;   // LDS of a CU less the kernel's own arrays
constexpr int kResMaxBlocks = 512;    // eight eighths of a wavefront's lanes

// Blocks and rows of a block for n rows on a chip of `cus` blocks, at most
// rows_per_thread x kResThreads rows in a block; grid 0 when the chip does
// not hold them.
struct ResidentShape {
    int grid = 0, rows = 0;
};
ResidentShape resident_shape(int n, int rows_per_thread, int cus);

// rows of a thread that the registers hold: FP64 8 (14 of 256 registers per
// row's values) and FP32 16 of a shared-offset matrix, half where every entry
// also has its column (the locality order)
template <typename T>
constexpr int resident_rows_per_thread(bool reordered) {
    return (sizeof(T) == 8 ? 8 : 16) / (reordered ? 2 : 1);
}
// the rows per thread of the kernel that runs R of them
constexpr int window_kernel_rows(int R) { return R <= 1 ? R : R <= 8 ? (R + 1) / 2 * 2 : (R + 3) / 4 * 4; }
// D in LDS, too, where a thread's rows would take too many registers
template <typename T>
constexpr bool window_d_in_lds(int kernel_rows) {
    return kernel_rows * sizeof(T) >= 48;
}
// entries of a row k_cg_window keeps: those of a 7-point row, without the
// diagonal in the FP32 difference form
template <typename T>
constexpr int window_slots() {
    return sizeof(T) == 8 ? 7 : 6;
}
// rows of a halo of `need` rows: whole granules of 16 bytes
constexpr int halo_rows(int need) { return need <= 0 ? 0 : (need + 3) / 4 * 4; }

// LDS of k_cg_window.  The halo of a block of a shared-offset matrix: column
// offsets shorter than a block lie within `lo` rows of the block; each longer
// one (far) has a region of its own, as many rows as the block.
constexpr int kMaxFar = 4;
constexpr int kMaxWindowSlots = 7;
struct WindowShape {
    int lo = 0, nfar = 0, nslots = 0;
    int farbase = 0;                          // LDS index of the first far region
    int far[kMaxFar] = {};
    int offset[kMaxWindowSlots] = {};         // the matrix's column offsets, ascending
    int disp[kMaxWindowSlots] = {};           // LDS distance of each from the row's own p
    size_t lds = 0;                           // bytes
};
// The shapes of a shared-offset matrix (its distinct column offsets) and of
// any other (deps read back); false when the LDS does not hold them.
template <typename T>
bool window_shape(const ResidentShape& sh, const std::vector<int>& offsets, WindowShape& w);
template <typename T>
bool window_shape(const ResidentShape& sh, const std::vector<int>& deps, int n, WindowShape& w);

// Rows [first, last] of the matrix, empty where last < first.
struct RowRange {
    int first, last;
};
constexpr RowRange add_rows(RowRange r, int from, int to, int n) {   // r and [from, to) within the matrix
    from = from < 0 ? 0 : from;
    to = to > n ? n : to;
    if (from >= to) return r;
    if (r.last < r.first) return RowRange{from, to - 1};
    return RowRange{from < r.first ? from : r.first, to - 1 > r.last ? to - 1 : r.last};
}
// Every row that the halo of the block of rows rb .. rb + rows - 1 reads: its
// columns (`deps`) and, for shared offsets, all rows of the near and far
// runs.  A run is loaded whole, so it goes beyond the columns where rows lack
// entries (the last plane of a zone numbered before another), and its values
// are multiplied by 0 there: a form that waits for some blocks only has to
// wait for these rows' blocks.
constexpr RowRange halo_reach(const WindowShape& w, bool shared, RowRange deps, int rb, int rows, int n) {
    if (!shared) return deps;
    RowRange r = add_rows(deps, rb - w.lo, rb, n);
    r = add_rows(r, rb + rows, rb + rows + w.lo, n);
    for (int q = 0; q < w.nfar; ++q) r = add_rows(r, rb + w.far[q], rb + w.far[q] + rows, n);
    return r;
}

}  // namespace tflows
