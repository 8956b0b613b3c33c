// Host check of the on-chip solvers' block and halo shapes
// (t-flows-old-compressible_amd/csrc/resident_window.cpp).
//
// For generated patterns of shared column offsets -- single boxes, several
// boxes numbered one after another, planes and lines -- it takes the shapes
// from the library's own functions and repeats, row by row, what the kernels
// of cg_resident.hip keep in LDS and read from it, and checks:
//   * every LDS index read (threads past a block's rows included) lies inside
//     the block's allocation;
//   * the index a slot reads holds the column of that slot;
//   * every row that the halo's loads touch belongs to a block that
//     halo_reach names, so that CGS, which waits for those only, reads no row
//     that has not been published in this product.
//
// Prints "case <name> grid=<n> rows=<n> beyond=<blocks whose halo reads blocks
// their columns do not reach> ok" or "FAIL ..."; "ALL OK" at the end; exits
// non-zero on a failure.
#include <algorithm>
#include <cstdio>
#include <string>
#include <vector>

#include "resident_window.h"

using namespace tflows;

namespace {

struct Box {
    int nx, ny, nz;
};
struct Pattern {
    int n = 0;
    std::vector<std::vector<int>> cols;
    std::vector<int> offsets;
};

// 7-point boxes in natural order, numbered one after another
Pattern stacked(const std::vector<Box>& boxes, bool diag) {
    Pattern p;
    for (const Box& b : boxes) {
        const int r0 = p.n, nxy = b.nx * b.ny;
        for (int i = 0; i < nxy * b.nz; ++i) {
            const int x = i % b.nx, y = i / b.nx % b.ny, z = i / nxy, c = r0 + i;
            std::vector<int> r;
            if (z > 0) r.push_back(c - nxy);
            if (y > 0) r.push_back(c - b.nx);
            if (x > 0) r.push_back(c - 1);
            if (diag) r.push_back(c);
            if (x + 1 < b.nx) r.push_back(c + 1);
            if (y + 1 < b.ny) r.push_back(c + b.nx);
            if (z + 1 < b.nz) r.push_back(c + nxy);
            for (int v : r) p.offsets.push_back(v - c);
            p.cols.push_back(r);
        }
        p.n += nxy * b.nz;
    }
    std::sort(p.offsets.begin(), p.offsets.end());
    p.offsets.erase(std::unique(p.offsets.begin(), p.offsets.end()), p.offsets.end());
    return p;
}

int g_fail = 0;
void fail(const std::string& name, const char* what, int a, int b) {
    if (g_fail++ < 20) std::printf("FAIL %s: %s (%d, %d)\n", name.c_str(), what, a, b);
}

template <typename T>
void check(const std::string& name, const Pattern& p, int rows_per_thread, int cus) {
    const ResidentShape sh = resident_shape(p.n, rows_per_thread, cus);
    WindowShape w;
    if (!sh.grid || !window_shape<T>(sh, p.offsets, w)) {
        std::printf("case %s not held\n", name.c_str());
        return;
    }
    const int rows = sh.rows, R = window_kernel_rows((rows + kResThreads - 1) / kResThreads);
    if (sh.grid > cus || sh.grid > kResMaxBlocks || (int64_t)sh.grid * rows < p.n) fail(name, "grid", sh.grid, rows);
    const int d_elems = window_d_in_lds<T>(R) ? R * kResThreads : 0, elems = (int)(w.lds / sizeof(T)) - d_elems;
    if (w.lds > kResLdsBytes) fail(name, "lds", (int)w.lds, 0);
    int beyond = 0;
    for (int blk = 0; blk < sh.grid; ++blk) {
        const int rb = std::min(blk * rows, p.n), nloc = std::min(p.n - rb, rows);
        std::vector<int> held(elems, -1);           // the row at each LDS index
        std::vector<int> loaded;                    // rows of other blocks
        for (int l = 0; l < nloc; ++l) held[w.lo + l] = rb + l;
        auto run = [&](int at, int row, int count) {
            for (int e = 0; e < count; ++e) {
                if (at + e < 0 || at + e >= elems) {
                    fail(name, "halo outside the LDS", blk, at + e);
                    continue;
                }
                if (row + e < 0 || row + e >= p.n) continue;
                held[at + e] = row + e;
                loaded.push_back(row + e);
            }
        };
        run(0, rb - w.lo, w.lo);
        run(w.lo + rows, rb + rows, w.lo);
        for (int q = 0; q < w.nfar; ++q) run(w.farbase + q * rows, rb + w.far[q], rows);
        for (int t = 0; t < R * kResThreads; ++t)
            for (int j = 0; j < w.nslots; ++j)
                if (w.lo + t + w.disp[j] < 0 || w.lo + t + w.disp[j] >= elems) fail(name, "read outside the LDS", blk, t);
        int lo = p.n, hi = 0;
        for (int l = 0; l < nloc; ++l)
            for (int c : p.cols[rb + l]) {
                lo = std::min(lo, c);
                hi = std::max(hi, c);
                const int j = (int)(std::find(w.offset, w.offset + w.nslots, c - rb - l) - w.offset);
                if (j == w.nslots || held[w.lo + l + w.disp[j]] != c) fail(name, "slot reads another row", rb + l, c);
            }
        if (nloc <= 0) lo = hi = std::min(blk * rows, p.n - 1);
        const RowRange reach = halo_reach(w, true, RowRange{lo, hi}, rb, rows, p.n);
        bool more = false;
        for (int c : loaded) {
            const int b = c / rows;
            if (b < reach.first / rows || b > reach.last / rows) fail(name, "halo row of a block not waited for", blk, b);
            more = more || b < lo / rows || b > hi / rows;
        }
        if (reach.first > lo || reach.last < hi || reach.first < 0 || reach.last >= p.n) fail(name, "reach", blk, 0);
        beyond += more;
    }
    std::printf("case %s grid=%d rows=%d beyond=%d ok\n", name.c_str(), sh.grid, rows, beyond);
}

}  // namespace

int main() {
    const std::vector<std::pair<std::string, std::vector<Box>>> cases = {
        {"box_40x40x41", {{40, 40, 41}}},
        {"box_67x53x59", {{67, 53, 59}}},
        {"box_101x99x98", {{101, 99, 98}}},
        {"line_9000", {{9000, 1, 1}}},
        {"plane_300x170", {{300, 170, 1}}},
        {"thin_2000x3x9", {{2000, 3, 9}}},
        {"tall_5x4x3001", {{5, 4, 3001}}},
        {"eight_16", std::vector<Box>(8, Box{16, 16, 16})},
        {"two_40x40x41", std::vector<Box>(2, Box{40, 40, 41})},
        {"three_70x60x25", std::vector<Box>(3, Box{70, 60, 25})},
        {"five_33x31x7", std::vector<Box>(5, Box{33, 31, 7})},
        {"uneven_lines", {{64, 40, 3}, {64, 40, 1}, {64, 40, 9}}},
    };
    for (const auto& c : cases) {
        check<double>(c.first + "_cg", stacked(c.second, true), resident_rows_per_thread<double>(false), 256);
        check<double>(c.first + "_cgs", stacked(c.second, true), 4, 256);
        check<float>(c.first + "_f32", stacked(c.second, false), resident_rows_per_thread<float>(false), 256);
        check<double>(c.first + "_cgs_80cus", stacked(c.second, true), 4, 80);
    }
    if (g_fail) return 1;
    std::printf("ALL OK\n");
    return 0;
}
