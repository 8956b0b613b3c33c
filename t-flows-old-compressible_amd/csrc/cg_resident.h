// cg_resident.h -- the on-chip CG (cg_resident.hip): its arguments, sizes and
// launchers.
#pragma once
#include <vector>

#include "krylov_kernels.h"

namespace tflows {

constexpr int kResThreads = 512;      // threads of a block
constexpr size_t kResLdsBytes = 160 * 1024 - 16 * 1024;   // LDS of a CU less the kernel's own arrays
constexpr int kResChunk = 1024;       // iterations of a launch: bounds how long it holds the CUs
constexpr int kResMaxBlocks = 512;    // eight eighths of a wavefront's lanes
constexpr int kPostWords = 4;         // 64-bit words a block posts at a site (two FP64 values)
constexpr int kPostStride = kResMaxBlocks;            // words between two words of a block
constexpr int kPostSite = kPostWords * kPostStride;   // words of a copy of a site's posts
constexpr int kPostCopies = 8;                        // one per XCD
constexpr int kPostSecond = 128;                      // words of a copy of the eighths' sums
constexpr int kPostTotal = 2 * kPostCopies * (kPostSite + kPostSecond);

// the mixed-precision forms pause the FP32 recurrence for a residual
// replacement once it has dropped this far below the last FP64 norm
constexpr double kReplaceDrop = 1e-2;

// Blocks and rows of a block for n rows on the current device, at most
// rows_per_thread x kResThreads rows in a block; grid 0 when the chip does
// not hold them.
struct ResidentShape {
    int grid = 0, rows = 0;
};
ResidentShape resident_shape(int n, int rows_per_thread);
// the most blocks of a launch: one per CU
int resident_blocks();

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
__host__ __device__ constexpr int halo_rows(int need) { return need <= 0 ? 0 : (need + 3) / 4 * 4; }

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

template <typename T>
struct ResidentArgs {
    int n;
    int rows;              // rows of a block, a multiple of the slice height
    int chunk;             // iterations of this launch
    uint32_t tag;          // number of the last synchronisation before this launch
    T* x;
    T* r;
    T* p;                  // carries p from launch to launch (k_cg_stream: published here)
    T* z;                  // k_cg_window: published z
    const T* D;
    T* keep;               // when not null: x and r of the launch's start (2 n)
    uint64_t* slotB;       // kPostTotal / 2 words a site
    uint64_t* slotC;
    uint32_t* flags;       // one per block
    const int* deps;       // smallest and largest column of each block's rows
    const double* partE;   // mixed precision: (r, r) of the last replacement, nE partial sums
    int nE;
    HostMirror* hm;
    uint64_t wait_ticks;
    SolverState* st;       // its `fault` word ends every wait of the launch
};
// CSR rows of one system of a block-diagonal matrix (rowptr at its first
// row, columns counted over the whole matrix)
struct CsrRows {
    int n, row0;
    const int* __restrict__ rowptr;
    const int* __restrict__ col;
    const double* __restrict__ val;
};
// One system of a batched launch: blocks blk0 .. blk0 + grid - 1.
struct ResidentSystem {
    CsrRows A;
    ResidentArgs<double> a;
    WindowShape w;
    int grid, blk0;
};
// synchronisations a launch of `chunk` iterations may number
inline uint32_t resident_tags(int chunk) { return 4u * (uint32_t)chunk + 4u; }

// TFLOWS_CG_RESIDENT=0, or an explicit kernel-per-phase form (TFLOWS_CG_FORM,
// TFLOWS_CG_CARRY), turns the on-chip CG off (read at every solve)
bool cg_resident_enabled();
// longest wait of a synchronisation in wall-clock ticks (TFLOWS_BARRIER_WAIT_MS)
uint64_t resident_wait_ticks();

// Launches whose blocks wait for each other need the CUs of all their blocks
// at once.  Two of them started from two host threads could each hold a part
// of the chip and wait for the rest, so such launches take their share of
// the device's CUs here first, in order of arrival, and give it back when
// they have ended (blocks < 0: the whole device).
class CuShare {
   public:
    explicit CuShare(int blocks);
    ~CuShare();
    CuShare(const CuShare&) = delete;
    CuShare& operator=(const CuShare&) = delete;

   private:
    int dev_, blocks_;
};

void launch_resident_deps(int n, int rows, int grid, const int* rowptr, const int* col, int* deps, hipStream_t s);
// false (nothing launched) when the device cannot hold the grid at once
template <typename Op, typename T>
bool launch_cg_stream(const Op& A, const ResidentArgs<T>& a, int grid, hipStream_t s);
template <typename Op, typename T>
bool launch_cg_window(const Op& A, const ResidentArgs<T>& a, const WindowShape& w, int grid, hipStream_t s);
// CGS: rows of a thread (seven vectors and the matrix rows in registers)
constexpr int kCgsRows = 4;
bool launch_cgs_window(const Sell<double>& A, const ResidentArgs<double>& a, const WindowShape& w, const double* r2,
                       double* q, double* u2, int grid, hipStream_t s);
// LDS of system s in a launch of R rows per thread (the most of any system)
size_t batch_window_lds(const ResidentSystem& s, int R);
bool launch_cg_window_batch(const ResidentSystem* sys, const int* blk_sys, int grid, int R, size_t lds, uint32_t tag,
                            hipStream_t s);

}  // namespace tflows
