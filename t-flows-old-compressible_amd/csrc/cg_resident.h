// cg_resident.h -- the on-chip CG (cg_resident.hip): its arguments, sizes and
// launchers.
#pragma once
#include <vector>

#include "krylov_kernels.h"
#include "resident_window.h"

namespace tflows {

constexpr int kResChunk = 1024;       // iterations of a launch: bounds how long it holds the CUs
constexpr int kPostWords = 4;         // 64-bit words a block posts at a site (two FP64 values)
constexpr int kPostStride = kResMaxBlocks;            // words between two words of a block
constexpr int kPostSite = kPostWords * kPostStride;   // words of a copy of a site's posts
constexpr int kPostCopies = 8;                        // one per XCD
constexpr int kPostSecond = 128;                      // words of a copy of the eighths' sums
constexpr int kPostTotal = 2 * kPostCopies * (kPostSite + kPostSecond);

// the mixed-precision forms pause the FP32 recurrence for a residual
// replacement once it has dropped this far below the last FP64 norm
constexpr double kReplaceDrop = 1e-2;

// resident_shape on the current device
ResidentShape resident_shape(int n, int rows_per_thread);
// the most blocks of a launch: one per CU
int resident_blocks();

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
// longest wait of a synchronisation in wall-clock ticks
// (TFLOWS_BARRIER_WAIT_MS; 0: a poll that finds a post missing gives up)
uint64_t resident_wait_ticks();
// TFLOWS_BARRIER_WAIT_MS below 0: a solve's first launch starts with its
// fault word raised, as for a block that starts after another gave up
bool resident_starts_given_up();

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
// (alone: every system is one block, so that no block waits and the grid
// need not be on the device at once)
bool launch_cg_window_batch(const ResidentSystem* sys, const int* blk_sys, int grid, int R, size_t lds, bool alone,
                            uint32_t tag, hipStream_t s);

}  // namespace tflows
