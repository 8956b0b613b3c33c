// cg_resident.hip -- Jacobi (or unpreconditioned) CG with the vectors of the
// solve kept on the chip: one launch runs many iterations, one block per CU.
//
// What bounds the kernel-per-phase form (cg_fused.hip) is not arithmetic:
// every iteration moves x, r, z, p, q and D through memory (10 N values
// beside the SpMV) and pays three kernel starts.  The register files and the
// LDS of 256 CUs hold 168 MB, so here x, r, D, z / q and the matrix rows of a
// block stay in registers and p in LDS for the whole launch.
//
// k_cg_window, the form of the meshes: a block also keeps p of the rows of
// other blocks that its columns reach (its halo), and advances it itself:
// p = z + beta p needs only their z, which is published before the
// reduction that gives beta.  Per iteration:
//
//   C  ||r||^2 and rho = (r, z) over all blocks, z published
//                                      -> stopping test, beta, own and halo p
//   B  (p, q) over all blocks          -> alfa
//
// so an iteration costs two synchronisations, one write of z, one read of
// the halo's z, and gathers from LDS.
//
// k_cg_stream: rows that k_cg_window does not hold (more than 7 entries, or
// columns beyond the halo): they are read every iteration and p is
// published, which takes a third synchronisation (A: a block waits for the
// blocks its columns reach).  It sums over the same rows in the same order,
// so both give the same bits.
//
// Process/CG.f90:113-259 per iteration, every value formed with the
// reference's operations in the reference's order (each row's products added
// in CSR order); only the dot-product summation order is the blocks'.
//
// Synchronisation without fences: values that cross blocks (z or p, and the
// partial sums) are stored and loaded with device-coherent accesses that
// bypass the non-coherent caches, so no L2 is written back or invalidated.
// A block posts its partial sums in words that carry the number of the
// synchronisation beside 32 bits of the value; a reader polls all blocks'
// words until every one carries that number, and adds the values in block
// order: every block gets the same bits.  B and C alternate and each waits
// for every block, so one set of words per site is enough: no block can post
// its next B before all have read the last C, and none posts C before all
// have read the last B.
//
// Measured, us per iteration, one launch per kernel -> on the chip (FP64,
// Jacobi): natural order 65,600 rows 12.9 -> 6.5, 230,580 17.0 -> 8.2,
// 491,111 26.1 -> 9.1, 979,902 35.8 -> 12.6; locality order 230,580 rows
// 18.2 -> 8.5, 506,880 28.9 -> 10.4; k_cg_stream (CSR rows) 65,600 rows
// 14.8 -> 11.7, 491,111 28.5 -> 20.7, 979,902 40.8 -> 34.3.  At 491,111 rows
// (256 blocks, 2.35 GHz) an iteration is 20,900 cycles: 5900 to 7400 of
// synchronisation C, 6100 of B, 3200 to 4400 of halo, 1100 of row sums, 1100
// of waiting for the published z and 2100 of the rest: latency of
// device-scope accesses, not bandwidth, bounds it.
//
// Every wait ends: the grid is at most one block per CU (the host checks
// that the device holds it at once; a batch of one-block systems has no wait
// and may have more), and a wait longer than wait_ticks
// (another process held the CUs) raises the fault word, on which every
// block stops; the host then restores the vectors and runs the
// kernel-per-phase form.
#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "cg_resident.h"

namespace tflows {

namespace {

constexpr int kResWaves = kResThreads / kWave;
__device__ __forceinline__ double coherent_load(const double* p) {
    const uint64_t u = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(double, u);
}
__device__ __forceinline__ float coherent_load(const float* p) {
    const uint32_t u = __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(float, u);
}
__device__ __forceinline__ void coherent_store(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void coherent_store(float* p, float v) {
    __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Posts of one site: word i of block b at i * stride + b, so that a
// wavefront polls 64 blocks' words in four cache lines, and where every
// block reads them in kPostCopies copies, one for the blocks of each XCD
// (one copy: 7500 cycles against 3700 at 32 blocks).  Each word carries 32
// bits of the value and the tag.
template <typename P> struct PostWords;
template <> struct PostWords<double> { static constexpr int n = 2; };
template <> struct PostWords<float> { static constexpr int n = 1; };

__device__ __forceinline__ void post_word(uint64_t* w, uint32_t v, uint32_t tag) {
    __hip_atomic_store(w, ((uint64_t)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void post_value(uint64_t* w, int stride, double v, uint32_t tag) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    post_word(w, (uint32_t)b, tag);
    post_word(w + stride, (uint32_t)(b >> 32), tag);
}
__device__ __forceinline__ void post_value(uint64_t* w, int, float v, uint32_t tag) {
    post_word(w, __builtin_bit_cast(uint32_t, v), tag);
}
// true (and v) when every word of the value carries the tag
__device__ __forceinline__ bool read_value(const uint64_t* w, int stride, uint32_t tag, double& v) {
    const uint64_t a = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t b = __hip_atomic_load(w + stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = __builtin_bit_cast(double, (a & 0xffffffffu) | (b << 32));
    return (uint32_t)(a >> 32) == tag && (uint32_t)(b >> 32) == tag;
}
__device__ __forceinline__ bool read_value(const uint64_t* w, int, uint32_t tag, float& v) {
    const uint64_t a = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = __builtin_bit_cast(float, (uint32_t)a);
    return (uint32_t)(a >> 32) == tag;
}

// Waits of one launch: bounded by the wall clock and the fault word.
struct Waiter {
    int* fault;
    uint64_t ticks;
    HostMirror* hm;                 // told, too, so that a host that paces itself on it stops
    // false when the wait must be given up
    __device__ __forceinline__ bool keep_waiting(unsigned& polls, uint64_t& t0) const {
        if ((++polls & 127u) != 0 && ticks != 0) return true;
        const uint64_t now = (uint64_t)wall_clock64();
        if (polls == 128u) t0 = now;
        if (now - t0 > ticks || __hip_atomic_load(fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
            __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            publish(hm, 1, 0);
            return false;
        }
        return true;
    }
};

// Sum over the block of value k of every thread, in wavefront k's lanes.  The
// values go through LDS and one wavefront adds them: a cross-lane sum in
// every wavefront cost 4 x 40 instructions on each SIMD.
template <typename T, int NV>
__device__ __forceinline__ T block_partial(int tid, const T (&v)[NV], T* sm) {
    const int lane = tid & (kWave - 1), w = tid / kWave;
#pragma unroll
    for (int k = 0; k < NV; ++k) sm[k * kResThreads + tid] = v[k];
    __syncthreads();
    T s = T(0);
    if (w < NV) {
        T t[kResWaves];
#pragma unroll
        for (int i = 0; i < kResWaves; ++i) t[i] = sm[w * kResThreads + i * kWave + lane];
        s = t[0];
#pragma unroll
        for (int i = 1; i < kResWaves; ++i) s += t[i];
        s = wave_sum(s);
    }
    return s;
}

// Sums of NV values over the block, valid in every thread.
template <int NV>
__device__ __forceinline__ void block_total(double (&v)[NV], double* sm) {
    __shared__ double tot[NV];
    const double s = block_partial<double, NV>(threadIdx.x, v, sm);
    if (threadIdx.x % kWave == 0 && threadIdx.x / kWave < NV) tot[threadIdx.x / kWave] = s;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = tot[k];
}

// wave_sum of values in the first eight lanes, 0 in the others: the same bits
__device__ __forceinline__ double octet_sum(double v) {
    v += dpp_d<kQuadSwap1>(v);
    v += dpp_d<kQuadSwap2>(v);
    v += dpp_d<kRowHalfMirror>(v);
    return readlane_d(v, 0);
}

// Polls block b's post of value k where `use`, and returns the FP64 sum over
// the wavefront's lanes (OCTET: the first eight) in every one of them.
template <typename P, bool OCTET = false>
__device__ __forceinline__ double poll_sum(const uint64_t* slots, int k, int stride, int b, bool use, uint32_t tag,
                                           const Waiter& wt, int* s_fail) {
    P got = P(0);
    if (use) {
        const uint64_t* s = slots + k * PostWords<P>::n * stride + b;
        unsigned polls = 0;
        uint64_t t0 = 0;
        while (!read_value(s, stride, tag, got))
            if (!wt.keep_waiting(polls, t0)) {
                *s_fail = 1;
                break;
            }
    }
    return OCTET ? octet_sum((double)got) : wave_sum((double)got);
}

// Sums of NV values over the block, then over the `nblk` blocks: posted in
// `slots` in the values' type, added in FP64.  Valid in every thread; false
// when the wait was given up (the whole block agrees).  Up to a wavefront of
// blocks each reads all posts; above that the first block of each eighth adds
// its eighth's posts and posts the sum, and every block reads eight: all
// blocks reading all posts took 10,000 cycles at 256 blocks, two steps take
// 6000 (one at 32 blocks: 3500).
template <typename T, int NV>
__device__ __forceinline__ bool resident_sum(int tid, const T (&v)[NV], double (&sum)[NV], uint64_t* slots, int nblk,
                                             int blk, uint32_t tag, const Waiter& wt, int* s_fail, T* sm) {
    __shared__ double tot[NV];
    constexpr int kWords = PostWords<T>::n;
    const int lane = tid & (kWave - 1), w = tid / kWave;
    const T mine = block_partial<T, NV>(tid, v, sm);
    double s = mine;
    if (w < NV && nblk > 1) {
        if (nblk <= kWave) {
            if (lane < kPostCopies)
                post_value(slots + lane * kPostSite + w * kWords * kPostStride + blk, kPostStride, mine, tag);
            s = poll_sum<T>(slots + (blockIdx.x & (kPostCopies - 1)) * kPostSite, w, kPostStride, lane, lane < nblk, tag,
                            wt, s_fail);
        } else {
            const int m = nblk / kNumXcd, g = blk / m;       // above kWave blocks, a multiple of 8
            if (lane == 0) post_value(slots + w * kWords * kPostStride + blk, kPostStride, mine, tag);
            uint64_t* const second = slots + kPostCopies * kPostSite;
            if (blk == g * m) {
                s = poll_sum<T>(slots, w, kPostStride, blk + lane, lane < m, tag, wt, s_fail);
                if (lane < kPostCopies)
                    post_value(second + lane * kPostSecond + w * kWords * kNumXcd + g, kNumXcd, (T)s, tag);
            }
            s = poll_sum<T, true>(second + (blockIdx.x & (kPostCopies - 1)) * kPostSecond, w, kNumXcd, lane,
                                  lane < kNumXcd, tag, wt, s_fail);
        }
    }
    if (w < NV && lane == 0) tot[w] = s;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) sum[k] = tot[k];
    return *s_fail == 0;
}

// Synchronisation A: this block's published rows have reached memory, and
// those of the blocks its columns reach (alo .. ahi) have.  False when the
// wait was given up (the whole block agrees).
static_assert(kResMaxBlocks <= kResThreads, "a thread for each block waited for");
__device__ __forceinline__ bool neighbour_sync(uint32_t* flags, int blk, int alo, int ahi, uint32_t tag,
                                               const Waiter& wt, int* s_fail) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int tid = threadIdx.x;
    if (tid == 0) __hip_atomic_store(flags + blk, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int b = alo + tid;
    if (b <= ahi && b != blk) {
        unsigned polls = 0;
        uint64_t t0 = 0;
        while ((int)(__hip_atomic_load(flags + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - tag) < 0)
            if (!wt.keep_waiting(polls, t0)) {
                *s_fail = 1;
                break;
            }
    }
    __syncthreads();
    return *s_fail == 0;
}

// A vector of other blocks' values, read W (16 bytes of) rows at a time with
// device-coherent loads (the same cache policy as the atomic loads above: a
// wider access needs no atomicity, since the rows of a granule are complete
// before the synchronisation that precedes the load).
template <typename T>
struct CoherentVec {
    static constexpr int W = 16 / (int)sizeof(T);
    static constexpr int kSc1 = 16;                  // device scope, in the builtin's policy bits
    __amdgpu_buffer_rsrc_t rsrc;
    const T* v;
    int n;
    __device__ __forceinline__ CoherentVec(const T* vec, int n_)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(vec), 0, n_ * (int)sizeof(T), 0x00027000)), v(vec),
          n(n_) {}
    // rows c .. c + W - 1, which lie in the vector
    __device__ __forceinline__ void load(int c, T (&out)[W]) const {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, c * (int)sizeof(T), 0, kSc1);
        __builtin_memcpy(out, &q, sizeof(out));
    }
};

// `count` granules of consecutive rows from `row` on, at lp[at] (16-byte
// aligned).
struct HaloRun {
    int at, row, count;
};

// The first NB granules of a run that a thread moves: loaded, then applied
// as p = z + beta p.  A run that reaches outside the matrix (the first and
// last blocks') is left to apply, row by row.
template <typename T, int NB>
struct HaloLoad {
    static constexpr int W = CoherentVec<T>::W;
    T z[NB][W];
    __device__ __forceinline__ static bool inside(const CoherentVec<T>& v, const HaloRun& h) {
        return h.row >= 0 && h.row + h.count * W <= v.n;
    }
    __device__ __forceinline__ void load(int tid, const CoherentVec<T>& v, const HaloRun& h, int e0 = 0) {
        if (!inside(v, h)) return;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int e = e0 + i * kResThreads + tid;
            if (e < h.count) v.load(h.row + e * W, z[i]);
        }
    }
    __device__ __forceinline__ void apply(int tid, const CoherentVec<T>& v, T* lp, const HaloRun& h, bool first, T beta,
                                          int e0 = 0) {
        if (inside(v, h)) {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int e = e0 + i * kResThreads + tid;
                if (e < h.count)
#pragma unroll
                    for (int u = 0; u < W; ++u)
                        lp[h.at + e * W + u] = first ? z[i][u] : z[i][u] + beta * lp[h.at + e * W + u];
            }
            return;
        }
        for (int e = e0 * W + tid; e < min(h.count, e0 + NB * kResThreads) * W; e += kResThreads) {
            const int c = h.row + e;
            if (c < 0 || c >= v.n) continue;
            const T zc = coherent_load(v.v + c);
            lp[h.at + e] = first ? zc : zc + beta * lp[h.at + e];
        }
    }
    __device__ __forceinline__ void rest(int tid, const CoherentVec<T>& v, T* lp, const HaloRun& h, bool first, T beta) {
        for (int e0 = NB * kResThreads; e0 < h.count; e0 += NB * kResThreads) {
            load(tid, v, h, e0);
            apply(tid, v, lp, h, first, beta, e0);
        }
    }
};

// p of a column: this block's rows in LDS, others from memory with
// device-coherent loads (a row the entry lacks reads LDS slot 0: unused).
template <typename T>
struct ResGather {
    const T* lp;
    const T* __restrict__ pg;
    int rb, nloc;
    __device__ __forceinline__ T operator()(bool has, int c) const {
        const unsigned o = (unsigned)(c - rb);
        const bool loc = o < (unsigned)nloc;
        T g = lp[loc ? o : 0];
        // a 32-bit byte offset from a scalar base (n * sizeof(T) < 2^32)
        if (has && !loc)
            g = coherent_load(reinterpret_cast<const T*>(reinterpret_cast<const char*>(pg) +
                                                         (uint32_t)c * (uint32_t)sizeof(T)));
        return g;
    }
};

// The slots of a row kept in registers: values and where the column's p is
// in LDS, in CSR order.  A slot the row lacks has the value 0 and a finite p
// (its own row, or the place of a row outside the matrix, which holds 0), so
// it adds +-0 to a sum that is never -0: the sum's bits are those of the
// slots it has.
template <typename Op> struct OpDiff { static constexpr bool value = false; };
template <> struct OpDiff<DiffSell32> { static constexpr bool value = true; };
template <typename T, bool SHARED>
struct RowSlots {
    static constexpr int N = window_slots<T>();
    T a[N];
    int c[SHARED ? 1 : N];
    T rs;                           // difference form: the row sum
};

// Row `row` (every thread of the block calls it, with live = false past the
// block's rows: the slice is the wavefront's, clamped to the last one).
// Shared offsets: slot j is the matrix's j-th column offset, whose p lies
// w.disp[j] from the row's own in LDS, so no index is kept.  Otherwise c is
// an index of lp (own: the row's).
template <bool SHARED, typename Op, typename T>
__device__ __forceinline__ void load_row(const Op& A, int row, bool live, const WindowShape& w, int base, int own,
                                         RowSlots<T, SHARED>& s) {
    constexpr int N = RowSlots<T, SHARED>::N;
    const int lane = (int)threadIdx.x & (kSlice - 1);
    const int sl = __builtin_amdgcn_readfirstlane(min(row, A.n - 1) / kSlice);
    row = sl * kSlice + lane;
    const int b = A.off[sl];
    const int stored = (A.off[sl + 1] - b) / kSlice;
    if constexpr (OpDiff<Op>::value) s.rs = live ? A.rs[row] : T(0);
#pragma unroll
    for (int j = 0; j < N; ++j) s.a[j] = T(0);
    if constexpr (SHARED) {
        const bool sym = A.lbase != nullptr;
        const int sb = sym ? A.sidx[sl] : b / kSlice;
        const int ws = sym ? A.sidx[sl + 1] - sb : stored;
        const int nl = ws - stored;
        const unsigned m = live ? A.mask[row] : 0u;
        for (int i = 0; i < ws; ++i) {               // the slice's slots; both lists ascend
            const int d = __builtin_amdgcn_readfirstlane(A.soff[sb + i]);
            if (!((m >> i) & 1u)) continue;
            const T v = A.val[i < nl ? sym_mirror_pos(A.lbase, sb, i, sl, row, d) : b + lane + (i - nl) * kSlice];
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (j < w.nslots && d == w.offset[j]) s.a[j] = v;
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            s.c[j] = own;
            if (!live || j >= stored) continue;
            const int at = b + lane + j * kSlice;
            int c = -1;
            if (A.dc) {
                const short d = A.dc[at];
                if (d != kPad16) c = row + (int)d;
            } else {
                c = A.col[at];
            }
            if (c >= 0) {
                s.c[j] = c - base;
                s.a[j] = A.val[at];
            }
        }
    }
}

// The same from the CSR arrays (a system of a block-diagonal batch): every
// column offset of the row is one of w.offset.
template <bool SHARED, typename T>
__device__ __forceinline__ void load_row(const CsrRows& A, int row, bool live, const WindowShape& w, int, int,
                                         RowSlots<T, SHARED>& s) {
    static_assert(SHARED, "rows of known offsets");
    constexpr int N = RowSlots<T, SHARED>::N;
#pragma unroll
    for (int j = 0; j < N; ++j) s.a[j] = T(0);
    if (!live) return;
    const int e1 = A.rowptr[row + 1];
    for (int e = A.rowptr[row]; e < e1; ++e) {
        const int d = A.col[e] - A.row0 - row;
        const T v = A.val[e];
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (j < w.nslots && d == w.offset[j]) s.a[j] = v;
    }
}

// Products added to 0 in CSR order (CG.f90:193-199), or the terms of the
// difference form, gathered from LDS; `off` is an opaque 0.  Row k of a thread lies k * kResThreads above its first, an
// immediate offset of the LDS reads.
template <bool SHARED, typename Op, typename T>
__device__ __forceinline__ T row_sum(const RowSlots<T, SHARED>& s, int k, int own, int off, const WindowShape& w,
                                     const T* lp) {
    constexpr int N = RowSlots<T, SHARED>::N;
    T acc = T(0);
    T pv[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        if constexpr (SHARED) pv[j] = (lp + own + w.disp[j])[k * kResThreads];
        else pv[j] = lp[off + s.c[j]];
    }
    const T pi = OpDiff<Op>::value ? (lp + own)[k * kResThreads] : T(0);
#pragma unroll
    for (int j = 0; j < N; ++j)
        acc = acc + s.a[j] * (OpDiff<Op>::value ? pv[j] - pi : pv[j]);
    if constexpr (OpDiff<Op>::value) acc = acc + s.rs * pi;
    return acc;
}

// A row of any length, read from memory.
template <typename T>
__device__ __forceinline__ T stream_row(const Csr<T>& A, int row, const ResGather<T>& g) {
    T acc = T(0);
    const int e1 = A.rowptr[row + 1];
#pragma unroll 4
    for (int e = A.rowptr[row]; e < e1; ++e) acc = acc + A.val[e] * g(true, A.col[e]);
    return acc;
}

}  // namespace

template <typename Op, int R, typename T = typename OpValue<Op>::type>
__global__ __launch_bounds__(kResThreads) void k_cg_stream(Op A, ResidentArgs<T> a) {
    extern __shared__ __align__(16) char res_lds[];
    T* lp = reinterpret_cast<T*>(res_lds);           // p of this block's rows
    __shared__ T sm[2 * kResThreads];
    __shared__ int s_fail, s_done;
    SolverState* st = a.st;
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_fail = 0;
        s_done = st->done;
    }
    const int G = gridDim.x, blk = logical_block();
    const int rb = min(blk * a.rows, a.n), nloc = min(a.n - rb, a.rows);
    const bool lead = blk == 0 && tid == 0;
    const double tol = st->tol;
    const int cap = st->cap, it0 = st->it;
    T rho_old = (T)st->rho[it0 & 1];
    __syncthreads();
    if (s_done) return;
    const Waiter wt{&st->fault, a.wait_ticks, a.hm};
    const ResGather<T> g{lp, a.p, rb, nloc};
    const int alo = G > 1 ? a.deps[2 * blk] / a.rows : 0, ahi = G > 1 ? a.deps[2 * blk + 1] / a.rows : 0;
    T xv[R], rv[R], dv[R], zq[R];   // zq: z, then q of the iteration
#pragma unroll
    for (int k = 0; k < R; ++k) {   // past the block's rows: x = r = p = 0, D = 1, no entries
        const int l = k * kResThreads + tid;
        T d = T(1), p = T(0);
        xv[k] = rv[k] = zq[k] = T(0);
        if (l < nloc) {
            xv[k] = a.x[rb + l];
            rv[k] = a.r[rb + l];
            d = a.D[rb + l];
            if (it0 > 0) p = a.p[rb + l];
            if (a.keep) {           // the state a fallback starts from
                a.keep[rb + l] = xv[k];
                a.keep[(size_t)a.n + rb + l] = rv[k];
            }
        }
        lp[l] = p;
        dv[k] = d;
    }
    uint32_t tag = a.tag;
    int it = it0, niter = 0;
    bool stop = false;
    double err = 0.0;
    for (;;) {
        T v[2] = {T(0), T(0)};
#pragma unroll
        for (int k = 0; k < R; ++k) {
            zq[k] = rv[k] / dv[k];                       // z, CG.f90:126
            v[0] += rv[k] * rv[k];                       // ||r||^2, CG.f90:250
            v[1] += rv[k] * zq[k];                       // rho, CG.f90:174
        }
        double sum[2];
        if (!resident_sum(tid, v, sum, a.slotC, G, blk, ++tag, wt, &s_fail, sm)) return;
        err = sqrt(sum[0]);
        if (err < tol) {                                 // CG.f90:93-108, :248-255
            stop = true;
            niter = it;
            break;
        }
        if (it + 1 > cap) {                              // CG.f90:259-262
            stop = true;
            niter = (cap > 0 ? cap : 0) + 1;
            break;
        }
        if (it - it0 == a.chunk) break;
        const T rho = (T)sum[1];
        const bool first = it == 0;
        const T beta = first ? T(0) : rho / rho_old;     // CG.f90:183
        rho_old = rho;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + tid;
            const T p = first ? zq[k] : zq[k] + beta * lp[l];       // CG.f90:180, :185
            lp[l] = p;
            if (G > 1 && l < nloc) coherent_store(a.p + rb + l, p);
        }
        if (G > 1) {
            if (!neighbour_sync(a.flags, blk, alo, ahi, ++tag, wt, &s_fail)) return;
        } else {
            __syncthreads();
        }
        T pq[1] = {T(0)};
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + tid;
            zq[k] = l < nloc ? stream_row(A, rb + l, g) : T(0);     // CG.f90:193-199
            pq[0] += lp[l] * zq[k];                                 // CG.f90:216
        }
        double spq[1];
        if (!resident_sum(tid, pq, spq, a.slotB, G, blk, ++tag, wt, &s_fail, sm)) return;
        const T alfa = rho / (T)spq[0];                  // CG.f90:219
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + tid;
            if (l >= nloc) continue;                     // alfa may be infinite
            xv[k] = xv[k] + alfa * lp[l];                // CG.f90:227
            rv[k] = rv[k] - alfa * zq[k];                // CG.f90:228
        }
        ++it;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int l = k * kResThreads + tid;
        if (l < nloc) {
            a.x[rb + l] = xv[k];
            a.r[rb + l] = rv[k];
            if (G == 1) a.p[rb + l] = lp[l];
        }
    }
    if (lead) {
        st->it = it;
        st->rho[it & 1] = (double)rho_old;
        st->error = err;
        if (stop) {
            st->done = 1;
            st->niter_out = niter;
        }
    }
}

template <typename T>
__device__ __forceinline__ HaloRun far_run(const WindowShape& w, int rb, int rows, int q) {
    return HaloRun{w.farbase + q * rows, rb + w.far[q], q < w.nfar ? rows / CoherentVec<T>::W : 0};
}

// The halo's p = z + beta p (z when first): every run's loads in flight
// together, R rows per thread.
template <bool SHARED, int R, typename T>
__device__ __forceinline__ void halo_update(int t, const CoherentVec<T>& zin, T* lp, const HaloRun& below,
                                            const HaloRun& above, const WindowShape& w, int rb, int rows, bool first,
                                            T beta) {
    constexpr int NF = (R + CoherentVec<T>::W - 1) / CoherentVec<T>::W;   // granules of a far run per thread
    if constexpr (SHARED) {
        auto far = [&](int q) { return far_run<T>(w, rb, rows, q); };
        HaloLoad<T, NF> f0, f1;
        HaloLoad<T, 1> n0, n1;
        f0.load(t, zin, far(0));
        f1.load(t, zin, far(1));
        n0.load(t, zin, below);
        n1.load(t, zin, above);
        f0.apply(t, zin, lp, far(0), first, beta);
        f1.apply(t, zin, lp, far(1), first, beta);
        n0.apply(t, zin, lp, below, first, beta);
        n1.apply(t, zin, lp, above, first, beta);
        n0.rest(t, zin, lp, below, first, beta);
        n1.rest(t, zin, lp, above, first, beta);
        if (w.nfar > 2) {
            f0.load(t, zin, far(2));
            f1.load(t, zin, far(3));
            f0.apply(t, zin, lp, far(2), first, beta);
            f1.apply(t, zin, lp, far(3), first, beta);
        }
    } else {
        HaloLoad<T, 4> n0, n1;
        n0.load(t, zin, below);
        n1.load(t, zin, above);
        n0.apply(t, zin, lp, below, first, beta);
        n1.apply(t, zin, lp, above, first, beta);
        n0.rest(t, zin, lp, below, first, beta);
        n1.rest(t, zin, lp, above, first, beta);
    }
}

// SHARED: shared-offset matrix, the halo being `lo` rows either side and the
// far regions of w; else the halo is the window of columns the block reaches
// (deps).  LDS: halo below, own rows, halo above, far regions.
//
// MIXED: the FP32 iterations of a residual-replacement solve.  A block's sum
// and the posts are FP32, the posts are added in FP64: the mean error of x
// against 64 bits over 26 solves of 0.26 to 2.1 M rows is 3.0e-7, with every
// sum in FP32 3.8e-7 (one launch per kernel 4.0e-7), with FP64 posts 3.1e-7,
// with the threads' sums in FP64, too, 2.9e-7.  Against every sum in FP32 300
// iterations take 1.0 % more at 614,125 rows (FP64 posts 3.6 %), none at 2.1 M.
template <typename Op, bool SHARED, int R, bool MIXED, typename T>
__device__ __forceinline__ void cg_window(const Op& A, const ResidentArgs<T>& a, const WindowShape& w, const int G,
                                          const int blk) {
    extern __shared__ __align__(16) char res_lds[];
    __shared__ T sm[2 * kResThreads];
    __shared__ int s_fail, s_done;
    SolverState* st = a.st;
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_fail = 0;
        // a launch that keeps the state a fallback starts from keeps all of
        // it: a block that starts after another has given up does so, too,
        // and gives up at its first long wait
        s_done = st->done | st->suspend | (a.keep ? 0 : st->fault);
    }
    const int rb = min(blk * a.rows, a.n), nloc = min(a.n - rb, a.rows);
    const bool lead = blk == 0 && tid == 0;
    const double tol = st->tol;
    const int cap = st->cap, it0 = st->it;
    double err_rep = st->err_rep;
    T rho_old = (T)st->rho[it0 & 1];
    __syncthreads();
    if (s_done) return;
    const Waiter wt{&st->fault, a.wait_ticks, a.hm};
    int lo = w.lo, hi = w.lo;
    if (!SHARED) {                  // the columns this block reaches
        lo = G > 1 && nloc > 0 ? halo_rows(rb - a.deps[2 * blk]) : 0;
        hi = G > 1 && nloc > 0 ? halo_rows(a.deps[2 * blk + 1] + 1 - (rb + a.rows)) : 0;
    }
    constexpr bool kLdsD = window_d_in_lds<T>(R);
    T* const ld = reinterpret_cast<T*>(res_lds);     // D where it is in LDS, else nothing
    T* const lp = ld + (kLdsD ? R * kResThreads : 0);
    T* const own = lp + lo;
    for (size_t i = tid; i < w.lds / sizeof(T); i += kResThreads) ld[i] = T(0);   // read as a finite p (times 0) too
    __syncthreads();
    T xv[R], rv[R], dv[kLdsD ? 1 : R], zq[R];        // zq: z, then q of the iteration
    RowSlots<T, SHARED> rows[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {   // past the block's rows: x = r = 0, D = 1, no entries
        const int l = k * kResThreads + tid;
        T d = T(1);
        xv[k] = rv[k] = zq[k] = T(0);
        if (l < nloc) {
            xv[k] = a.x[rb + l];
            rv[k] = a.r[rb + l];
            d = a.D[rb + l];
            if (a.keep) {           // the state a fallback starts from
                a.keep[rb + l] = xv[k];
                a.keep[(size_t)a.n + rb + l] = rv[k];
            }
        }
        if (it0 > 0 && l < nloc) own[l] = a.p[rb + l];
        if (kLdsD) ld[l] = d;
        else dv[kLdsD ? 0 : k] = d;
        load_row(A, rb + l, l < nloc, w, rb - lo, lo + min(l, a.rows - 1), rows[k]);
    }
    // The halo: runs of rows in LDS order, moved W rows (16 bytes) at a time.
    // A run's rows may lie partly outside the matrix.
    constexpr int W = 16 / (int)sizeof(T);
    const CoherentVec<T> zin(a.z, a.n);
    const HaloRun below{0, rb - lo, lo / W}, above{lo + a.rows, rb + a.rows, hi / W};
    auto first_p = [&](const HaloRun& h) {
        for (int e = tid; it0 > 0 && e < h.count * W; e += kResThreads)
            if (h.row + e >= 0 && h.row + e < a.n) lp[h.at + e] = a.p[h.row + e];
    };
    first_p(below);
    first_p(above);
    if (SHARED)
        for (int q = 0; q < w.nfar; ++q) first_p(far_run<T>(w, rb, a.rows, q));
    double err64 = 0.0;
    if (MIXED) {                    // the FP64 norm of the replacement before this launch (site E)
        __shared__ double sm64[kResThreads];
        double e[1] = {0.0};
        for (int b = tid; b < a.nE; b += kResThreads) e[0] += a.partE[b];
        block_total<1>(e, sm64);
        err64 = sqrt(e[0]);
    }
    uint32_t tag = a.tag;
    int it = it0, niter = 0;
    bool stop = false, pause = false;
    double err = 0.0;
    for (;;) {
        // opaque, as the same every iteration the compiler would keep all
        // addresses formed from it in registers
        int t = tid;
        asm volatile("" : "+v"(t));
        T v[2] = {T(0), T(0)};
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + t;
            zq[k] = rv[k] / (kLdsD ? ld[l] : dv[kLdsD ? 0 : k]);    // z, CG.f90:126
            v[0] += rv[k] * rv[k];                                  // ||r||^2, CG.f90:250
            v[1] += rv[k] * zq[k];                                  // rho, CG.f90:174
            if (G > 1 && l < nloc) coherent_store(a.z + rb + l, zq[k]);
        }
        __builtin_amdgcn_s_waitcnt(0);               // this wave's z has reached memory before the block posts
        double sum[2];
        if (!resident_sum(t, v, sum, a.slotC, G, blk, ++tag, wt, &s_fail, sm)) return;
        err = sqrt(sum[0]);
        if (MIXED && it == it0) {                    // after a replacement the FP64 norm decides
            err = err_rep = err64;
            if (lead) {
                st->error = st->err_rep = err;
                if (it == 0) {
                    st->ini_res = err;
                    st->ini_written = 1;
                }
            }
        } else if (MIXED) {
            pause = err < kReplaceDrop * err_rep || err < tol;      // the next replacement verifies
            if (pause) break;
        }
        if (err < tol) {                             // CG.f90:93-108, :248-255
            stop = true;
            niter = it;
            break;
        }
        if (it + 1 > cap) {                          // CG.f90:259-262
            stop = true;
            niter = (cap > 0 ? cap : 0) + 1;
            break;
        }
        if (it - it0 == a.chunk) break;
        const T rho = (T)sum[1];
        const bool first = it == 0;
        const T beta = first ? T(0) : rho / rho_old;                // CG.f90:183
        rho_old = rho;
        if (G > 1) halo_update<SHARED, R>(t, zin, lp, below, above, w, rb, a.rows, first, beta);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + t;
            if (l < nloc) own[l] = first ? zq[k] : zq[k] + beta * own[l];
        }
        __syncthreads();
        T pq[1] = {T(0)};
        int at = lo + t, off = 0;
        asm volatile("" : "+v"(off));
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + t;
            zq[k] = row_sum<SHARED, Op>(rows[k], k, at, off, w, lp);
            if (l < nloc) pq[0] += own[l] * zq[k];                  // CG.f90:216
            if (R > 2) asm volatile("" : "+v"(zq[k]));              // one row's gathers in registers at a time
        }
        double spq[1];
        if (!resident_sum(t, pq, spq, a.slotB, G, blk, ++tag, wt, &s_fail, sm)) return;
        const T alfa = rho / (T)spq[0];                             // CG.f90:219
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kResThreads + t;
            if (l < nloc) xv[k] = xv[k] + alfa * own[l];            // CG.f90:227
            // an infinite alfa must not turn FinRes into NaN past the rows
            // (a replacement's norm is FinRes in the mixed solve)
            if (MIXED || l < nloc) rv[k] = rv[k] - alfa * zq[k];    // CG.f90:228
        }
        ++it;
        if (MIXED && it - it0 == a.chunk) break;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int l = k * kResThreads + tid;
        if (l < nloc) {
            a.x[rb + l] = xv[k];
            a.r[rb + l] = rv[k];
            a.p[rb + l] = own[l];
        }
    }
    if (lead) {
        st->it = it;
        st->rho[it & 1] = (double)rho_old;
        if (!MIXED) st->error = err;
        if (pause) st->suspend = 1;
        if (stop) {
            st->done = 1;
            st->niter_out = niter;
            publish(a.hm, 1, it);
        }
    }
}

template <typename Op, bool SHARED, int R, bool MIXED, typename T = typename OpValue<Op>::type>
__global__ __launch_bounds__(kResThreads) void k_cg_window(Op A, ResidentArgs<T> a, WindowShape w) {
    cg_window<Op, SHARED, R, MIXED, T>(A, a, w, gridDim.x, logical_block());
}

// CGS (Process/CGS.f90:112-334) in the same form: x, r, the shadow r2, q, u1,
// u2, D and the matrix rows in registers, the vector of the next product
// (own rows and halo) in LDS.  Its two products an iteration act on vectors
// that need the scalar just reduced and a division by D, so each is
// published after that (synchronisation A):
//
//   C  ||r||^2, rho = (r, r2)  -> stopping test, beta; u1, u2; u2 / D published
//   A  -> halo, v = A (u2 / D)
//   B  (r2, v)                 -> alfa; q; w = (u1 + q) / D published
//   A  -> halo, x += alfa w, r -= alfa A w
//
// A waits for every block whose rows the halo loads, those multiplied by 0
// included (halo_reach): what they publish is finite, what the vector holds
// before that need not be.
//
// qg, u2g carry q and u2 from launch to launch.  The grid is two blocks or more.
template <typename Op, bool SHARED, int R, typename T = typename OpValue<Op>::type>
__global__ __launch_bounds__(kResThreads) void k_cgs_window(Op A, ResidentArgs<T> a, WindowShape w,
                                                            const T* __restrict__ shadow, T* __restrict__ qg,
                                                            T* __restrict__ u2g) {
    extern __shared__ __align__(16) char res_lds[];
    __shared__ T sm[2 * kResThreads];
    __shared__ int s_fail, s_done;
    SolverState* st = a.st;
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_fail = 0;
        s_done = st->done | (a.keep ? 0 : st->fault);   // as in cg_window
    }
    const int G = gridDim.x, blk = logical_block();
    const int rb = min(blk * a.rows, a.n), nloc = min(a.n - rb, a.rows);
    const bool lead = blk == 0 && tid == 0;
    const double tol = st->tol;
    const int cap = st->cap, it0 = st->it;
    T rho_old = (T)st->rho[it0 & 1];
    __syncthreads();
    if (s_done) return;
    const Waiter wt{&st->fault, a.wait_ticks, a.hm};
    int lo = w.lo, hi = w.lo;
    if (!SHARED) {                  // the columns this block reaches
        lo = nloc > 0 ? halo_rows(rb - a.deps[2 * blk]) : 0;
        hi = nloc > 0 ? halo_rows(a.deps[2 * blk + 1] + 1 - (rb + a.rows)) : 0;
    }
    // the blocks whose rows the halo reads (neighbour_sync has a thread for
    // each: at most kResMaxBlocks)
    const RowRange reach = halo_reach(w, SHARED, RowRange{a.deps[2 * blk], a.deps[2 * blk + 1]}, rb, a.rows, a.n);
    const int alo = reach.first / a.rows, ahi = reach.last / a.rows;
    T* const lp = reinterpret_cast<T*>(res_lds);
    T* const own = lp + lo;
    for (size_t i = tid; i < w.lds / sizeof(T); i += kResThreads) lp[i] = T(0);   // read as a finite p (times 0) too
    __syncthreads();
    T xv[R], rv[R], sv[R], qv[R], u1[R], u2[R], dv[R];
    RowSlots<T, SHARED> rows[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {   // past the block's rows: every vector 0, D = 1, no entries
        const int l = k * kResThreads + tid;
        xv[k] = rv[k] = sv[k] = qv[k] = u1[k] = u2[k] = T(0);
        dv[k] = T(1);
        if (l < nloc) {
            xv[k] = a.x[rb + l];
            rv[k] = a.r[rb + l];
            sv[k] = shadow[rb + l];
            dv[k] = a.D[rb + l];
            if (it0 > 0) {
                qv[k] = qg[rb + l];
                u2[k] = u2g[rb + l];
            }
            if (a.keep) {           // the state a fallback starts from
                a.keep[rb + l] = xv[k];
                a.keep[(size_t)a.n + rb + l] = rv[k];
            }
        }
        load_row(A, rb + l, l < nloc, w, rb - lo, lo + min(l, a.rows - 1), rows[k]);
    }
    constexpr int W = CoherentVec<T>::W;
    const CoherentVec<T> zin(a.z, a.n);
    const HaloRun below{0, rb - lo, lo / W}, above{lo + a.rows, rb + a.rows, hi / W};
    uint32_t tag = a.tag;
    int it = it0, niter = 0;
    bool stop = false;
    double err = 0.0;
    for (;;) {
        int t = tid;                // opaque, as in cg_window
        asm volatile("" : "+v"(t));
        // the product with the vector f(k) of row k: LDS, memory, halo, row sums into y
        auto product = [&](auto&& f, auto&& y) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int l = k * kResThreads + t;
                const T p = f(k);
                if (l < nloc) {
                    own[l] = p;
                    coherent_store(a.z + rb + l, p);
                }
            }
            if (!neighbour_sync(a.flags, blk, alo, ahi, ++tag, wt, &s_fail)) return false;
            halo_update<SHARED, R>(t, zin, lp, below, above, w, rb, a.rows, true, T(0));
            __syncthreads();
            int at = lo + t, off = 0;
            asm volatile("" : "+v"(off));
#pragma unroll
            for (int k = 0; k < R; ++k) y(k, row_sum<SHARED, Op>(rows[k], k, at, off, w, lp));
            return true;
        };
        T v[2] = {T(0), T(0)};
#pragma unroll
        for (int k = 0; k < R; ++k) {
            v[0] += rv[k] * rv[k];
            v[1] += rv[k] * sv[k];                                  // rho, CGS.f90:118-122
        }
        double sum[2];
        if (!resident_sum(t, v, sum, a.slotC, G, blk, ++tag, wt, &s_fail, sm)) return;
        err = sqrt(sum[0]);
        if (err < tol) {
            stop = true;
            niter = it;
            break;
        }
        if (it + 1 > cap) {
            stop = true;
            niter = (cap > 0 ? cap : 0) + 1;
            break;
        }
        if (it - it0 == a.chunk) break;
        const T rho = (T)sum[1];
        const bool first = it == 0;
        const T beta = first ? T(0) : rho / rho_old;
        rho_old = rho;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            u1[k] = first ? rv[k] : rv[k] + beta * qv[k];
            u2[k] = first ? rv[k] : u1[k] + beta * (qv[k] + beta * u2[k]);
        }
        T rs[1] = {T(0)};
        if (!product([&](int k) { return u2[k] / dv[k]; },
                     [&](int k, T y) {
                         qv[k] = y;                                 // v, until alfa is known
                         rs[0] += sv[k] * y;                        // (r2, v)  :215-219
                     }))
            return;
        double srs[1];
        if (!resident_sum(t, rs, srs, a.slotB, G, blk, ++tag, wt, &s_fail, sm)) return;
        const T alfa = rho / (T)srs[0];                                 // :220
        if (!product(
                [&](int k) {
                    qv[k] = u1[k] - alfa * qv[k];                   // :226-228
                    const T p = (u1[k] + qv[k]) / dv[k];            // :238-241
                    xv[k] = xv[k] + alfa * p;                       // :286-288
                    return p;
                },
                [&](int k, T y) {
                    if (k * kResThreads + t < nloc) rv[k] = rv[k] - alfa * y;      // :315-317; alfa may be infinite
                }))
            return;
        ++it;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int l = k * kResThreads + tid;
        if (l < nloc) {
            a.x[rb + l] = xv[k];
            a.r[rb + l] = rv[k];
            qg[rb + l] = qv[k];
            u2g[rb + l] = u2[k];
        }
    }
    if (lead) {
        st->it = it;
        st->rho[it & 1] = (double)rho_old;
        st->error = err;
        if (stop) {
            st->done = 1;
            st->niter_out = niter;
        }
    }
}

// Many systems in one launch: each has its own blocks, posts and state, and
// goes its own way (a system that has stopped, or whose blocks stop early,
// leaves the others alone).
template <int R>
__global__ __launch_bounds__(kResThreads) void k_cg_window_batch(const ResidentSystem* __restrict__ sys,
                                                                 const int* __restrict__ blk_sys, uint32_t tag) {
    const ResidentSystem& s = sys[blk_sys[blockIdx.x]];
    ResidentArgs<double> a = s.a;
    a.tag = tag;
    cg_window<CsrRows, true, R, false, double>(s.A, a, s.w, s.grid, (int)blockIdx.x - s.blk0);
}

// Smallest and largest column of each block's rows.
__global__ __launch_bounds__(kBlock) void k_resident_deps(int n, int rows, const int* __restrict__ rowptr,
                                                          const int* __restrict__ col, int* __restrict__ deps) {
    __shared__ int lo, hi;
    if (threadIdx.x == 0) {
        lo = n;
        hi = 0;
    }
    __syncthreads();
    const int b = blockIdx.x;
    const int rb = min(b * rows, n), re = min(n, rb + rows);
    int l = n, h = 0;
    if (rb < re)
        for (int e = rowptr[rb] + (int)threadIdx.x; e < rowptr[re]; e += kBlock) {
            l = min(l, col[e]);
            h = max(h, col[e]);
        }
    atomicMin(&lo, l);
    atomicMax(&hi, h);
    __syncthreads();
    if (threadIdx.x == 0) {
        deps[2 * b] = rb < re ? lo : min(b * rows, n - 1);
        deps[2 * b + 1] = rb < re ? hi : min(b * rows, n - 1);
    }
}

bool cg_resident_enabled() {
    const char* e = std::getenv("TFLOWS_CG_RESIDENT");
    return !(e && e[0] == '0') && !std::getenv("TFLOWS_CG_FORM") && !std::getenv("TFLOWS_CG_CARRY");
}

static int device_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    return cus;
}

static long wait_ms_from_env() {
    const char* e = std::getenv("TFLOWS_BARRIER_WAIT_MS");
    return e ? std::atol(e) : 2000;
}
bool resident_starts_given_up() { return wait_ms_from_env() < 0; }
uint64_t resident_wait_ticks() {
    const long ms = wait_ms_from_env();
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
        khz = 100000;
    return (uint64_t)khz * (uint64_t)(ms < 0 ? 0 : ms);
}

int resident_blocks() {
    const int cus = std::min(device_cus(), kResMaxBlocks);
    return cus >= kNumXcd ? cus / kNumXcd * kNumXcd : cus;   // whole shares of the XCDs
}

ResidentShape resident_shape(int n, int rows_per_thread) {
    return resident_shape(n, rows_per_thread, resident_blocks());
}

namespace {
struct CuPool {
    std::mutex m;
    std::condition_variable cv;
    uint64_t next = 0, serving = 0;
    int used = 0, cap = 0;
};
CuPool g_cu_pools[64];
}  // namespace

CuShare::CuShare(int blocks) : dev_(0), blocks_(blocks) {
    if (hipGetDevice(&dev_) != hipSuccess || dev_ < 0 || dev_ >= 64) dev_ = 0;
    CuPool& p = g_cu_pools[dev_];
    std::unique_lock<std::mutex> lk(p.m);
    if (p.cap == 0) p.cap = std::max(1, device_cus());
    // blocks go to the XCDs in turn: as many of each XCD as the fullest one
    // gets, so that no launch waits for a CU of one XCD that another launch
    // holds while that waits for a CU of another XCD
    if (blocks_ >= 0) blocks_ = std::min(p.cap, (blocks_ + kNumXcd - 1) / kNumXcd * kNumXcd);
    else blocks_ = p.cap;
    const uint64_t mine = p.next++;
    p.cv.wait(lk, [&] { return p.serving == mine && p.used + blocks_ <= p.cap; });
    p.used += blocks_;
    ++p.serving;
    p.cv.notify_all();
}
CuShare::~CuShare() {
    CuPool& p = g_cu_pools[dev_];
    std::lock_guard<std::mutex> lk(p.m);
    p.used -= blocks_;
    p.cv.notify_all();
}

void launch_resident_deps(int n, int rows, int grid, const int* rowptr, const int* col, int* deps, hipStream_t s) {
    hipLaunchKernelGGL(k_resident_deps, dim3(grid), dim3(kBlock), 0, s, n, rows, rowptr, col, deps);
}

// Launches `kernel` on `grid` blocks if the device holds `at_once` of them.
template <class K, class... Args>
static bool launch_resident_of(int at_once, K kernel, int grid, size_t lds, hipStream_t s, const Args&... args) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)kernel, kResThreads, lds) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (per_cu <= 0 || at_once > per_cu * cus) return false;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kResThreads), lds, s, args...);
    return true;
}
template <class K, class... Args>
static bool launch_resident(K kernel, int grid, size_t lds, hipStream_t s, const Args&... args) {
    return launch_resident_of(grid, kernel, grid, lds, s, args...);
}

template <typename Op, typename T>
bool launch_cg_stream(const Op& A, const ResidentArgs<T>& a, int grid, hipStream_t s) {
    const int R = (a.rows + kResThreads - 1) / kResThreads;
    const size_t lds = sizeof(T) * (size_t)((R + 1) / 2 * 2) * kResThreads;
    if (R <= 2) return launch_resident(k_cg_stream<Op, 2>, grid, lds, s, A, a);
    if (R <= 4) return launch_resident(k_cg_stream<Op, 4>, grid, lds, s, A, a);
    if (R <= 6) return launch_resident(k_cg_stream<Op, 6>, grid, lds, s, A, a);
    return launch_resident(k_cg_stream<Op, 8>, grid, lds, s, A, a);
}
template bool launch_cg_stream<Csr<double>, double>(const Csr<double>&, const ResidentArgs<double>&, int, hipStream_t);

// the kernel of the fewest rows per thread that hold R (even ones, the FP32
// ones above 8 by fours)
template <bool SHARED, int N, typename Op, typename T>
static bool launch_window(std::integral_constant<int, N>, int R, const Op& A, const ResidentArgs<T>& a,
                          const WindowShape& w, int grid, hipStream_t s) {
    if constexpr (N > resident_rows_per_thread<T>(!SHARED)) {
        return false;
    } else {
        if (R <= N) return launch_resident(k_cg_window<Op, SHARED, N, OpDiff<Op>::value>, grid, w.lds, s, A, a, w);
        return launch_window<SHARED>(std::integral_constant<int, window_kernel_rows(N + 1)>{}, R, A, a, w,
                                     grid, s);
    }
}

template <typename Op, typename T>
bool launch_cg_window(const Op& A, const ResidentArgs<T>& a, const WindowShape& w, int grid, hipStream_t s) {
    const int R = (a.rows + kResThreads - 1) / kResThreads;
    return A.soff ? launch_window<true>(std::integral_constant<int, 1>{}, R, A, a, w, grid, s)
                  : launch_window<false>(std::integral_constant<int, 1>{}, R, A, a, w, grid, s);
}
template <bool SHARED>
static bool launch_cgs(int R, const Sell<double>& A, const ResidentArgs<double>& a, const WindowShape& w,
                       const double* r2, double* q, double* u2, int grid, hipStream_t s) {
    if (R <= 2) return launch_resident(k_cgs_window<Sell<double>, SHARED, 2>, grid, w.lds, s, A, a, w, r2, q, u2);
    if (R <= kCgsRows) return launch_resident(k_cgs_window<Sell<double>, SHARED, 4>, grid, w.lds, s, A, a, w, r2, q, u2);
    return false;
}
bool launch_cgs_window(const Sell<double>& A, const ResidentArgs<double>& a, const WindowShape& w, const double* r2,
                       double* q, double* u2, int grid, hipStream_t s) {
    const int R = (a.rows + kResThreads - 1) / kResThreads;
    return A.soff ? launch_cgs<true>(R, A, a, w, r2, q, u2, grid, s) : launch_cgs<false>(R, A, a, w, r2, q, u2, grid, s);
}

template <int N>
static bool launch_batch(std::integral_constant<int, N>, int R, int grid, size_t lds, bool alone,
                         const ResidentSystem* sys, const int* blk_sys, uint32_t tag, hipStream_t s) {
    if constexpr (N > resident_rows_per_thread<double>(false)) {
        return false;
    } else {
        if (R <= N) return launch_resident_of(alone ? 1 : grid, k_cg_window_batch<N>, grid, lds, s, sys, blk_sys, tag);
        return launch_batch(std::integral_constant<int, window_kernel_rows(N + 1)>{}, R, grid, lds, alone, sys, blk_sys,
                            tag, s);
    }
}
size_t batch_window_lds(const ResidentSystem& s, int R) {
    const int K = window_kernel_rows(std::max(R, 2));
    return sizeof(double) * (2 * (size_t)s.w.lo + (size_t)s.w.nfar * s.a.rows +
                             (size_t)K * kResThreads * (window_d_in_lds<double>(K) ? 2 : 1));
}
bool launch_cg_window_batch(const ResidentSystem* sys, const int* blk_sys, int grid, int R, size_t lds, bool alone,
                            uint32_t tag, hipStream_t s) {
    return launch_batch(std::integral_constant<int, 2>{}, R, grid, lds, alone, sys, blk_sys, tag, s);
}

template bool launch_cg_window<Sell<double>, double>(const Sell<double>&, const ResidentArgs<double>&,
                                                     const WindowShape&, int, hipStream_t);
template bool launch_cg_window<DiffSell32, float>(const DiffSell32&, const ResidentArgs<float>&, const WindowShape&,
                                                  int, hipStream_t);

}  // namespace tflows
