// Local SpGEMM C = A*B on gfx950 (int32 CSR, fp64 values).
//
// Replaces LocalMatrix::spgemm / KokkosSparse::spgemm
// (include/KokkosWrap.hpp:367-391, call at :375).  Pipeline:
//
//  1. row analysis   flops_i = sum_{k in A_i} nnz(B_k), summed in equal units
//                    of entries by the pass that also checks the operands
//                    (k_check.hip); rows are binned by flops (empty / six
//                    light classes / short rows / two heavy classes).
//  2. symbolic       light rows (flops <= the tuned cut): one wave per row, LDS
//                    open-addressing hash of column keys; short rows eight to
//                    a wave;
//                    heavy rows: one 512- or 1024-thread block per row, a
//                    bitmap of 2^18, 2^19 or 2^20 columns in LDS (128 KiB of
//                    the 160 KiB at most), popcounted per 128-column fine
//                    block; the block packs fine blocks into column windows of
//                    at most H+127 entries and appends them to a device work
//                    list (heavy_items.h).
//  3. scan           row counts -> 64-bit row offsets; C is cut into int32
//                    tiles (panels) when it exceeds INT32_MAX entries.
//  4. numeric        light rows: all products of a row at once, sorted in
//                    registers by (column, position in A-order) and summed
//                    run by run; short rows of at most 32 entries eight to a
//                    wave, B row after B row;
//                    compact heavy rows (at most 128 entries): one wave per
//                    row, LDS hash of (key, fp64), compacted and sorted;
//                    heavy rows: one workgroup per item (a run of windows of
//                    one row) sharing one LDS table per window, products of
//                    the window flattened in A-order into groups of 64, which
//                    its waves prepare together and add in turn, lanes that
//                    share a column one after the other; sorted ranks from a
//                    presence bitmap.
//
// Every output entry therefore receives c = fma(a_ik, b_kj, c) in the order
// of A's stored entries, starting from +0.0: the results are bit-identical to
// the CPU oracle and do not depend on scheduling.
#include "dev_common.h"
#include "tr_internal.h"
#include "spgemm_types.h"

#include <algorithm>
#include <cstring>
#include <vector>


namespace tr {


namespace {

using namespace dev;

__device__ __forceinline__ int32_t lower_bound_dev(const TR_GLOBAL int32_t *__restrict__ a, int32_t lo, int32_t hi,
                                                   int32_t key) {
    while (lo < hi) {
        int32_t mid = lo + ((hi - lo) >> 1);
        if (a[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// first q in (lo, e] with a[q] >= key (q == e if none), galloping from lo,
// where a[lo] < key is known; vq receives a[q] (INT32_MAX when q == e), the
// column the next window of a heavy row starts from.  A round probes 2, 8 and
// 32 entries ahead with independent loads (then 128, 512, 2048, ...): the
// search is a fifth of the heavy numeric, bound by its slowest lane's round
// trips.  num_heavy of R-MAT s19: one probe a round, doubling 88.2 ms;
// quadrupling 86.0; two probes (1, 4 / 2, 8) 84.9 / 84.6; three 84.1; with a
// binary search of two probes a round 86.3.
__device__ __forceinline__ int32_t gallop_from(const TR_GLOBAL int32_t *__restrict__ a, int32_t lo, int32_t e,
                                               int32_t key, int32_t &vq) {
    int32_t step = 2, hi;
    vq = INT32_MAX;
    while (true) {
        const int32_t rem = e - lo;  // (distances, so that no position overflows)
        const int32_t v1 = step < rem ? a[lo + step] : INT32_MAX;
        const int32_t v2 = 4 * step < rem ? a[lo + 4 * step] : INT32_MAX;
        const int32_t v3 = 16 * step < rem ? a[lo + 16 * step] : INT32_MAX;
        if (v1 >= key) {
            vq = v1;
            hi = lo + min(step, rem);
            break;
        }
        if (v2 >= key) {
            vq = v2;
            hi = lo + min(4 * step, rem);
            lo += step;
            break;
        }
        if (v3 >= key) {
            vq = v3;
            hi = lo + min(16 * step, rem);
            lo += 4 * step;
            break;
        }
        lo += 16 * step;
        step <<= 6;
    }
    while (hi - lo > 1) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        const int32_t v = a[mid];
        if (v < key) {
            lo = mid;
        } else {
            hi = mid;
            vq = v;
        }
    }
    return hi;
}

// Visit the column indices of B row segment [s, e) with the wave's lanes,
// four loads in flight per lane before the first is consumed.
template <typename F>
__device__ __forceinline__ void stream_cols(const TR_GLOBAL int32_t *__restrict__ bi, int32_t s, int32_t e, F &&f) {
    int32_t q = s + lane_id();
    for (; q + 3 * kWave < e; q += 4 * kWave) {
        const int32_t j0 = bi[q], j1 = bi[q + kWave], j2 = bi[q + 2 * kWave], j3 = bi[q + 3 * kWave];
        f(j0);
        f(j1);
        f(j2);
        f(j3);
    }
    for (; q < e; q += kWave) f(bi[q]);
}

// Same visit with 16-byte loads for the aligned body of the segment (four
// columns per lane per load, four loads in flight), scalar head and tail.
// Alignment is taken from the address: caller tiles may place indices at any
// 4-byte offset.  Rows of up to 1024 columns, and the rest of longer ones, cost
// one round trip: head, tail and the last four groups per lane are loaded
// together (two to five trips before: the heavy symbolic of R-MAT s17 2245 ->
// 1896 us, Galerkin 96^3 445 -> 380 us).
template <typename F>
__device__ __forceinline__ void stream_cols_v4(const TR_GLOBAL int32_t *__restrict__ bi, int32_t s, int32_t e,
                                               F &&f) {
    const int l = lane_id();
    const int32_t mis = (int32_t)(((uintptr_t)(bi + s) >> 2) & 3);  // dwords past a 16-byte boundary
    const int32_t sa = min(e, s + ((4 - mis) & 3));                  // first 16-byte aligned index
    const int32_t nv = (e - sa) >> 2;                                // whole int4 groups
    typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
    const TR_GLOBAL i32x4 *__restrict__ b4 = (const TR_GLOBAL i32x4 *)(bi + sa);
    const int32_t ta = sa + (nv << 2);
    int32_t v = l;
    for (; v + 3 * kWave < nv; v += 4 * kWave) {
        const i32x4 x0 = b4[v], x1 = b4[v + kWave], x2 = b4[v + 2 * kWave], x3 = b4[v + 3 * kWave];
        f(x0.x), f(x0.y), f(x0.z), f(x0.w);
        f(x1.x), f(x1.y), f(x1.z), f(x1.w);
        f(x2.x), f(x2.y), f(x2.z), f(x2.w);
        f(x3.x), f(x3.y), f(x3.z), f(x3.w);
    }
    const bool p0 = v < nv, p1 = v + kWave < nv, p2 = v + 2 * kWave < nv, p3 = v + 3 * kWave < nv;
    const bool ph = s + l < sa, pt = ta + l < e;
    i32x4 x0 = {0, 0, 0, 0}, x1 = x0, x2 = x0, x3 = x0;
    int32_t xt = 0, xh = 0;
    if (ph) xh = bi[s + l];
    if (pt) xt = bi[ta + l];
    if (p0) x0 = b4[v];
    if (p1) x1 = b4[v + kWave];
    if (p2) x2 = b4[v + 2 * kWave];
    if (p3) x3 = b4[v + 3 * kWave];
    if (ph) f(xh);
    if (pt) f(xt);
    if (p0) f(x0.x), f(x0.y), f(x0.z), f(x0.w);
    if (p1) f(x1.x), f(x1.y), f(x1.z), f(x1.w);
    if (p2) f(x2.x), f(x2.y), f(x2.z), f(x2.w);
    if (p3) f(x3.x), f(x3.y), f(x3.z), f(x3.w);
}

// Same visit of the B rows of up to kShortB columns that the lanes in `rows`
// hold (first position, length), four rows at a time with 16 lanes each: a row
// by itself is a round trip that fills few lanes.  The order of the rows is
// free.  (One row at a time, then rows of up to 32, 64, 128, 192 columns by
// four, up to 256 by two: product of 15013 vertices 665, 628, 608, 590, 595,
// 608 us; R-MAT s17 10.60, 10.60, 10.54, 10.45, 10.43, 10.49 ms; Galerkin 96^3
// 2078, 2025, 2030, 2022, 2018, 2019 us.)
constexpr int kShortB = 128, kShortBLanes = 16;
template <typename F>
__device__ __forceinline__ void stream_short_rows(const TR_GLOBAL int32_t *__restrict__ bi, int32_t bs, int32_t len,
                                                  uint64_t rows, F &&f) {
    constexpr int kAtOnce = kWave / kShortBLanes, kLoads = kShortB / kShortBLanes;
    const int l = lane_id(), grp = l / kShortBLanes;
    while (rows) {
        int t = -1;
#pragma unroll
        for (int g = 0; g < kAtOnce; ++g) {
            if (rows) t = grp == g ? __ffsll((unsigned long long)rows) - 1 : t;
            rows &= rows - 1;
        }
        const int32_t s = __shfl(bs, t & (kWave - 1), kWave), all = __shfl(len, t & (kWave - 1), kWave);
        const int32_t n = t >= 0 ? all : 0;
        int32_t j[kLoads];
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int32_t e = q * kShortBLanes + l % kShortBLanes;
            if (e < n) j[q] = bi[s + e];
        }
#pragma unroll
        for (int q = 0; q < kLoads; ++q)
            if (q * kShortBLanes + l % kShortBLanes < n) f(j[q]);
    }
}

// Streaming of B rows with their loads one round trip ahead, for kernels
// whose LDS leaves registers to spare (the 2^20-bit heavy symbolic runs one
// 16-wave workgroup per CU): each row's first round trip (its unaligned head
// and tail and its first two 16-byte groups per lane)
// is issued while the previous row is applied, and a long row's next 1024
// columns while the current ones are.
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

struct RowHead {
    int32_t s, e, sa, nv, jh, jt;
    i32x4_t g0, g1;
};

// Loads below are issued unconditionally so that the compiler can keep the
// next round trip's loads in flight while it waits for the current ones (a
// branch around a load makes it wait for every load): a lane with nothing to
// read loads the aligned 16 bytes around an element known to exist (the
// row's first, or bi[0], which a heavy row's operand always has), which
// stays on a mapped page, and its value is dropped.
__device__ __forceinline__ const TR_GLOBAL i32x4_t *safe_block(const TR_GLOBAL int32_t *__restrict__ bi, int32_t s,
                                                             int32_t e) {
    return (const TR_GLOBAL i32x4_t *)((uintptr_t)(bi + (e > s ? s : 0)) & ~(uintptr_t)15);
}

__device__ __forceinline__ RowHead row_head_issue(const TR_GLOBAL int32_t *__restrict__ bi, int32_t s, int32_t e) {
    RowHead h;
    const int l = lane_id();
    const int32_t mis = (int32_t)(((uintptr_t)(bi + s) >> 2) & 3);
    h.s = s;
    h.e = e;
    h.sa = min(e, s + ((4 - mis) & 3));
    h.nv = (e - h.sa) >> 2;
    const int32_t ta = h.sa + (h.nv << 2);
    const TR_GLOBAL i32x4_t *__restrict__ b4 = (const TR_GLOBAL i32x4_t *)(bi + h.sa);
    const TR_GLOBAL i32x4_t *__restrict__ sb = safe_block(bi, s, e);
    const TR_GLOBAL int32_t *__restrict__ s1 = (const TR_GLOBAL int32_t *)sb;
    h.jh = *(s + l < h.sa ? bi + s + l : s1);
    h.jt = *(ta + l < e ? bi + ta + l : s1);
    h.g0 = *(l < h.nv ? b4 + l : sb);
    h.g1 = *(l + kWave < h.nv ? b4 + l + kWave : sb);
    return h;
}

template <typename F>
__device__ __forceinline__ void row_stream_apply(const TR_GLOBAL int32_t *__restrict__ bi, const RowHead &h, F &f) {
    const int l = lane_id();
    const int32_t ta = h.sa + (h.nv << 2);
    if (h.s + l < h.sa) f(h.jh);
    if (ta + l < h.e) f(h.jt);
    if (l < h.nv) f(h.g0.x), f(h.g0.y), f(h.g0.z), f(h.g0.w);
    if (l + kWave < h.nv) f(h.g1.x), f(h.g1.y), f(h.g1.z), f(h.g1.w);
    if (h.nv <= 2 * kWave) return;  // wave-uniform
    const TR_GLOBAL i32x4_t *__restrict__ b4 = (const TR_GLOBAL i32x4_t *)(bi + h.sa);
    const TR_GLOBAL i32x4_t *__restrict__ sb = safe_block(bi, h.s, h.e);
    i32x4_t c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int32_t v = 2 * kWave + k * kWave + l;
        c[k] = *(v < h.nv ? b4 + v : sb);
    }
    for (int32_t base = 2 * kWave; base < h.nv; base += 4 * kWave) {  // wave-uniform
        i32x4_t n[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int32_t v = base + 4 * kWave + k * kWave + l;
            n[k] = *(v < h.nv ? b4 + v : sb);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (base + k * kWave + l < h.nv) f(c[k].x), f(c[k].y), f(c[k].z), f(c[k].w);
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = n[k];
    }
}

// the nk rows [bs, be) held by lanes 0..nk-1, each streamed over the wave
template <typename F>
__device__ __forceinline__ void stream_rows_ahead(const TR_GLOBAL int32_t *__restrict__ bi, int32_t bs, int32_t be,
                                                  int nk, F &&f) {
    if (nk <= 0) return;
    RowHead cur = row_head_issue(bi, __shfl(bs, 0, kWave), __shfl(be, 0, kWave));
    for (int t = 0; t < nk; ++t) {
        RowHead nxt = cur;
        if (t + 1 < nk) nxt = row_head_issue(bi, __shfl(bs, t + 1, kWave), __shfl(be, t + 1, kWave));
        row_stream_apply(bi, cur, f);
        cur = nxt;
    }
}

// Same with the values (all entries of one B row have distinct columns, so
// the order in which one lane applies them does not matter).
template <typename F>
__device__ __forceinline__ void stream_entries(const TR_GLOBAL int32_t *__restrict__ bi,
                                               const TR_GLOBAL double *__restrict__ bv, int32_t s, int32_t e, F &&f) {
    int32_t q = s + lane_id();
    for (; q + kWave < e; q += 2 * kWave) {
        const int32_t j0 = bi[q], j1 = bi[q + kWave];
        const double b0 = bv[q], b1 = bv[q + kWave];
        f(j0, b0);
        f(j1, b1);
    }
    for (; q < e; q += kWave) f(bi[q], bv[q]);
}

// task owning global row g (largest t with row_base <= g)
__device__ __forceinline__ int task_of(const TaskDev *__restrict__ tasks, int nt, int32_t g) {
    int lo = 0, hi = nt - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tasks[mid].row_base <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ const Panel &find_panel(const Panel *__restrict__ panels, int np, int32_t row) {
    int lo = 0, hi = np - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (panels[mid].row_begin <= row) lo = mid;
        else hi = mid - 1;
    }
    return panels[lo];
}

// ---------------------------------------------------------------- analysis
// k_check.hip sums every row's multiplications; here a thread takes four global
// rows and puts them into their classes.  Class counters are aggregated in LDS
// so there is one global atomic per class per workgroup; they all meet in one
// cache line, so a workgroup takes 1024 rows (256: 77 us on 2^19 rows, now
// 23 us).
constexpr int kRowsPerBlock = 1024;
constexpr int kClassThreads = 256;

__global__ void k_zero_counters(Counters *__restrict__ cnt) {
    if (threadIdx.x < sizeof(Counters) / 4) ((int32_t *)cnt)[threadIdx.x] = 0;
}

// start of a plain product: its one task, from the kernel's argument, and the
// counters
__global__ void k_put_task(TaskDev *__restrict__ dst, const TaskDev t, Counters *__restrict__ cnt) {
    if (threadIdx.x < sizeof(Counters) / 4) ((int32_t *)cnt)[threadIdx.x] = 0;
    if (threadIdx.x == 0) *dst = t;
}

// light class of n: the smallest c with 2 n <= 64 << c
__device__ __forceinline__ int light_class(int64_t n) {
    int c = 0;
    while ((int64_t)(64 << c) < 2 * n) ++c;
    return c;
}

// Rows of up to 128 multiplications over many B rows of 2 to 10 entries (at
// least twice as many as entries in one; a Laplacian times a prolongator: 27 of
// 4.5): eight to a wave (k_num_short).  Few B rows meet in few columns, which
// suits the sorted classes (ER n = 200000, 8 of 8: 302 against 394 us), longer
// B rows would leave eight lanes several turns, emptier ones turns of nothing.
__device__ __forceinline__ bool is_short(int64_t f, int32_t len) {
    return f <= kShortMaxF && f >= 2 * (int64_t)len && f <= 10 * (int64_t)len && 2 * f <= (int64_t)len * len;
}

__global__ __launch_bounds__(kClassThreads) void k_classify(const TaskDev *__restrict__ tasks, int nt,
                                                            int32_t rows_total, const int64_t *__restrict__ flops,
                                                            int64_t *__restrict__ rownnz,
                                                            int32_t *__restrict__ lists, Counters *__restrict__ cnt,
                                                            int32_t light_max, int allow_short) {
    constexpr int kPer = kRowsPerBlock / kClassThreads;
    __shared__ int32_t s_cnt[kNumClasses], s_base[kNumClasses];
    __shared__ unsigned long long s_f, s_hf;
    const int tid = threadIdx.x, l = lane_id();
    const int32_t g0 = blockIdx.x * kRowsPerBlock + tid;
    if (tid < kNumClasses) s_cnt[tid] = 0;
    if (tid == 0) s_f = s_hf = 0ull;
    __syncthreads();
    int64_t f[kPer], sf = 0, shf = 0;
    int32_t len[kPer];  // A entries
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int32_t g = g0 + u * kClassThreads;
        f[u] = 0;
        len[u] = 0;
        if (g < rows_total) {
            const TaskDev &T = tasks[task_of(tasks, nt, g)];
            const int32_t *p = T.ap + (g - T.row_base);
            len[u] = p[1] - p[0];
            f[u] = flops[g];
            rownnz[g] = 0;
        }
    }
    int c[kPer], lpos[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        c[u] = -1;
        lpos[u] = 0;
        if (f[u] > 0) {
            if (f[u] <= light_max) {
                c[u] = allow_short && is_short(f[u], len[u]) ? kShortClass : light_class(f[u]);
            } else {
                c[u] = f[u] <= kMidMaxF ? kMidClass : kHeavyClass;
                shf += f[u];
            }
            lpos[u] = atomicAdd(&s_cnt[c[u]], 1);
            sf += f[u];
        }
    }
    const unsigned long long wf = (unsigned long long)wave_sum(sf);
    const unsigned long long whf = (unsigned long long)wave_sum(shf);
    if (l == 0) {
        atomicAdd(&s_f, wf);
        atomicAdd(&s_hf, whf);
    }
    __syncthreads();
    if (tid < kNumClasses && s_cnt[tid] > 0) s_base[tid] = atomicAdd(&cnt->cls[tid], s_cnt[tid]);
    if (tid == 0) {
        if (s_f) atomicAdd(&cnt->flops, s_f);
        if (s_hf) atomicAdd(&cnt->heavy_flops, s_hf);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (c[u] >= 0) lists[(int64_t)c[u] * rows_total + s_base[c[u]] + lpos[u]] = g0 + u * kClassThreads;
}

// ---------------------------------------------------------------- symbolic, light rows
// One wave per row, rows taken from the class list (grid-stride, count read
// on the device so the launch can be replayed from a graph).
template <int T>
__device__ __forceinline__ void sym_light_rows(int32_t *lds, int32_t block, int32_t blocks,
                                               const TaskDev *__restrict__ tasks, int nt,
                                               const int32_t *__restrict__ rows, const Counters *__restrict__ cnt,
                                               int cls, int64_t *__restrict__ rownnz) {
    constexpr uint32_t kLog = __builtin_ctz(T);
    // (marking the row wave-uniform here moves its values to scalar
    // registers, 101 SGPRs: 7 waves per SIMD instead of 8, and slower)
    const int w = threadIdx.x / kWave, l = lane_id();
    int32_t *tab = lds + w * T;
    const int32_t nrows = cnt->cls[cls];
    for (int32_t li = block * 4 + w; li < nrows; li += blocks * 4) {
        const int32_t g = rows[li];
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
        const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
        const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
        for (int t = l; t < T; t += kWave) tab[t] = kEmpty;
        wave_sync();
        const int32_t a0 = as_global(TK.ap)[r], a1 = as_global(TK.ap)[r + 1];
        int cntv = 0;
        auto insert = [&](int32_t j) {
            uint32_t h = hash_slot(j, kLog);
            for (int probe = 0; probe < T; ++probe) {
                const int32_t old = atomicCAS(&tab[h], kEmpty, j);
                if (old == kEmpty) {
                    ++cntv;
                    break;
                }
                if (old == j) break;
                h = (h + 1) & (T - 1);
            }
        };
        for (int32_t pb = a0; pb < a1; pb += kWave) {
            int32_t bs = 0, be = 0;
            if (pb + l < a1) {
                const int32_t k = ai[pb + l];
                bs = bp[k];
                be = bp[k + 1];
            }
            const int nk = min(kWave, a1 - pb);
            const int32_t len = be - bs;
            const int32_t inc = wave_incl_scan(len);
            const int32_t total = __shfl(inc, kWave - 1, kWave);
            if (total >= 32 * nk) {
                // long B rows: lanes stream one B row at a time
                for (int t = 0; t < nk; ++t) {
                    const int32_t s = __shfl(bs, t, kWave), e = __shfl(be, t, kWave);
                    stream_cols(bi, s, e, insert);
                }
            } else {
                // short B rows: the chunk's products flattened over the lanes
                // (counting distinct columns does not depend on the order);
                // product x belongs to the last lane whose prefix is <= x
                const int32_t excl = inc - len;
                for (int32_t x0 = 0; x0 < total; x0 += kWave) {
                    const int32_t x = x0 + l;
                    int t = 0;
#pragma unroll
                    for (int step = kWave / 2; step > 0; step >>= 1)
                        if (__shfl(excl, t + step, kWave) <= x) t += step;
                    const int32_t q = __shfl(bs, t, kWave) + (x - __shfl(excl, t, kWave));
                    if (x < total) insert(bi[q]);
                }
            }
        }
        cntv = wave_sum(cntv);
        if (l == 0) rownnz[g] = cntv;
        wave_sync();
    }
}

template <int T>
__global__ __launch_bounds__(256) void k_sym_light(const TaskDev *__restrict__ tasks, int nt,
                                                   const int32_t *__restrict__ rows, const Counters *__restrict__ cnt,
                                                   int cls, int64_t *__restrict__ rownnz) {
    __shared__ int32_t tabs[4 * T];
    sym_light_rows<T>(tabs, blockIdx.x, gridDim.x, tasks, nt, rows, cnt, cls, rownnz);
}

// Workgroups of the light classes in one launch: class c has [end[c + 1],
// end[c]), the longest rows first.
struct LightBlocks {
    int32_t end[kNumLight + 1];
};

// class of this workgroup (block-uniform)
__device__ __forceinline__ int light_block_class(const LightBlocks &lb) {
    int c = kNumLight - 1;
    while (c > 0 && (int32_t)blockIdx.x >= lb.end[c]) --c;
    return c;
}

// All light classes at once, where they are few rows (light_blocks); 32 KiB of
// LDS, five workgroups a CU
__global__ __launch_bounds__(256) void k_sym_light_all(const TaskDev *__restrict__ tasks, int nt,
                                                       const int32_t *__restrict__ lists, int32_t rows_total,
                                                       const Counters *__restrict__ cnt, const LightBlocks lb,
                                                       int64_t *__restrict__ rownnz) {
    __shared__ int32_t tabs[4 * 2048];
    const int c = light_block_class(lb);
    const int32_t block = (int32_t)blockIdx.x - lb.end[c + 1], blocks = lb.end[c] - lb.end[c + 1];
    const int32_t *rows = lists + (int64_t)c * rows_total;
    if (c == 5) sym_light_rows<2048>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
    else if (c == 4) sym_light_rows<1024>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
    else if (c == 3) sym_light_rows<512>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
    else if (c == 2) sym_light_rows<256>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
    else if (c == 1) sym_light_rows<128>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
    else sym_light_rows<64>(tabs, block, blocks, tasks, nt, rows, cnt, c, rownnz);
}

// ---------------------------------------------------------------- short rows
// Eight rows to a wave, eight lanes to a row: a row's A entries are taken in
// order, the lanes over one short B row at a time, into the row's own LDS table.
//
// What bounds it: vector instructions, about 35 per A entry for eight rows
// together.  With a wave per row and its products flattened over 64 lanes, the
// products that meet in a column (27 B rows over 17 columns) had to be put back
// in order afterwards: A*P of Galerkin 96^3 (885 k rows, 105 M products)
// 434 and 1150 us (symbolic, numeric), now 228 and 732 us.
constexpr int kShortLanes = 8;
constexpr int kShortRows = kWave / kShortLanes;  // rows per wave

// value of lane kLane of the calling lane's group of eight
template <int kLane>
__device__ __forceinline__ int32_t group_lane(int32_t v) {
    return __builtin_amdgcn_ds_swizzle(v, 0x18 | kLane << 5);
}
template <int kLane>
__device__ __forceinline__ double group_lane(double v) {
    return by_words(v, [](uint32_t u) { return (uint32_t)__builtin_amdgcn_ds_swizzle((int)u, 0x18 | kLane << 5); });
}

// A entries [pb, pb + 8) of a short row, one per lane of its group
struct ShortChunk {
    int32_t bs, len;
    double a;
};

// The first kShortLanes entries of the chunk's B rows, loaded together
template <bool kVals>
struct ShortB {
    int32_t s[kShortLanes], n[kShortLanes], j[kShortLanes];
    double b[kVals ? kShortLanes : 1];
};

template <bool kVals, int kLane = 0>
__device__ __forceinline__ void short_load(const ShortChunk &c, const TR_GLOBAL int32_t *__restrict__ bi,
                                           const TR_GLOBAL double *__restrict__ bv, int q, ShortB<kVals> &x) {
    x.s[kLane] = group_lane<kLane>(c.bs);
    x.n[kLane] = group_lane<kLane>(c.len);
    x.j[kLane] = 0;
    if (q < x.n[kLane]) {
        x.j[kLane] = bi[x.s[kLane] + q];
        if constexpr (kVals) x.b[kLane] = bv[x.s[kLane] + q];
    }
    if constexpr (kLane + 1 < kShortLanes) short_load<kVals, kLane + 1>(c, bi, bv, q, x);
}

// f(column, A value, B value) for every product of the chunk, B row after B
// row (the lanes of a group hold distinct columns of one B row)
template <bool kVals, int kLane = 0, typename F>
__device__ __forceinline__ void short_apply(const ShortChunk &c, const TR_GLOBAL int32_t *__restrict__ bi,
                                            const TR_GLOBAL double *__restrict__ bv, int q, const ShortB<kVals> &x,
                                            F &f) {
    double a = 0.0;
    if constexpr (kVals) a = group_lane<kLane>(c.a);
    if (q < x.n[kLane]) f(x.j[kLane], a, kVals ? x.b[kVals ? kLane : 0] : 0.0);
    for (int32_t o = q + kShortLanes; ballot(o < x.n[kLane]); o += kShortLanes)
        if (o < x.n[kLane]) f(bi[x.s[kLane] + o], a, kVals ? bv[x.s[kLane] + o] : 0.0);
    wave_sync();  // the next B row sees this one's entries
    if constexpr (kLane + 1 < kShortLanes) short_apply<kVals, kLane + 1>(c, bi, bv, q, x, f);
}

// all products of the row [a0, a1) of each group
template <bool kVals, typename F>
__device__ __forceinline__ void short_products(const TaskDev &TK, int32_t a0, int32_t a1, int q, F &&f) {
    const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
    const TR_GLOBAL double *__restrict__ av = as_global(TK.av);
    const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
    const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
    const TR_GLOBAL double *__restrict__ bv = as_global(TK.bv);
    for (int32_t pb = a0; ballot(pb < a1); pb += kShortLanes) {
        ShortChunk c{0, 0, 0.0};
        if (pb + q < a1) {
            const int32_t k = ai[pb + q];
            if constexpr (kVals) c.a = av[pb + q];
            c.bs = bp[k];
            c.len = bp[k + 1] - c.bs;
        }
        ShortB<kVals> x;
        short_load<kVals>(c, bi, bv, q, x);
        short_apply<kVals>(c, bi, bv, q, x, f);
    }
}

// slot of column j in the table (claimed, if it is new; then fresh), or -1
template <int T>
__device__ __forceinline__ int table_slot(int32_t *keys, int32_t j, bool &fresh) {
    uint32_t h = hash_slot(j, __builtin_ctz(T));
    for (int probe = 0; probe < T; ++probe) {
        const int32_t old = atomicCAS(&keys[h], kEmpty, j);
        if (old == kEmpty || old == j) {
            fresh = old == kEmpty;
            return (int)h;
        }
        h = (h + 1) & (T - 1);
    }
    return -1;
}

// Entries per row of the short class.  Rows of more entries than k_num_short's
// table takes are counted too, so that the numeric launches only what it needs.
__global__ __launch_bounds__(256) void k_sym_short(const TaskDev *__restrict__ tasks, int nt,
                                                   const int32_t *__restrict__ rows, Counters *__restrict__ cnt,
                                                   int64_t *__restrict__ rownnz) {
    constexpr int T = kShortMaxF;  // at most that many columns
    __shared__ __align__(16) int32_t keys_s[4][kShortRows][T];
    __shared__ int32_t sizes[2];
    const int w = threadIdx.x / kWave, l = lane_id(), grp = l / kShortLanes, q = l % kShortLanes;
    int32_t *keys = keys_s[w][grp];
    if (threadIdx.x < 2) sizes[threadIdx.x] = 0;
    __syncthreads();
    const int32_t nrows = cnt->cls[kShortClass];
    for (int32_t base = (blockIdx.x * 4 + w) * kShortRows; base < nrows; base += gridDim.x * 4 * kShortRows) {
        const bool valid = base + grp < nrows;
        const int32_t g = rows[valid ? base + grp : base];
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const int32_t a0 = as_global(TK.ap)[r], a1 = valid ? as_global(TK.ap)[r + 1] : a0;
        for (int t = q * 4; t < T; t += kShortLanes * 4)
            *reinterpret_cast<int4 *>(&keys[t]) = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
        wave_sync();
        int32_t n = 0;
        short_products<false>(TK, a0, a1, q, [&](int32_t j, double, double) {
            bool fresh = false;
            (void)table_slot<T>(keys, j, fresh);
            n += fresh ? 1 : 0;
        });
        n += lane_xor<1>(n);
        n += lane_xor<2>(n);
        n += lane_xor<4>(n);
        if (valid && q == 0) {
            rownnz[g] = n;
            atomicAdd(&sizes[n <= kShortMaxNnz ? 0 : 1], 1);
        }
        wave_sync();
    }
    __syncthreads();
    if (threadIdx.x < 2 && sizes[threadIdx.x]) atomicAdd(&cnt->short_rows[threadIdx.x], sizes[threadIdx.x]);
}

// Values of the short rows of at most kShortMaxNnz entries.
__global__ __launch_bounds__(256, 6) void k_num_short(const TaskDev *__restrict__ tasks, int nt,
                                                      const int32_t *__restrict__ rows, Counters *__restrict__ cnt,
                                                      const int64_t *__restrict__ rowptr,
                                                      const Panel *__restrict__ panels, int npanels) {
    constexpr int T = 2 * kShortMaxNnz;
    constexpr int kSlots = T / kShortLanes;  // table slots per lane
    constexpr int kOut = kSlots / 2;         // entries per lane
    __shared__ __align__(16) int32_t keys_s[4][kShortRows][T];
    __shared__ double vals_s[4][kShortRows][T];
    __shared__ uint16_t slot_s[4][kShortRows][T / 2];
    const int w = threadIdx.x / kWave, l = lane_id(), grp = l / kShortLanes, q = l % kShortLanes;
    int32_t *keys = keys_s[w][grp];
    double *vals = vals_s[w][grp];
    uint16_t *slots = slot_s[w][grp];
    const int32_t nrows = cnt->cls[kShortClass];
    for (int32_t base = (blockIdx.x * 4 + w) * kShortRows; base < nrows; base += gridDim.x * 4 * kShortRows) {
        const int32_t g = rows[base + grp < nrows ? base + grp : base];
        const int64_t rs = rowptr[g];
        const int32_t expect = (int32_t)(rowptr[g + 1] - rs);
        const bool valid = base + grp < nrows && expect <= T / 2;
        if (!ballot(valid)) continue;
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const int32_t a0 = as_global(TK.ap)[r], a1 = valid ? as_global(TK.ap)[r + 1] : a0;
        for (int t = q * 4; t < T; t += kShortLanes * 4)
            *reinterpret_cast<int4 *>(&keys[t]) = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
        wave_sync();
        short_products<true>(TK, a0, a1, q, [&](int32_t j, double a, double b) {
            bool fresh = false;
            const int h = table_slot<T>(keys, j, fresh);
            if (h >= 0) vals[h] = __fma_rn(a, b, fresh ? 0.0 : vals[h]);
        });
        // occupied slots to the front (keys, and the slots their values are in)
        int32_t k[kSlots];
#pragma unroll
        for (int u = 0; u < kSlots; ++u) k[u] = keys[u * kShortLanes + q];
        wave_sync();
        int n = 0;
#pragma unroll
        for (int u = 0; u < kSlots; ++u) {
            const uint32_t m = (uint32_t)(ballot(k[u] != kEmpty) >> (grp * kShortLanes)) & 0xffu;
            const int at = n + __popc(m & ((1u << q) - 1u));
            if (k[u] != kEmpty && at < T / 2) {
                keys[at] = k[u];
                slots[at] = (uint16_t)(u * kShortLanes + q);
            }
            n += __popc(m);
        }
        if (valid && q == 0 && n != expect) atomicOr(&cnt->overflow, 2);
        n = min(n, T / 2);
        wave_sync();
        // each lane's entries, ranked by the smaller columns of their row
        int32_t c[kOut], rank[kOut];
        double v[kOut];
#pragma unroll
        for (int i = 0; i < kOut; ++i) {
            const int e = q + i * kShortLanes;
            c[i] = INT32_MAX;
            v[i] = 0.0;
            rank[i] = 0;
            if (valid && e < n) {
                c[i] = keys[e];
                v[i] = vals[slots[e]];
            }
        }
        for (int x = 0; ballot(valid && x < n); ++x) {
            const int32_t o = x < n ? keys[x] : INT32_MAX;
#pragma unroll
            for (int i = 0; i < kOut; ++i) rank[i] += o < c[i] ? 1 : 0;
        }
        const Panel &PN = find_panel(panels, npanels, g);
        TR_GLOBAL int32_t *oi = as_global(PN.idx) + (rs - PN.nnz_begin);
        TR_GLOBAL double *ov = as_global(PN.val) + (rs - PN.nnz_begin);
#pragma unroll
        for (int i = 0; i < kOut; ++i)
            if (valid && q + i * kShortLanes < n && rank[i] < expect) {
                oi[rank[i]] = c[i];
                ov[rank[i]] = v[i];
            }
        wave_sync();
    }
}

// LDS word of presence-bitmap word wd: with kSwz, its bank bits (the low
// five) XORed with the next two groups of five, a bijection on each aligned
// group of 32 words (clearing whole groups clears every word in use)
template <bool kSwz>
__device__ __forceinline__ int32_t bm_word(int32_t wd) {
    return kSwz ? wd ^ (((wd >> 5) ^ (wd >> 10)) & 31) : wd;
}

// ---------------------------------------------------------------- symbolic, heavy rows
// One NTH-thread block per row (grid-stride over the heavy list): a bitmap
// of 2^PB columns in LDS per pass, popcounts per 128-column fine block, and
// the row's column windows (<= win_h + 127 entries, <= kWinMaxWidth columns)
// appended to the device work lists.
template <int PB, int NTH>
// Narrow bitmaps (2^18 bits on 512 threads, 2^19 on 1024) leave LDS for 32
// waves per CU; the register budget is held to that too (64 VGPRs and a
// few spilled bytes per lane): Galerkin 128^3 12.5 -> 12.0 ms, R-MAT s19
// (2^19 columns) 17.8 -> 15.0 ms.
__global__ __launch_bounds__(NTH, (PB <= 18 || (PB == 19 && NTH == 1024)) ? 8 : 1) void k_sym_heavy(
    const TaskDev *__restrict__ tasks, int nt, Counters *__restrict__ cnt, int cls, int cls2,
    int64_t *__restrict__ rownnz, int emit, int32_t win_h, int32_t item_windows, int64_t item_flops,
    const int64_t *__restrict__ flops, Window *__restrict__ wins,
    int32_t win_cap, Item *__restrict__ items, int32_t item_cap, int32_t *__restrict__ lists, int32_t rows_total) {
    constexpr int kWords = 1 << (PB - 5);          // bitmap words of one pass
    constexpr int kFine = 1 << (PB - kFineShift);  // fine blocks of one pass
    constexpr int kPerThread = kFine / NTH;        // consecutive fine blocks per thread: 2..8
    constexpr int kWavesB = NTH / kWave;
    static_assert(kPerThread >= 1 && kPerThread <= 8 && (kPerThread & (kPerThread - 1)) == 0, "fine blocks per thread");
    // B rows are streamed with eager loads where the bitmap's LDS already
    // limits the kernel to four waves per SIMD (2^20 bits), so the extra
    // registers cost no occupancy
    constexpr bool kEagerB = PB == 20 || (PB == 19 && NTH == 512);
    // R-MAT column bits are mostly 0, so a quarter of the marks would share a
    // bank; the 2^20-bit kernel XORs the word's bank bits with higher ones
    // (R-MAT s20: 34.8 -> 33.2 ms).  In the 64-VGPR kernels the extra work
    // costs more than it saves (2^19 bits: 16.0 -> 18.4 ms).
    constexpr bool kSwizzle = PB == 20;
    static_assert(kWords % 32 == 0, "the bitmap holds whole 32-word swizzle groups");
    __shared__ __align__(16) uint32_t bm[kWords];
    __shared__ int32_t wsum[kWavesB];
    __shared__ int32_t sh_wbase;

    const int tid = threadIdx.x, w = tid / kWave, l = lane_id();
    int32_t *fex_lds = (int32_t *)bm;            // [0, kFine) after marking
    int32_t *first_lds = (int32_t *)bm + kFine;  // [kFine, 2 kFine)
    // rows of class cls, then those of class cls2 (the same class: none)
    const int32_t nfirst = cnt->cls[cls];
    const int32_t nheavy = nfirst + (cls2 != cls ? cnt->cls[cls2] : 0);
    for (int32_t hi = blockIdx.x; hi < nheavy; hi += gridDim.x) {
        const int32_t g = hi < nfirst ? lists[(int64_t)cls * rows_total + hi]
                                      : lists[(int64_t)cls2 * rows_total + (hi - nfirst)];
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
        const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
        const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
        const int32_t ncols = TK.n;
        const int32_t a0 = as_global(TK.ap)[r], a1 = as_global(TK.ap)[r + 1];
        int32_t row_total = 0;
        for (int64_t base = 0; base < ncols; base += (1 << PB)) {
            const int32_t width = (int32_t)min<int64_t>(1 << PB, (int64_t)ncols - base);
            const int32_t nwords = (width + 31) >> 5;
            const int32_t nfine = (width + (1 << kFineShift) - 1) >> kFineShift;
            // only the pass's words are marked and counted (a narrow matrix
            // leaves the rest of the bitmap unused)
            for (int t = tid; t < (kSwizzle ? ((nwords + 31) & ~31) : ((nwords + 3) & ~3)); t += NTH) bm[t] = 0u;
            __syncthreads();
            // mark: entry pb + w + 16 t goes to wave w
            for (int32_t pb = a0; pb < a1; pb += kWavesB * kWave) {
                int32_t bs = 0, be = 0;
                const int32_t p = pb + w + kWavesB * l;
                if (p < a1) {
                    const int32_t k = ai[p];
                    bs = bp[k];
                    be = bp[k + 1];
                }
                const int32_t rem = a1 - (pb + w);
                const int nk = rem <= 0 ? 0 : min(kWave, (rem + kWavesB - 1) / kWavesB);
                auto mark = [&](int32_t j) {
                    const uint32_t jj = (uint32_t)j - (uint32_t)base;  // (wraps for columns of earlier passes)
                    if (jj < (uint32_t)width) atomicOr(&bm[bm_word<kSwizzle>((int32_t)(jj >> 5))], 1u << (jj & 31));
                };
                if constexpr (kEagerB) {
                    stream_rows_ahead(bi, bs, be, nk, mark);
                } else {
                    const int32_t len = be - bs;
                    stream_short_rows(bi, bs, len, ballot(len > 0 && len <= kShortB), mark);
                    for (uint64_t rows = ballot(len > kShortB); rows; rows &= rows - 1) {
                        const int t = __ffsll((unsigned long long)rows) - 1;
                        stream_cols_v4(bi, read_lane(bs, t), read_lane(be, t), mark);
                    }
                }
            }
            __syncthreads();
            // fine-block counts, kPerThread consecutive fine blocks per thread.
            // A fine block's four words are one 16-byte read (the swizzle
            // keeps them in their aligned 16 bytes), and read k of lane l
            // takes block (k + l / (8 / kPerThread)) mod kPerThread: eight
            // consecutive lanes then read eight different 16-byte bank groups
            // (in order, lanes kPerThread blocks apart would share one or two:
            // a 32- or 64-way conflict on every read)
            int32_t c[kPerThread];
            int32_t tsum = 0;
#pragma unroll
            for (int u = 0; u < kPerThread; ++u) c[u] = 0;
#pragma unroll
            for (int k = 0; k < kPerThread; ++k) {
                const int u = (k + l / (8 / kPerThread)) & (kPerThread - 1);
                const int f = tid * kPerThread + u;
                int32_t v = 0;
                if (f < nfine) {
                    const uint4 x = *reinterpret_cast<const uint4 *>(&bm[bm_word<kSwizzle>(f * 4) & ~3]);
                    v = __popc(x.x) + __popc(x.y) + __popc(x.z) + __popc(x.w);
                }
#pragma unroll
                for (int uu = 0; uu < kPerThread; ++uu) c[uu] = uu == u ? v : c[uu];
                tsum += v;
            }
            const int32_t inc = wave_incl_scan(tsum);
            if (l == kWave - 1) wsum[w] = inc;
            __syncthreads();
            int32_t off = 0, pass_total = 0;
            for (int v = 0; v < kWavesB; ++v) {
                if (v < w) off += wsum[v];
                pass_total += wsum[v];
            }
            int32_t fex[kPerThread];
            {
                int32_t run = off + inc - tsum;
#pragma unroll
                for (int u = 0; u < kPerThread; ++u) {
                    fex[u] = run;
                    run += c[u];
                }
            }
            if (pass_total == 0 || !emit) {
                row_total += pass_total;
                __syncthreads();
                continue;
            }
            // A row done in one pass whose product has few entries (many
            // multiplications per entry: the coarse Galerkin product has about
            // 55) goes to the hashed light numeric, whose small table and
            // lane-mask ordering suit it, instead of to windows: appended to
            // the compact class whose table holds twice its entries.
            if (ncols <= (1 << PB) && pass_total <= kCompactMax) {
                if (tid == 0) {
                    const int c = kCompactClass + (pass_total <= 32 ? 0 : pass_total <= 64 ? 1 : 2);
                    const int32_t pos = atomicAdd(&cnt->cls[c], 1);
                    lists[(int64_t)c * rows_total + pos] = g;
                }
                row_total += pass_total;
                __syncthreads();
                continue;
            }
            // 16-byte writes: a thread's offsets are consecutive words
            if constexpr (kPerThread % 4 == 0) {
#pragma unroll
                for (int u = 0; u < kPerThread; u += 4)
                    *reinterpret_cast<int4 *>(&fex_lds[tid * kPerThread + u]) =
                        make_int4(fex[u], fex[u + 1], fex[u + 2], fex[u + 3]);
            } else {
#pragma unroll
                for (int u = 0; u < kPerThread; ++u) fex_lds[tid * kPerThread + u] = fex[u];
            }
            __syncthreads();
            // window starts: a count quantum or a width quantum begins.  A
            // sparse pass (few entries per width quantum) is cut by a smaller
            // count quantum only; its windows may be as wide as the pass and
            // are ranked without a bitmap by the numeric kernel.
            const bool sparse_pass = (int64_t)pass_total * (1 << kWidthShift) <= (int64_t)kSparseAvg * nfine;
            const int32_t q = sparse_pass ? kSparseH : win_h;
            int flags = 0, nflag = 0;
#pragma unroll
            for (int u = 0; u < kPerThread; ++u) {
                const int f = tid * kPerThread + u;
                bool first = false;
                // the previous block's offset is this thread's, except for its first block
                const int32_t prev = u == 0 ? (f > 0 ? fex_lds[f - 1] : 0) : fex[u - 1];
                if (f < nfine)
                    first = (f == 0) || (fex[u] / q != prev / q) ||
                            (!sparse_pass && ((f >> kWidthShift) != ((f - 1) >> kWidthShift)));
                if (first) {
                    flags |= 1 << u;
                    ++nflag;
                }
            }
            const int32_t finc = wave_incl_scan(nflag);
            __syncthreads();
            if (l == kWave - 1) wsum[w] = finc;
            __syncthreads();
            int32_t foff = 0, nwin = 0;
            for (int v = 0; v < kWavesB; ++v) {
                if (v < w) foff += wsum[v];
                nwin += wsum[v];
            }
            int32_t rk = foff + finc - nflag;
#pragma unroll
            for (int u = 0; u < kPerThread; ++u)
                if (flags & (1 << u)) first_lds[rk++] = tid * kPerThread + u;
            const int32_t iw = heavy_item_windows(item_windows, a1 - a0, item_flops, flops[g], heavy_passes(ncols, PB), nwin);
            if (tid == 0) {
                const int32_t nitems = (nwin + iw - 1) / iw;
                const int32_t wb = atomicAdd(&cnt->windows, nwin);
                const int32_t ib = atomicAdd(&cnt->items, nitems);
                if (wb + nwin > win_cap || ib + nitems > item_cap) {
                    atomicOr(&cnt->overflow, 1);
                    // taken back, so that refused rows, however many, never
                    // carry a count past 2^31 (an overflowed list is not read)
                    atomicSub(&cnt->windows, nwin);
                    atomicSub(&cnt->items, nitems);
                    sh_wbase = -1;
                } else {
                    sh_wbase = wb;
                    for (int32_t it = 0; it < nitems; ++it) {
                        Item I;
                        I.row = g;
                        I.wbeg = wb + it * iw;
                        I.wend = min(wb + nwin, I.wbeg + iw);
                        I.pad = 0;
                        items[ib + it] = I;
                    }
                }
            }
            __syncthreads();
            const int32_t wbase = sh_wbase;
            if (wbase >= 0) {
                for (int32_t rr = tid; rr < nwin; rr += NTH) {
                    const int32_t f = first_lds[rr];
                    const int32_t fn = (rr + 1 < nwin) ? first_lds[rr + 1] : nfine;
                    Window W;
                    W.c0 = (int32_t)(base + ((int64_t)f << kFineShift));
                    W.c1 = (int32_t)min<int64_t>(base + ((int64_t)fn << kFineShift), base + width);
                    W.off = row_total + fex_lds[f];
                    W.cnt = (fn < nfine ? fex_lds[fn] : pass_total) - fex_lds[f];
                    wins[wbase + rr] = W;
                }
            }
            row_total += pass_total;
            __syncthreads();
        }
        if (tid == 0) rownnz[g] = row_total;
        __syncthreads();
    }
}

// Items of the work list.  A list that would not fit (a batch's replay on
// operands with another sparsity pattern than the planned one) holds none:
// refused rows leave gaps that were never written, and rows that came while
// another was refused may lie over each other.
__device__ __forceinline__ int32_t listed_items(const Counters *__restrict__ cnt) {
    return (cnt->overflow & 1) ? 0 : cnt->items;
}

// per item: cursor slots it needs (multi-window items of rows longer than
// reg_max entries; shorter rows keep their cursors in registers)
__global__ void k_item_cursor_len(const Item *__restrict__ items, const Counters *__restrict__ cnt,
                                  const TaskDev *__restrict__ tasks, int nt, int32_t cap, int32_t reg_max,
                                  int32_t *__restrict__ len) {
    const int32_t it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= cap) return;
    int32_t v = 0;
    if (it < listed_items(cnt)) {
        const Item I = items[it];
        if (I.wend - I.wbeg > 1) {
            const TaskDev &TK = tasks[task_of(tasks, nt, I.row)];
            const int32_t r = I.row - TK.row_base;
            v = as_global(TK.ap)[r + 1] - as_global(TK.ap)[r];
            if (v <= reg_max) v = 0;
        }
    }
    len[it] = v;
}

// ---------------------------------------------------------------- heavy item order
// Heavy items are processed in the column order of their first window, so
// the workgroups resident at one time work in one column region of B and
// share its lines through L2 (the items of one row still run left to right
// within their item).  Counting sort by column bucket: a block-aggregated
// histogram, a scan, and a scatter with block-local ranks.
// bucket = first window's c0 >> shift; the host picks the smallest shift
// that maps the widest operand onto the buckets
constexpr int kOrderBuckets = 4096;

__global__ void k_fill_u64(unsigned long long *__restrict__ p, int32_t n) {
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0ull;
}

__device__ __forceinline__ int item_bucket(const Item *__restrict__ items, const Window *__restrict__ wins,
                                           int32_t it, int shift) {
    const int32_t c0 = wins[items[it].wbeg].c0;
    return min(c0 >> shift, kOrderBuckets - 1);
}

__global__ __launch_bounds__(256) void k_item_hist(const Item *__restrict__ items, const Window *__restrict__ wins,
                                                   const Counters *__restrict__ cnt, int shift,
                                                   unsigned long long *__restrict__ hist) {
    __shared__ int32_t h[kOrderBuckets];
    for (int t = threadIdx.x; t < kOrderBuckets; t += 256) h[t] = 0;
    __syncthreads();
    const int32_t n = listed_items(cnt);
    for (int32_t it = blockIdx.x * 256 + threadIdx.x; it < n; it += gridDim.x * 256)
        atomicAdd(&h[item_bucket(items, wins, it, shift)], 1);
    __syncthreads();
    for (int t = threadIdx.x; t < kOrderBuckets; t += 256)
        if (h[t]) atomicAdd(&hist[t], (unsigned long long)h[t]);
}

// hist[0..kOrderBuckets) -> exclusive offsets, in place (one block)
__global__ __launch_bounds__(1024) void k_item_hist_scan(unsigned long long *__restrict__ hist) {
    __shared__ unsigned long long part[1024 / kWave];
    constexpr int kPer = kOrderBuckets / 1024;
    const int tid = threadIdx.x, w = tid / kWave, l = lane_id();
    unsigned long long v[kPer], sum = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        v[u] = hist[tid * kPer + u];
        sum += v[u];
    }
    const unsigned long long inc = wave_incl_scan(sum);
    if (l == kWave - 1) part[w] = inc;
    __syncthreads();
    unsigned long long off = 0;
    for (int u = 0; u < w; ++u) off += part[u];
    unsigned long long run = off + inc - sum;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        hist[tid * kPer + u] = run;
        run += v[u];
    }
}

// The same grid walk as k_item_hist: block-local ranks per bucket, one
// global cursor bump per (block, bucket)
__global__ __launch_bounds__(256) void k_item_scatter(const Item *__restrict__ items, const Window *__restrict__ wins,
                                                      const Counters *__restrict__ cnt, int shift,
                                                      unsigned long long *__restrict__ cursor,
                                                      int32_t *__restrict__ order) {
    __shared__ int32_t h[kOrderBuckets];
    __shared__ unsigned long long base[kOrderBuckets];
    const int32_t n = listed_items(cnt);
    for (int32_t it0 = blockIdx.x * 256; it0 < n; it0 += gridDim.x * 256) {
        for (int t = threadIdx.x; t < kOrderBuckets; t += 256) h[t] = 0;
        __syncthreads();
        const int32_t it = it0 + threadIdx.x;
        int b = 0, r = 0;
        if (it < n) {
            b = item_bucket(items, wins, it, shift);
            r = atomicAdd(&h[b], 1);
        }
        __syncthreads();
        for (int t = threadIdx.x; t < kOrderBuckets; t += 256)
            if (h[t]) base[t] = atomicAdd(&cursor[t], (unsigned long long)h[t]);
        __syncthreads();
        if (it < n) order[base[b] + r] = it;
        __syncthreads();
    }
}

// int32 row pointers of the tile that holds global rows [r0, r0 + n], rebased,
// and its entry of the panel table
__global__ void k_tile_ptr(const int64_t *__restrict__ rowptr, int32_t r0, int32_t n, int32_t *__restrict__ ptr,
                           const Panel panel, Panel *__restrict__ dst) {
    const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) *dst = panel;
    if (t <= n) ptr[t] = (int32_t)(rowptr[r0 + t] - rowptr[r0]);
}

// ---------------------------------------------------------------- numeric, compact rows
// Rows of many multiplications over at most 128 columns (found by the heavy
// symbolic): one wave per row with a hash table of at least twice its entries.
constexpr int kLightPre = 4;  // B rows prefetched together per batch of a row

template <int T, int WPB>
// The tables leave LDS for 8 waves per SIMD; the registers are held to that
// too (63 VGPRs, 12 spilled bytes per lane; about 1% on Galerkin 128^3 against
// 65 VGPRs and 7 waves).
__global__ __launch_bounds__(WPB * kWave, 8) void k_num_light(const TaskDev *__restrict__ tasks, int nt,
                                                           const int32_t *__restrict__ rows,
                                                           Counters *__restrict__ cnt, int cls,
                                                           const int64_t *__restrict__ rowptr,
                                                           const Panel *__restrict__ panels, int npanels) {
    // chunks of short B rows are flattened over the lanes; a lane mask per slot
    // orders the chunk's products
    static_assert(T <= 256, "lane masks of larger tables would cost occupancy");
    __shared__ int32_t keys_s[WPB][T];
    __shared__ double vals_s[WPB][T];
    __shared__ unsigned long long own_s[WPB][T];
    constexpr uint32_t kLog = __builtin_ctz(T);
    // the wave index and everything per row are wave-uniform (scalar loads
    // and registers)
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), l = lane_id();
    int32_t *keys = keys_s[w];
    double *vals = vals_s[w];
    unsigned long long *own = own_s[w];
    for (int t = l; t < T; t += kWave) own[t] = 0ull;
    const int32_t nrows = cnt->cls[cls];
    const int32_t stride = gridDim.x * WPB;
    int32_t g_next = 0;
    if (blockIdx.x * WPB + w < nrows) g_next = rows[blockIdx.x * WPB + w];
    for (int32_t li = blockIdx.x * WPB + w; li < nrows; li += stride) {
        // a row is a chain of dependent loads (row, A entries, B row
        // pointers, B entries); the next row's index and this row's output
        // place are loaded early so that their latency overlaps the chain
        const int32_t g = __builtin_amdgcn_readfirstlane(g_next);
        if (li + stride < nrows) g_next = rows[li + stride];
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
        const TR_GLOBAL double *__restrict__ av = as_global(TK.av);
        const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
        const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
        const TR_GLOBAL double *__restrict__ bv = as_global(TK.bv);
        const int32_t a0 = as_global(TK.ap)[r], a1 = as_global(TK.ap)[r + 1];
        const int64_t rs = rowptr[g];
        const int64_t re = rowptr[g + 1];
        const Panel P = find_panel(panels, npanels, g);
        for (int t = l; t < T; t += kWave) keys[t] = kEmpty;
        wave_sync();
        for (int32_t pb = a0; pb < a1; pb += kWave) {
            int32_t bs = 0, be = 0;
            double a = 0.0;
            if (pb + l < a1) {
                const int32_t k = ai[pb + l];
                a = av[pb + l];
                bs = bp[k];
                be = bp[k + 1];
            }
            const int nk = min(kWave, a1 - pb);
            const int32_t len = be - bs;
            const int32_t inc = wave_incl_scan(len);
            const int32_t total = __shfl(inc, kWave - 1, kWave);
            if (total < 24 * nk) {
                // Short B rows: 64 products of the chunk per round, flattened
                // in A-order over the lanes (product x belongs to the last
                // lane whose prefix is <= x).  Products that meet in a slot
                // are applied in lane (= A) order: each pass, the lowest
                // pending lane of every slot applies its product.
                const int32_t excl = inc - len;
                for (int32_t x0 = 0; x0 < total; x0 += kWave) {
                    const int32_t x = x0 + l;
                    int t = 0;
                    int32_t q;
                    if constexpr (T >= 2 * kWave) {
                        // The lanes whose B rows meet this round write (lane,
                        // B offset) at the position where their rows start in
                        // it (or 0) and mark it in a start mask; position x
                        // belongs to the highest start at or below it.  The
                        // first 65 lane-mask words, all zero between rounds,
                        // hold both and are cleared again before the round
                        // uses them.  Three round trips instead of the six
                        // dependent shuffles of a search over the lanes.
                        const bool meets = len > 0 && excl < x0 + kWave && excl + len > x0;
                        const int32_t pos = max(excl - x0, 0);
                        if (meets) {
                            own[pos] = ((unsigned long long)(uint32_t)l << 32) | (uint32_t)(bs - excl);
                            atomicOr(&own[kWave], 1ull << pos);
                        }
                        wave_sync();
                        const unsigned long long starts = own[kWave] & (~0ull >> (63 - l));
                        const unsigned long long e = own[63 - __clzll((long long)starts)];
                        t = (int)(e >> 32);
                        q = (int32_t)(uint32_t)e + x;
                        wave_sync();
                        own[l] = 0ull;
                        if (l == 0) own[kWave] = 0ull;
                        wave_sync();
                    } else {
#pragma unroll
                        for (int step = kWave / 2; step > 0; step >>= 1)
                            if (__shfl(excl, t + step, kWave) <= x) t += step;
                        q = __shfl(bs, t, kWave) + (x - __shfl(excl, t, kWave));
                    }
                    const double at = __shfl(a, t, kWave);
                    bool pend = x < total;
                    uint32_t h = 0;
                    double b = 0.0;
                    if (pend) {
                        const int32_t j = bi[q];
                        b = bv[q];
                        h = hash_slot(j, kLog);
                        bool placed = false;
                        for (int probe = 0; probe < T; ++probe) {
                            const int32_t old = atomicCAS(&keys[h], kEmpty, j);
                            if (old == kEmpty) {
                                vals[h] = 0.0;
                                placed = true;
                                break;
                            }
                            if (old == j) {
                                placed = true;
                                break;
                            }
                            h = (h + 1) & (T - 1);
                        }
                        if (!placed) {
                            atomicOr(&cnt->overflow, 2);  // table full: symbolic counts were wrong
                            pend = false;
                        }
                    }
                    wave_sync();
                    // each slot's lanes as a mask; its lowest lane
                    // applies them all in lane order, fetching the
                    // other lanes' operands across the wave
                    if (pend) atomicOr(&own[h], 1ull << l);
                    wave_sync();
                    unsigned long long rem = 0ull;
                    double v = 0.0;
                    if (pend) {
                        const unsigned long long m = own[h];
                        if (__ffsll(m) - 1 == l) {
                            rem = m;
                            v = vals[h];
                        }
                    }
                    while (ballot(rem != 0ull)) {  // every lane takes part in the fetches
                        const int t = rem ? __ffsll(rem) - 1 : l;
                        const double ta = __shfl(at, t, kWave);
                        const double tb = __shfl(b, t, kWave);
                        if (rem) {
                            v = __fma_rn(ta, tb, v);
                            rem &= rem - 1ull;
                        }
                    }
                    wave_sync();
                    if (pend && (__ffsll(own[h]) - 1 == l)) {
                        vals[h] = v;
                        own[h] = 0ull;
                    }
                    wave_sync();
                }
                continue;
            }
            auto ins = [&](int32_t j, double b, double at) {
                uint32_t h = hash_slot(j, kLog);
                for (int probe = 0; probe < T; ++probe) {
                    const int32_t old = atomicCAS(&keys[h], kEmpty, j);
                    if (old == kEmpty) {
                        vals[h] = __fma_rn(at, b, 0.0);
                        break;
                    }
                    if (old == j) {
                        vals[h] = __fma_rn(at, b, vals[h]);
                        break;
                    }
                    h = (h + 1) & (T - 1);
                }
            };
            // the first 64 entries of the first kLightPre B rows are loaded
            // together (one round trip instead of one per row), then applied
            // row by row in A-order
            int32_t pj[kLightPre];
            double pv[kLightPre];
#pragma unroll
            for (int t = 0; t < kLightPre; ++t) {
                pj[t] = 0;
                pv[t] = 0.0;
                const int32_t s = __shfl(bs, t, kWave), e = __shfl(be, t, kWave);
                if (t < nk && s + l < e) {
                    pj[t] = bi[s + l];
                    pv[t] = bv[s + l];
                }
            }
#pragma unroll
            for (int t = 0; t < kLightPre; ++t) {
                if (t < nk) {
                    const int32_t s = __shfl(bs, t, kWave), e = __shfl(be, t, kWave);
                    const double at = __shfl(a, t, kWave);
                    if (s + l < e) ins(pj[t], pv[t], at);
                    stream_entries(bi, bv, s + kWave, e, [&](int32_t j, double b) { ins(j, b, at); });
                }
            }
            for (int t = kLightPre; t < nk; ++t) {
                const int32_t s = __shfl(bs, t, kWave), e = __shfl(be, t, kWave);
                const double at = __shfl(a, t, kWave);
                stream_entries(bi, bv, s, e, [&](int32_t j, double b) { ins(j, b, at); });
            }
        }
        wave_sync();
        const int n = wave_compact_lds<double>(keys, vals, T);
        wave_sort_lds<double>(keys, vals, n);
        const int expect = (int)(re - rs);
        if (l == 0 && n != expect) atomicOr(&cnt->overflow, 2);
        const int nw = n < expect ? n : expect;  // never write past the row
        TR_GLOBAL int32_t *oi = as_global(P.idx) + (rs - P.nnz_begin);
        TR_GLOBAL double *ov = as_global(P.val) + (rs - P.nnz_begin);
        for (int t = l; t < nw; t += kWave) {
            oi[t] = keys[t];
            ov[t] = vals[t];
        }
        wave_sync();
    }
}

// ---------------------------------------------------------------- numeric, light rows by sorting
// Rows of up to 1024 multiplications that did not come from the heavy symbolic:
// all products of a row at once, P per thread (one wave a row with P = 1, 2 or 4
// products, or 128 or 256 threads with 4).  The products are flattened in A-order, sorted in registers by
// (column, position), and every column's run is summed in position (= A) order
// by the thread that holds its first product; the runs in order are the sorted
// output.
//
// What bounds it: the sort, about 3.5 vector instructions per product and step
// (strides inside a thread are minimum and maximum, inside a wave DPP moves and
// permlane swaps; only strides of a wave and more go through LDS).  The hash
// tables that these rows had held one wave to 12 or 24 KiB of LDS (6 to 13 waves
// per CU), walked A's entries one after the other and sorted the table in LDS:
// stage of R-MAT s18 2671 us for the three classes, now 481 us (22 KiB for a row
// of 256 threads: 28 waves per CU); tile accumulate of R-MAT s16 154 -> 33 us.
constexpr int kSortIdBits = 10;    // product positions < 1024

template <typename K>
__device__ __forceinline__ void order_pair(K &a, K &b, bool up) {
    const K lo = a < b ? a : b, hi = a < b ? b : a;
    a = up ? lo : hi;
    b = up ? hi : lo;
}

// One step of the bitonic sort of NT * P keys, key u of thread t at position
// t * P + u, then the smaller strides of the same size.
template <int NT, int kSize, int kStride, int P, typename K>
__device__ __forceinline__ void sort_step(K (&key)[P], K *lds, int t) {
    if constexpr (kStride < P) {
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (!(u & kStride)) {
                const bool up = kSize < P ? (u & kSize) == 0 : (t & (kSize / P)) == 0;
                order_pair(key[u], key[u | kStride], up);
            }
    } else {
        constexpr int X = kStride / P;  // thread distance
        const bool keep_min = ((t & X) == 0) == ((t & (kSize / P)) == 0);
        if constexpr (X < kWave) {
#pragma unroll
            for (int u = 0; u < P; ++u) {
                const K o = lane_xor<X>(key[u]);
                key[u] = (o < key[u]) == keep_min ? o : key[u];
            }
        } else {
#pragma unroll
            for (int u = 0; u < P; ++u) lds[u * NT + t] = key[u];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < P; ++u) {
                const K o = lds[u * NT + (t ^ X)];
                key[u] = (o < key[u]) == keep_min ? o : key[u];
            }
            __syncthreads();
        }
    }
    if constexpr (kStride > 1) sort_step<NT, kSize, kStride / 2, P>(key, lds, t);
}

template <int NT, int P, int kSize = 2, typename K>
__device__ __forceinline__ void sort_products(K (&key)[P], K *lds, int t) {
    sort_step<NT, kSize, kSize / 2, P>(key, lds, t);
    if constexpr (kSize < NT * P) sort_products<NT, P, kSize * 2>(key, lds, t);
}

// barrier of a row's threads
template <int NT>
__device__ __forceinline__ void row_sync() {
    if constexpr (NT > kWave) __syncthreads();
    else wave_sync();
}

template <int NT, int P, typename K>
struct SortLds {
    static constexpr int kMax = NT * P;
    double pa[kMax];  // by a B row's first position: its A value; then by position: the product's
    double pb[kMax];
    union {
        int32_t sq[kMax];  // by a B row's first position: B position minus product position
        K key[kMax];       // sorted keys
    };
    __align__(8) uint16_t mark[kMax];  // a B row's first position + 1, else 0
    int32_t part[2][NT / kWave];
};

template <int NT, int WPB, int P, typename K>
__device__ __forceinline__ void num_sort_rows(SortLds<NT, P, K> *lds_s, int32_t block, int32_t blocks,
                                              const TaskDev *__restrict__ tasks, int nt,
                                              const int32_t *__restrict__ rows, Counters *__restrict__ cnt, int cls,
                                              int32_t lo, const int64_t *__restrict__ rowptr,
                                              const Panel *__restrict__ panels, int npanels) {
    static_assert(NT > kWave ? WPB == 1 : NT == kWave, "a row's threads are a workgroup or a wave of it");
    constexpr int kMax = NT * P, kWaves = NT / kWave;
    static_assert(kMax <= 1 << kSortIdBits, "positions fit their key bits");
    constexpr K kIdMask = ((K)1 << kSortIdBits) - 1;
    const int sub = NT > kWave ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // row of the workgroup
    const int t = threadIdx.x % NT, l = lane_id();
    const int w = NT > kWave ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : 0;    // wave of the row
    SortLds<NT, P, K> &L = lds_s[sub];
    const int32_t nrows = cnt->cls[cls];
    for (int32_t li = block * WPB + sub; li < nrows; li += blocks * WPB) {
        const int32_t g = __builtin_amdgcn_readfirstlane(rows[li]);
        const int64_t rs = rowptr[g];
        const int32_t expect = (int32_t)(rowptr[g + 1] - rs);
        if (expect <= lo) continue;  // uniform over the row's threads: not this launch's (short rows)
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
        const TR_GLOBAL double *__restrict__ av = as_global(TK.av);
        const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
        const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
        const TR_GLOBAL double *__restrict__ bv = as_global(TK.bv);
        const int32_t a0 = as_global(TK.ap)[r], a1 = as_global(TK.ap)[r + 1];
#pragma unroll
        for (int u = 0; u < P; ++u) L.mark[t * P + u] = 0;
        row_sync<NT>();
        // B rows of A's entries, flattened: each non-empty one is entered at its
        // first product position
        int32_t total = 0;
        for (int32_t pb = a0, turn = 0; pb < a1; pb += NT, turn ^= 1) {
            int32_t bs = 0, len = 0;
            double a = 0.0;
            if (pb + t < a1) {
                const int32_t k = ai[pb + t];
                a = av[pb + t];
                bs = bp[k];
                len = bp[k + 1] - bs;
            }
            const int32_t inc = wave_incl_scan(len);
            int32_t pos = total + inc - len;
            if constexpr (kWaves > 1) {
                if (l == kWave - 1) L.part[turn][w] = inc;
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kWaves; ++u) {
                    const int32_t s = L.part[turn][u];
                    pos += u < w ? s : 0;
                    total += s;
                }
            } else {
                total += read_lane(inc, kWave - 1);
            }
            if (len > 0 && pos < kMax) {
                L.mark[pos] = (uint16_t)(pos + 1);
                L.sq[pos] = bs - pos;
                L.pa[pos] = a;
            }
        }
        total = min(total, kMax);  // (the row's class bounds it)
        row_sync<NT>();
        // this thread's products t P .. t P + P - 1: the last mark at or below
        uint32_t m[P];
        {
#pragma unroll
            for (int u = 0; u < P; ++u) {
                m[u] = L.mark[t * P + u];
                if (u) m[u] = max(m[u], m[u - 1]);
            }
            const uint32_t inc = wave_incl_max(m[P - 1]);
            uint32_t before = dpp<0x138>(inc);  // the lane below; 0 for lane 0
            if constexpr (kWaves > 1) {
                // (the entries' last use of `part` is behind the barrier above)
                if (l == kWave - 1) L.part[0][w] = (int32_t)inc;
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kWaves - 1; ++u) before = max(before, u < w ? (uint32_t)L.part[0][u] : 0u);
            }
#pragma unroll
            for (int u = 0; u < P; ++u) m[u] = max(m[u], before);
        }
        K key[P];
        double pa[P], pbv[P];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const int32_t x = t * P + u;
            key[u] = ~(K)0;
            pa[u] = pbv[u] = 0.0;
            if (x < total) {
                const uint32_t s = m[u] - 1;
                const int32_t q = L.sq[s] + x;
                pa[u] = L.pa[s];
                key[u] = (K)(uint32_t)bi[q] << kSortIdBits | (K)x;
                pbv[u] = bv[q];
            }
        }
        row_sync<NT>();  // sq and the A values by first position are read
#pragma unroll
        for (int u = 0; u < P; ++u) {
            L.pa[t * P + u] = pa[u];
            L.pb[t * P + u] = pbv[u];
        }
        sort_products<NT, P>(key, L.key, t);
#pragma unroll
        for (int u = 0; u < P; ++u) L.key[t * P + u] = key[u];
        row_sync<NT>();
        // columns that begin in this thread, and their places
        K prev = t > 0 ? L.key[t * P - 1] : 0;
        int32_t nhead = 0, first = P;
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const int32_t x = t * P + u;
            if (x < total && (x == 0 || (prev >> kSortIdBits) != (key[u] >> kSortIdBits))) {
                if (nhead == 0) first = u;
                ++nhead;
            }
            prev = key[u];
        }
        const int32_t inc = wave_incl_scan(nhead);
        int32_t rank = inc - nhead, n = 0;
        if constexpr (kWaves > 1) {
            if (l == kWave - 1) L.part[1][w] = inc;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kWaves; ++u) {
                const int32_t s = L.part[1][u];
                rank += u < w ? s : 0;
                n += s;
            }
        } else {
            n = read_lane(inc, kWave - 1);
        }
        const Panel &PN = find_panel(panels, npanels, g);
        if (t == 0 && n != expect) atomicOr(&cnt->overflow, 2);
        TR_GLOBAL int32_t *oi = as_global(PN.idx) + (rs - PN.nnz_begin);
        TR_GLOBAL double *ov = as_global(PN.val) + (rs - PN.nnz_begin);
        if (nhead > 0) {
            int32_t x = t * P + first;
            K col = L.key[x] >> kSortIdBits;
            double v = 0.0;
            while (true) {
                const K k = L.key[x];
                const uint32_t id = (uint32_t)(k & kIdMask);
                v = __fma_rn(L.pa[id], L.pb[id], v);
                ++x;
                const bool more = x < total;
                const K next = more ? L.key[x] >> kSortIdBits : 0;
                if (!more || next != col) {
                    if (rank < expect) {  // never write past the row
                        oi[rank] = (int32_t)col;
                        ov[rank] = v;
                    }
                    ++rank;
                    if (!more || x >= t * P + P) break;  // the next column begins in another thread
                    col = next;
                    v = 0.0;
                }
            }
        }
        row_sync<NT>();  // the next row rewrites the arrays
    }
}

template <int NT, int WPB, int P, typename K>
__global__ __launch_bounds__(NT *WPB) void k_num_sort(const TaskDev *__restrict__ tasks, int nt,
                                                      const int32_t *__restrict__ rows, Counters *__restrict__ cnt,
                                                      int cls, int32_t lo, const int64_t *__restrict__ rowptr,
                                                      const Panel *__restrict__ panels, int npanels) {
    __shared__ SortLds<NT, P, K> lds_s[WPB];
    num_sort_rows<NT, WPB, P, K>(lds_s, blockIdx.x, gridDim.x, tasks, nt, rows, cnt, cls, lo, rowptr, panels, npanels);
}

// All light classes at once, where they are few rows (light_blocks); a
// workgroup is 256 threads in every class (a row of 257 to 512 products takes
// two a thread instead of four of half as many threads).
template <typename K>
__global__ __launch_bounds__(256) void k_num_sort_all(const TaskDev *__restrict__ tasks, int nt,
                                                      const int32_t *__restrict__ lists, int32_t rows_total,
                                                      Counters *__restrict__ cnt, const LightBlocks lb,
                                                      const int64_t *__restrict__ rowptr,
                                                      const Panel *__restrict__ panels, int npanels) {
    __shared__ union {
        SortLds<64, 1, K> a[4];
        SortLds<64, 2, K> b[4];
        SortLds<64, 4, K> c[4];
        SortLds<256, 2, K> d[1];
        SortLds<256, 4, K> e[1];
    } L;
    const int c = light_block_class(lb);
    const int32_t block = (int32_t)blockIdx.x - lb.end[c + 1], blocks = lb.end[c] - lb.end[c + 1];
    const int32_t *rows = lists + (int64_t)c * rows_total;
    if (c == 5) num_sort_rows<256, 1, 4, K>(L.e, block, blocks, tasks, nt, rows, cnt, c, 0, rowptr, panels, npanels);
    else if (c == 4) num_sort_rows<256, 1, 2, K>(L.d, block, blocks, tasks, nt, rows, cnt, c, 0, rowptr, panels, npanels);
    else if (c == 3) num_sort_rows<64, 4, 4, K>(L.c, block, blocks, tasks, nt, rows, cnt, c, 0, rowptr, panels, npanels);
    else if (c == 2) num_sort_rows<64, 4, 2, K>(L.b, block, blocks, tasks, nt, rows, cnt, c, 0, rowptr, panels, npanels);
    else num_sort_rows<64, 4, 1, K>(L.a, block, blocks, tasks, nt, rows, cnt, c, 0, rowptr, panels, npanels);
}

// ---------------------------------------------------------------- numeric, heavy rows (workgroup)
// One NT-thread workgroup per item (a run of windows of one row),
// sharing one T-slot LDS table per window.  For each window the row's A
// entries are taken NT at a time (one per thread): each thread finds the
// part of B_k inside the window (register cursor for rows with <= NT
// entries, the item's cursor array otherwise) and a workgroup scan flattens
// the products in A-order.
//
// The waves take the products in groups of 64 and work on their groups at the
// same time, but for the sum itself: finding the slots, the operands' loads
// and the search for lanes that meet in a slot need no order (a free slot
// holds 0, whoever claims it).  Only the addition to the slots waits for its
// turn, a count in LDS that every group passes on, so that every slot sums in
// A-order; lanes of a group that share a slot add one after the other.  The
// turn is a read, an fma and a write, so the wait is short: it has no cost
// that a raised wave priority, a sleep in the wait or weaker fences change.
// (Steps of NT products between barriers, where a slot's last pusher walked a
// list of the step's products: product of R-MAT s17 12.1 ms, with turns 10.5;
// s19 95.5 and 82.5.  With tags of each wave's own, T/2 or T/4 of them, s17
// 11.1 and 11.9: a shared tag costs a round of the search below.  Also slower,
// s19: buckets of four keys read at once 85.9, a second hash for the step 83.6,
// B as 16-byte records 89.)
// A presence bitmap over the window, built after the window's last group,
// gives every entry its sorted rank (prefix popcounts) for the write-out.
//
// Occupancy: the kernel is bound by the latency of its dependent LDS and
// memory chains, so resident waves matter most: product of R-MAT s19 97.6 ms
// with four workgroups per CU, 82.4 with five, 75.0 with six (s17 12.3, 10.5,
// 9.6).  For the six, a 2048-slot, 256-thread workgroup keeps to 26.4 KB: the
// tags are the keys' upper bits, the bitmap takes the keys' space once they
// are in registers, and the segments of a round of 4096 products are one bit
// per start.  The register budget is held to 80 VGPRs; the 4096-slot table (53
// KB, 512 threads) fits three workgroups per CU.
constexpr int kRegSlots = 1;  // register-held A entries per thread in the heavy numeric kernel
constexpr int kSmallNT = 256;  // threads of the 2048-slot heavy numeric
constexpr uint32_t kSlotFree = 0xffffffffu;
constexpr int kOffBits = 20;  // a slot's key: column offset, the last thread that met it above
constexpr uint32_t kOffMask = (1u << kOffBits) - 1u;
constexpr int kRound = kWave * kWave;  // products of a round of marks

template <int T, int NT>
struct HeavyWgLds {
    union {
        __align__(16) uint32_t key[T];  // kSlotFree in free slots
        struct {  // extraction of a window: presence bitmap and its prefix counts
            unsigned long long bm[kBmWords];
            uint16_t wpre[kBmWords];
        };
    };
    double vals[T];                     // 0 in free slots
    // segments (A entries with products in the window) of a batch, in A-order
    int32_t seg_d[NT];                  // B position minus flattened product position
    uint64_t starts[kRound / kWave];    // positions of the round where a segment starts
    typename std::conditional<(NT <= 256), uint8_t, uint16_t>::type seg_o[NT];  // its A entry, from the batch's first
    int32_t wsum[NT / kWave];
    int32_t nocc;
    int32_t turn;                       // group of 64 products that is applied next
};
static_assert(sizeof(HeavyWgLds<2048, 256>) <= 26880, "six workgroups per CU");

// LDS only: loads in flight from global memory are not waited for
__device__ __forceinline__ void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
__device__ __forceinline__ void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }

// workgroup exclusive scan of v; returns the exclusive prefix, *total = sum
template <int NT>
__device__ __forceinline__ int32_t wg_excl_scan(int32_t v, int32_t *wsum, int32_t *total) {
    const int w = threadIdx.x / kWave, l = lane_id();
    const int32_t inc = wave_incl_scan(v);
    if (l == kWave - 1) wsum[w] = inc;
    __syncthreads();
    int32_t off = 0, tot = 0;
#pragma unroll
    for (int u = 0; u < NT / kWave; ++u) {
        const int32_t s = wsum[u];
        off += (u < w) ? s : 0;
        tot += s;
    }
    *total = tot;
    return off + inc - v;
}

template <int T, int NT>
__global__ __launch_bounds__(NT, 6) void k_num_heavy_wg(const TaskDev *__restrict__ tasks, int nt,
                                                     const Item *__restrict__ items, Counters *__restrict__ cnt,
                                                     const Window *__restrict__ wins,
                                                     const int32_t *__restrict__ order,
                                                     const int64_t *__restrict__ cursor_base,
                                                     int4 *__restrict__ cursors, const int64_t *__restrict__ rowptr,
                                                     const Panel *__restrict__ panels, int npanels,
                                                     int32_t dense_width) {
    constexpr uint32_t kLog = __builtin_ctz(T);
    __shared__ HeavyWgLds<T, NT> L;
    constexpr int kWaves = NT / kWave;
    const int tid = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (int t = tid; t < T; t += NT) {
        L.key[t] = kSlotFree;
        L.vals[t] = 0.0;
    }
    if (tid == 0) L.nocc = L.turn = 0;
    __syncthreads();
    const int32_t nitems = cnt->items;
    const int32_t slot = (int32_t)blockIdx.x;
    for (int32_t ord = slot; ord < nitems; ord += gridDim.x) {
        const int32_t itx = order[ord];
        const Item I = items[itx];
        const int32_t g = I.row;
        const TaskDev &TK = tasks[task_of(tasks, nt, g)];
        const int32_t r = g - TK.row_base;
        const TR_GLOBAL int32_t *__restrict__ ai = as_global(TK.ai);
        const TR_GLOBAL double *__restrict__ av = as_global(TK.av);
        const TR_GLOBAL int32_t *__restrict__ bp = as_global(TK.bp);
        const TR_GLOBAL int32_t *__restrict__ bi = as_global(TK.bi);
        const TR_GLOBAL double *__restrict__ bv = as_global(TK.bv);
        const int32_t ncols = TK.n;
        const int32_t a0 = as_global(TK.ap)[r], a1 = as_global(TK.ap)[r + 1];
        // cursor of A entry p: (first B position at or after the next window,
        // its column, end of B_k)
        int4 *cur = cursors + cursor_base[itx];
        const int64_t rs = rowptr[g];
        const Panel &P = find_panel(panels, npanels, g);
        TR_GLOBAL int32_t *oi_row = as_global(P.idx) + (rs - P.nnz_begin);
        TR_GLOBAL double *ov_row = as_global(P.val) + (rs - P.nnz_begin);
        // rows with <= NT * kRegSlots entries: the B ranges of thread tid's A
        // entries (slots tid, tid + NT, ...) and their cursors live in
        // registers; longer rows keep cursors in the item's cursor array
        const bool reg_row = (a1 - a0) <= NT * kRegSlots;
        // (before the item's first window the cursor holds the start of B_k)
        int32_t rk_be[kRegSlots], rk_cur[kRegSlots], rk_nxt[kRegSlots];
#pragma unroll
        for (int u = 0; u < kRegSlots; ++u) {
            rk_be[u] = rk_cur[u] = rk_nxt[u] = 0;
            const int32_t p = a0 + u * NT + tid;
            if (reg_row && p < a1) {
                const int32_t k = ai[p];
                rk_cur[u] = bp[k];
                rk_be[u] = bp[k + 1];
            }
        }
        bool have_cursor = false;
        for (int32_t wi = I.wbeg; wi < I.wend; ++wi) {
            const Window W = wins[wi];
            if (W.cnt == 0) continue;  // block-uniform
            const bool full = (W.c0 == 0 && W.c1 >= ncols);
            const bool last = (wi == I.wend - 1);
            // windows up to kWinMaxWidth columns are ranked by presence
            // bitmaps of kBmWidth columns, one pass each; wider (sparse)
            // windows hold <= kSparseH + 127 entries and are ranked by
            // counting smaller keys
            const bool dense = (W.c1 - W.c0) <= kWinMaxWidth;
            // windows no wider than dense_width (<= T) address their slots by
            // column offset: no probing, no ranking pass.  The slot is
            // (off * hmul) >> (32 - kLog) either way, with hmul = 2^(32 - kLog)
            // for the identity and the golden-ratio multiplier for the hash.
            const uint32_t hmul = (W.c1 - W.c0) <= dense_width ? (1u << (32 - kLog)) : 0x9E3779B1u;
            int nfresh = 0;
            for (int32_t pb = a0, slot = 0; pb < a1; pb += NT, ++slot) {
                if (tid < kRound / kWave) L.starts[tid] = 0;
                // this thread's k-slot: A entry p, B segment [s, e) inside the window
                const int32_t p = pb + tid;
                int32_t s = 0, e = 0;
                if (p < a1) {
                    // c: cursor (first entry at or after this window's start),
                    // v: its column (INT32_MAX at the end of B_k); known once the
                    // item's first window has been visited
                    int32_t bs = 0, be = 0, c = 0, v = 0;
                    if (reg_row) {
                        // uniform slot index: selects, not dynamic register indexing
#pragma unroll
                        for (int u = 0; u < kRegSlots; ++u)
                            if (u == slot) {
                                be = rk_be[u];
                                c = rk_cur[u];
                                v = rk_nxt[u];
                            }
                        bs = c;
                    } else if (have_cursor && !full) {
                        const int4 cv = cur[p - a0];
                        c = cv.x;
                        v = cv.y;
                        be = cv.z;
                    } else {
                        const int32_t k = ai[p];
                        bs = bp[k];
                        be = bp[k + 1];
                    }
                    if (full) {
                        s = bs;
                        e = be;
                    } else {
                        if (!have_cursor) {
                            // an item that starts at the row's first column
                            // starts at the front of B_k: no search
                            c = W.c0 == 0 ? bs : lower_bound_dev(bi, bs, be, W.c0);
                            v = c < be ? bi[c] : INT32_MAX;
                        }
                        s = c;
                        // an A entry with nothing in this window costs no load
                        e = v >= W.c1 ? s : gallop_from(bi, s, be, W.c1, v);
                        if (reg_row) {
#pragma unroll
                            for (int u = 0; u < kRegSlots; ++u)
                                if (u == slot) {
                                    rk_cur[u] = e;
                                    rk_nxt[u] = v;
                                }
                        } else if (!last) {
                            cur[p - a0] = make_int4(e, v, be, 0);
                        }
                    }
                }
                // one scan for the products and the segments before this one
                // (a segment's columns are entries of the window, 3/4 T at most)
                constexpr int kSegShift = 21;
                static_assert(3 * T / 4 * NT < 1 << kSegShift, "packed counts");
                int32_t packed;
                const int32_t slen = e - s;
                const uint32_t ex = (uint32_t)wg_excl_scan<NT>(slen > 0 ? slen + (1 << kSegShift) : 0, L.wsum, &packed);
                const int32_t total = packed & ((1 << kSegShift) - 1);
                const int32_t excl = (int32_t)(ex & ((1u << kSegShift) - 1u));
                if (slen > 0) {
                    const uint32_t rank = ex >> kSegShift;
                    L.seg_d[rank] = s - excl;
                    L.seg_o[rank] = tid;
                    // (cleared before the scan's barrier)
                    if (excl < kRound) atomicOr((unsigned long long *)&L.starts[excl / kWave], 1ull << (excl % kWave));
                }
                __syncthreads();
                // products flattened in A-order, in groups of 64: the waves take
                // the groups in turn
                const int32_t ngroups = (total + kWave - 1) / kWave;
                int32_t segs = -1;  // last segment that starts before the round
                for (int32_t base = 0; base < total; base += kRound) {
                    if (base > 0) {
                        __syncthreads();
                        if (tid < kRound / kWave) L.starts[tid] = 0;
                        __syncthreads();
                        if (slen > 0 && excl >= base && excl < base + kRound)
                            atomicOr((unsigned long long *)&L.starts[(excl - base) / kWave], 1ull << (excl % kWave));
                        __syncthreads();
                    }
                    // lane i: the starts in the round's group i, and the last
                    // segment that starts before it
                    const uint64_t word = L.starts[l];
                    const int32_t upto = wave_incl_scan((int32_t)__popcll(word));
                    const int32_t before = segs + upto - __popcll(word);
                    segs += read_lane(upto, kWave - 1);
                    const int32_t gend = min(ngroups, (base + kRound) / kWave);
                    int32_t grp = base / kWave + w;
                    int32_t jn = 0;
                    double bn = 0.0, an = 0.0;
                    // product of group q that is this lane's
                    auto load = [&](int32_t q) {
                        if (q >= gend) return;
                        const int32_t x = q * kWave + l;
                        const uint64_t starts = read_lane(word, q - base / kWave);
                        const int32_t o = read_lane(before, q - base / kWave) + rank_below(starts) +
                                          (int32_t)__builtin_amdgcn_inverse_ballot_w64(starts);
                        if (x < total) {
                            const int32_t t = L.seg_d[o] + x;
                            an = av[pb + L.seg_o[o]];
                            jn = bi[t];
                            bn = bv[t];
                        }
                    };
                    load(grp);
                    for (; grp < gend; grp += kWaves) {
                        bool act = grp * kWave + l < total;
                        const double a = an, b = bn;
                        // find or claim the slot: in any order, a free slot holds 0
                        const uint32_t off = (uint32_t)(jn - W.c0);
                        uint32_t h = (off * hmul) >> (32 - kLog);
                        bool more = act;
                        for (int probe = 0; probe < T && ballot(more); ++probe) {
                            if (more) {
                                const uint32_t old = atomicCAS(&L.key[h], kSlotFree, off | (uint32_t)tid << kOffBits);
                                nfresh += old == kSlotFree ? 1 : 0;
                                more = old != kSlotFree && (old & kOffMask) != off;
                                if (more) h = (h + 1) & (T - 1);
                            }
                        }
                        if (more) {
                            atomicOr(&cnt->overflow, 8);  // table full: symbolic counts were wrong
                            act = false;
                        }
                        // lanes of the group that meet in a slot: every lane
                        // writes itself to the upper half of the slot's key
                        // (the offset's bits there are the same), and one that reads
                        // another may share the slot (or another wave came in
                        // between): of lanes that share one, all but one do.
                        // turn_of: lanes of the same slot before this one.
                        // A round takes the slots of the lowest and the
                        // highest such lane (one slot a round: product of
                        // R-MAT s17 9.54 ms, two 9.15, the lowest two, three
                        // or four lanes 9.31, 9.46, 9.50)
                        static_assert(NT <= 1 << (32 - kOffBits) && kOffBits >= 16, "a thread above the offset");
                        if (act) ((volatile uint16_t *)&L.key[h])[1] = (uint16_t)(off >> 16 | (uint32_t)tid << (kOffBits - 16));
                        wave_sync();
                        uint64_t shared = ballot(act && ((volatile uint32_t *)L.key)[h] >> kOffBits != (uint32_t)tid);
                        int turn_of = 0, turns = 1;
                        const uint32_t hm = act ? h : ~0u;
                        while (shared) {
                            const uint32_t hf = read_lane(hm, __ffsll((unsigned long long)shared) - 1);
                            const uint32_t hf2 = read_lane(hm, 63 - __clzll((long long)shared));
                            const bool same = hm == hf, same2 = hm == hf2;
                            const uint64_t m = ballot(same), m2 = ballot(same2);
                            if (same) turn_of = rank_below(m);
                            if (same2) turn_of = rank_below(m2);
                            turns = max(turns, max(__popcll(m), __popcll(m2)));
                            shared &= ~(m | m2);
                        }
                        load(grp + kWaves);
                        // wait for the groups before this one, which other waves hold
                        while (__hip_atomic_load(&L.turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != grp) {
                        }
                        lds_acquire();
                        for (int q = 0; q < turns; ++q) {
                            if (act && turn_of == q) L.vals[h] = __fma_rn(a, b, L.vals[h]);
                            wave_sync();
                        }
                        lds_release();
                        if (l == 0) __hip_atomic_store(&L.turn, grp + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
                __syncthreads();  // seg_d and the marks are rewritten by the next batch
                if (tid == 0) L.turn = 0;
            }
            if (!full) have_cursor = true;
            // entries created in this window (each thread counted its fresh inserts)
            const int32_t wf = wave_sum(nfresh);
            if (l == 0 && wf) atomicAdd(&L.nocc, wf);
            TR_GLOBAL int32_t *oi = oi_row + W.off;
            TR_GLOBAL double *ov = ov_row + W.off;
            // Each thread's entries as rank << 20 | column offset (kNone: no
            // entry) and value.  The table's first three quarters [0, kStage)
            // are also the staging area (a window holds at most kStage
            // entries): their values are stashed in registers before a
            // barrier, the last quarter is read and staged after it.
            constexpr int kSt = (T + NT - 1) / NT;
            constexpr int kStage = 3 * T / 4;
            constexpr int kLo = (kStage + NT - 1) / NT;
            constexpr int kSp = (kSparseH + 127 + NT - 1) / NT;  // sparse entries per thread
            constexpr int kStash = kLo > kSp ? kLo : kSp;
            static_assert(kSp <= kSt && kStage % NT == 0, "stash slots are exactly the staging area's");
            constexpr uint32_t kNone = 0xffffffffu;
            uint32_t st_rk[kSt];
            double st_v[kStash];
            const int32_t lim = min(W.cnt, kStage);  // never write past the window
            int32_t *sidx = reinterpret_cast<int32_t *>(L.key);
            // the thread's slots (h = tid + u NT) by column offset; the keys'
            // space is the bitmap's from here on
#pragma unroll
            for (int u = 0; u < kSt; ++u) {
                const int h = tid + u * NT;
                const uint32_t kt = h < T ? L.key[h] : kSlotFree;
                st_rk[u] = kt == kSlotFree ? kNone : kt & kOffMask;
            }
            __syncthreads();
            if (dense) {
                // ranked one kBmWidth-column pass at a time with a presence
                // bitmap.  A direct window's slots are its column offsets, so a
                // ballot over 64 consecutive slots is its presence word, and its
                // one pass (width <= T < kBmWidth) needs no clearing or atomics.
                const int32_t width = W.c1 - W.c0;
                const bool direct = width <= dense_width;
                if (direct) {
#pragma unroll
                    for (int u = 0; u < kSt; ++u) {
                        const uint64_t m = ballot(st_rk[u] != kNone);
                        if (l == 0) L.bm[u * (NT / kWave) + w] = m;
                    }
                }
                static_assert(T / kWave <= kBmWords, "a direct window's slots fit one pass");
                int32_t base_rank = 0;
                for (int32_t lo = 0; lo < width; lo += kBmWidth) {  // block-uniform
                    const int nwords = min(kBmWords, (width - lo + 63) >> 6);
                    if (!direct) {
                        for (int t = tid; t < nwords; t += NT) L.bm[t] = 0ull;
                        __syncthreads();
#pragma unroll
                        for (int u = 0; u < kSt; ++u) {
                            const uint32_t rel = st_rk[u] - (uint32_t)lo;  // kNone wraps past kBmWidth
                            if (rel < (uint32_t)kBmWidth) atomicOr(&L.bm[rel >> 6], 1ull << (rel & 63));
                        }
                    }
                    __syncthreads();
                    // prefix popcounts of the presence words
                    constexpr int kPer = (kBmWords + NT - 1) / NT;
                    int32_t wc[kPer];
                    int32_t tsum = 0;
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const int wd = tid * kPer + u;
                        wc[u] = (wd < nwords) ? __popcll(L.bm[wd]) : 0;
                        tsum += wc[u];
                    }
                    int32_t tot;
                    int32_t run = wg_excl_scan<NT>(tsum, L.wsum, &tot);
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const int wd = tid * kPer + u;
                        if (wd < kBmWords) L.wpre[wd] = (uint16_t)run;
                        run += wc[u];
                    }
                    __syncthreads();
#pragma unroll
                    for (int u = 0; u < kSt; ++u) {
                        const uint32_t rel = st_rk[u] - (uint32_t)lo;
                        if (rel < (uint32_t)kBmWidth) {
                            const int wd = (int)(rel >> 6);
                            const uint32_t rr = (uint32_t)(base_rank + L.wpre[wd]) +
                                                __popcll(L.bm[wd] & ((1ull << (rel & 63)) - 1ull));
                            st_rk[u] |= rr << 20;
                        }
                    }
                    base_rank += tot;
                    __syncthreads();  // wsum, bm and wpre are reused by the next pass
                }
            }
            if (dense) {
                if (tid == 0 && L.nocc != W.cnt) atomicOr(&cnt->overflow, 4);
#pragma unroll
                for (int u = 0; u < kStash; ++u) {
                    const int h = tid + u * NT;
                    if (u < kLo && h < kStage && st_rk[u] != kNone) st_v[u] = L.vals[h];
                }
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kSt; ++u) {
                    const int h = tid + u * NT;
                    if (h < kStage || h >= T || st_rk[u] == kNone) continue;
                    const int32_t rr = (int32_t)(st_rk[u] >> 20);
                    if (rr < lim) {
                        const double v = L.vals[h];
                        sidx[rr] = W.c0 + (int32_t)(st_rk[u] & 0xfffffu);
                        L.vals[rr] = v;
                    }
                }
            } else {
                // compact the occupied slots (keys into the bitmap's space,
                // slot numbers into the prefix array), then rank each entry by
                // the number of smaller keys
                uint32_t *lkey = reinterpret_cast<uint32_t *>(L.bm);
                uint16_t *lslot = L.wpre;
                int32_t mine = 0;
#pragma unroll
                for (int u = 0; u < kSt; ++u) mine += st_rk[u] != kNone ? 1 : 0;
                int32_t tot;
                int32_t pos = wg_excl_scan<NT>(mine, L.wsum, &tot);
                const bool fits = tot <= kSparseH + 127;  // bound of a sparse window
                if (fits)
#pragma unroll
                    for (int u = 0; u < kSt; ++u) {
                        if (st_rk[u] == kNone) continue;
                        lkey[pos] = st_rk[u];
                        lslot[pos] = (uint16_t)(tid + u * NT);
                        ++pos;
                    }
                __syncthreads();
                if (tid == 0 && (L.nocc != W.cnt || !fits)) atomicOr(&cnt->overflow, 4);
#pragma unroll
                for (int u = 0; u < kStash; ++u) {
                    const int e = tid + u * NT;
                    st_rk[u] = kNone;
                    if (u >= kSp || !fits || e >= tot) continue;
                    const uint32_t k = lkey[e];
                    uint32_t rr = 0;
                    for (int q = 0; q < tot; ++q) rr += lkey[q] < k ? 1u : 0u;
                    st_rk[u] = (rr << 20) | k;
                    st_v[u] = L.vals[lslot[e]];
                }
                __syncthreads();
            }
            // stage the stashed entries in rank order, then write the window
            // out with coalesced stores
#pragma unroll
            for (int u = 0; u < kStash; ++u) {
                const int32_t rr = (int32_t)(st_rk[u] >> 20);
                if (st_rk[u] != kNone && rr < lim) {
                    sidx[rr] = W.c0 + (int32_t)(st_rk[u] & 0xfffffu);
                    L.vals[rr] = st_v[u];
                }
            }
            __syncthreads();
            // streaming stores: C is written once and should not evict the B
            // rows that later windows read again
            for (int e = tid; e < W.cnt; e += NT) {
                __builtin_nontemporal_store(sidx[e], &oi[e]);
                __builtin_nontemporal_store(L.vals[e], &ov[e]);
            }
            __syncthreads();
            for (int t = tid; t < T; t += NT) {
                L.key[t] = kSlotFree;
                L.vals[t] = 0.0;
            }
            if (tid == 0) L.nocc = 0;
            __syncthreads();
        }
    }
}

}  // namespace

// ======================================================================= host side

void *Workspace::get(int slot, size_t bytes) {
    req[slot] = std::max(req[slot], bytes);
    if (!owned) return scratch(ctx, slot, bytes);
    if (bytes == 0) bytes = 1;
    if (sz[slot] < bytes) {
        if (p[slot]) ctx->pool.release(p[slot]);
        p[slot] = nullptr;
        sz[slot] = 0;
        p[slot] = ctx->pool.alloc(bytes);
        sz[slot] = bytes;
    }
    return p[slot];
}

void Workspace::drop(int slot) {
    if (!owned) return scratch_drop(ctx, slot);
    if (p[slot]) ctx->pool.release(p[slot]);
    p[slot] = nullptr;
    sz[slot] = 0;
}

void Workspace::release() {
    if (!owned || !ctx) return;
    for (size_t s = 0; s < p.size(); ++s)
        if (p[s]) {
            try {
                ctx->pool.release(p[s]);
            } catch (...) {
            }
            p[s] = nullptr;
            sz[s] = 0;
        }
}

namespace {

uint32_t cap_grid(int64_t need, int64_t cap) {
    if (need <= 0) return 0;
    return (uint32_t)std::min<int64_t>(need, cap);
}


// Workgroups of the light classes if they go into one launch: more than one
// class has rows, and together they are at most kLightPerCu workgroups a CU.
// `wide`: classes 4 and 5 take a workgroup a row.
// A class of few rows leaves most CUs idle for the whole chain of its longest
// row, so up to six such launches wait for each other (5 to 22 us each); in one
// they overlap.  Every workgroup then holds the LDS of the largest class, which
// costs occupancy once the rows fill the chip several times.  (Separate
// launches, then one launch up to 4, 16 and 32 a CU: tile accumulate of R-MAT
// s16 347, 339, 270, 271 us; Galerkin 19^3 345, 279, 261, 264 us; product of
// 15013 vertices 568, 561, 493, 497 us.)
constexpr int kLightPerCu = 16;
bool light_blocks(tr_ctx *ctx, const MulPlan &pl, bool wide, LightBlocks &lb) {
    int64_t all = 0;
    int used = 0;
    lb.end[kNumLight] = 0;
    for (int c = kNumLight - 1; c >= 0; --c) {
        const int64_t n = pl.h.cls[c];
        all += wide && c >= 4 ? n : (n + 3) / 4;
        used += n > 0 ? 1 : 0;
        lb.end[c] = (int32_t)std::min<int64_t>(all, INT32_MAX);
    }
    return used > 1 && all <= (int64_t)ctx->cu_count * kLightPerCu;
}

template <int T>
void launch_sym_light(tr_ctx *ctx, MulPlan &pl, int c) {
    const int32_t n = pl.h.cls[c];
    TR_LAUNCH(ctx, "sym_light", k_sym_light<T>, cap_grid(div_up((uint64_t)n, 4), 1 << 20), 256, 0, pl.d_tasks,
              pl.nt, pl.lists + (int64_t)c * pl.rows_total, pl.cnt, c, pl.rownnz);
}

template <int T>
void launch_num_light(tr_ctx *ctx, MulPlan &pl, int c, Panel *panels, int np) {
    constexpr int kWpb = 4;
    const int32_t n = pl.h.cls[c];
    if (n) TR_LAUNCH(ctx, "num_light", (k_num_light<T, kWpb>), cap_grid(div_up((uint64_t)n, kWpb), 1 << 20), kWpb * kWave,
              0, pl.d_tasks, pl.nt, pl.lists + (int64_t)c * pl.rows_total, pl.cnt, c, pl.rowptr, panels, np);
}

}  // namespace

namespace {

// buffers of a plan over pl.h_tasks
void mul_buffers(tr_ctx *ctx, Workspace &ws, MulPlan &pl) {
    pl.nt = (int)pl.h_tasks.size();
    pl.tune = ctx->tune;
    int64_t rows = 0;
    for (auto &t : pl.h_tasks) {
        t.row_base = (int32_t)rows;
        rows += t.m;
    }
    TR_REQUIRE(rows < INT32_MAX, "spgemm: total rows of the batch exceed INT32_MAX");
    pl.rows_total = (int32_t)rows;
    const size_t R = (size_t)rows + 1, nt = (size_t)std::max(pl.nt, 1);
    pl.d_tasks = (TaskDev *)ws.get(S_PANELS + 0, (sizeof(TaskDev) + sizeof(CheckJob)) * nt);
    pl.flops = (int64_t *)ws.get(S_FLOPS, sizeof(int64_t) * R);
    pl.lists = (int32_t *)ws.get(S_BINS, sizeof(int32_t) * (size_t)kNumClasses * R);
    pl.cnt = (Counters *)ws.get(S_BINCNT, sizeof(Counters));
    pl.rownnz = (int64_t *)ws.get(S_ROWNNZ, sizeof(int64_t) * R);
    pl.rowptr = (int64_t *)ws.get(S_ROWPTR64, sizeof(int64_t) * R);
    pl.scan_tmp = ws.owned ? (int64_t *)ws.get(S_SCAN_TMP, scan_tmp_bytes(rows)) : nullptr;
}

CheckJob flops_job(const MulPlan &pl, const TaskDev &t) {
    CheckJob j{};
    j.ptr = t.ap;
    j.idx = t.ai;
    j.bp = t.bp;
    j.flops = pl.flops + t.row_base;
    j.cap = t.a_cap;
    j.n = t.m;
    j.other = t.k;
    return j;
}

TaskDev task_of_pair(const tr_csx_t *A, const tr_csx_t *B) {
    TaskDev t{};
    t.ap = A->ptr_vec;
    t.ai = A->idx_vec;
    t.av = A->val;
    t.bp = B->ptr_vec;
    t.bi = B->idx_vec;
    t.bv = B->val;
    t.m = A->nrows;
    t.n = B->ncols;
    t.k = A->ncols;
    t.a_cap = A->nnz;
    return t;
}

}  // namespace

void mul_setup(tr_ctx *ctx, Workspace &ws, MulPlan &pl, const std::vector<TaskDev> &tasks) {
    pl.h_tasks = tasks;
    mul_buffers(ctx, ws, pl);
    std::vector<CheckJob> jobs;
    for (auto &t : pl.h_tasks) {
        jobs.push_back(flops_job(pl, t));
        check_place(jobs.back(), pl.check_grid);
    }
    pl.njobs = pl.nt;
    pl.jobs = (CheckJob *)(pl.d_tasks + pl.nt);
    TR_HIP(hipMemcpyAsync(pl.d_tasks, pl.h_tasks.data(), sizeof(TaskDev) * (size_t)pl.nt, hipMemcpyHostToDevice,
                          ctx->stream));
    TR_HIP(hipMemcpyAsync(pl.jobs, jobs.data(), sizeof(CheckJob) * jobs.size(), hipMemcpyHostToDevice, ctx->stream));
    TR_HIP(hipStreamSynchronize(ctx->stream));  // `jobs` ends here
}

void mul_setup_plain(tr_ctx *ctx, Workspace &ws, MulPlan &pl, const tr_csx_t *A, const tr_csx_t *B) {
    check_operand_shapes(A, B);
    pl.h_tasks = {task_of_pair(A, B)};
    mul_buffers(ctx, ws, pl);
    pl.pair.j[0] = flops_job(pl, pl.h_tasks[0]);
    check_place(pl.pair.j[0], pl.check_grid);
    pl.njobs = 1;
    if (!same_tile(A, B)) {
        pl.pair.j[1] = check_job(B);
        check_place(pl.pair.j[1], pl.check_grid);
        pl.njobs = 2;
    }
}

void mul_analyze(tr_ctx *ctx, MulPlan &pl) {
    if (pl.jobs) {
        TR_LAUNCH(ctx, "zero_counters", k_zero_counters, 1, 64, 0, pl.cnt);
    } else {
        TR_LAUNCH(ctx, "put_task", k_put_task, 1, 64, 0, pl.d_tasks, pl.h_tasks[0], pl.cnt);
        check_open(ctx);
        ctx->check_twin = pl.njobs == 1;
    }
    launch_check(ctx, pl.jobs, pl.njobs, pl.pair, pl.check_grid);
    TR_LAUNCH(ctx, "classify", k_classify, div_up((uint64_t)pl.rows_total, kRowsPerBlock), kClassThreads, 0,
              pl.d_tasks, pl.nt, pl.rows_total, pl.flops, pl.rownnz, pl.lists, pl.cnt, pl.tune.light_max_flops,
              pl.rows_total >= kShortMinRows ? 1 : 0);
}

namespace {

void require_sorted_operands(const int32_t (&hs)[2]) {
    if (hs[0] & 3) fail(TR_ERR_INVALID, "spgemm: A is not a valid CSR (ptr or column index out of range)");
    if (hs[1] & 3) fail(TR_ERR_INVALID, "spgemm: B is not a valid CSR (ptr or column index out of range)");
    if (hs[1] & 4) fail(TR_ERR_INVALID, "spgemm: B has unsorted or duplicate columns; call tr_csx_sort_rows");
    if (hs[0] & 4) fail(TR_ERR_INVALID, "spgemm: A has unsorted or duplicate columns; call tr_csx_sort_rows");
}

}  // namespace

void mul_checked(tr_ctx *ctx) {
    int32_t hs[2];
    check_result(ctx, hs, 2);
    require_sorted_operands(hs);
}

void mul_read_counts(tr_ctx *ctx, MulPlan &pl) { read_array(ctx, &pl.h, pl.cnt, sizeof(Counters)); }

int64_t item_flops(const tr_ctx *ctx, const MulPlan &pl) {
    return heavy_item_flops((int64_t)pl.h.heavy_flops, ctx->cu_count);
}

template <int PB, int NTH>
void launch_sym_heavy(tr_ctx *ctx, MulPlan &pl, int cls, int cls2, int per_cu, bool emit) {
    const int64_t n = (int64_t)pl.h.cls[cls] + (cls2 != cls ? pl.h.cls[cls2] : 0);
    TR_LAUNCH(ctx, "sym_heavy", (k_sym_heavy<PB, NTH>), cap_grid(n, (int64_t)ctx->cu_count * per_cu), NTH,
              0, pl.d_tasks, pl.nt, pl.cnt, cls, cls2, pl.rownnz, emit ? 1 : 0,
              pl.tune.window_entries, pl.tune.item_windows, item_flops(ctx, pl), pl.flops, pl.wins, pl.win_cap,
              pl.items, pl.item_cap, pl.lists, pl.rows_total);
}

namespace {

int32_t widest(const MulPlan &pl) {
    int32_t n = 0;
    for (const TaskDev &t : pl.h_tasks) n = std::max(n, t.n);
    return n;
}

int heavy_pass_bits(int32_t max_n) { return max_n <= (1 << 18) ? 18 : max_n <= (1 << 19) ? 19 : kPassBits; }

}  // namespace

void mul_symbolic(tr_ctx *ctx, Workspace &ws, MulPlan &pl, bool emit, bool capture) {
    LightBlocks lb;
    if (light_blocks(ctx, pl, false, lb)) {
        TR_LAUNCH(ctx, "sym_light", k_sym_light_all, (uint32_t)lb.end[0], 256, 0, pl.d_tasks, pl.nt, pl.lists,
                  pl.rows_total, pl.cnt, lb, pl.rownnz);
    } else {
        if (pl.h.cls[0]) launch_sym_light<64>(ctx, pl, 0);
        if (pl.h.cls[1]) launch_sym_light<128>(ctx, pl, 1);
        if (pl.h.cls[2]) launch_sym_light<256>(ctx, pl, 2);
        if (pl.h.cls[3]) launch_sym_light<512>(ctx, pl, 3);
        if (pl.h.cls[4]) launch_sym_light<1024>(ctx, pl, 4);
        if (pl.h.cls[5]) launch_sym_light<2048>(ctx, pl, 5);
    }
    if (pl.h.cls[kShortClass])
        TR_LAUNCH(ctx, "sym_light", k_sym_short,
                  cap_grid(div_up((uint64_t)pl.h.cls[kShortClass], 4 * kShortRows), (int64_t)ctx->cu_count * 32), 256, 0,
                  pl.d_tasks, pl.nt, pl.lists + (int64_t)kShortClass * pl.rows_total, pl.cnt, pl.rownnz);
    const int32_t nh = pl.h.cls[kHeavyClass] + pl.h.cls[kMidClass];
    if (nh) {
        const int32_t max_n = widest(pl);
        if (emit && !capture) {
            const HeavyLists cap = heavy_lists((int64_t)pl.h.heavy_flops, nh, max_n, pl.tune.window_entries,
                                               pl.tune.item_windows, item_flops(ctx, pl));
            TR_REQUIRE(cap.windows < INT32_MAX && cap.items < INT32_MAX, "spgemm: heavy work list exceeds int32 capacity");
            pl.win_cap = (int32_t)cap.windows;
            pl.item_cap = (int32_t)cap.items;
            pl.wins = (Window *)ws.get(S_WINDOWS, sizeof(Window) * (size_t)cap.windows);
            pl.items = (Item *)ws.get(S_ITEMS, sizeof(Item) * (size_t)cap.items);
        }
        // The bitmap covers 2^PB columns per pass and its LDS bounds the
        // resident workgroups: 2^20 bits (128 KiB) hold one per CU, 2^19 two,
        // 2^18 four.  The narrowest pass that still covers the widest
        // operand in one pass is used (same windows, same results).  The
        // grids hold many more workgroups than fit at once: rows differ
        // widely in cost, and queued workgroups go to whichever CU frees
        // first (Galerkin 128^3: 12.9 -> 12.3 ms against one resident wave
        // of workgroups).
        const int pb = heavy_pass_bits(max_n);
        // Up to 2^19 columns both classes share a kernel, the heaviest rows
        // first, in one launch: the lighter rows fill the end of the heavier
        // ones (R-MAT s17 1896 -> 1410 us, 15013 vertices 218 -> 179 us).
        if (pb == 18) launch_sym_heavy<18, kMidThreads>(ctx, pl, kHeavyClass, kMidClass, 64, emit);
        else if (pb == 19) launch_sym_heavy<19, kHeavyThreads>(ctx, pl, kHeavyClass, kMidClass, 32, emit);
        else {
            launch_sym_heavy<kPassBits, kHeavyThreads>(ctx, pl, kHeavyClass, kHeavyClass, 32, emit);
            launch_sym_heavy<kMidPassBits, kHeavyThreads>(ctx, pl, kMidClass, kMidClass, 32, emit);
        }
    }
    launch_exclusive_scan_i64(ctx, pl.rownnz, pl.rowptr, pl.rows_total, pl.scan_tmp);
}

void mul_cursor_prep(tr_ctx *ctx, Workspace &ws, MulPlan &pl, bool capture) {
    if (!pl.h.cls[kHeavyClass] && !pl.h.cls[kMidClass]) return;
    if (!capture) {
        pl.clen = (int32_t *)ws.get(S_MISC, sizeof(int32_t) * ((size_t)pl.item_cap + 1));
        pl.cbase = (int64_t *)ws.get(S_MISC2, sizeof(int64_t) * ((size_t)pl.item_cap + 1));
    }
    if (ws.owned && !capture) pl.scan_tmp = (int64_t *)ws.get(S_SCAN_TMP, scan_tmp_bytes(std::max<int64_t>(pl.item_cap, pl.rows_total)));
    TR_LAUNCH(ctx, "item_cursor_len", k_item_cursor_len, div_up((uint64_t)pl.item_cap, 256), 256, 0, pl.items, pl.cnt,
              pl.d_tasks, pl.nt, pl.item_cap, (pl.tune.heavy_table == 4096 ? 512 : kSmallNT) * kRegSlots, pl.clen);
    // column order of the items
    if (!capture) {
        pl.order = (int32_t *)ws.get(S_ORDER, sizeof(int32_t) * ((size_t)pl.item_cap + 1));
        pl.order_hist = (unsigned long long *)ws.get(S_ORDER_HIST, sizeof(unsigned long long) * kOrderBuckets);
    }
    const uint32_t og = cap_grid(div_up((uint64_t)pl.item_cap, 256), (int64_t)ctx->cu_count * 8);
    const int32_t maxn = widest(pl);
    int shift = 0;
    while (((int64_t)kOrderBuckets << shift) < (int64_t)maxn) ++shift;
    TR_LAUNCH(ctx, "item_order", k_fill_u64, div_up((uint64_t)kOrderBuckets, 256), 256, 0, pl.order_hist,
              kOrderBuckets);
    TR_LAUNCH(ctx, "item_order", k_item_hist, og, 256, 0, pl.items, pl.wins, pl.cnt, shift, pl.order_hist);
    TR_LAUNCH(ctx, "item_order", k_item_hist_scan, 1, 1024, 0, pl.order_hist);
    TR_LAUNCH(ctx, "item_order", k_item_scatter, og, 256, 0, pl.items, pl.wins, pl.cnt, shift, pl.order_hist,
              pl.order);
    launch_exclusive_scan_i32_to_i64(ctx, pl.clen, pl.cbase, pl.item_cap, pl.scan_tmp);
}

void mul_read_totals(tr_ctx *ctx, MulPlan &pl, int64_t *nnz, int64_t *ncur) {
    const bool heavy = pl.h.cls[kHeavyClass] || pl.h.cls[kMidClass];
    *ncur = 0;
    const ReadPart parts[3] = {{&pl.h, pl.cnt, sizeof(Counters)},
                               {nnz, pl.rowptr + pl.rows_total, sizeof(int64_t)},
                               {ncur, pl.cbase + pl.item_cap, sizeof(int64_t)}};
    read_parts(ctx, parts, heavy ? 3 : 2);
}

namespace {

__global__ void k_task_offsets(const TaskDev *__restrict__ tasks, int nt, const int64_t *__restrict__ rowptr,
                               int32_t rows, int64_t *__restrict__ out) {
    for (int t = threadIdx.x; t <= nt; t += blockDim.x) out[t] = rowptr[t < nt ? tasks[t].row_base : rows];
}

}  // namespace

void mul_read_task_offsets(tr_ctx *ctx, MulPlan &pl, int64_t *host) {
    if (sizeof(int64_t) * ((size_t)pl.nt + 1) > kPinnedValues) {
        for (int t = 0; t <= pl.nt; ++t)
            host[t] = read_scalar<int64_t>(ctx, pl.rowptr + (t < pl.nt ? pl.h_tasks[t].row_base : pl.rows_total));
        return;
    }
    TR_LAUNCH(ctx, "publish", k_task_offsets, 1, 64, 0, pl.d_tasks, pl.nt, pl.rowptr, pl.rows_total,
              (int64_t *)ctx->pinned);
    TR_HIP(hipStreamSynchronize(ctx->stream));
    std::memcpy(host, ctx->pinned, sizeof(int64_t) * ((size_t)pl.nt + 1));
}

namespace {

template <int NT, int P, typename K>
void launch_num_sort_as(tr_ctx *ctx, MulPlan &pl, int c, int32_t lo, Panel *panels, int np) {
    constexpr int kWpb = NT > kWave ? 1 : 4;
    const int32_t n = pl.h.cls[c];
    TR_LAUNCH(ctx, "num_light", (k_num_sort<NT, kWpb, P, K>), cap_grid(div_up((uint64_t)n, kWpb), 1 << 20), NT * kWpb,
              0, pl.d_tasks, pl.nt, pl.lists + (int64_t)c * pl.rows_total, pl.cnt, c, lo, pl.rowptr,
              panels, np);
}

// (column, position) keys of 32 bits hold every column
bool narrow_keys(const MulPlan &pl) {
    return widest(pl) <= 1 << (32 - kSortIdBits);
}

// class c of rows of up to NT * P products, those of more than lo entries
template <int NT, int P>
void launch_num_sort(tr_ctx *ctx, MulPlan &pl, int c, int32_t lo, Panel *panels, int np) {
    if (!pl.h.cls[c]) return;
    if (narrow_keys(pl)) launch_num_sort_as<NT, P, uint32_t>(ctx, pl, c, lo, panels, np);
    else launch_num_sort_as<NT, P, uint64_t>(ctx, pl, c, lo, panels, np);
}

}  // namespace

void mul_numeric(tr_ctx *ctx, MulPlan &pl, Panel *dp, int np) {
    LightBlocks lb;
    if (light_blocks(ctx, pl, true, lb)) {
        if (narrow_keys(pl))
            TR_LAUNCH(ctx, "num_light", k_num_sort_all<uint32_t>, (uint32_t)lb.end[0], 256, 0, pl.d_tasks, pl.nt,
                      pl.lists, pl.rows_total, pl.cnt, lb, pl.rowptr, dp, np);
        else
            TR_LAUNCH(ctx, "num_light", k_num_sort_all<uint64_t>, (uint32_t)lb.end[0], 256, 0, pl.d_tasks, pl.nt,
                      pl.lists, pl.rows_total, pl.cnt, lb, pl.rowptr, dp, np);
    } else {
        launch_num_sort<64, 1>(ctx, pl, 0, 0, dp, np);
        launch_num_sort<64, 1>(ctx, pl, 1, 0, dp, np);
        launch_num_sort<64, 2>(ctx, pl, 2, 0, dp, np);
        launch_num_sort<64, 4>(ctx, pl, 3, 0, dp, np);
        launch_num_sort<128, 4>(ctx, pl, 4, 0, dp, np);
        launch_num_sort<256, 4>(ctx, pl, 5, 0, dp, np);
    }
    // short rows of more entries than their table takes are sorted
    if (pl.h.short_rows[0])
        TR_LAUNCH(ctx, "num_light", k_num_short,
                  cap_grid(div_up((uint64_t)pl.h.cls[kShortClass], 4 * kShortRows), 1 << 20), 256, 0, pl.d_tasks, pl.nt,
                  pl.lists + (int64_t)kShortClass * pl.rows_total, pl.cnt, pl.rowptr, dp, np);
    if (pl.h.short_rows[1]) launch_num_sort<64, 2>(ctx, pl, kShortClass, kShortMaxNnz, dp, np);
    launch_num_light<64>(ctx, pl, kCompactClass, dp, np);
    launch_num_light<128>(ctx, pl, kCompactClass + 1, dp, np);
    launch_num_light<256>(ctx, pl, kCompactClass + 2, dp, np);
    if (pl.h.items > 0) {
        // one workgroup per item, grid-stride beyond 2^22 workgroups (the
        // dispatch packet counts work-items in 32 bits)
        const uint32_t grid = cap_grid(pl.h.items, 1 << 22);
        if (pl.tune.heavy_table == 4096)
            TR_LAUNCH(ctx, "num_heavy", (k_num_heavy_wg<4096, 512>), grid, 512, 0, pl.d_tasks, pl.nt, pl.items,
                      pl.cnt, pl.wins, pl.order, pl.cbase, pl.cursors, pl.rowptr, dp, np, pl.tune.dense_width);
        else
            TR_LAUNCH(ctx, "num_heavy", (k_num_heavy_wg<2048, kSmallNT>), grid, kSmallNT, 0, pl.d_tasks, pl.nt, pl.items,
                      pl.cnt, pl.wins, pl.order, pl.cbase, pl.cursors, pl.rowptr, dp, np, pl.tune.dense_width);
    }
}

// A class that had no row gets no launch; the two heavy classes share theirs
// where they share a kernel.
uint32_t mul_taken(const MulPlan &pl) {
    uint32_t m = 0;
    for (int c = 0; c < kNumClasses; ++c) m |= pl.h.cls[c] > 0 ? 1u << c : 0u;
    if (heavy_pass_bits(widest(pl)) != kPassBits && (m & (1u << kHeavyClass | 1u << kMidClass)))
        m |= 1u << kHeavyClass | 1u << kMidClass;
    for (int i = 0; i < 2; ++i) m |= pl.h.short_rows[i] > 0 ? 1u << (kShortRowsBit + i) : 0u;
    return m | (pl.h.items > 0 ? 1u << kItemsBit : 0u);
}

void mul_check(tr_ctx *ctx, MulPlan &pl) {
    const int32_t ov = read_scalar<int32_t>(ctx, &pl.cnt->overflow);
    if (ov & 1) fail(TR_ERR_HIP, "spgemm: heavy work list capacity exceeded (internal bound violated)");
    if (ov & 14) fail(TR_ERR_HIP, "spgemm: numeric row counts disagree with the symbolic phase (internal error)");
}

void check_operand_shapes(const tr_csx_t *A, const tr_csx_t *B) {
    check_csx(A, "A");
    check_csx(B, "B");
    TR_REQUIRE(A->majordim == TR_ROWS && B->majordim == TR_ROWS, "spgemm operands must be CSR (TR_ROWS)");
    TR_REQUIRE(A->ncols == B->nrows, "spgemm: A.ncols != B.nrows");
}

void validate_operands(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *B) {
    check_operand_shapes(A, B);
    const tr_csx_t *m[2] = {A, B};
    int32_t hs[2];
    check_tiles(ctx, m, 2, hs);
    require_sorted_operands(hs);
}

int64_t spgemm_flops(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *B) {
    Workspace ws(ctx, false);
    MulPlan pl;
    mul_setup_plain(ctx, ws, pl, A, B);
    mul_analyze(ctx, pl);
    mul_read_counts(ctx, pl);
    mul_checked(ctx);
    return (int64_t)pl.h.flops;
}

void spgemm_symbolic_only(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *B, int64_t *nnz, size_t *bytes) {
    Workspace ws(ctx, false);
    MulPlan pl;
    mul_setup_plain(ctx, ws, pl, A, B);
    mul_analyze(ctx, pl);
    mul_read_counts(ctx, pl);
    mul_checked(ctx);
    // the same steps as the product up to its numeric phase, so every work
    // list and the cursor array are sized exactly as the product sizes them
    mul_symbolic(ctx, ws, pl, true, false);
    mul_cursor_prep(ctx, ws, pl, false);
    int64_t total = 0, ncur = 0;
    mul_read_totals(ctx, pl, &total, &ncur);
    if (nnz) *nnz = total;
    if (bytes) {
        // Upper bound of the device memory tr_spgemm takes from a context
        // pool with nothing cached: every scratch slot at the size the product
        // requests (grown to 1.25x, in pool granules), the cursor array and the
        // output tile.  A batch places the product in
        // two blocks (indices, values) and its row pointers in a third.
        std::vector<size_t> req = ws.req;
        if (pl.h.items > 0) req[S_CURSORS] = std::max(req[S_CURSORS], sizeof(int4) * (size_t)std::max<int64_t>(ncur, 1));
        req[S_TMP_CSX] = std::max(req[S_TMP_CSX], std::max<size_t>(64, sizeof(Panel)));
        size_t b = 0;
        for (size_t r : req)
            if (r) b += scratch_block_bytes(r);
        const size_t rows1 = (size_t)pl.rows_total + 1;
        b += pool_block_bytes((size_t)total * 12 + rows1 * 4);
        b += pool_block_bytes((size_t)total * 4) + pool_block_bytes((size_t)total * 8) + pool_block_bytes(rows1 * 4) +
             2 * pool_block_bytes(sizeof(Panel) + rows1 * 4);
        *bytes = b;
    }
}

int spgemm_panels(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *B, int64_t max_panel_nnz, tr_csx_t *panels,
                  int32_t *row_begin, int32_t max_panels, int32_t *npanels) {
    TR_REQUIRE(panels && row_begin && npanels && max_panels >= 1, "spgemm: null panel outputs");
    TR_REQUIRE(max_panel_nnz >= 1 && max_panel_nnz <= INT32_MAX, "spgemm: max_panel_nnz must be in [1, INT32_MAX]");
    Workspace ws(ctx, false);
    MulPlan pl;
    mul_setup_plain(ctx, ws, pl, A, B);
    mul_analyze(ctx, pl);
    mul_read_counts(ctx, pl);
    mul_checked(ctx);
    mul_symbolic(ctx, ws, pl, true, false);
    mul_cursor_prep(ctx, ws, pl, false);
    const int32_t m = pl.rows_total;
    int64_t total = 0, ncur = 0;
    mul_read_totals(ctx, pl, &total, &ncur);
    if (pl.h.overflow & 1) fail(TR_ERR_HIP, "spgemm: heavy work list capacity exceeded (internal bound violated)");

    // panel split
    std::vector<int32_t> rb{0};
    std::vector<int64_t> hrp;
    if (total > max_panel_nnz) {
        hrp.resize((size_t)m + 1);
        read_array(ctx, hrp.data(), pl.rowptr, sizeof(int64_t) * ((size_t)m + 1));
        int64_t start = 0;
        for (int32_t r = 0; r < m; ++r) {
            if (hrp[r + 1] - hrp[r] > max_panel_nnz)
                fail(TR_ERR_OVERFLOW, "spgemm: a single row of C exceeds the panel capacity");
            if (hrp[r + 1] - start > max_panel_nnz) {
                rb.push_back(r);
                start = hrp[r];
            }
        }
    }
    rb.push_back(m);
    const int32_t np = (int32_t)rb.size() - 1;
    if (np > max_panels) {
        *npanels = np;
        fail(TR_ERR_OVERFLOW, "spgemm: nnz(C) = " + std::to_string(total) + " needs " + std::to_string(np) +
                                  " panels of at most " + std::to_string(max_panel_nnz) + " entries");
    }
    Panel *dp = (Panel *)ws.get(S_TMP_CSX, sizeof(Panel) * (size_t)np);
    for (int32_t p = 0; p < np; ++p) {
        const int64_t nb0 = np == 1 ? 0 : hrp[rb[p]];
        const int64_t nb1 = np == 1 ? total : hrp[rb[p + 1]];
        tr_csx_t *C = &panels[p];
        alloc_tile(ctx, TR_ROWS, rb[p + 1] - rb[p], pl.h_tasks[0].n, nb1 - nb0, C);
        const Panel hp{nb0, rb[p], 0, C->idx_vec, C->val};
        TR_LAUNCH(ctx, "tile_ptr", k_tile_ptr, div_up((uint64_t)(rb[p + 1] - rb[p]) + 1, 256), 256, 0, pl.rowptr,
                  rb[p], rb[p + 1] - rb[p], C->ptr_vec, hp, dp + p);
        row_begin[p] = rb[p];
    }
    row_begin[np] = m;
    *npanels = np;
    if (pl.h.items > 0)
        pl.cursors = (int4 *)ws.get(S_CURSORS, sizeof(int4) * (size_t)std::max<int64_t>(ncur, 1));
    mul_numeric(ctx, pl, dp, np);
    mul_check(ctx, pl);
    return TR_OK;
}

}  // namespace tr
