// Well-formedness checks of compressed tiles and the row analysis of a
// product, on gfx950.
//
// The reference trusts its tiles; here every operand is checked before a
// kernel indexes through it.  One pass over the segment pointers, one over the
// entries (csr_units.h: equal units of segments plus entries), which for A of
// a product also sums the lengths of the B rows that a row's entries meet.
//
// What bounds it: 4 bytes read per entry, and for a product the gather of two
// row pointers of B per entry.  Before, the checks marked row starts in a
// bitmap in memory (a clear, an atomic per row and a pass per tile), and the
// sums took a wave per long row, so that an R-MAT's hub rows decided their
// time: R-MAT s19 (8 M entries) 1220 us for the sums and 73 us for the checks,
// now 46 us for both; 95 M entries of an add 268 -> 138 us (2.8 TB/s).
#include "csr_units.h"
#include "dev_common.h"
#include "tr_internal.h"

namespace tr {
namespace {

using namespace dev;

// findings[4 * tile + f], f: 0 ptr malformed, 1 index out of range, 2 order
__device__ __forceinline__ void report(uint8_t *findings, int tile, int f) {
    if (findings) findings[4 * tile + f] = 1;
}

template <int32_t CheckJob::*kFirst>
__device__ __forceinline__ int job_of(const CheckJob *jobs, int nj) {
    int lo = 0, hi = nj - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].*kFirst <= (int32_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(256) void k_check_ptr(const CheckJob *__restrict__ tab, int nj, const CheckPair pair,
                                                   uint8_t *__restrict__ findings) {
    const int t = tab ? job_of<&CheckJob::block0>(tab, nj) : (nj > 1 && (int32_t)blockIdx.x >= pair.j[1].block0);
    const CheckJob J = tab ? tab[t] : pair.j[t];
    const int64_t i = (int64_t)((int32_t)blockIdx.x - J.block0) * 256 + threadIdx.x;
    if (i > J.n) return;
    const int32_t v = J.ptr[i];
    bool bad = v < 0 || (int64_t)v > J.cap;
    if (i == 0 && v != 0) bad = true;
    if (i == J.n && (int64_t)v != J.cap) bad = true;
    if (i < J.n) {
        if (J.ptr[i + 1] < v) bad = true;
        if (J.bp) J.flops[i] = 0;
    }
    if (bad) report(findings, t, 0);
}

__global__ __launch_bounds__(kUnitThreads) void k_check_entries(const CheckJob *__restrict__ tab, int nj,
                                                               const CheckPair pair, uint8_t *__restrict__ findings) {
    constexpr int kPer = kUnit / kUnitThreads;
    constexpr int kWaves = kUnitThreads / kWave;
    __shared__ unsigned long long starts[kUnitWords];  // entries that start a segment
    __shared__ uint32_t sum[kUnit + 1];                // B row lengths of the unit's first x entries
    __shared__ uint32_t tot[kWaves];
    __shared__ int32_t split[2];
    const int tid = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int t = tab ? job_of<&CheckJob::unit0>(tab, nj) : (nj > 1 && (int32_t)blockIdx.x >= pair.j[1].unit0);
    const CheckJob J = tab ? tab[t] : pair.j[t];
    if (tid < kUnitWords) starts[tid] = 0ull;
    // (a compressed tile may hold fewer entries than its arrays)
    const int64_t nnz = min(max((int64_t)J.ptr[J.n], (int64_t)0), J.cap);
    const Unit U = find_unit(J.ptr, J.n, nnz, (int32_t)blockIdx.x - J.unit0, split);
    if (U.len == 0) return;  // block-uniform
    // entry x of the unit: wave w holds x = w * 64 kPer + 64 u + lane
    const int32_t x0 = w * (kPer * kWave) + l;
    int32_t c[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int32_t x = x0 + u * kWave;
        c[u] = x < U.len ? J.idx[U.j0 + x] : 0;
    }
    int32_t before = -1;  // lane 0: the entry before the wave's first
    if (l == 0 && x0 < U.len && U.j0 + x0 > 0) before = J.idx[U.j0 + x0 - 1];
    if (J.bp) {
        uint32_t v[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            v[u] = 0;
            if (x0 + u * kWave < U.len && (uint32_t)c[u] < (uint32_t)J.other)
                v[u] = (uint32_t)(J.bp[c[u] + 1] - J.bp[c[u]]);
        }
        // sums modulo 2^32: a row's own sum is at most nnz(B) < 2^31
        uint32_t run = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const uint32_t inc = wave_incl_scan(v[u]);
            v[u] = run + inc;
            run += read_lane(inc, kWave - 1);
        }
        if (l == 0) tot[w] = run;
        __syncthreads();
        uint32_t off = 0;
#pragma unroll
        for (int u = 0; u < kWaves - 1; ++u) off += u < w ? tot[u] : 0u;
        if (tid == 0) sum[0] = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u) sum[x0 + u * kWave + 1] = off + v[u];
    }
    __syncthreads();
    for (int32_t i = U.i0 + tid; i <= U.i1 && i < J.n; i += kUnitThreads) {
        const int64_t b = (int64_t)J.ptr[i] - U.j0, e = (int64_t)J.ptr[i + 1] - U.j0;
        if (findings && b >= 0 && b < U.len) atomicOr(&starts[b >> 6], 1ull << (b & 63));
        if (!J.bp) continue;
        const int32_t xb = (int32_t)min(max(b, (int64_t)0), (int64_t)U.len);
        const int32_t xe = (int32_t)min(max(e, (int64_t)0), (int64_t)U.len);
        if (xe <= xb) continue;
        const uint32_t f = sum[xe] - sum[xb];
        if (b >= 0 && e <= U.len) J.flops[i] = f;  // the whole segment
        else atomicAdd((unsigned long long *)&J.flops[i], (unsigned long long)f);
    }
    if (!findings) return;  // block-uniform
    __syncthreads();
    bool range = false, order = false;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int32_t x = x0 + u * kWave;
        int32_t prev = __shfl_up(c[u], 1, kWave);
        if (l == 0) prev = before;
        before = read_lane(c[u], kWave - 1);
        if (x >= U.len) continue;
        range |= c[u] < 0 || c[u] >= J.other;
        const bool start = (starts[x >> 6] >> (x & 63)) & 1ull;
        order |= !start && U.j0 + x > 0 && c[u] <= prev;
    }
    if (range) report(findings, t, 1);
    if (order) report(findings, t, 2);
}

// Units need monotone pointers.  The entries of a tile whose pointers are not
// well formed are checked by position: a segment starts where a sound,
// non-empty pair of pointers says so.
__global__ __launch_bounds__(256) void k_mark_starts(const CheckJob J, uint32_t *__restrict__ starts) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= J.n) return;
    const int32_t v = J.ptr[i];
    if (v < 0 || (int64_t)v >= J.cap || (i == 0 && v != 0) || J.ptr[i + 1] <= v) return;
    atomicOr(&starts[v >> 5], 1u << (v & 31));
}

__global__ __launch_bounds__(256) void k_check_positions(const CheckJob J, const uint32_t *__restrict__ starts,
                                                         uint8_t *__restrict__ findings) {
    bool range = false, order = false;
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < J.cap; p += (int64_t)gridDim.x * 256) {
        const int32_t c = J.idx[p];
        range |= c < 0 || c >= J.other;
        order |= p > 0 && !((starts[p >> 5] >> (p & 31)) & 1u) && c <= J.idx[p - 1];
    }
    if (range) report(findings, 0, 1);
    if (order) report(findings, 0, 2);
}

}  // namespace

CheckJob check_job(const tr_csx_t *m) {
    CheckJob j{};
    j.ptr = m->ptr_vec;
    j.idx = m->idx_vec;
    j.cap = m->nnz;
    j.n = ptrdim(m);
    j.other = otherdim(m);
    return j;
}

void check_place(CheckJob &j, CheckGrid &g) {
    j.block0 = (int32_t)g.blocks;
    j.unit0 = (int32_t)g.units;
    g.blocks += ((int64_t)j.n + 256) / 256;
    g.units += unit_count(j.n, j.cap);
    TR_REQUIRE(g.blocks < INT32_MAX && g.units < INT32_MAX, "operands too large to check in one launch");
}

void launch_check(tr_ctx *ctx, const CheckJob *jobs, int nj, const CheckPair &pair, const CheckGrid &g) {
    uint8_t *findings = jobs ? nullptr : ctx->status;
    TR_LAUNCH(ctx, "check_ptr", k_check_ptr, (uint32_t)g.blocks, 256, 0, jobs, nj, pair, findings);
    TR_LAUNCH(ctx, "check_entries", k_check_entries, (uint32_t)g.units, kUnitThreads, 0, jobs, nj, pair, findings);
}

// the status bytes are zero when a check starts: one that was begun and never
// asked for its result (a call that failed in between) is waited for first
void check_open(tr_ctx *ctx) {
    if (ctx->check_running) {
        TR_HIP(hipStreamSynchronize(ctx->stream));
        for (int i = 0; i < 4 * kCheckTiles; ++i) ctx->status[i] = 0;
    }
    ctx->check_running = true;
}

bool same_tile(const tr_csx_t *a, const tr_csx_t *b) {
    return a->ptr_vec == b->ptr_vec && a->idx_vec == b->idx_vec && a->nnz == b->nnz && ptrdim(a) == ptrdim(b) &&
           otherdim(a) == otherdim(b);
}

void check_begin(tr_ctx *ctx, const tr_csx_t *const *m, int n) {
    CheckPair pair{};
    CheckGrid g;
    check_open(ctx);
    ctx->check_twin = n > 1 && same_tile(m[0], m[1]);
    const int k = ctx->check_twin ? 1 : n;
    for (int t = 0; t < k; ++t) {
        pair.j[t] = check_job(m[t]);
        check_place(pair.j[t], g);
    }
    launch_check(ctx, nullptr, k, pair, g);
}

void check_pointers(tr_ctx *ctx, const tr_csx_t *const *m, int n) {
    CheckPair pair{};
    CheckGrid g;
    check_open(ctx);
    ctx->check_twin = false;
    for (int t = 0; t < n; ++t) {
        pair.j[t] = check_job(m[t]);
        check_place(pair.j[t], g);
    }
    TR_LAUNCH(ctx, "check_ptr", k_check_ptr, (uint32_t)g.blocks, 256, 0, (const CheckJob *)nullptr, n, pair,
              ctx->status);
}

void check_result(tr_ctx *ctx, int32_t *status, int n) {
    for (int t = 0; t < n; ++t) {
        const uint8_t *f = ctx->status + 4 * (t > 0 && ctx->check_twin ? 0 : t);
        status[t] = (f[0] ? 1 : 0) | (f[1] ? 2 : 0) | (f[2] ? 4 : 0);
    }
    for (int i = 0; i < 4 * kCheckTiles; ++i) ctx->status[i] = 0;
    ctx->check_running = false;
}

void check_tiles(tr_ctx *ctx, const tr_csx_t *const *m, int n, int32_t *status) {
    check_begin(ctx, m, n);
    TR_HIP(hipStreamSynchronize(ctx->stream));
    check_result(ctx, status, n);
}

int32_t check_positions(tr_ctx *ctx, const tr_csx_t *m) {
    const CheckJob j = check_job(m);
    const int64_t words = j.cap / 32 + 1;
    uint32_t *starts = (uint32_t *)scratch(ctx, S_MISC2, sizeof(uint32_t) * (size_t)words);
    check_open(ctx);
    ctx->check_twin = false;
    launch_fill_i32(ctx, (int32_t *)starts, 0, words);
    TR_LAUNCH(ctx, "mark_starts", k_mark_starts, div_up((uint64_t)j.n, 256), 256, 0, j, starts);
    TR_LAUNCH(ctx, "check_positions", k_check_positions, (uint32_t)std::min<int64_t>((j.cap + 255) / 256, 16384), 256,
              0, j, (const uint32_t *)starts, ctx->status);
    TR_HIP(hipStreamSynchronize(ctx->stream));
    int32_t status = 0;
    check_result(ctx, &status, 1);
    return status;
}

}  // namespace tr
