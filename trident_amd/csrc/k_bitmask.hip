// Bitmask tile compression on gfx950.
//
// Replaces SpaComm::gen_bitmask (include/spacomm.cuh:29-117),
// intersect_bitmasks (:126-148) and SpaCommHandler::Compress (:962-1091,
// with select_entries_cuda :808-889 and select_ptrs :556-623).
//
// Mask words are 64 bits: one wave64 ballot over 64 consecutive segments
// produces one word directly (the reference builds 8-bit words with a
// transform, a segmented reduction and a host round trip).  Compression cuts
// a tile into units of equal segments plus entries; there is no per-entry
// binary search over the pointer array and values and indices move in the
// same pass.
#include "csr_units.h"
#include "dev_common.h"
#include "tr_internal.h"

namespace tr {
namespace {

using namespace dev;

__global__ void k_bitmask_gen(const int32_t *__restrict__ ptr, int32_t n, uint64_t *__restrict__ mask) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool nonempty = false;
    if (i < n) nonempty = ptr[i] != ptr[i + 1];
    uint64_t word = ballot(nonempty);
    if (lane_id() == 0 && i < n) mask[i >> 6] = word;
}

__global__ void k_bitmask_and(const uint64_t *__restrict__ a, const uint64_t *__restrict__ b, int32_t words,
                              uint64_t *__restrict__ out) {
    int32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w < words) out[w] = a[w] & b[w];
}

// ---- entry filter ----
// Keeps a subset of a tile's entries in their order: those of masked segments
// (Compress; the B side of a stage) or those whose index is masked (the A
// side).  A workgroup takes one work unit (csr_units.h): one wave per 64
// segments, the split before, left the hub segments of an R-MAT to one wave
// (2^18 segments, 4 M entries: 1110 us a tile; now 9 us to count, 23 us to
// write 90 MB at about 4 TB/s).  A unit's kept entries are 64-entry bit words
// in LDS, from which every entry's place and every segment's new start are a
// popcount away.  Pass 1 counts per unit, a scan over the units gives their
// first output entry, pass 2 writes.  Jobs of one launch come from a table, or
// as one job by value (njobs == 0).

template <bool kWrite>
__global__ __launch_bounds__(kUnitThreads) void k_filter(const FilterJob *__restrict__ jobs, int njobs,
                                                           const FilterJob one, int32_t *__restrict__ counts,
                                                           const int64_t *__restrict__ first) {
    __shared__ unsigned long long bits[kUnitWords];
    __shared__ int32_t before[kUnitWords];
    __shared__ int32_t split[2];
    const int tid = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].tile0 <= (int32_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const FilterJob J = njobs ? jobs[lo] : one;
    const int32_t unit = (int32_t)blockIdx.x - J.tile0;
    if (tid < kUnitWords) bits[tid] = 0ull;
    const Unit U = find_unit(J.ptr, J.n, J.nnz, unit, split);
    const int32_t i0 = U.i0, i1 = U.i1, len = U.len;
    const int64_t j0 = U.j0;
    if (J.by_index) {
        for (int u = w; u < kUnitWords; u += kUnitThreads / kWave) {
            const int32_t x = u * 64 + l;
            bool keep = false;
            if (x < len) {
                const int32_t c = J.idx[j0 + x];
                keep = (uint32_t)c < (uint32_t)J.nmask && ((J.mask[c >> 6] >> (c & 63)) & 1ull);
            }
            const uint64_t m = ballot(keep);
            if (l == 0) bits[u] = m;
        }
    } else {
        // segment i1's end lies beyond the unit, some of its entries may not
        for (int32_t i = i0 + tid; i <= i1 && i < J.n; i += kUnitThreads) {
            if (!(J.bytes ? ((const uint8_t *)J.mask)[i] : ((J.mask[i >> 6] >> (i & 63)) & 1ull))) continue;
            const int32_t x0 = (int32_t)max((int64_t)J.ptr[i] - j0, (int64_t)0);
            const int32_t x1 = (int32_t)min((int64_t)J.ptr[i + 1] - j0, (int64_t)len);
            for (int32_t x = x0; x < x1; x = (x | 63) + 1) {
                const unsigned long long from = ~0ull << (x & 63);
                const unsigned long long upto = x1 - (x & ~63) >= 64 ? ~0ull : (1ull << (x1 & 63)) - 1ull;
                atomicOr(&bits[x >> 6], from & upto);
            }
        }
    }
    __syncthreads();
    if (w == 0) {
        const int32_t c = l < kUnitWords ? __popcll(bits[l]) : 0;
        const int32_t inc = wave_incl_scan(c);
        if (l < kUnitWords) before[l] = inc - c;
        if (!kWrite && l == kWave - 1) counts[blockIdx.x] = inc;
    }
    if constexpr (kWrite) {
        __syncthreads();
        const int64_t base = first[blockIdx.x] - first[J.tile0];
        auto place = [&](int32_t x) {  // kept entries of the unit before its entry x
            if (x >= kUnit) return before[kUnitWords - 1] + __popcll(bits[kUnitWords - 1]);
            return before[x >> 6] + __popcll(bits[x >> 6] & ((1ull << (x & 63)) - 1ull));
        };
        for (int32_t i = i0 + tid; i < i1; i += kUnitThreads) {
            const int64_t x = (int64_t)J.ptr[i + 1] - j0;
            J.optr[i + 1] = (int32_t)(base + place((int32_t)min(max(x, (int64_t)0), (int64_t)len)));
        }
        if (unit == 0 && tid == 0) J.optr[0] = 0;
        if (before[kUnitWords - 1] + __popcll(bits[kUnitWords - 1]) == 0) return;  // block-uniform
        // all loads before the first store; a dropped entry's lane reads the
        // unit's first entry, which exists
        constexpr int kPer = kUnit / kUnitThreads;
        int32_t ci[kPer];
        double cv[kPer];
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            const int32_t x = t * kUnitThreads + tid;
            const int64_t p = j0 + (((bits[x >> 6] >> (x & 63)) & 1ull) ? x : 0);
            ci[t] = J.idx[p];
            cv[t] = J.val[p];
        }
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            const int32_t x = t * kUnitThreads + tid;
            if (!((bits[x >> 6] >> (x & 63)) & 1ull)) continue;
            const int64_t q = base + place(x);
            if (q < J.cap) {
                J.oidx[q] = ci[t];
                J.oval[q] = cv[t];
            }
        }
    }
}

}  // namespace

void launch_bitmask_gen(tr_ctx *ctx, const int32_t *ptr, int32_t n, uint64_t *mask) {
    if (n <= 0) return;
    TR_LAUNCH(ctx, "bitmask_gen", k_bitmask_gen, div_up((uint64_t)n, 256), 256, 0, ptr, n, mask);
}

void launch_bitmask_and(tr_ctx *ctx, const uint64_t *a, const uint64_t *b, int32_t words, uint64_t *out) {
    if (words <= 0) return;
    TR_LAUNCH(ctx, "bitmask_and", k_bitmask_and, div_up((uint64_t)words, 256), 256, 0, a, b, words, out);
}

// counts and first: one entry per work unit (first: one more)
void launch_filter_count(tr_ctx *ctx, const FilterJob *jobs, int njobs, const FilterJob &one, int32_t ntiles,
                         int32_t *counts, int64_t *first, int64_t *scan_tmp) {
    TR_LAUNCH(ctx, "filter_count", k_filter<false>, ntiles, kUnitThreads, 0, jobs, njobs, one, counts,
              (const int64_t *)nullptr);
    launch_exclusive_scan_i32_to_i64(ctx, counts, first, ntiles, scan_tmp);
}

void launch_filter_write(tr_ctx *ctx, const FilterJob *jobs, int njobs, const FilterJob &one, int32_t ntiles,
                         const int64_t *first) {
    TR_LAUNCH(ctx, "filter_write", k_filter<true>, ntiles, kUnitThreads, 0, jobs, njobs, one, (int32_t *)nullptr,
              first);
}

int64_t compress(tr_ctx *ctx, const tr_csx_t *m, const uint64_t *mask, tr_csx_t *out) {
    FilterJob j{};
    j.ptr = m->ptr_vec;
    j.idx = m->idx_vec;
    j.val = m->val;
    j.mask = mask;
    j.n = ptrdim(m);
    j.nnz = m->nnz;
    const int32_t nt = (int32_t)unit_count(j.n, j.nnz);
    int32_t *counts = (int32_t *)scratch(ctx, S_MISC, sizeof(int32_t) * (size_t)nt);
    int64_t *first = (int64_t *)scratch(ctx, S_ROWPTR64, sizeof(int64_t) * ((size_t)nt + 1));
    launch_filter_count(ctx, nullptr, 0, j, nt, counts, first, nullptr);
    const int64_t nnz = read_scalar<int64_t>(ctx, first + nt);
    alloc_tile(ctx, m->majordim, m->nrows, m->ncols, nnz, out);
    j.optr = out->ptr_vec;
    j.oidx = out->idx_vec;
    j.oval = out->val;
    j.cap = nnz;
    launch_filter_write(ctx, nullptr, 0, j, nt, first);
    return nnz;
}

}  // namespace tr
