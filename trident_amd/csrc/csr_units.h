// Equal work units of a compressed tile, whatever its segment lengths are.
//
// The merge of a tile's segment ends with its entries (segment i's end comes
// before entry ptr[i + 1]) is cut every kUnit steps, so a unit has at most
// kUnit segments and kUnit entries: hub segments are spread over workgroups
// and runs of empty segments are too.  Reads stay in [0, n] of ptr and the
// entries of a unit in [0, nnz) whatever ptr holds.
#pragma once

#include "dev_common.h"

namespace tr {

constexpr int kUnit = 2048;         // segments plus entries per work unit
constexpr int kUnitThreads = 256;
constexpr int kUnitWords = kUnit / 64;

// work units of a tile of n segments and nnz entries (at least one)
inline int64_t unit_count(int64_t n, int64_t nnz) {
    const int64_t u = (n + nnz + kUnit - 1) / kUnit;
    return u > 0 ? u : 1;
}

namespace dev {

// Number of segment ends among the first d steps, searched 64 probes at a
// time (wave-uniform).  In [max(0, d - nnz), min(d, n)] whatever ptr holds.
__device__ __forceinline__ int32_t merge_rows(const int32_t *__restrict__ ptr, int32_t n, int64_t nnz, int64_t d) {
    int64_t lo = d > nnz ? d - nnz : 0, hi = d < n ? d : n;
    while (lo < hi) {
        const int64_t step = (hi - lo + kWave - 1) / kWave;
        const int64_t mid = lo + lane_id() * step;
        const bool past = mid < hi && (int64_t)ptr[mid + 1] <= d - 1 - mid;
        const int c = __popcll(ballot(past));
        if (c == 0) break;
        const int64_t up = lo + c * step;
        lo = up - step + 1;
        hi = up < hi ? up : hi;
    }
    return (int32_t)lo;
}

// Segments whose end lies in the unit are [i0, i1); its entries are
// [j0, j0 + len), of segments i0 .. i1 (the ends of i0 and i1 may lie in
// other units).
struct Unit {
    int32_t i0, i1, len;
    int64_t j0;
};

// The unit's place, found by two waves; `split` is LDS of the workgroup.
// Contains a workgroup barrier.
__device__ __forceinline__ Unit find_unit(const int32_t *__restrict__ ptr, int32_t n, int64_t nnz, int64_t unit,
                                          int32_t *split) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t steps = (int64_t)n + nnz;
    const int64_t d0 = min(unit * kUnit, steps), d1 = min(d0 + kUnit, steps);
    if (w < 2) {
        const int32_t i = merge_rows(ptr, n, nnz, w ? d1 : d0);
        if (lane_id() == 0) split[w] = i;
    }
    __syncthreads();
    Unit u;
    u.i0 = split[0];
    u.i1 = max(split[1], u.i0);  // (below i0 only if ptr is not monotone)
    u.j0 = d0 - u.i0;
    u.len = (int32_t)max((int64_t)0, d1 - u.i1 - u.j0);
    return u;
}

}  // namespace dev
}  // namespace tr
