// Exclusive prefix sum of a function of the index, into 64-bit offsets.
//
// out[i] = sum of in(0) .. in(i - 1) for i in [0, n], out[n] the total.  `in`
// is a device functor, so a count that is cheap to recompute (a row length, a
// masked segment length) is scanned without an array or a launch of its own.
//
// What bounds it: at the sizes of this library (row pointers of 10^3..10^6
// entries) launches and dependent latencies, not bandwidth.  A wave owns 1024
// consecutive items and loads its 16 groups of 64 together; the groups are
// scanned in registers and joined by one barrier, where the kernels before
// walked 16 groups with three barriers each (11 us for their last launch alone
// at any size; the one launch now 6.5 us for 1024 items, 8.2 for 15013).
// One workgroup does up to 16384 items in one launch (three before); up to
// kScanDirect tiles every tile sums the tile totals before it by itself (two
// launches); beyond, a third launch scans the totals, so that the totals read
// stay a small part of the input.
// No workspace needs clearing and no workgroup waits for another, so the
// launches can be recorded into a graph as they are.
#pragma once

#include "dev_common.h"
#include "tr_internal.h"

namespace tr {
namespace scan {

using namespace dev;

constexpr int kGroups = 16;                      // groups of 64 items per wave
constexpr int kWaveItems = kGroups * kWave;      // 1024
constexpr int kTileWaves = 4;
constexpr int kTile = kTileWaves * kWaveItems;   // items of one 256-thread workgroup
constexpr int kOneWaves = 16;
constexpr int kOneItems = kOneWaves * kWaveItems;  // items of the one-launch scan
constexpr int kScanDirect = 2048;                // tiles whose totals every tile sums by itself

template <typename T>
struct ArrayIn {
    const T *p;
    __device__ __forceinline__ int64_t operator()(int64_t i) const { return (int64_t)p[i]; }
};

template <typename In>
__device__ __forceinline__ int64_t wave_load(const In &in, int64_t base, int64_t n, int64_t (&v)[kGroups]) {
    int64_t s = 0;
#pragma unroll
    for (int t = 0; t < kGroups; ++t) {
        const int64_t i = base + t * kWave + lane_id();
        v[t] = i < n ? in(i) : 0;
        s += v[t];
    }
    return wave_sum(s);
}

// stores the wave's exclusive sums, its first item's being `run`
__device__ __forceinline__ void wave_store(int64_t *__restrict__ out, int64_t base, int64_t n,
                                           const int64_t (&v)[kGroups], int64_t run) {
#pragma unroll
    for (int t = 0; t < kGroups; ++t) {
        const int64_t i = base + t * kWave + lane_id();
        const int64_t inc = wave_incl_scan(v[t]);
        if (i < n) out[i] = run + inc - v[t];
        run += read_lane(inc, kWave - 1);
    }
}

template <typename In>
__global__ __launch_bounds__(kOneWaves *kWave) void k_scan_one(In in, int64_t n, int64_t *__restrict__ out) {
    __shared__ int64_t tot[kOneWaves];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t base = (int64_t)w * kWaveItems;
    int64_t v[kGroups];
    const int64_t s = wave_load(in, base, n, v);
    if (lane_id() == 0) tot[w] = s;
    __syncthreads();
    int64_t run = 0, all = 0;
#pragma unroll
    for (int u = 0; u < kOneWaves; ++u) {
        run += u < w ? tot[u] : 0;
        all += tot[u];
    }
    wave_store(out, base, n, v, run);
    if (threadIdx.x == 0) out[n] = all;
}

template <typename In>
__global__ __launch_bounds__(kTileWaves *kWave) void k_scan_reduce(In in, int64_t n, int64_t *__restrict__ tile_sums) {
    __shared__ int64_t tot[kTileWaves];
    const int w = threadIdx.x / kWave;
    int64_t v[kGroups];
    const int64_t s = wave_load(in, (int64_t)blockIdx.x * kTile + (int64_t)w * kWaveItems, n, v);
    if (lane_id() == 0) tot[w] = s;
    __syncthreads();
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot[0] + tot[1] + tot[2] + tot[3];
}

// Exclusive scan of the tile totals in place, single workgroup.
__global__ void k_scan_tiles(int64_t *__restrict__ sums, int64_t ntiles);

// kScanned: tile_sums hold exclusive offsets; otherwise the tiles' totals
template <typename In, bool kScanned>
__global__ __launch_bounds__(kTileWaves *kWave) void k_scan_apply(In in, int64_t n,
                                                                  const int64_t *__restrict__ tile_sums,
                                                                  int64_t *__restrict__ out) {
    __shared__ int64_t tot[kTileWaves], before[kTileWaves];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t base = (int64_t)blockIdx.x * kTile + (int64_t)w * kWaveItems;
    int64_t b = 0;
    if constexpr (kScanned) {
        if (threadIdx.x == 0) b = tile_sums[blockIdx.x];
    } else {
        for (int64_t t = threadIdx.x; t < (int64_t)blockIdx.x; t += kTileWaves * kWave) b += tile_sums[t];
    }
    int64_t v[kGroups];
    const int64_t s = wave_load(in, base, n, v);
    b = wave_sum(b);
    if (lane_id() == 0) {
        tot[w] = s;
        before[w] = b;
    }
    __syncthreads();
    int64_t run = 0, all = 0;
#pragma unroll
    for (int u = 0; u < kTileWaves; ++u) {
        run += before[u] + (u < w ? tot[u] : 0);
        all += before[u] + tot[u];
    }
    wave_store(out, base, n, v, run);
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) out[n] = all;
}

inline int64_t tiles(int64_t n) { return (n + kTile - 1) / kTile; }

// tmp: caller-owned temp of scan_tmp_bytes(n) bytes, or nullptr to use the
// context scratch
template <typename In>
void launch(tr_ctx *ctx, const In &in, int64_t *out, int64_t n, int64_t *tmp) {
    if (n <= kOneItems) {
        TR_LAUNCH(ctx, "scan", (k_scan_one<In>), 1, kOneWaves * kWave, 0, in, n, out);
        return;
    }
    const int64_t nt = tiles(n);
    int64_t *sums = tmp ? tmp : (int64_t *)scratch(ctx, S_SCAN_TMP, scan_tmp_bytes(n));
    TR_LAUNCH(ctx, "scan_reduce", (k_scan_reduce<In>), (uint32_t)nt, kTileWaves * kWave, 0, in, n, sums);
    if (nt <= kScanDirect) {
        TR_LAUNCH(ctx, "scan_apply", (k_scan_apply<In, false>), (uint32_t)nt, kTileWaves * kWave, 0, in, n, sums, out);
    } else {
        TR_LAUNCH(ctx, "scan_tiles", k_scan_tiles, 1, 1024, 0, sums, nt);
        TR_LAUNCH(ctx, "scan_apply", (k_scan_apply<In, true>), (uint32_t)nt, kTileWaves * kWave, 0, in, n, sums, out);
    }
}

}  // namespace scan
}  // namespace tr
