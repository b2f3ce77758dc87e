// Utility kernels of libtrident_hip: scans and per-row
// sorting.  These are not the hot path; they are written for
// correctness with coalesced access and no host round trips.
#include "dev_common.h"
#include "scan.h"
#include "tr_internal.h"

namespace tr {

namespace scan {

__global__ __launch_bounds__(1024) void k_scan_tiles(int64_t *__restrict__ sums, int64_t ntiles) {
    __shared__ int64_t tot[1024 / kWave];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int64_t carry = 0;
    for (int64_t base = 0; base < ntiles; base += 1024) {
        const int64_t i = base + threadIdx.x;
        const int64_t v = i < ntiles ? sums[i] : 0;
        const int64_t inc = wave_incl_scan(v);
        if (lane_id() == kWave - 1) tot[w] = inc;
        __syncthreads();
        int64_t off = carry;
#pragma unroll
        for (int u = 0; u < 1024 / kWave; ++u) {
            off += u < w ? tot[u] : 0;
            carry += tot[u];
        }
        if (i < ntiles) sums[i] = off + inc - v;
        __syncthreads();
    }
}

}  // namespace scan

namespace {

using namespace dev;

// plain streaming copy, 16 bytes per lane per iteration (counter calibration)
__global__ void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int64_t n16) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

__global__ void k_fill_i32(int32_t *p, int32_t v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

__global__ void k_rowptr_rebase(const int64_t *__restrict__ rp, int32_t r0, int32_t n, int32_t *__restrict__ o) {
    int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t <= n) o[t] = (int32_t)(rp[r0 + t] - rp[r0]);
}

// ---- per-row sort (keys with original positions, values gathered after) ----
// wave per row for rows up to kSortWaveMax entries
constexpr int kSortWaveMax = 2048;
constexpr int kSortBlockMax = 16384;

constexpr int kSortWaves = 4;

__global__ void k_sort_rows_wave(const int32_t *__restrict__ ptr, int32_t *__restrict__ idx,
                                 double *__restrict__ val, const double *__restrict__ val_copy,
                                 const int32_t *__restrict__ rows, int32_t nrows_list) {
    __shared__ int32_t smem[kSortWaves * 2 * kSortWaveMax];
    const int w = threadIdx.x / kWave;
    const int l = lane_id();
    int32_t li = blockIdx.x * (blockDim.x / kWave) + w;
    if (li >= nrows_list) return;
    int32_t *keys = smem + (size_t)w * 2 * kSortWaveMax;
    int32_t *pos = keys + kSortWaveMax;
    const int32_t r = rows[li];
    const int32_t b = ptr[r];
    const int n = ptr[r + 1] - b;
    for (int t = l; t < n; t += kWave) {
        keys[t] = idx[b + t];
        pos[t] = b + t;
    }
    wave_sync();
    wave_sort_lds<int32_t>(keys, pos, n);
    for (int t = l; t < n; t += kWave) {
        idx[b + t] = keys[t];
        val[b + t] = val_copy[pos[t]];
    }
}

// block-level bitonic over (key, pos) pairs in LDS or in a global scratch
// region for longer rows
template <bool kGlobal>
__global__ void k_sort_rows_block(const int32_t *__restrict__ ptr, int32_t *__restrict__ idx,
                                  double *__restrict__ val, const double *__restrict__ val_copy,
                                  const int32_t *__restrict__ rows, int32_t nrows_list,
                                  int32_t *__restrict__ gkeys, int32_t *__restrict__ gpos, int64_t gcap) {
    __shared__ int32_t smem[kGlobal ? 1 : 2 * kSortBlockMax];
    const int32_t r = rows[blockIdx.x];
    const int32_t b = ptr[r];
    const int n = ptr[r + 1] - b;
    int N = 64;
    while (N < n) N <<= 1;
    int32_t *keys;
    int32_t *pos;
    if (kGlobal) {
        if ((int64_t)N > gcap) return;  // host sizes gcap for the longest row
        keys = gkeys;
        pos = gpos;
    } else {
        keys = smem;
        pos = smem + kSortBlockMax;
    }
    for (int t = threadIdx.x; t < N; t += blockDim.x) {
        if (t < n) {
            keys[t] = idx[b + t];
            pos[t] = b + t;
        } else {
            keys[t] = kKeyPad;
            pos[t] = 0;
        }
    }
    __syncthreads();
    for (int size = 2; size <= N; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = threadIdx.x; i < (N >> 1); i += blockDim.x) {
                int lo = ((i & ~(stride - 1)) << 1) | (i & (stride - 1));
                int hi = lo + stride;
                bool up = ((lo & size) == 0);
                int32_t ka = keys[lo], kb = keys[hi];
                if ((ka > kb) == up) {
                    int32_t pa = pos[lo];
                    keys[lo] = kb;
                    keys[hi] = ka;
                    pos[lo] = pos[hi];
                    pos[hi] = pa;
                }
            }
            if (kGlobal) __threadfence_block();
            __syncthreads();
        }
    }
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        idx[b + t] = keys[t];
        val[b + t] = val_copy[pos[t]];
    }
}

// classify rows by length for the sort kernels
__global__ void k_sort_classify(const int32_t *__restrict__ ptr, int32_t m, int32_t *__restrict__ lists,
                                int32_t *__restrict__ counts, int32_t *__restrict__ maxlen) {
    int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    int32_t n = ptr[i + 1] - ptr[i];
    if (n <= 1) return;
    int c = n <= kSortWaveMax ? 0 : (n <= kSortBlockMax ? 1 : 2);
    int32_t slot = atomicAdd(&counts[c], 1);
    lists[(int64_t)c * m + slot] = i;
    if (c == 2) atomicMax(maxlen, n);
}

}  // namespace

size_t scan_tmp_bytes(int64_t n) { return sizeof(int64_t) * (size_t)(scan::tiles(n) + 1); }
void launch_exclusive_scan_i64(tr_ctx *ctx, const int64_t *in, int64_t *out, int64_t n, int64_t *tmp) {
    scan::launch(ctx, scan::ArrayIn<int64_t>{in}, out, n, tmp);
}
void launch_exclusive_scan_i32_to_i64(tr_ctx *ctx, const int32_t *in, int64_t *out, int64_t n, int64_t *tmp) {
    scan::launch(ctx, scan::ArrayIn<int32_t>{in}, out, n, tmp);
}

void launch_copy16(tr_ctx *ctx, void *dst, const void *src, size_t bytes) {
    const int64_t n16 = (int64_t)(bytes / 16);
    if (n16 <= 0) return;
    const uint32_t g = (uint32_t)std::min<int64_t>((n16 + 255) / 256, (int64_t)ctx->cu_count * 32);
    TR_LAUNCH(ctx, "copy16", k_copy16, g, 256, 0, (const uint4 *)src, (uint4 *)dst, n16);
}

void launch_fill_i32(tr_ctx *ctx, int32_t *p, int32_t v, int64_t n) {
    if (n <= 0) return;
    uint32_t g = (uint32_t)std::min<int64_t>((n + 255) / 256, 65536);
    TR_LAUNCH(ctx, "fill_i32", k_fill_i32, g, 256, 0, p, v, n);
}

void launch_rowptr_i64_to_i32(tr_ctx *ctx, const int64_t *rp64, int32_t r0, int32_t r1, int32_t *out) {
    // out[t] = rp64[r0 + t] - rp64[r0], t in [0, r1-r0]
    int32_t n = r1 - r0;
    TR_LAUNCH(ctx, "rowptr_to_i32", k_rowptr_rebase, div_up((uint64_t)n + 1, 256), 256, 0, rp64, r0, n, out);
}

void launch_sort_rows(tr_ctx *ctx, tr_csx_t *m) {
    const int32_t P = ptrdim(m);
    if (m->nnz <= 1 || P == 0) return;
    int32_t *lists = (int32_t *)scratch(ctx, S_BINS, sizeof(int32_t) * 3 * (size_t)P);
    int32_t *cnt = (int32_t *)scratch(ctx, S_BINCNT, sizeof(int32_t) * 4);
    TR_HIP(hipMemsetAsync(cnt, 0, sizeof(int32_t) * 4, ctx->stream));
    TR_LAUNCH(ctx, "sort_classify", k_sort_classify, div_up((uint64_t)P, 256), 256, 0, m->ptr_vec, P, lists, cnt,
              cnt + 3);
    int32_t hc[4];
    read_array(ctx, hc, cnt, sizeof(hc));
    double *vcopy = (double *)scratch(ctx, S_TMP_CSX, sizeof(double) * (size_t)m->nnz);
    TR_HIP(hipMemcpyAsync(vcopy, m->val, sizeof(double) * (size_t)m->nnz, hipMemcpyDeviceToDevice, ctx->stream));
    if (hc[0] > 0) {
        TR_LAUNCH(ctx, "sort_rows_wave", k_sort_rows_wave, div_up((uint64_t)hc[0], kSortWaves), kSortWaves * kWave, 0,
                  m->ptr_vec, m->idx_vec, m->val, vcopy, lists, hc[0]);
    }
    if (hc[1] > 0) {
        TR_LAUNCH(ctx, "sort_rows_block", (k_sort_rows_block<false>), (uint32_t)hc[1], 1024, 0, m->ptr_vec,
                  m->idx_vec, m->val, vcopy, lists + P, hc[1], (int32_t *)nullptr, (int32_t *)nullptr, (int64_t)0);
    }
    if (hc[2] > 0) {
        int64_t N = 64;
        while (N < hc[3]) N <<= 1;
        int32_t *g = (int32_t *)scratch(ctx, S_MISC, sizeof(int32_t) * 2 * (size_t)N);
        // one row at a time: the global scratch is shared
        for (int32_t t = 0; t < hc[2]; ++t) {
            TR_LAUNCH(ctx, "sort_rows_global", (k_sort_rows_block<true>), 1, 1024, 0, m->ptr_vec, m->idx_vec, m->val,
                      vcopy, lists + 2 * (int64_t)P + t, 1, g, g + N, N);
        }
    }
}

}  // namespace tr
