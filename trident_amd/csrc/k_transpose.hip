// Transposition (CSC <-> CSR) on gfx950: a stable radix sort of the entries by
// destination segment.
//
// Replaces cusparse_csc_to_csr (include/cusparse_helpers.cuh:607-705) and
// LocalMatrix::csc_to_csr (include/KokkosWrap.hpp:441-531).
//
// The input lists its entries by source segment, so a stable sort by
// destination leaves every destination segment ordered by source: no sort per
// row follows.  Digits of at most 10 bits, least significant first: two passes
// up to 2^20 destinations.  A pass counts digits per tile of 4096 entries,
// scans the counts (digit major) and scatters 16-byte records (destination,
// source, value); the first pass reads the matrix itself, the last writes it.
//
// What bounds it: the scattered 16-byte stores and the traffic of two passes,
// about 76 bytes an entry against the 24 that a transposition must move.  The
// form before (a global atomic per entry to count, one to place, then a sort
// of every row in LDS, long rows one workgroup at a time) was bound by atomics
// on the hub columns of an R-MAT and by its longest rows: 8 M entries on
// 500009 columns 7450 us, now 423 us (131 us of it the last scatter, 108 us the
// first).
#include <algorithm>

#include "dev_common.h"
#include "scan.h"
#include "tr_internal.h"

namespace tr {
namespace {

using namespace dev;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kRounds = 16;
constexpr int kTileEntries = kThreads * kRounds;  // a wave owns kRounds * 64 consecutive entries
constexpr int kMaxDigitBits = 10;
constexpr int kMaxDigits = 1 << kMaxDigitBits;
constexpr int kXcds = 8;
constexpr int32_t kMarkSegs = 8192;  // source segments a tile marks; beyond, a search per entry

struct __align__(16) Rec {
    int32_t key, src;
    double val;
};

struct Pass {
    const int32_t *ptr, *idx;  // the matrix (first pass)
    const double *val;
    const Rec *in;             // the pass before
    Rec *out;                  // to the next pass
    int32_t *okey, *oidx;      // the result (last pass)
    double *oval;
    int32_t *hist;             // digit counts, [digit][tile]
    const int64_t *off;        // their exclusive sums
    int64_t n;                 // entries read
    int32_t nseg;              // source segments
    int32_t klo, kspan;        // destinations [klo, klo + kspan) take part (first pass)
    int32_t shift, nbits, ntiles;
};

// Consecutive workgroups go to different XCDs.  Tiles whose runs of one digit
// meet in a cache line should not, so each XCD takes consecutive tiles.
__device__ __forceinline__ int32_t tile_of_block(int32_t ntiles) {
    const int32_t per = (ntiles + kXcds - 1) / kXcds;
    return (int32_t)(blockIdx.x % kXcds) * per + (int32_t)(blockIdx.x / kXcds);
}

inline uint32_t tile_blocks(int32_t ntiles) { return div_up((uint64_t)ntiles, kXcds) * kXcds; }

template <bool kFirst>
__global__ __launch_bounds__(kThreads) void k_radix_count(const Pass a) {
    __shared__ int32_t h[kMaxDigits];
    const int32_t tile = tile_of_block(a.ntiles);
    if (tile >= a.ntiles) return;
    const int ndig = 1 << a.nbits;
    for (int d = threadIdx.x; d < ndig; d += kThreads) h[d] = 0;
    __syncthreads();
    int32_t key[kRounds];
#pragma unroll
    for (int t = 0; t < kRounds; ++t) {
        const int64_t e = (int64_t)tile * kTileEntries + t * kThreads + threadIdx.x;
        key[t] = -1;
        if (e < a.n) key[t] = kFirst ? a.idx[e] - a.klo : a.in[e].key;
    }
#pragma unroll
    for (int t = 0; t < kRounds; ++t)
        if ((uint32_t)key[t] < (uint32_t)a.kspan) atomicAdd(&h[(key[t] >> a.shift) & (ndig - 1)], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < ndig; d += kThreads) a.hist[(int64_t)d * a.ntiles + tile] = h[d];
}

// Last source segment that starts at or before entry e < ptr[nseg], searched
// 64 probes at a time (wave-uniform)
__device__ __forceinline__ int32_t segment_of(const int32_t *__restrict__ ptr, int32_t nseg, int64_t e) {
    int32_t lo = 0, hi = nseg;  // ptr[lo] <= e < ptr[hi]
    while (hi - lo > 1) {
        const int32_t step = (hi - lo + kWave - 1) / kWave;
        const int64_t mid = (int64_t)lo + (int64_t)lane_id() * step;
        const int c = __popcll(ballot(mid < hi && (int64_t)ptr[mid] <= e));  // lane 0's is true
        const int64_t up = (int64_t)lo + (int64_t)c * step;
        lo = (int32_t)(up - step);
        hi = (int32_t)(up < hi ? up : hi);
    }
    return lo;
}

template <bool kFirst, bool kLast>
__global__ __launch_bounds__(kThreads) void k_radix_scatter(const Pass a) {
    // entries of a digit in the tile's waves before, then in the rounds before
    __shared__ uint16_t cnt[kWaves][kMaxDigits];
    __shared__ int64_t base[kMaxDigits];
    __shared__ __align__(16) int32_t owner[kFirst ? kTileEntries : 4];
    __shared__ int32_t seg[2], top[kWaves];
    const int tid = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int32_t tile = tile_of_block(a.ntiles);
    if (tile >= a.ntiles) return;
    const int64_t e0 = (int64_t)tile * kTileEntries;
    const int64_t e1 = min(e0 + kTileEntries, a.n);
    const int ndig = 1 << a.nbits;
    for (int d = tid; d < ndig; d += kThreads) {
#pragma unroll
        for (int u = 0; u < kWaves; ++u) cnt[u][d] = 0;
        base[d] = a.off[(int64_t)d * a.ntiles + tile];
    }
    // the entries, and their source segments
    int32_t key[kRounds], src[kRounds];
    double val[kRounds];
    const int64_t we = e0 + (int64_t)w * (kRounds * kWave) + l;
#pragma unroll
    for (int t = 0; t < kRounds; ++t) {
        const int64_t e = min(we + t * kWave, e1 - 1);
        if constexpr (kFirst) {
            key[t] = a.idx[e] - a.klo;
            val[t] = a.val[e];
        } else {
            const Rec r = a.in[e];
            key[t] = r.key;
            src[t] = r.src;
            val[t] = r.val;
        }
    }
    if constexpr (kFirst) {
        if (w < 2) {
            const int32_t s = segment_of(a.ptr, a.nseg, w ? e1 - 1 : e0);
            if (l == 0) seg[w] = s;
        }
        for (int t = tid; t < kTileEntries; t += kThreads) owner[t] = 0;
        __syncthreads();
        const int32_t s0 = seg[0], s1 = seg[1];
        if (s1 - s0 <= kMarkSegs) {  // block-uniform
            // non-empty segments mark their first entry; a running maximum
            // gives every entry its segment
            for (int32_t s = s0 + 1 + tid; s <= s1; s += kThreads) {
                const int32_t p = a.ptr[s];
                if (a.ptr[s + 1] > p) owner[p - e0] = s - s0;
            }
            __syncthreads();
            constexpr int kPer = kTileEntries / kThreads;
            int32_t m[kPer];
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                m[u] = owner[tid * kPer + u];
                if (u) m[u] = max(m[u], m[u - 1]);
            }
            const int32_t inc = (int32_t)wave_incl_max((uint32_t)m[kPer - 1]);
            int32_t run = __shfl_up(inc, 1, kWave);
            if (l == 0) run = 0;
            if (l == kWave - 1) top[w] = inc;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kWaves - 1; ++u) run = max(run, u < w ? top[u] : 0);
#pragma unroll
            for (int u = 0; u < kPer; ++u) owner[tid * kPer + u] = max(m[u], run);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < kRounds; ++t) src[t] = s0 + owner[w * (kRounds * kWave) + t * kWave + l];
        } else {
            for (int t = 0; t < kRounds; ++t) {
                const int64_t e = min(we + t * kWave, e1 - 1);
                int32_t lo = s0, hi = s1;
                while (lo < hi) {
                    const int32_t mid = lo + ((hi - lo + 1) >> 1);
                    if ((int64_t)a.ptr[mid] <= e) lo = mid;
                    else hi = mid - 1;
                }
                owner[w * (kRounds * kWave) + t * kWave + l] = lo;
            }
#pragma unroll
            for (int t = 0; t < kRounds; ++t) src[t] = owner[w * (kRounds * kWave) + t * kWave + l];
        }
    }
    __syncthreads();
    // rank of each entry among its digit's in the wave: lanes with the same
    // digit are found by a ballot per digit bit; the rounds go in order
    uint16_t rank[kRounds];
    uint32_t valid = 0;
    uint16_t *wc = cnt[w];
#pragma unroll
    for (int t = 0; t < kRounds; ++t) {
        const bool ok = we + t * kWave < e1 && (!kFirst || (uint32_t)key[t] < (uint32_t)a.kspan);
        const int d = (key[t] >> a.shift) & (ndig - 1);
        uint64_t peers = ballot(ok);
        for (int b = 0; b < a.nbits; ++b) {
            const bool bit = (d >> b) & 1;
            const uint64_t m = ballot(bit);
            peers &= bit ? m : ~m;
        }
        if (ok) {
            valid |= 1u << t;
            const int below = rank_below(peers);
            const uint16_t c = wc[d];
            rank[t] = (uint16_t)(c + below);
            wave_sync();
            if (below == 0) wc[d] = (uint16_t)(c + __popcll(peers));
        }
        wave_sync();
    }
    __syncthreads();
    for (int d = tid; d < ndig; d += kThreads) {
        int run = 0;
#pragma unroll
        for (int u = 0; u < kWaves; ++u) {
            const int c = cnt[u][d];
            cnt[u][d] = (uint16_t)run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kRounds; ++t) {
        if (!(valid & (1u << t))) continue;
        const int d = (key[t] >> a.shift) & (ndig - 1);
        const int64_t q = base[d] + wc[d] + rank[t];
        if constexpr (kLast) {
            a.okey[q] = key[t];
            a.oidx[q] = src[t];
            a.oval[q] = val[t];
        } else {
            Rec r;
            r.key = key[t];
            r.src = src[t];
            r.val = val[t];
            a.out[q] = r;
        }
    }
}

// optr[klo + k] = base + first sorted entry of destination k, k in [0, n]
__global__ void k_segment_starts(const int32_t *__restrict__ key, int32_t cnt, int64_t base, int32_t klo, int32_t n,
                                 int32_t *__restrict__ optr) {
    const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > n) return;
    int32_t lo = 0, hi = cnt;
    while (lo < hi) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (key[mid] < k) lo = mid + 1;
        else hi = mid;
    }
    optr[klo + k] = (int32_t)(base + lo);
}

// A pool block for the length of one call (work on it is ordered on the
// context's stream, so its release needs no wait)
struct Temp {
    tr_ctx *ctx;
    void *p;
    Temp(tr_ctx *c, size_t bytes) : ctx(c), p(c->pool.alloc(bytes)) {}
    ~Temp() { ctx->pool.release(p); }
    Temp(const Temp &) = delete;
    Temp &operator=(const Temp &) = delete;
};

int bits_for(int32_t n) {
    int b = 1;
    while (b < 31 && ((int64_t)1 << b) < n) ++b;
    return b;
}

template <bool kFirst>
void count_digits(tr_ctx *ctx, const Pass &a, int64_t *off) {
    TR_LAUNCH(ctx, "transpose_count", k_radix_count<kFirst>, tile_blocks(a.ntiles), kThreads, 0, a);
    scan::launch(ctx, scan::ArrayIn<int32_t>{a.hist}, off, (int64_t)a.ntiles << a.nbits, nullptr);
}

template <bool kFirst, bool kLast>
void scatter(tr_ctx *ctx, const Pass &a) {
    TR_LAUNCH(ctx, "transpose_scatter", (k_radix_scatter<kFirst, kLast>), tile_blocks(a.ntiles), kThreads, 0, a);
}

int32_t tiles_of(int64_t n) { return (int32_t)((n + kTileEntries - 1) / kTileEntries); }

// Sorts the entries of the destinations [a.klo, a.klo + a.kspan) into the
// result from entry `done` on, and returns how many they are.  all: they are
// all entries, so that nothing is read back to learn it.  cnt: their number, as
// soon as it is known.
int64_t transpose_range(tr_ctx *ctx, Pass a, const tr_csx_t *out, int64_t done, bool all, int64_t &cnt) {
    const int bits = bits_for(a.kspan), passes = (bits + kMaxDigitBits - 1) / kMaxDigitBits;
    a.nbits = (bits + passes - 1) / passes;
    const size_t cells = (size_t)a.ntiles << a.nbits;
    Temp hist(ctx, sizeof(int32_t) * cells), offsets(ctx, sizeof(int64_t) * (cells + 1));
    int64_t *off = (int64_t *)offsets.p;
    a.hist = (int32_t *)hist.p;
    a.off = off;
    cnt = a.n;
    if (!all) {
        count_digits<true>(ctx, a, off);
        cnt = read_scalar<int64_t>(ctx, off + cells);
    }
    const size_t n = (size_t)std::max<int64_t>(cnt, 1);
    Temp keys(ctx, sizeof(int32_t) * n), r0(ctx, passes > 1 ? sizeof(Rec) * n : 1),
        r1(ctx, passes > 2 ? sizeof(Rec) * n : 1);
    a.okey = (int32_t *)keys.p;
    a.oidx = out->idx_vec + done;
    a.oval = out->val + done;
    if (all) count_digits<true>(ctx, a, off);
    a.out = (Rec *)r0.p;
    if (cnt > 0) passes > 1 ? scatter<true, false>(ctx, a) : scatter<true, true>(ctx, a);
    a.n = cnt;
    a.ntiles = tiles_of(cnt);
    for (int p = 1; p < passes && cnt > 0; ++p) {
        a.shift = p * a.nbits;
        a.in = (const Rec *)(p % 2 ? r0.p : r1.p);
        a.out = (Rec *)(p % 2 ? r1.p : r0.p);
        count_digits<false>(ctx, a, off);
        p + 1 < passes ? scatter<false, false>(ctx, a) : scatter<false, true>(ctx, a);
    }
    TR_LAUNCH(ctx, "transpose_starts", k_segment_starts, div_up((uint64_t)a.kspan + 1, 256), 256, 0, a.okey,
              (int32_t)cnt, done, a.klo, a.kspan, out->ptr_vec);
    return cnt;
}

}  // namespace

// out receives the segments of m's other dimension (for a CSR m: the CSR of
// m^T); its descriptor and storage are prepared by the caller and m is valid.
//
// Scratch: 20 bytes an entry (36 beyond 2^20 destinations) plus 12 << digit
// bits a tile.  Where that cannot be had, the destinations are taken in ranges
// that are halved until one's entries fit, down to 1024 destinations (4 bytes
// an entry, straight from the matrix to the result).  A range costs one read
// of the matrix and a wait, so their number follows from the room that is
// missing and not from the number of destinations; ranges grow again where
// they held few entries.  (With room for 10 bytes an entry: 2 M entries over
// 2^20 destinations 53.4 ms by 1024 destinations a range, now 0.44; 8 M over
// 2^22 372 ms, now 0.83.)
void launch_transpose(tr_ctx *ctx, const tr_csx_t *m, tr_csx_t *out) {
    const int64_t O = otherdim(m);
    if (m->nnz == 0) {
        launch_fill_i32(ctx, out->ptr_vec, 0, O + 1);
        return;
    }
    Pass a{};
    a.ptr = m->ptr_vec;
    a.idx = m->idx_vec;
    a.val = m->val;
    a.n = m->nnz;
    a.nseg = ptrdim(m);
    a.ntiles = tiles_of(m->nnz);
    int64_t done = 0, span = O, refused = INT64_MAX;  // refused: entries of the least range that did not fit
    for (int64_t k = 0; k < O;) {
        a.klo = (int32_t)k;
        a.kspan = (int32_t)std::min(span, O - k);
        int64_t cnt = 0;
        try {
            done += transpose_range(ctx, a, out, done, a.kspan == O, cnt);
        } catch (const Error &e) {
            if (e.code != TR_ERR_OOM || a.kspan <= kMaxDigits) throw;
            if (cnt > 0) refused = std::min(refused, cnt);
            span = kMaxDigits;
            while (2 * span < a.kspan) span *= 2;
            continue;
        }
        k += a.kspan;
        if (cnt <= refused / 4) span *= 2;
    }
}

}  // namespace tr
