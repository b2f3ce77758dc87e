// Device-side helpers shared by the gfx950 kernels: wave64 primitives,
// LDS ordering and the sorting network used to emit sorted rows.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tr {
namespace dev {

constexpr int kWave = 64;
constexpr int32_t kEmpty = -1;          // empty hash slot (columns are >= 0)
constexpr int32_t kKeyPad = 0x7fffffff;  // sort padding key

// Global-memory (address space 1) view of a device pointer.  Accesses
// through it are global instructions, which count on vmcnt only; a flat
// access (what a pointer read from memory compiles to) also counts on
// lgkmcnt, so every wait for an LDS result would wait for it as well.
#define TR_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ TR_GLOBAL T *as_global(T *p) {
    return (TR_GLOBAL T *)p;
}

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Order this wave's LDS accesses across the call (and wait for outstanding
// LDS operations); no cross-wave synchronisation.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint64_t ballot(bool p) { return (uint64_t)__ballot(p ? 1 : 0); }

// Number of set bits of `mask` below this lane.
__device__ __forceinline__ int rank_below(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// ---- lane exchange in registers ----
// Fixed lane patterns go through DPP moves and gfx950's permlane swaps:
// vector instructions on registers.  __shfl is an LDS round trip
// (ds_bpermute) per 32 bits and step, which made the six dependent steps of a
// scan cost several hundred cycles in kernels that wait on LDS anyway
// (Galerkin 96^3 4.74 -> 4.20 ms, R-MAT s17 15.85 -> 15.57 ms, an add of 95 M
// entries 1.53 -> 1.49 ms, products the same bits).
// Lanes that a DPP pattern leaves out (row edges, masked rows) read 0.
template <int kCtrl, int kRowMask = 0xf>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRowMask, 0xf, false);
}

// Value of a 32-bit or 64-bit type moved through a 32-bit lane exchange f.
template <typename T, typename F>
__device__ __forceinline__ T by_words(T v, F &&f) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32-bit or 64-bit values");
    if constexpr (sizeof(T) == 4) {
        uint32_t u;
        __builtin_memcpy(&u, &v, 4);
        u = f(u);
        __builtin_memcpy(&v, &u, 4);
    } else {
        uint32_t u[2];
        __builtin_memcpy(u, &v, 8);
        u[0] = f(u[0]);
        u[1] = f(u[1]);
        __builtin_memcpy(&v, u, 8);
    }
    return v;
}

template <int kCtrl, int kRowMask = 0xf, typename T>
__device__ __forceinline__ T dpp(T v) {
    return by_words(v, [](uint32_t u) { return dpp_u32<kCtrl, kRowMask>(u); });
}

// Value of lane `l` (wave-uniform), as a wave-uniform value.
template <typename T>
__device__ __forceinline__ T read_lane(T v, int l) {
    return by_words(v, [l](uint32_t u) { return (uint32_t)__builtin_amdgcn_readlane((int)u, l); });
}

// Inclusive prefix sum over the wave: shifts by 1, 2, 4, 8 inside each row of
// 16 lanes, then the row totals broadcast to the rows above.
template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v) {
    v += dpp<0x111>(v);       // row_shr:1
    v += dpp<0x112>(v);       // row_shr:2
    v += dpp<0x114>(v);       // row_shr:4
    v += dpp<0x118>(v);       // row_shr:8
    v += dpp<0x142, 0xa>(v);  // lane 15 of rows 0, 2 to rows 1, 3
    v += dpp<0x143, 0xc>(v);  // lane 31 to rows 2, 3
    return v;
}

// Inclusive running maximum over the wave of unsigned values.
__device__ __forceinline__ uint32_t wave_incl_max(uint32_t v) {
    v = max(v, dpp<0x111>(v));
    v = max(v, dpp<0x112>(v));
    v = max(v, dpp<0x114>(v));
    v = max(v, dpp<0x118>(v));
    v = max(v, dpp<0x142, 0xa>(v));
    return max(v, dpp<0x143, 0xc>(v));
}

// Sum over the wave, wave-uniform.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    return read_lane(wave_incl_scan(v), kWave - 1);
}

// Value of lane (this lane ^ kX), kX a power of two.
template <int kX, typename T>
__device__ __forceinline__ T lane_xor(T v) {
    static_assert(kX == 1 || kX == 2 || kX == 4 || kX == 8 || kX == 16 || kX == 32, "power of two");
    if constexpr (kX == 1) return dpp<0xb1>(v);  // quad_perm 1,0,3,2
    if constexpr (kX == 2) return dpp<0x4e>(v);  // quad_perm 2,3,0,1
    if constexpr (kX == 4) return dpp<0x1b>(dpp<0x141>(v));  // half-row mirror (xor 7), then quad mirror (xor 3)
    if constexpr (kX == 8) return dpp<0x128>(v);  // row_ror:8
    if constexpr (kX == 16) {
        const bool odd = (lane_id() & 16) != 0;
        return by_words(v, [odd](uint32_t u) {
            const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
            return odd ? (uint32_t)r[0] : (uint32_t)r[1];
        });
    }
    const bool high = (lane_id() & 32) != 0;
    return by_words(v, [high](uint32_t u) {
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return high ? (uint32_t)r[0] : (uint32_t)r[1];
    });
}

// Multiplicative hash of a column index into a table of 2^log2T slots.
__device__ __forceinline__ uint32_t hash_slot(int32_t key, uint32_t log2T) {
    return ((uint32_t)key * 0x9E3779B1u) >> (32u - log2T);
}

template <int kSize, int kStride, typename V>
__device__ __forceinline__ void bitonic_step(int32_t &k, V &v, int l) {
    const int32_t pk = lane_xor<kStride>(k);
    const V pv = lane_xor<kStride>(v);
    const bool take_min = ((l & kStride) == 0) == ((l & kSize) == 0);
    if (take_min ? (pk < k) : (pk > k)) {
        k = pk;
        v = pv;
    }
    if constexpr (kStride > 1) bitonic_step<kSize, kStride / 2>(k, v, l);
}

// Ascending register bitonic sort of one (key, value) per lane.
template <int kSize = 2, typename V>
__device__ __forceinline__ void bitonic_wave(int32_t &k, V &v) {
    bitonic_step<kSize, kSize / 2>(k, v, lane_id());
    if constexpr (kSize < kWave) bitonic_wave<kSize * 2>(k, v);
}

// Sort keys[0..n) (with vals) ascending in LDS by one wave.  The table
// region must hold at least N = max(64, next_pow2(n)) entries; entries
// [n, N) are overwritten with padding.
template <typename V>
__device__ void wave_sort_lds(int32_t *keys, V *vals, int n) {
    const int l = lane_id();
    int N = 64;
    while (N < n) N <<= 1;
    for (int t = n + l; t < N; t += kWave) keys[t] = kKeyPad;
    wave_sync();
    if (N == 64) {
        // register bitonic sort, one entry per lane
        int32_t k = keys[l];
        V v = vals[l];
        bitonic_wave(k, v);
        wave_sync();
        keys[l] = k;
        vals[l] = v;
        wave_sync();
        return;
    }
    for (int size = 2; size <= N; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = l; i < (N >> 1); i += kWave) {
                int lo = ((i & ~(stride - 1)) << 1) | (i & (stride - 1));
                int hi = lo + stride;
                bool up = ((lo & size) == 0);
                int32_t ka = keys[lo], kb = keys[hi];
                if ((ka > kb) == up) {
                    V va = vals[lo], vb = vals[hi];
                    keys[lo] = kb;
                    keys[hi] = ka;
                    vals[lo] = vb;
                    vals[hi] = va;
                }
            }
            wave_sync();
        }
    }
}

// Move the occupied slots of a hash table to its front, preserving nothing
// about order.  Returns the number of occupied slots (wave-uniform).
template <typename V>
__device__ int wave_compact_lds(int32_t *keys, V *vals, int T) {
    const int l = lane_id();
    int n = 0;
    for (int base = 0; base < T; base += kWave) {
        int32_t k = keys[base + l];
        V v = vals[base + l];
        bool occ = (k != kEmpty);
        uint64_t m = ballot(occ);
        int r = rank_below(m);
        wave_sync();
        if (occ) {
            keys[n + r] = k;
            vals[n + r] = v;
        }
        wave_sync();
        n += __popcll(m);
    }
    return n;
}

}  // namespace dev
}  // namespace tr
