// Sorted sparse add C = X + Y on gfx950 (partial-C accumulation).
//
// Replaces the spadd of LocalMatrix::spadd / sp_mma
// (include/KokkosWrap.hpp:341-352, :394-439: KokkosSparse spadd with
// alpha = beta = 1) and cusparse_spgeam (include/cusparse_helpers.cuh:
// 799-905: csrgeam2 bufferSize / Nnz / compute with a host sync after each).
//
// The rows of a tile are merged as one sequence: row ends and merged entries
// (every row's X and Y entries in column order, ties X first, so that an equal
// column appears as an adjacent (X, Y) pair that becomes one entry x + y) are
// cut into units of kAddUnit steps.  A unit takes consecutive entries of X and
// of Y, whatever the row lengths are, so its loads are contiguous, every entry
// is read once and every thread has four merged positions to do.
//  1. split   per unit boundary, the row and the X entry it falls on;
//  2. merge   of the columns, a wave per unit in registers: two bits per merged
//             position say what it is, and the kept ones are counted; for
//             caller tiles also the column range and order checks, since every
//             entry passes by once;
//  3. scan    over the units;
//  4. write   entries and row pointers, from the bits and the values alone.
//
// What bounds it: HBM bandwidth in the write pass, vector instructions in the
// merge.  262144 rows, 95 M entries: split 46, merge with checks 221, write
// 447 us (24 bytes moved an entry); a wave per chunk of one row, which searched
// its share of the merge in LDS in both passes, took 133 for the checks, 343
// and 795 us.
//
// Like the multiply, the add runs over a table of tasks (a plain call passes
// its one task by value; the batched stage executor adds all tile products
// into their partial-C tiles in one pass).  X rows are addressed either by an
// int32 pointer per task or by a 64-bit pointer over the global row space (the
// product arena of a batch).
#include "csr_units.h"
#include "dev_common.h"
#include "tr_internal.h"
#include "spgemm_types.h"

#include <algorithm>

namespace tr {
namespace {

using namespace dev;

constexpr int kWords = 8;               // 64 merged positions each
constexpr int kAddUnit = kWords * kWave;  // row ends plus merged entries of a work unit
constexpr int kAddWaves = 4;
constexpr int kAddThreads = kAddWaves * kWave;
// Units whose merge is kept from the count to the write pass (128 bytes each,
// 1% of what their entries take); an add of more units is merged again, this
// many units at a time.  (A stage that adds 1.4e9 products into 7.2e9 entries:
// kept by 2^22 units, merged twice, 25.6 ms of merges.)
constexpr int64_t kMaxKept = 1 << 25, kMinKept = 1 << 10;

// Where row i of X and Y begins, counted from the task's first entry
__device__ __forceinline__ int64_t x_row(const AddTaskDev &T, int32_t i) {
    return T.xp64 ? as_global(T.xp64)[T.row_base + i] - as_global(T.xp64)[T.row_base] : (int64_t)as_global(T.xp)[i];
}
__device__ __forceinline__ int64_t y_row(const AddTaskDev &T, int32_t i) { return (int64_t)as_global(T.yp)[i]; }

__device__ __forceinline__ const TR_GLOBAL int32_t *x_idx(const AddTaskDev &T) {
    return as_global(T.xi) + (T.xp64 ? as_global(T.xp64)[T.row_base] : 0);
}
__device__ __forceinline__ const TR_GLOBAL double *x_val(const AddTaskDev &T) {
    return as_global(T.xv) + (T.xp64 ? as_global(T.xp64)[T.row_base] : 0);
}

__device__ __forceinline__ int add_task_of(const AddTaskDev *__restrict__ tasks, int nt, int32_t unit) {
    int lo = 0, hi = nt - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tasks[mid].unit0 <= unit) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// number of X entries among the first t merged positions of a row (ties take
// X first)
template <typename P>
__device__ __forceinline__ int32_t merge_split(P xi, int32_t lx, P yi, int32_t ly, int32_t t) {
    int32_t lo = t - ly > 0 ? t - ly : 0;
    int32_t hi = t < lx ? t : lx;
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (xi[mid] <= yi[t - 1 - mid]) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int64_t clamp64(int64_t v, int64_t lo, int64_t hi) { return min(max(v, lo), hi); }

// First of the task's rows [lo, hi] whose end is among the merged steps from d
// on, found by a whole wave: 64 rows are probed at a time.
__device__ __forceinline__ int64_t row_of(const AddTaskDev &T, int64_t d, int l) {
    int64_t lo = max((int64_t)0, d - T.nx - T.ny), hi = min(d, (int64_t)T.m);
    while (lo < hi) {
        const int64_t step = (hi - lo + kWave - 1) / kWave;
        const int64_t p = lo + (l + 1) * step - 1;  // the last row of this lane's share
        const bool before = p < hi && x_row(T, (int32_t)p + 1) + y_row(T, (int32_t)p + 1) <= d - 1 - p;
        const int64_t q = lo + __popcll(ballot(before)) * step;
        hi = min(hi, q + step - 1);
        lo = min(q, hi);
    }
    return lo;
}

// First row whose end the unit holds, and first X entry, of every unit.  In
// bounds whatever the row pointers hold.  A wave's 64 boundaries lie between
// its first and its last, which it looks up together: the rows between are few
// and near (186 k units over 262144 rows: 46 us, 56 with a search of all rows
// by every lane; the columns that the split of a row reads are most of it).
__global__ __launch_bounds__(256) void k_add_split(const AddTaskDev *__restrict__ tasks, int nt, const AddTaskDev one,
                                                   int32_t nunits, const int32_t *__restrict__ guard,
                                                   int2 *__restrict__ split) {
    const int32_t u = blockIdx.x * 256 + threadIdx.x;
    const int l = lane_id();
    const int32_t ua = __builtin_amdgcn_readfirstlane(u), ub = min(ua + kWave, nunits) - 1;
    if (ua >= nunits || (guard && *guard)) return;
    const int ta = tasks ? add_task_of(tasks, nt, ua) : 0;
    int64_t row_a = 0, row_b = INT32_MAX;
    if (!tasks || add_task_of(tasks, nt, ub) == ta) {
        const AddTaskDev &S = tasks ? tasks[ta] : one;
        const int64_t steps = (int64_t)S.m + S.nx + S.ny;
        row_a = row_of(S, min((int64_t)(ua - S.unit0) * kAddUnit, steps), l);
        row_b = row_of(S, min((int64_t)(ub - S.unit0) * kAddUnit, steps), l);
    }
    if (u >= nunits) return;
    const AddTaskDev &T = tasks ? tasks[add_task_of(tasks, nt, u)] : one;
    const int64_t d = min((int64_t)(u - T.unit0) * kAddUnit, (int64_t)T.m + T.nx + T.ny);
    int64_t lo = max(max((int64_t)0, d - T.nx - T.ny), row_a), hi = min(min(d, (int64_t)T.m), row_b);
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (x_row(T, (int32_t)mid + 1) + y_row(T, (int32_t)mid + 1) <= d - 1 - mid) lo = mid + 1;
        else hi = mid;
    }
    const int32_t row = (int32_t)lo;
    const int64_t j = d - row;  // merged entries before the unit
    int64_t xa = T.nx;
    if (row < T.m) {
        const int64_t x0 = clamp64(x_row(T, row), 0, T.nx), x1 = clamp64(x_row(T, row + 1), x0, T.nx);
        const int64_t y0 = clamp64(y_row(T, row), 0, T.ny), y1 = clamp64(y_row(T, row + 1), y0, T.ny);
        const int64_t t = clamp64(j - x0 - y0, 0, x1 - x0 + y1 - y0);
        xa = x0 + merge_split(x_idx(T) + x0, (int32_t)(x1 - x0), as_global(T.yi) + y0, (int32_t)(y1 - y0), (int32_t)t);
    }
    xa = clamp64(xa, max((int64_t)0, j - T.ny), min(j, T.nx));
    split[u] = make_int2(row, (int32_t)xa);
}

// A wave-uniform pointer in scalar registers
template <typename P>
__device__ __forceinline__ P *uniform_ptr(P *p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return (P *)((uint64_t)hi << 32 | lo);
}

// What a unit takes: its rows [i0, i1] (the ends of [i0, i1) are its own), X
// entries [xa, xa + nx) and Y entries [ya, ya + ny).  false: row pointers that
// are not monotone, or rows that are not sorted.
struct AddUnit {
    int64_t xa, ya;
    int32_t i0, i1, nx, ny;
    bool first, last;  // of its task
};

__device__ __forceinline__ bool add_unit(const AddTaskDev &T, int32_t u, const int2 *__restrict__ split, AddUnit &U) {
    const int64_t steps = (int64_t)T.m + T.nx + T.ny;
    const int64_t d0 = min((int64_t)(u - T.unit0) * kAddUnit, steps), d1 = min(d0 + kAddUnit, steps);
    U.first = u == T.unit0;
    U.last = d1 == steps;
    const int2 s0 = split[u];
    const int2 s1 = U.last ? make_int2(T.m, (int32_t)T.nx) : split[u + 1];
    auto uniform = [](int32_t v) { return __builtin_amdgcn_readfirstlane(v); };  // (a unit is a wave's)
    U.i0 = uniform(s0.x);
    U.i1 = uniform(s1.x);
    U.xa = uniform(s0.y);
    U.ya = d0 - U.i0 - U.xa;
    U.nx = uniform(s1.y) - (int32_t)U.xa;
    U.ny = uniform((int32_t)(d1 - d0)) - (U.i1 - U.i0) - U.nx;
    return U.i1 >= U.i0 && U.nx >= 0 && U.ny >= 0 && U.nx + U.ny <= kAddUnit;
}

template <typename K>
__device__ __forceinline__ K less_of(K a, K b) {
    return a < b ? a : b;
}
template <typename K>
__device__ __forceinline__ K greater_of(K a, K b) {
    return a < b ? b : a;
}

// One exchange of a bitonic merge between lanes kX apart: the lower lane takes
// the lesser key, the upper one the greater.  32-bit keys: lanes 32 and 16
// apart by swapping halves of two registers, so that one minimum and one
// maximum serve both; 8 and 4 apart by shifts that write only the lanes they
// are for (four instructions a pair of registers instead of up to fourteen).
template <int kX, typename K>
__device__ __forceinline__ void exchange(K (&k)[kWords], int l) {
    if constexpr (sizeof(K) == 4 && kX >= 16) {
#pragma unroll
        for (int r = 0; r < kWords; r += 2) {
            const auto v = kX == 32 ? __builtin_amdgcn_permlane32_swap(k[r], k[r + 1], false, false)
                                    : __builtin_amdgcn_permlane16_swap(k[r], k[r + 1], false, false);
            const uint32_t a = less_of<uint32_t>(v[0], v[1]), b = greater_of<uint32_t>(v[0], v[1]);
            const auto o = kX == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false)
                                    : __builtin_amdgcn_permlane16_swap(a, b, false, false);
            k[r] = o[0];
            k[r + 1] = o[1];
        }
    } else if constexpr (sizeof(K) == 4 && kX >= 4) {
        // banks of four lanes: 0 and 1 (or 0 and 2) are the lower lanes
        constexpr int kLow = kX == 8 ? 0x3 : 0x5;
#pragma unroll
        for (int r = 0; r < kWords; ++r) {
            const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)k[r], 0x100 + kX, 0xf, kLow, false);
            const uint32_t down = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[r], 0x110 + kX, 0xf, 0xf ^ kLow, false);
            k[r] = greater_of<uint32_t>(down, less_of<uint32_t>(up, k[r]));
        }
    } else {
        const bool upper = (l & kX) != 0;
#pragma unroll
        for (int r = 0; r < kWords; ++r) {
            const K o = lane_xor<kX>(k[r]);
            const K a = less_of(k[r], o), b = greater_of(k[r], o);
            k[r] = upper ? b : a;
        }
    }
}

// The value of the lane below; `first` for lane 0
template <typename K>
__device__ __forceinline__ K lane_below(K v, K first, int l) {
    if constexpr (sizeof(K) == 4) return (K)__builtin_amdgcn_update_dpp((int)first, (int)v, 0x138, 0xf, 0xf, false);
    const K p = dpp<0x138>(v);
    return l == 0 ? first : p;
}

// bits [lo, hi) of a unit's positions that lie in its word r
__device__ __forceinline__ uint64_t word_span(int32_t lo, int32_t hi, int r) {
    const int32_t a = max(lo - r * kWave, 0), b = min(hi - r * kWave, kWave);
    return a >= b ? 0 : (~0ull >> (kWave - (b - a))) << a;
}

// Merges each unit's X and Y entries, a wave per unit, and stores for each of
// its merged positions one bit "from Y" and one bit "folded into the X entry
// before it" (kWords words of each), and the number that is kept.
//
// An entry's key is (row of the unit, column, side).  X ascending from the
// front and Y descending from the back are a bitonic sequence, so the merge is
// 9 exchange steps in registers, 3 between a lane's own 8 keys and 6 between
// lanes: no search, no LDS and no barrier, and a wave reads X and Y in whole
// lines.  Vector instructions bound it (78% of the cycles, scalar ones 64%; a
// block that searched each thread's merge split in LDS: 627 us where this takes
// 221).
// Only a unit with row ends goes through LDS, for the entries' rows.
// K: 32-bit keys hold 513 rows and 21 bits of column, which is all that the
// exchanges move; wider tiles take 64-bit keys.
//
// kCheck: findings[4 * {X: 0, Y: 1} + {1: column out of range, 2: order}]
template <typename K, bool kCheck>
__global__ __launch_bounds__(kAddThreads) void k_add_merge(const AddTaskDev *__restrict__ tasks, int nt,
                                                          const AddTaskDev one, int32_t u0, int32_t u1,
                                                          const int2 *__restrict__ split,
                                                          const int32_t *__restrict__ guard,
                                                          uint64_t *__restrict__ bits, int32_t *__restrict__ counts,
                                                          uint8_t *__restrict__ findings) {
    constexpr int kRowShift = sizeof(K) == 4 ? 22 : 32;
    constexpr K kPad = ~(K)0;
    __shared__ __align__(16) int32_t ends[kAddWaves][kAddUnit];
    const int l = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int32_t u = u0 + (int32_t)blockIdx.x * kAddWaves + w;
    if (u >= u1) return;
    if (guard && *guard) {  // a replay that met another pattern than the planned one
        if (counts && l == 0) counts[u] = 0;
        return;
    }
    AddTaskDev T = one;
    if (tasks) T = tasks[add_task_of(tasks, nt, u)];
    AddUnit U;
    if (!add_unit(T, u, split, U)) {
        if (counts && l == 0) counts[u] = 0;
        if (kCheck && l == 0) findings[2] = 1;
        return;
    }
    const int32_t nx = U.nx, ny = U.ny, n = nx + ny;
    const TR_GLOBAL int32_t *xi = uniform_ptr(x_idx(T) + U.xa);
    const TR_GLOBAL int32_t *yi = uniform_ptr(as_global(T.yi) + U.ya);
    // position e: X entry e, or from the back Y entry kAddUnit - 1 - e
    int32_t c[kWords], cy[kWords];
#pragma unroll
    for (int r = 0; r < kWords; ++r) {
        c[r] = cy[r] = -1;
        if (r * kWave + l < nx) c[r] = xi[r * kWave + l];
    }
    const TR_GLOBAL int32_t *const yb = yi + (kAddUnit - kWave);  // (64 entries a word, the lanes backwards)
#pragma unroll
    for (int r = 0; r < kWords; ++r)
        if (r * kWave + l >= kAddUnit - ny) cy[r] = (yb - r * kWave)[(uint32_t)(kWave - 1 - l)];
#pragma unroll
    for (int r = 0; r < kWords; ++r)
        if (r * kWave + l >= nx) c[r] = cy[r];
    // the entries before the unit, where its first row began earlier
    K before_x = kPad, before_y = kPad;
    if (U.i0 < T.m && n > 0) {
        if (U.xa > 0 && x_row(T, U.i0) < U.xa) before_x = (K)((K)(uint32_t)xi[-1] << 1);
        if (kCheck && U.ya > 0 && y_row(T, U.i0) < U.ya) before_y = (K)((K)(uint32_t)yi[-1] << 1) | 1u;
    }
    // an entry's row, counted from the unit's first: row ends up to its position
    uint32_t row[kWords] = {};
    if (n > 0 && U.i1 > U.i0) {
        // Y runs backwards: all row ends, less those that are behind the entry
        int32_t *const E = ends[w];
#pragma unroll
        for (int q = 0; q < kWords / 4; ++q) *reinterpret_cast<int4 *>(&E[4 * (q * kWave + l)]) = make_int4(0, 0, 0, 0);
        wave_sync();
        int32_t sum_x = 0, sum_y = 0;
        for (int32_t i = U.i0 + l; i - l < U.i1; i += kWave) {
            const bool in = i < U.i1;
            const int64_t ex = in ? x_row(T, i + 1) - U.xa : nx, ey = in ? y_row(T, i + 1) - U.ya : ny;
            if (ex < nx) atomicAdd(&E[max(ex, (int64_t)0)], 1);
            if (ey < ny && ey > 0) atomicAdd(&E[kAddUnit - (int32_t)ey], -1);
            sum_x += __popcll(ballot(ex < nx));
            sum_y += __popcll(ballot(ey < ny));
        }
        wave_sync();
        int32_t carry = 0;
#pragma unroll
        for (int r = 0; r < kWords; ++r) {
            const int32_t s = wave_incl_scan(E[r * kWave + l]) + carry;
            carry = read_lane(s, kWave - 1);
            row[r] = (uint32_t)(r * kWave + l < nx ? s : s - sum_x + sum_y);
        }
    }
    K k[kWords];
#pragma unroll
    for (int r = 0; r < kWords; ++r) {
        const int32_t e = r * kWave + l;
        k[r] = ((K)row[r] << kRowShift) | ((K)(uint32_t)c[r] << 1) | (e < nx ? 0u : 1u);
        if (e >= nx && e < kAddUnit - ny) k[r] = kPad;
    }
    if constexpr (kCheck) {
        // X ascends from e = 0, Y descends to the last e (masks of e, wave-uniform)
        uint64_t range_x = 0, range_y = 0, order_x = 0, order_y = 0;
        const int32_t y0 = kAddUnit - ny;
        K carry = kPad;
#pragma unroll
        for (int r = 0; r < kWords; ++r) {
            const K p = lane_below(k[r], carry, l);
            carry = read_lane(k[r], kWave - 1);
            const uint64_t range = ballot((uint32_t)c[r] >= (uint32_t)T.n);
            range_x |= range & word_span(0, nx, r);
            range_y |= range & word_span(y0, kAddUnit, r);
            order_x |= ballot(k[r] <= p) & word_span(1, nx, r);
            order_y |= ballot(k[r] >= p) & word_span(y0 + 1, kAddUnit, r);
        }
        // and against the entries before the unit
        if (nx > 0 && before_x != kPad && read_lane(k[0], 0) <= before_x) order_x = 1;
        if (ny > 0 && before_y != kPad && carry <= before_y) order_y = 1;
        if (l == 0) {
            if (range_x) findings[1] = 1;
            if (order_x) findings[2] = 1;
            if (range_y) findings[5] = 1;
            if (order_y) findings[6] = 1;
        }
    }
#pragma unroll
    for (int s = kWords / 2; s > 0; s >>= 1)
#pragma unroll
        for (int r = 0; r < kWords; ++r)
            if (!(r & s)) {
                const K a = less_of(k[r], k[r + s]), b = greater_of(k[r], k[r + s]);
                k[r] = a;
                k[r + s] = b;
            }
    exchange<32>(k, l);
    exchange<16>(k, l);
    exchange<8>(k, l);
    exchange<4>(k, l);
    exchange<2>(k, l);
    exchange<1>(k, l);
    uint32_t lo = 0, hi = 0;  // lane q: word q
    int32_t kept = n;
    K carry = before_x;
#pragma unroll
    for (int r = 0; r < kWords; ++r) {
        const K p = lane_below(k[r], carry, l);
        carry = read_lane(k[r], kWave - 1);
        const uint64_t from_y = ballot((k[r] & 1u) != 0);
        const uint64_t fold = ballot((k[r] & 1u) != 0 && (k[r] ^ 1u) == p);
        kept -= __popcll(fold);
        const bool is_y = __builtin_amdgcn_inverse_ballot_w64(1ull << r);
        const bool is_f = __builtin_amdgcn_inverse_ballot_w64(1ull << (kWords + r));
        lo = is_y ? (uint32_t)from_y : is_f ? (uint32_t)fold : lo;
        hi = is_y ? (uint32_t)(from_y >> 32) : is_f ? (uint32_t)(fold >> 32) : hi;
    }
    if (l < 2 * kWords) bits[(int64_t)(u - u0) * (2 * kWords) + l] = (uint64_t)hi << 32 | lo;
    if (counts && l == 0) counts[u] = kept;
}

// Entries and row pointers of the units [u0, u1), a wave each, from the merge's
// bits (of [u0, min(u1 + 1, all)): an X entry's partner may be the next unit's
// first).  Straight from global memory to global memory: a word's positions
// come from one run of X and one of Y and go to one run of the output.
__global__ __launch_bounds__(kAddThreads) void k_add_write(const AddTaskDev *__restrict__ tasks, int nt,
                                                          const AddTaskDev one, int32_t u0, int32_t u1,
                                                          const int2 *__restrict__ split,
                                                          const int32_t *__restrict__ guard,
                                                          const uint64_t *__restrict__ bits,
                                                          const int64_t *__restrict__ first, int32_t *__restrict__ oi,
                                                          double *__restrict__ ov) {
    const int l = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int32_t u = u0 + (int32_t)blockIdx.x * kAddWaves + w;
    if (u >= u1 || (guard && *guard)) return;
    AddTaskDev T = one;
    if (tasks) T = tasks[add_task_of(tasks, nt, u)];
    AddUnit U;
    if (!add_unit(T, u, split, U)) return;
    const int32_t nx = U.nx, ny = U.ny, n = nx + ny;
    const TR_GLOBAL int32_t *xi = x_idx(T) + U.xa;
    const TR_GLOBAL double *xv = x_val(T) + U.xa;
    const TR_GLOBAL int32_t *yi = as_global(T.yi) + U.ya;
    const TR_GLOBAL double *yv = as_global(T.yv) + U.ya;
    const uint64_t *W = bits + (int64_t)(u - u0) * (2 * kWords);
    const int64_t out = first[u];
    int32_t *const po = oi + out;
    double *const pv = ov + out;
    int32_t c[kWords];
    double v[kWords + 1];
    int32_t ys = 0;
#pragma unroll
    for (int r = 0; r < kWords; ++r) {
        const uint64_t from_y = W[r];
        const int32_t p = r * kWave + l, j = ys + rank_below(from_y);
        const bool y = (from_y >> l) & 1;
        c[r] = 0;
        v[r] = 0.0;
        if (p < n) {
            const TR_GLOBAL int32_t *ip = y ? yi + j : xi + (p - j);
            const TR_GLOBAL double *vp = y ? yv + j : xv + (p - j);
            c[r] = *ip;
            v[r] = *vp;
        }
        ys += __popcll(from_y);
    }
    // the first entry beyond the unit, if it is folded into the unit's last
    const uint64_t beyond = U.last ? 0 : W[3 * kWords] & 1;
    v[kWords] = beyond && U.ya + ny < T.ny ? yv[ny] : 0.0;
    int32_t folds = 0;
#pragma unroll
    for (int r = 0; r < kWords; ++r) {
        const int32_t p = r * kWave + l;
        const uint64_t fold = W[kWords + r];
        const uint64_t next = fold >> 1 | (r + 1 < kWords ? W[kWords + r + 1] : beyond) << 63;
        double z = dpp<0x130>(v[r]);  // the value behind: the lane above
        if (next >> (kWave - 1)) z = l == kWave - 1 ? read_lane(v[r + 1], 0) : z;
        bool pair = (next >> l) & 1;
        if (beyond && p == n - 1) {
            z = v[kWords];
            pair = true;
        }
        const double s = pair ? v[r] + z : v[r];
        if (p < n && !((fold >> l) & 1)) {
            const int32_t at = p - folds - rank_below(fold);
            __builtin_nontemporal_store(c[r], &po[at]);
            __builtin_nontemporal_store(s, &pv[at]);
        }
        folds += __popcll(fold);
    }
    // row pointers of the rows that end in the unit, rebased to the task
    TR_GLOBAL int32_t *optr = as_global(T.optr);
    if (U.first && l == 0) optr[0] = 0;
    if (U.i1 == U.i0) return;
    const int64_t base = out - first[T.unit0];
    const uint64_t fw = l < kWords ? W[kWords + l] : 0;
    const int32_t upto = wave_incl_scan((int32_t)__popcll(fw));
    for (int32_t i = U.i0 + l; i - l < U.i1; i += kWave) {
        int32_t e = 0;
        if (i < U.i1) e = (int32_t)clamp64(x_row(T, i + 1) - U.xa + y_row(T, i + 1) - U.ya, 0, n);
        const int q = e / kWave;
        const uint64_t word = __shfl(fw, q);
        const int32_t f = __shfl(upto, q) - __popcll(word >> (e % kWave));
        if (i < U.i1) optr[i + 1] = (int32_t)(base + e - f);
    }
}

// Replay guard of a planned add (a batch's graph): every task's output must
// start where the plan put it.  On a mismatch the guard word records it and the
// write pass writes nothing.
__global__ void k_add_guard_output(const AddTaskDev *__restrict__ tasks, int nt, const int64_t *__restrict__ first,
                                   int32_t nunits, const int64_t *__restrict__ expect, int32_t *__restrict__ guard) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t <= nt && *guard == 0) {
        // expect[t]: planned first output entry of task t (expect[nt]: total)
        const int64_t got = first[t < nt ? tasks[t].unit0 : nunits];
        if (got != expect[t]) atomicOr(guard, 4);
    }
}

constexpr size_t kAlign = 256;
inline size_t align_up(size_t b) { return (b + kAlign - 1) & ~(kAlign - 1); }

int64_t add_units(const AddTaskDev &t) { return std::max<int64_t>(((int64_t)t.m + t.nx + t.ny + kAddUnit - 1) / kAddUnit, 1); }

// The one task of A + C
AddTaskDev add_task(const tr_csx_t *A, const tr_csx_t *C, int32_t *optr) {
    AddTaskDev t{};
    t.xp = A->ptr_vec;
    t.xi = A->idx_vec;
    t.xv = A->val;
    t.yp = C->ptr_vec;
    t.yi = C->idx_vec;
    t.yv = C->val;
    t.m = A->nrows;
    t.n = A->ncols;
    t.nx = A->nnz;
    t.ny = C->nnz;
    t.optr = optr;
    return t;
}

// Places the plan's units; bytes of split, counts, first and the scan's temp
void add_place(AddPlan &ap, size_t (&bytes)[4]) {
    int64_t units = 0, rows = 0;
    for (auto &t : ap.h) {
        t.row_base = (int32_t)rows;
        t.unit0 = (int32_t)units;
        rows += t.m;
        units += add_units(t);
        ap.wide = ap.wide || t.n > 1 << 21;
    }
    TR_REQUIRE(rows < INT32_MAX, "spadd: total rows exceed INT32_MAX");
    TR_REQUIRE(units < INT32_MAX / 2, "spadd: operands too large for one launch");
    ap.nt = (int)ap.h.size();
    ap.nunits = (int32_t)units;
    bytes[0] = sizeof(int2) * (size_t)units;
    bytes[1] = sizeof(int32_t) * (size_t)units;
    bytes[2] = sizeof(int64_t) * ((size_t)units + 1);
    bytes[3] = scan_tmp_bytes(units);
}

// bytes of the merge bits of k units (and the one behind them)
size_t kept_bytes(int64_t k) { return sizeof(uint64_t) * 2 * kWords * (size_t)(k + 1); }

// The plan's arrays, in a workspace; the merge bits of fewer units if there is
// no room for all.
void add_arrays(Workspace &ws, AddPlan &ap, const size_t (&b)[4]) {
    ap.split = (int2 *)ws.get(S_ROWPTR64, b[0]);
    ap.counts = (int32_t *)ws.get(S_MISC, b[1]);
    ap.first = (int64_t *)ws.get(S_FLOPS, b[2]);
    if (ws.owned) ap.scan_tmp = (int64_t *)ws.get(S_SCAN_TMP, b[3]);
    for (int64_t k = std::min<int64_t>(ap.nunits, kMaxKept);; k = std::max(k / 2, kMinKept)) {
        try {
            ap.bits = (uint64_t *)ws.get(S_BINS, kept_bytes(k));
            ap.kept = (int32_t)k;
            return;
        } catch (const Error &e) {
            if (e.code != TR_ERR_OOM || k <= kMinKept) throw;
        }
    }
}

void add_merge(tr_ctx *ctx, AddPlan &ap, int32_t u0, int32_t u1, const int32_t *guard, int32_t *counts,
               uint8_t *findings) {
    auto go = [&](auto kernel) {
        TR_LAUNCH(ctx, "add_count", kernel, div_up((uint64_t)(u1 - u0), kAddWaves), kAddThreads, 0, ap.d, ap.nt,
                  ap.h[0], u0, u1, ap.split, guard, ap.bits, counts, findings);
    };
    if (ap.wide) findings ? go(k_add_merge<uint64_t, true>) : go(k_add_merge<uint64_t, false>);
    else findings ? go(k_add_merge<uint32_t, true>) : go(k_add_merge<uint32_t, false>);
}

void add_plain(Workspace &ws, AddPlan &ap, const AddTaskDev &t) {
    size_t b[4];
    ap.h = {t};
    add_place(ap, b);
    add_arrays(ws, ap, b);
}

}  // namespace

void add_setup(tr_ctx *ctx, Workspace &ws, AddPlan &ap, const std::vector<AddTaskDev> &tasks) {
    size_t b[4];
    ap.h = tasks;
    add_place(ap, b);
    ap.d = (AddTaskDev *)ws.get(S_PANELS, sizeof(AddTaskDev) * (size_t)std::max(ap.nt, 1));
    add_arrays(ws, ap, b);
    TR_HIP(hipMemcpyAsync(ap.d, ap.h.data(), sizeof(AddTaskDev) * (size_t)ap.nt, hipMemcpyHostToDevice,
                          ctx->stream));
}

// findings: the context's status bytes to check both operands on the way, or
// nullptr
void add_count(tr_ctx *ctx, AddPlan &ap, bool capture, uint8_t *findings) {
    const int32_t *guard = capture ? ap.guard : nullptr;
    TR_LAUNCH(ctx, "add_split", k_add_split, div_up((uint64_t)ap.nunits, 256), 256, 0, ap.d, ap.nt, ap.h[0], ap.nunits,
              guard, ap.split);
    for (int32_t u = 0; u < ap.nunits; u += ap.kept)
        add_merge(ctx, ap, u, std::min(u + ap.kept, ap.nunits), guard, ap.counts, findings);
    launch_exclusive_scan_i32_to_i64(ctx, ap.counts, ap.first, ap.nunits, ap.scan_tmp);
    if (capture && ap.guard && ap.expect)
        TR_LAUNCH(ctx, "add_guard", k_add_guard_output, div_up((uint64_t)ap.nt + 1, 64), 64, 0, ap.d, ap.nt, ap.first,
                  ap.nunits, ap.expect, ap.guard);
}

int64_t add_total(tr_ctx *ctx, AddPlan &ap) { return read_scalar<int64_t>(ctx, ap.first + ap.nunits); }

// Gives back the merge bits but those of a small part, which add_write fills
// again part by part.  false: there are no more than that.
bool add_make_room(Workspace &ws, AddPlan &ap) {
    if (ap.kept <= kMinKept) return false;
    ws.drop(S_BINS);
    ap.kept = (int32_t)kMinKept;
    ap.bits = (uint64_t *)ws.get(S_BINS, kept_bytes(kMinKept));
    return true;
}

void add_write(tr_ctx *ctx, AddPlan &ap, int32_t *oi, double *ov, bool capture) {
    const int32_t *guard = capture ? ap.guard : nullptr;
    for (int32_t u = 0; u < ap.nunits; u += ap.kept) {
        const int32_t end = std::min(u + ap.kept, ap.nunits);
        if (ap.kept < ap.nunits) add_merge(ctx, ap, u, std::min(end + 1, ap.nunits), guard, nullptr, nullptr);
        TR_LAUNCH(ctx, "add_write", k_add_write, div_up((uint64_t)(end - u), kAddWaves), kAddThreads, 0, ap.d, ap.nt,
                  ap.h[0], u, end, ap.split, guard, ap.bits, ap.first, oi, ov);
    }
}

namespace {

// nnz(A + C) of a plan of one task.  check: what a caller's operands are
// checked for; the pointers by a pass of their own, the entries by the count
// (which stays in bounds whatever they hold).
int64_t plain_count(tr_ctx *ctx, AddPlan &ap, const tr_csx_t *A, const tr_csx_t *C, const char *check) {
    if (check) {
        const tr_csx_t *m[2] = {A, C};
        check_pointers(ctx, m, 2);
    }
    add_count(ctx, ap, false, check ? ctx->status : nullptr);
    const int64_t nnz = add_total(ctx, ap);
    if (check) {
        int32_t hs[2];
        check_result(ctx, hs, 2);
        if (hs[0] | hs[1]) {  // units cut by a merge of unsorted rows may miss entries: look again
            const tr_csx_t *m[2] = {A, C};
            const std::string w(check);
            check_tiles(ctx, m, 2, hs);
            if ((hs[0] | hs[1]) & 3) fail(TR_ERR_INVALID, w + ": malformed CSR operand");
            fail(TR_ERR_INVALID, w + ": operands need sorted unique columns");
        }
    }
    return nnz;
}

}  // namespace

// optr/oi/ov = A + C (both CSR, sorted) into caller arrays with room for
// `capacity` entries; returns nnz(A + C) and writes nothing if it exceeds
// the capacity.
int64_t spadd_into(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *C, int32_t *optr, int32_t *oi, double *ov,
                   int64_t capacity, const char *check) {
    Workspace ws(ctx, false);
    AddPlan ap;
    add_plain(ws, ap, add_task(A, C, optr));
    const int64_t nnz = plain_count(ctx, ap, A, C, check);
    if (nnz <= capacity) add_write(ctx, ap, oi, ov, false);
    return nnz;
}

int64_t spadd_into_fixed(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *C, int32_t *optr, int32_t *oi, double *ov,
                         int64_t capacity, const char *check, char *base, size_t bytes) {
    AddPlan ap;
    ap.h = {add_task(A, C, optr)};
    size_t b[4];
    add_place(ap, b);
    char *p[5] = {base};
    for (int i = 0; i < 4; ++i) p[i + 1] = p[i] + align_up(b[i]);
    ap.split = (int2 *)p[0];
    ap.counts = (int32_t *)p[1];
    ap.first = (int64_t *)p[2];
    ap.scan_tmp = (int64_t *)p[3];
    ap.bits = (uint64_t *)p[4];  // for what is left
    ap.kept = (int32_t)std::min<int64_t>(ap.nunits, ((int64_t)bytes - (p[4] - base)) / (int64_t)kept_bytes(0) - 1);
    TR_REQUIRE(ap.kept > 0, "spadd: fixed scratch region too small");
    const int64_t nnz = plain_count(ctx, ap, A, C, check);
    if (nnz <= capacity) add_write(ctx, ap, oi, ov, false);
    return nnz;
}

// out = A + C (both CSR, sorted), out context-owned.
void spadd(tr_ctx *ctx, const tr_csx_t *A, const tr_csx_t *C, tr_csx_t *out, const char *check) {
    Workspace ws(ctx, false);
    AddPlan ap;
    add_plain(ws, ap, add_task(A, C, nullptr));
    const int64_t nnz = plain_count(ctx, ap, A, C, check);
    if (nnz > INT32_MAX) fail(TR_ERR_OVERFLOW, "spadd: nnz(A + C) exceeds INT32_MAX");
    add_output(ws, ap, [&] { alloc_tile(ctx, TR_ROWS, A->nrows, A->ncols, nnz, out); });
    ap.h[0].optr = out->ptr_vec;
    add_write(ctx, ap, out->idx_vec, out->val, false);
}

}  // namespace tr
