// How the heavy rows of a product are cut into column windows and items, and
// how many of both there can be at most.  Host and device share it (the
// symbolic kernel cuts, the host sizes the lists), and a host program without
// HIP can check one against the other.
#pragma once

#include <cstdint>

namespace tr {

constexpr int kMidMaxF = 16384;    // heavy rows of at most that many multiplications: the mid class
constexpr int kMidPassBits = 19;   // mid rows: at most 2^19-column passes, two blocks per CU
constexpr int kPassBits = 20;      // heavy bitmap covers 2^20 columns per pass
constexpr int kFineShift = 7;      // fine block = 128 columns
constexpr int kWinLog = 19;                                // window width cap: 2^19 columns
constexpr int kWinMaxWidth = 1 << kWinLog;                 // (column offsets stay below 2^20)
constexpr int kWidthShift = kWinLog - kFineShift;          // fine blocks per width quantum
constexpr int kSparseAvg = 192;    // a pass with <= this many entries per width quantum is sparse
constexpr int kSparseH = 256;      // sparse windows: count quantum (<= kSparseH + 127 entries, any width)
constexpr int kLongRow = 2048;     // heavy rows with more A entries take shorter items
static_assert(kWinMaxWidth <= (1 << 20) && kPassBits <= 20, "window column offsets fit 20 bits");

// Multiplications that one heavy item should hold at most.  A product with few
// heavy rows would leave the chip to the few items that tune.item_windows
// windows make of them: about kItemsPerCu items a CU, but no item below
// kMinItemFlops.  (40, 160, 320 and 640 a CU, measured with five workgroups
// resident and the heavy numeric in steps between barriers: R-MAT s17 14.43,
// 13.74, 14.06, 14.44 ms; 16 served requests 21.9, 20.8, 21.2, 21.7 ms; R-MAT
// s19, whose items the window count cuts, within 1%.  A minimum of 8192 costs
// the R-MAT of 15013 vertices 3%.)
constexpr int kItemsPerCu = 160;
constexpr int64_t kMinItemFlops = 2048;
constexpr int64_t heavy_item_flops(int64_t heavy_flops, int cus) {
    const int64_t f = heavy_flops / ((int64_t)cus * kItemsPerCu);
    return f > kMinItemFlops ? f : kMinItemFlops;
}

// Column passes of 2^bits columns over a row of n
constexpr int64_t heavy_passes(int64_t n, int bits) { return (n + ((int64_t)1 << bits) - 1) >> bits; }

// Windows per item of a pass that cut `nwin` windows.  At most item_windows,
// and a quarter of them for rows of more than kLongRow A entries: their items
// are the longest, and the last of them would otherwise run alone at the end
// of the numeric.  And so many that an item holds about item_flops of the
// row's multiplications, taken as spread evenly over its passes and, in a pass,
// over its windows.  (Without the passes a row of P of them is cut P times too
// finely: 300 rows of 100 B rows of 5000 entries over 2^23 columns 2.28 ms, now
// 2.07; R-MAT s20 and s21, of one to four passes, within 0.3% either way.)
constexpr int32_t heavy_item_windows(int32_t item_windows, int32_t a_entries, int64_t item_flops, int64_t row_flops,
                                     int64_t passes, int32_t nwin) {
    const int64_t most = a_entries > kLongRow ? item_windows / 4 : item_windows;
    const int64_t even = item_flops * nwin * passes / row_flops;
    const int64_t w = even < most ? even : most;
    return w > 1 ? (int32_t)w : 1;
}

// Entries of the work lists that `rows` heavy rows with heavy_flops
// multiplications over at most n columns need at most.
//  windows: per pass one for each count quantum of its entries, one more, and
//  one for each width quantum (mid rows take the shorter passes).
//  items: a pass of w windows makes w / heavy_item_windows, rounded up.  Where
//  the window count decides, these are in all no more than the windows over
//  item_windows / 4.  Where item_flops decides, they are at most
//  2 * flops / (item_flops * P) a pass (rounding a quotient of at least 1 down
//  halves it at most; below 1, w itself is less than that), so
//  2 * flops / item_flops for the row's P passes.  And one a pass for rounding.
struct HeavyLists {
    int64_t windows, items;
};
constexpr HeavyLists heavy_lists(int64_t heavy_flops, int64_t rows, int64_t n, int32_t window_entries,
                                 int32_t item_windows, int64_t item_flops) {
    const int64_t passes = heavy_passes(n, kMidPassBits), wsplits = n / kWinMaxWidth + 1;
    const int64_t q = window_entries < kSparseH ? window_entries : kSparseH;
    const int64_t per_item = item_windows / 4 > 1 ? item_windows / 4 : 1;
    const int64_t windows = heavy_flops / q + rows * (2 * passes + wsplits) + 16;
    return {windows, windows / per_item + 2 * (heavy_flops / item_flops) + rows * passes + 16};
}

}  // namespace tr
