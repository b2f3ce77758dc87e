// CPU check of the heavy work lists' sizes (trident_amd/csrc/heavy_items.h):
// rows are cut pass by pass into windows by the rule of the symbolic kernel
// (a window starts where a count quantum or a width quantum of its fine blocks
// begins) and the windows into items; both counts stay within heavy_lists over
// the whole tuning range, for rows of one to nine passes, entries spread over
// the row or gathered in a few blocks, and one or many multiplications an
// entry.  Exact counts, so no tolerance.
#include "../../trident_amd/csrc/heavy_items.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

using namespace tr;

struct Row {
    int64_t flops;
    int32_t a_entries;
    std::vector<uint8_t> fine;  // entries per fine block of 128 columns
};

struct Tune {
    int32_t window_entries, item_windows;
};

// windows and items of one row, cut by passes of 2^bits columns
static HeavyLists cut(const Row &r, int64_t n, int bits, const Tune &t, int64_t item_flops) {
    HeavyLists made{0, 0};
    const int64_t per_pass = (int64_t)1 << (bits - kFineShift), blocks = (int64_t)r.fine.size();
    for (int64_t b0 = 0; b0 < blocks; b0 += per_pass) {
        const int64_t nfine = std::min(per_pass, blocks - b0);
        int64_t total = 0;
        for (int64_t f = 0; f < nfine; ++f) total += r.fine[b0 + f];
        if (total == 0) continue;
        const bool sparse = total * (1 << kWidthShift) <= (int64_t)kSparseAvg * nfine;
        const int64_t q = sparse ? kSparseH : t.window_entries;
        int64_t nwin = 0, before = 0, prev = 0;
        for (int64_t f = 0; f < nfine; ++f) {
            if (f == 0 || before / q != prev / q || (!sparse && (f >> kWidthShift) != ((f - 1) >> kWidthShift))) ++nwin;
            prev = before;
            before += r.fine[b0 + f];
        }
        const int64_t iw = heavy_item_windows(t.item_windows, r.a_entries, item_flops, r.flops, heavy_passes(n, bits),
                                              (int32_t)nwin);
        made.windows += nwin;
        made.items += (nwin + iw - 1) / iw;
    }
    return made;
}

static int fails = 0;

// `count` copies of every row, all of them heavy
static void check(const char *what, int64_t n, int64_t count, const std::vector<Row> &rows, const Tune &t, int cus) {
    int64_t flops = 0;
    for (const Row &r : rows) flops += count * r.flops;
    const int64_t item = heavy_item_flops(flops, cus);
    const HeavyLists cap = heavy_lists(flops, count * (int64_t)rows.size(), n, t.window_entries, t.item_windows, item);
    const int widest = n <= 1 << 18 ? 18 : n <= 1 << 19 ? 19 : kPassBits;
    HeavyLists made{0, 0};
    for (const Row &r : rows) {
        const HeavyLists m = cut(r, n, r.flops <= kMidMaxF ? std::min(widest, kMidPassBits) : widest, t, item);
        made.windows += count * m.windows;
        made.items += count * m.items;
    }
    if (made.windows > cap.windows || made.items > cap.items) {
        std::fprintf(stderr, "FAIL %s: n %lld, %lld rows, H %d, item_windows %d: %lld windows of %lld, %lld items of %lld\n",
                     what, (long long)n, (long long)(count * rows.size()), t.window_entries, t.item_windows,
                     (long long)made.windows, (long long)cap.windows, (long long)made.items, (long long)cap.items);
        if (++fails > 10) std::exit(1);
    }
}

// `entries` entries spread evenly over the fine blocks [from, to)
static Row even(int64_t n, int64_t entries, double mults, int64_t from, int64_t to) {
    Row r;
    r.fine.assign((size_t)((n + 127) >> kFineShift), 0);
    entries = std::min(entries, (to - from) * 128 - 128);
    for (int64_t f = from; f < to; ++f)
        r.fine[f] = (uint8_t)(entries * (f - from + 1) / (to - from) - entries * (f - from) / (to - from));
    r.flops = std::max<int64_t>((int64_t)(entries * mults), 65);
    r.a_entries = 100;
    return r;
}

int main() {
    // rows of many passes over distinct columns, at tunings an autotuner tries
    {
        const int64_t n = 1 << 23, blocks = n >> kFineShift;
        check("50 rows over 8.4 M columns", n, 50, {even(n, n - 4096, 1.0, 0, blocks)}, {1152, 32}, 256);
        check("4 mid rows", n, 4, {even(n, 16000, 1.0, 0, blocks)}, {64, 64}, 256);
        check("2300 rows", n, 2300, {even(n, 160000, 1.0, 0, blocks)}, {1152, 32}, 256);
    }
    std::mt19937_64 rng(7);
    auto uniform = [&](double lo, double hi) { return std::uniform_real_distribution<double>(lo, hi)(rng); };
    const int32_t h_values[] = {64, 128, 255, 256, 257, 512, 1152, 1409, 2945}, iw_values[] = {1, 2, 4, 7, 8, 16, 32, 64};
    for (int round = 0; round < 1500; ++round) {
        const int64_t n = (int64_t)std::exp2(uniform(12, 23.2));
        const int64_t blocks = (n + 127) >> kFineShift;
        std::vector<Row> rows;
        for (int k = 1 + (int)(rng() % 3); k > 0; --k) {
            // up to the whole row, in a range of its blocks
            const int64_t from = rng() % 2 ? 0 : (int64_t)uniform(0, (double)blocks);
            const int64_t to = rng() % 2 ? blocks : from + 1 + (int64_t)uniform(0, (double)(blocks - from - 1));
            Row r = even(n, (int64_t)std::exp2(uniform(5, 23)), std::max(1.0, std::exp2(uniform(-3, 7))), from, std::max(to, from + 1));
            if (r.flops <= 64) continue;
            r.a_entries = rng() % 2 ? 100 : 5000;
            if (rng() % 3 == 0) std::shuffle(r.fine.begin(), r.fine.end(), rng);
            rows.push_back(r);
        }
        if (rows.empty()) continue;
        const int64_t count = (int64_t)std::exp2(uniform(0, 14));
        check("drawn", n, count, rows, {h_values[rng() % 9], iw_values[rng() % 8]}, rng() % 2 ? 256 : 8);
    }
    if (fails) return 1;
    std::printf("heavy items ok\n");
    return 0;
}
