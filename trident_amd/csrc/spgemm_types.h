// Types shared by the multiply pipeline (k_spgemm.hip) and the batched
// stage executor (k_batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "heavy_items.h"

namespace tr {

// tuning constants
constexpr int kNumLight = 6;       // light classes: up to 32 << c multiplications, c < kNumLight
constexpr int kHeavyClass = kNumLight;      // heavy rows with more than kMidMaxF multiplications
constexpr int kMidClass = kNumLight + 1;    // heavy rows up to kMidMaxF multiplications
constexpr int kCompactClass = kNumLight + 2;  // + 0..2: heavy rows of <= 32, 64, 128 entries (found by the symbolic)
constexpr int kShortClass = kNumLight + 5;    // light rows of short B rows
constexpr int kNumClasses = kNumLight + 6;
constexpr int kShortMaxF = 128;               // multiplications of a short row
constexpr int kShortMaxNnz = 32;              // and its entries, for the table of the numeric
// rows of a product that looks for short ones: eight to a wave, fewer leave the
// chip idle (Galerkin n^3, short against sorted: 28 392 / 388 us, 32 385 / 394,
// 48 509 / 568, 64 874 / 1031)
constexpr int32_t kShortMinRows = 32768;
constexpr int kMidThreads = 512;
constexpr int kBmWidth = 32768;                            // columns ranked per presence-bitmap pass
constexpr int kBmWords = kBmWidth / 64;                    // presence words per pass
constexpr int kHeavyThreads = 1024;  // symbolic heavy block
constexpr int kCompactMax = 128;     // one-pass heavy rows with <= this many entries take the light numeric
static_assert(kCompactMax * 2 <= (64 << 2), "compact rows fit the light tables of classes 0..2");

struct Window {
    int32_t c0, c1;   // column range [c0, c1)
    int32_t off;      // offset of the window's first entry within the row
    int32_t cnt;      // entries in the window
};

struct Item {
    int32_t row;
    int32_t wbeg, wend;  // window index range
    int32_t pad;
};

struct Panel {
    int64_t nnz_begin;   // global offset of the panel's first entry
    int32_t row_begin;
    int32_t pad;
    int32_t *idx;
    double *val;
};

// One product C_t = A_t * B_t of a batch (a plain call is a batch of one).
// Rows of all tasks form one global row space: task t owns global rows
// [row_base, row_base + m).
struct TaskDev {
    const int32_t *ap, *ai;
    const double *av;
    const int32_t *bp, *bi;
    const double *bv;
    int32_t m;         // rows of A_t
    int32_t n;         // columns of B_t
    int32_t row_base;  // first global row
    int32_t k;         // columns of A_t, rows of B_t
    int64_t a_cap;     // entries of A_t's arrays (a compressed A_t holds ap[m] of them)
};

// device counters written by the symbolic phase
struct Counters {
    int32_t cls[kNumClasses];        // rows per class
    int32_t short_rows[2];           // rows of the short class with <= kShortMaxNnz and with more entries
    unsigned long long flops;        // total multiplications
    unsigned long long heavy_flops;  // multiplications of heavy rows
    int32_t windows;                 // windows appended
    int32_t items;                   // items appended
    int32_t overflow;                // capacity exceeded
    int32_t pad1;
};


// Buffers of one pipeline: the context's scratch slots for plain calls, or
// owned allocations for batches (a captured graph needs fixed addresses).
struct Workspace {
    tr_ctx *ctx = nullptr;
    bool owned = false;
    std::vector<void *> p;
    std::vector<size_t> sz;
    std::vector<size_t> req;  // largest request per slot (sizes the memory bound of a call)
    Workspace(tr_ctx *c, bool own)
        : ctx(c), owned(own), p(S_NUM_SLOTS, nullptr), sz(S_NUM_SLOTS, 0), req(S_NUM_SLOTS, 0) {}
    void *get(int slot, size_t bytes);
    void drop(int slot);
    void release();
    ~Workspace() { release(); }
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
};

// One multiply job over a table of tasks.
struct MulPlan {
    int nt = 0;
    int32_t rows_total = 0;
    std::vector<TaskDev> h_tasks;
    TaskDev *d_tasks = nullptr;
    // the pass over A's entries that sums the flops: a job per task, as a device
    // table, or by value with B's checks for a plain product
    CheckJob *jobs = nullptr;
    CheckPair pair{};
    int njobs = 0;
    CheckGrid check_grid;
    int64_t *flops = nullptr, *rownnz = nullptr, *rowptr = nullptr;
    int32_t *lists = nullptr;
    Counters *cnt = nullptr;
    Counters h{};
    Window *wins = nullptr;
    Item *items = nullptr;
    int32_t win_cap = 0, item_cap = 0;
    int32_t *clen = nullptr;
    int64_t *cbase = nullptr;
    int4 *cursors = nullptr;  // (cursor, column at the cursor, end of B_k) per A entry of multi-window items
    int32_t *order = nullptr;          // heavy items sorted by the column of their first window
    unsigned long long *order_hist = nullptr;
    int64_t cursor_cap = 0;
    int64_t *scan_tmp = nullptr;  // owned scan temp (graph mode)
    tr_tuning_t tune{};           // the context's tuning when the plan was set up
};

// One add X_t + Y_t of a batch.  X rows come from xp (int32, per task) or,
// when xp64 is set, from a 64-bit pointer over the global row space.
struct AddTaskDev {
    const int32_t *xp;
    const int64_t *xp64;
    const int32_t *xi;
    const double *xv;
    const int32_t *yp;
    const int32_t *yi;
    const double *yv;
    int32_t *optr;     // output row pointer (m + 1), rebased to the task
    int64_t nx, ny;    // entries of X_t and Y_t (planned)
    int32_t m;
    int32_t n;         // columns
    int32_t row_base;
    int32_t unit0;     // first work unit
};

// One add job.  No device table (d): the plan's one task goes by value.
struct AddPlan {
    int nt = 0;
    std::vector<AddTaskDev> h;
    AddTaskDev *d = nullptr;
    int32_t nunits = 0;
    int2 *split = nullptr;      // per unit: first row, first X entry
    int32_t *counts = nullptr;  // per unit: entries kept
    int64_t *first = nullptr;   // per unit: first output entry (and the total)
    uint64_t *bits = nullptr;   // the merge of `kept` units and the one behind them
    int32_t kept = 0;
    bool wide = false;          // columns beyond the 32-bit merge keys
    int64_t *scan_tmp = nullptr;
    // replay guard (batches): device word set on a mismatch with the plan,
    // and the planned first output entry of every task (nt + 1 entries)
    int32_t *guard = nullptr;
    const int64_t *expect = nullptr;
};

void add_setup(tr_ctx *ctx, Workspace &ws, AddPlan &ap, const std::vector<AddTaskDev> &tasks);
void add_count(tr_ctx *ctx, AddPlan &ap, bool capture, uint8_t *findings = nullptr);
int64_t add_total(tr_ctx *ctx, AddPlan &ap);
bool add_make_room(Workspace &ws, AddPlan &ap);
void add_write(tr_ctx *ctx, AddPlan &ap, int32_t *oi, double *ov, bool capture);

// Allocates an add's output; the merge bits make room if that fails.
template <typename F>
void add_output(Workspace &ws, AddPlan &ap, F &&alloc) {
    try {
        alloc();
        return;
    } catch (const Error &e) {
        if (e.code != TR_ERR_OOM || !add_make_room(ws, ap)) throw;
    }
    alloc();
}

// Pipeline steps.  In eager mode the host reads counts between steps to size
// grids and lists; in capture mode every size comes from a previous eager run
// on the same operands.
void mul_setup(tr_ctx *ctx, Workspace &ws, MulPlan &pl, const std::vector<TaskDev> &tasks);
// One product of operands that the analysis also checks: mul_checked, after
// the counts are read, fails if they are not sorted CSRs.
void mul_setup_plain(tr_ctx *ctx, Workspace &ws, MulPlan &pl, const tr_csx_t *A, const tr_csx_t *B);
void mul_checked(tr_ctx *ctx);
void mul_analyze(tr_ctx *ctx, MulPlan &pl);
void mul_read_counts(tr_ctx *ctx, MulPlan &pl);
void mul_symbolic(tr_ctx *ctx, Workspace &ws, MulPlan &pl, bool emit, bool capture);
void mul_cursor_prep(tr_ctx *ctx, Workspace &ws, MulPlan &pl, bool capture);
// After the symbolic phase, one read (eager): refreshes the counters, returns
// nnz(C) and the cursors that the heavy items need.
void mul_read_totals(tr_ctx *ctx, MulPlan &pl, int64_t *nnz, int64_t *ncur);
// The first product entry of every task, and the end (nt + 1 values).
void mul_read_task_offsets(tr_ctx *ctx, MulPlan &pl, int64_t *host);
void mul_numeric(tr_ctx *ctx, MulPlan &pl, Panel *d_panels, int np);
void mul_check(tr_ctx *ctx, MulPlan &pl);  // reads the consistency flags (eager)
// The rows that the plan's launches take (after its counts are read): a bit per
// class, then one per part of short_rows, then one for the heavy items.
constexpr int kShortRowsBit = kNumClasses, kItemsBit = kNumClasses + 2;
uint32_t mul_taken(const MulPlan &pl);

}  // namespace tr
