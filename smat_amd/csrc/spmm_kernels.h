// Internal interface between the C ABI (capi.hip) and the kernel launchers.
#pragma once
#include <hip/hip_runtime.h>

#include "devmem.h"
#include "sweep_format.h"
#include <mutex>
#include <utility>
#include <vector>
#include <stddef.h>
#include <stdint.h>

namespace smat {

// One unit of work for a wavefront: blocks [begin, end) of one block row.
struct WorkItem {
    int32_t block_row;
    int32_t begin;
    int32_t end;
    int32_t dst; // < 0: finished tile goes to C; >= 0: fp32 partial tile goes to this workspace slot
};

// A block row that was split over several work items: its partial tiles occupy
// workspace slots [slot_begin, slot_end), summed in that order.
struct SplitRow {
    int32_t block_row;
    int32_t slot_begin;
    int32_t slot_end;
    int32_t pad;
};

// How a launch over a work list deals its workgroups to the eight XCDs.  The dispatcher gives an XCD the workgroup
// ids that are equal modulo 8, whatever their work costs; the row-wise and the compact kernel lay the panel-major
// (panel, item) space out in runs of consecutive workgroups, counted as if of 4 items each, that the XCDs take in turn.
// One run per XCD keeps neighbouring block rows, which share rows of B, on one L2; short runs even out a list whose
// cost per item changes along it.
// choose_xcd_run: the longest run among {an eighth of the launch, 1024, 256, 64, 16, 4} that keeps the estimated load
// of the busiest XCD within 4 % of the mean (the best of them if none does); cost_prefix[i] = cost of the items
// before item i (n_items + 1 entries).
unsigned choose_xcd_run(const uint64_t *cost_prefix, uint64_t n_items, int n_panels);
struct XcdDeal {
    void set_costs(std::vector<uint64_t> &&prefix); // of another list: forgets the choices made for the old one
    // the choice for a launch of n_items x n_panels (kept once made); an eighth of the launch if the costs are not
    // those of a list of n_items
    unsigned run(size_t n_items, int n_panels) const;
private:
    std::vector<uint64_t> cost_prefix_;
    mutable std::mutex mutex_;
    mutable std::vector<std::pair<int, unsigned>> known_;
};

struct SpmmArgs {
    const uint16_t *vals;
    const int32_t *row_ptr;
    const int32_t *col_idx;
    const uint16_t *B;
    void *C;
    size_t M, N, K, nnzb;
    bool c_f32;
    int rule_items;        // work items of the whole matrix: with nnzb, what the choice of the kernel's shape looks at
    const WorkItem *items; // device; nullptr = one item per block row
    int n_items;
    const SplitRow *split_rows; // device
    int n_split_rows;
    float *workspace; // device, n_slots * 16 * N floats
    bool b_row_major;   // B[k * N + n], read in place (launch_rowwise); b_packed is not looked at
    uint16_t *b_packed; // device scratch of K * N halves, or nullptr: read the column-major B directly
    int max_item_blocks; // blocks of the longest work item, 0 = not known (no plan): lets short rows take the short-row kernel
    const XcdDeal *deal; // how to deal the items to the XCDs; nullptr = an eighth of the launch each
};

// Where chunk [begin, ..) of a split row begins in it, and the octave of a cost, as keys that lists with split rows are ordered by; ordered_by: the places of the keys
// from 0 to n_keys - 1, equal ones in the order they have (counted, not compared: ordering 10,000 items is 0.05 ms of a new plan, 0.2 when they were sorted).
constexpr int BEGIN_KEYS = 32768;
inline uint16_t begin_key(int32_t begin, int32_t row_begin, int32_t row_end)
{
    return (uint16_t)((int64_t)(begin - row_begin) * BEGIN_KEYS / (row_end - row_begin));
}
inline int octave_of(uint32_t cost) { return 31 - __builtin_clz(cost | 1u); }
inline std::vector<uint32_t> ordered_by(const std::vector<uint16_t> &keys, int n_keys)
{
    std::vector<uint32_t> next((size_t)n_keys + 1, 0), order(keys.size());
    for (uint16_t k : keys) next[(size_t)k + 1]++;
    for (int k = 0; k < n_keys; k++) next[(size_t)k + 1] += next[(size_t)k];
    for (size_t i = 0; i < keys.size(); i++) order[next[keys[i]]++] = (uint32_t)i;
    return order;
}

// Stream format and geometry of the sweep kernel: sweep_format.h (shared with the host-side plan builder).

struct SweepArgs {
    const uint16_t *vals;
    const uint16_t *B;
    void *C;
    size_t M, N, K, nnzb;
    bool c_f32;
    bool b_row_major;            // B[k*N + n]; ops are the streams for it
    bool whole = true;           // every block of vals is multiplied (not so in a plan of some of the block rows)
    const int32_t *rg_chunk_ptr; // device, n_rg + 1: range of the row group in chunk_ids
    const int32_t *chunk_ids;    // device: the K chunks in which the row group has blocks, ascending (+ SWEEP_CHUNK_PAD entries)
    const int32_t *op_ptr;       // device, n_rg * SWEEP_WAVES + 1: range of (row group, wavefront) in ops
    const SweepOp *ops;          // device, op streams (sweep_format.h)
    const int32_t *row_map;      // device, n_rg * SWEEP_G: block row of (row group, wavefront, local row), -1 = none
    int n_rg;
};

// Sums the fp32 partial tiles of split block rows (workspace[(slot*16 + i)*N + n]) in slot order.
hipError_t launch_reduce(const float *workspace, const SplitRow *split_rows, int n_split_rows, void *C, size_t N,
                         bool c_f32, hipStream_t st);

// ---- compacted-column kernel (spmm_compact.hip) ----
// For matrices whose blocks hold only a few nonzero columns: the nonzero columns of a block
// row are listed once (from the zero pattern of the values) and multiplied 32 at a time.
struct CompactPlan {
    int32_t *d_cols = nullptr;   // row of B (absolute column of A) of every listed column; block rows padded to 32
    // Where many rows of B meet no nonzero, the copy of a column-major B holds the others only: their places in it, -1 for a row
    // that has none (K int32), how many there are, and the list that names places instead of rows.
    int32_t *d_place = nullptr, *d_cols_placed = nullptr;
    int64_t n_placed = 0;
    uint16_t *d_acol = nullptr;  // the 16 values of every listed column, in MFMA operand order (32 bytes per column), or
    uint32_t *d_entries = nullptr;  // their nonzeros: value << 16 | byte in the step's operand
    int2 *d_step_range = nullptr;   // entries [x, y) of every step of 32 listed columns
    int entries_ahead = 0;          // loads of 64 entries that the product kernel asks for ahead: 1 or 2
    WorkItem *d_items = nullptr; // begin/end index the padded list
    int4 *d_tasks = nullptr;     // runs of items: first item, items, first and last column of the list (behind d_items, in their memory)
    SplitRow *d_split = nullptr;
    float *d_workspace = nullptr; // n_slots * 16 * n_cap floats
    int n_items = 0, n_tasks = 0, n_split_rows = 0, n_slots = 0;
    bool ordered = false;         // the tasks lie as order_tasks deals them: workgroup i to XCD i % 8
    bool by_name = false;         // the plan was asked for this kernel or for mixed dispatch, whose products have the same bits as it
    bool may_share = false;       // the steps of a task between wavefronts: every task is one item
    int64_t n_steps = 0;          // of 32 columns, of all block rows listed
    int64_t n_cols = 0;           // nonzero block columns listed (without padding)
    int64_t n_entries = 0;        // nonzeros listed one by one
    int64_t n_cols_all = 0;       // nonzero block columns of the whole matrix
    uint64_t values_checksum = 0; // of the block values the lists were made from
    XcdDeal deal;                 // of the tasks
    // Measured once, when the values are attached (compact_tune): the run length of the deal to the XCDs for
    // launches of tuned_n columns; 0 = not measured, the estimate from the costs decides.
    size_t tuned_n = 0;
    unsigned tuned_run = 0;
};
// What one pass over the block values tells: which columns of the blocks are nonzero, and the sums that the choice of
// the kernels looks at.
struct CompactCensus {
    size_t mb = 0, nnzb = 0;
    DevScratch mask;          // uint16 per block: its nonzero columns
    DevScratch single;        // uint32 per block: value << 16 | row of its only nonzero, 0 where it has none or more
    DevScratch count, offset; // uint64 per block: nonzero columns | nonzeros << 32, and their exclusive sums
    DevScratch rows;          // the same sums at the block rows (mb + 1)
    std::vector<uint64_t> raw; // rows on the host
    bool dropped = false;     // count, offset, rows and raw are those of the blocks that are not full
    uint64_t values_checksum = 0;
    int64_t n_cols_all = 0, nnz = 0;
    int64_t full_blocks = 0, cols_rest = 0; // blocks with at least 10 of their 16 columns nonzero, nonzero columns of the others
    void waited() { mask.idle = single.idle = count.idle = offset.idle = rows.idle = true; } // for all that uses them
    int64_t cols_of_row(size_t br) const { return (int64_t)(uint32_t)(raw[br + 1] - raw[br]); }
};
// vals / row_ptr / col_idx here and below: device BCSR arrays.  Synchronous.  widths != NULL: those of the windows of the pattern, kb block columns, too.
struct WindowCount;
hipError_t compact_census(const uint16_t *vals, const int32_t *row_ptr, size_t mb, size_t nnzb, CompactCensus &s, const int32_t *col_idx = nullptr, size_t kb = 0,
                          WindowCount *widths = nullptr);
hipError_t compact_full_blocks(const CompactCensus &s, std::vector<uint8_t> &full); // one flag per block
// The lists of a plan.  leave_rows != NULL: flagged block rows get no list and no work item (a dense kernel multiplies
// them).  drop_full: full blocks get no listed columns (another kernel multiplies them); from then on the census is
// that of the other blocks.
hipError_t compact_build(CompactCensus &s, const uint16_t *vals, const int32_t *row_ptr, const int32_t *col_idx, size_t K, size_t n_cap,
                         bool b_row_major, const std::vector<uint8_t> *leave_rows, bool drop_full, CompactPlan **out);
// out[j * 256 ..] = block ids_host[j] of vals (device to device, synchronous).
hipError_t copy_blocks(const uint16_t *vals, const int32_t *ids_host, size_t n, uint16_t *out);
void compact_destroy(CompactPlan *p);
// Order-independent checksum of nnzb * 256 block values on the device (synchronous, one pass over vals).
hipError_t values_checksum(const uint16_t *vals, size_t nnzb, uint64_t *out);
struct CompactArgs {
    const uint16_t *B; // column-major, or row-major with b_row_major
    bool b_row_major;  // B is already B[k*N + n]: no copy is made
    uint16_t *Bt;      // scratch, K * (N rounded up to 256) halves: the copy of B in panels of rows made at the start of the launch
    void *C;
    size_t M, N, K;
    bool c_f32;
    unsigned xcd_run = 0; // 0 = the plan's choice
    const CompactPlan *plan;
    bool accumulate = false; // C += A B instead of C = A B (plans without split rows only)
};
hipError_t launch_compact(const CompactArgs &a, hipStream_t st);
// Times launches of M x N x K with a few run lengths of the deal to the XCDs (the estimate's choice, an eighth of the
// launch, a half and a quarter of that) on zeros and keeps the fastest for launches of N columns (tuned_n, tuned_run);
// Bt is overwritten.  The deal decides where an item runs, not what it computes: the results do not depend on it.
// Synchronous, default stream; a plan too large for the temporary buffers, or whose single launch would take longer than
// 20 ms, keeps the estimate's choice.
hipError_t compact_tune(CompactPlan &p, uint16_t *Bt, size_t M, size_t N, size_t K, bool b_row_major, bool accumulate);
// Without trials, for plans that multiply from windows where they may: an even list of neighbouring block rows in runs of half or a quarter of an eighth of the launch.
void compact_deal_beside_windows(CompactPlan &p, size_t N, size_t K);
hipError_t launch_b_to_col_major(const uint16_t *B_row_major, uint16_t *out, size_t N, size_t K, hipStream_t st);

// What a launch of the row-wise kernel knows about the lengths of its items: no block row is much longer than the average
// (a plan found none to split), some were (and are split), or nothing (no plan).
enum class RowLengths { EVEN, SPLIT, UNKNOWN };
int rowwise_panel_tiles(size_t N, size_t n_items, size_t avg_blocks, RowLengths lengths, bool packed);
bool rowwise_shares_items(size_t N, size_t n_items, size_t avg_blocks);
size_t rowwise_row_major_width(size_t N); // columns of a panel on a row-major B in place
bool rowwise_row_major_fits(size_t n_items, size_t N); // whether such a launch has less than 2^32 threads
bool rowwise_takes_short_rows(size_t N, size_t n_items, int most_blocks); // by the short-row kernel: B in place, no split rows
// ---- whole blocks from windows of B in LDS (spmm_window.hip) ----
// For matrices whose neighbouring block rows use the same block columns.
constexpr int WINDOW_SIZES = 3;
struct WindowWidths { // over the groups of 4, 8 and 16 consecutive block rows: the most block columns that one uses, and all together
    uint32_t most[WINDOW_SIZES] = {};
    unsigned long long sum[WINDOW_SIZES] = {};
};
struct WindowLaunch {
    int tiles = 0; // 0: none
    int n_panels = 0, panels_per_unit = 0, workgroups = 0, rounds = 0;
    double us = 1e30; // estimate
};
struct WindowPlan {
    int rows = 0, cap = 0, n_groups = 0; // block rows of a group, block columns of the widest window (a multiple of 4)
    unsigned long long sum = 0;
    double share = 1.0, share4 = 1.0;    // window columns per block, in groups of this size and of 4
    int most_blocks = 0;                 // of a block row
    int32_t *d_window = nullptr, *d_count = nullptr; // window of group i: d_count[i] first columns from d_window[i * cap] on
    uint32_t *d_slot = nullptr;          // of every block: its place in the window, and its block column
    // With attached values: the nonzeros instead of the blocks, and the pattern as it was then (window_entries_kernel).
    int64_t nnz = -1;
    uint32_t *d_entries = nullptr, *d_table = nullptr;
    int32_t *d_blocks = nullptr;
    // The launch of the plan's own width, for C in fp16 and fp32: 0.9 us of estimates that a call does without.
    size_t n = 0;
    WindowLaunch own[2];
};
struct WindowProduct {
    size_t M, K, N, nnzb;
    int64_t nnz; // -1: whole blocks
    int most_blocks; // of a block row
    bool c_f32;
};
// The widths of a pattern's windows, counted on the host or by a kernel, which runs while its caller does other work, or with another kernel's results
// on their way to the host.  row_ptr / col_idx: device arrays; on the default stream.
struct WindowCount {
    static constexpr size_t FEW = 8192;      // blocks that the host counts sooner than it launches a kernel and fetches what that found
    static constexpr int PARTS = 256;        // workgroups a size, at most
    static constexpr size_t BYTES = WINDOW_SIZES * PARTS * 8;
    WindowWidths widths;
    bool there = false, begun = false;
    bool launch(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, void *to); // BYTES there; false: none to come
    void take(const void *parts); // what launch left, from host memory
    void begin(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb); // does not wait
    hipError_t end(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb); // of what has begun, or from the beginning
    void on_host(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb); // host arrays, columns checked
private:
    DevScratch parts;
};
// The size of group (index into the widths, -1 = none fits) that is fastest for a product of N columns, and its time in us.
double window_choose(const WindowWidths &widths, const WindowProduct &w, int *size);
// The launch of a product from windows of that size, of whole blocks, and their shares, before anything is built.
WindowLaunch window_launch_of(const WindowWidths &widths, int size, const WindowProduct &w, WindowPlan &shape);
double window_short_us(const WindowPlan &p, const WindowLaunch &l, size_t M, size_t K, size_t N, size_t nnzb); // of whole blocks, up to 14 us
// row_ptr / col_idx: device arrays.  Does not wait: the caller does, for the default stream, before a launch on another one.
hipError_t window_build(const WindowWidths &w, int size, const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, int most_blocks, WindowPlan **out);
void window_settle(WindowPlan &p, size_t M, size_t K, size_t N, size_t nnzb); // the launch of width N
void window_destroy(WindowPlan *p);
bool window_forced(); // by the test hook
bool window_takes_rows(int most_blocks); // block rows of so many blocks
// offset: of every block, the nonzeros before it in the upper half.  *taken: false where a pair of blocks has too many.  Synchronous.
hipError_t window_attach_entries(WindowPlan &p, const uint16_t *vals, const int32_t *row_ptr, const unsigned long long *offset, size_t mb, size_t nnzb, int64_t nnz,
                                 bool *taken);
double window_estimate_us(int rows, int cap, unsigned long long sum, int tiles, const WindowProduct &w);
double window_least_us(const WindowPlan &p); // no estimate is lower
WindowLaunch window_launch(const SpmmArgs &a, const WindowPlan &p); // of these sizes: the plan's own, or worked out
hipError_t launch_window(const SpmmArgs &a, const WindowPlan &p, const WindowLaunch &l, hipStream_t st); // column-major B

// ---- columns of B in LDS (spmm_resident.hip) ----
struct ResidentLaunch {
    int columns = 0; // that a workgroup holds, 0: none
    int groups = 0, shares = 0;
    double us = 1e30; // estimate
};
struct ResidentPlan {
    int n_slices = 0, longest = 0; // of 64 lanes each; nonzeros of the longest lane
    int64_t fours = 0;             // fours of nonzeros a lane, of all slices
    uint32_t *d_list = nullptr;    // of every lane its row and the lanes that share it, then value << 16 | row of B; 256 * d_first[s] before slice s
    uint32_t *d_first = nullptr;
    size_t n = 0; // the plan's own width, whose launch a call does not work out
    ResidentLaunch own;
};
// From the lists of the compact kernel, which must be all of the matrix; synchronous, on the default stream.  *out: NULL where they do not fit.
hipError_t resident_build(const CompactPlan &c, size_t M, size_t K, int64_t nnz, ResidentPlan **out);
void resident_destroy(ResidentPlan *p);
bool resident_forced(); // by the test hook
bool resident_holds(size_t K); // two columns of B
double resident_estimate_us(size_t M, size_t K, size_t N, int64_t nnz, bool long_rows); // before the lists are there; 1e30: K too long
void resident_settle(ResidentPlan &p, size_t K, size_t N); // the launch of width N
ResidentLaunch resident_launch(const ResidentPlan &p, size_t K, size_t N);
hipError_t launch_resident(const SpmmArgs &a, const ResidentPlan &p, const ResidentLaunch &l, hipStream_t st); // column-major B

hipError_t launch_sweep(const SweepArgs &a, hipStream_t st);
// Whether the sweep kernel reads a row-major B of this size in place; otherwise B is brought into column-major order first, one
// read and one write of it.  In place a row group reads 128 bytes of every row of B where it reads 512 of every column of the
// other order, which costs it more the more row groups there are and the less of B the caches hold, twice as much where the
// pieces straddle cache lines.  Of 39 products the rule takes the slower way in four, by 1 to 6 %; in place / column-major
// first, us: 8192^2, 10 %, N = 4096 105 / 119, N = 2048 46 / 72; 4096^2, N = 4088 30 / 50; 12288 x 8192, 8 %, N = 4096 132 / 145;
// 16384 rows, 16 row groups: K = 8192, N = 2048 96 / 101, N = 3072 153 / 140; K = 16384, N = 2040 185 / 155.
bool sweep_takes_row_major(size_t N, size_t K, int n_rg);
hipError_t launch_rowwise(const SpmmArgs &a, hipStream_t st);

} // namespace smat

struct smat_plan;
namespace smat {
// A plan that has no better kernel than the row-wise one gets windows where they are faster (row_ptr / col_idx: device arrays).  Does not wait, as window_build.
hipError_t plan_take_window(smat_plan *p, const int32_t *row_ptr, const int32_t *col_idx, WindowCount &count);
bool drop_in_may_take_window(size_t M, size_t K, size_t N, size_t nnzb, int most_blocks); // whether it may, as far as sizes tell
} // namespace smat
