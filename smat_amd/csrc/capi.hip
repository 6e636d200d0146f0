// C ABI over the HIP kernels: SpMM entry points, plans (work lists) and the thin
// runtime wrappers that let a g++-compiled host live without HIP headers.
// Interface contract: include/smat.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "../../include/smat.h"
#include "devmem.h"
#include "errors.h"
#include "spmm_kernels.h"
#include "sweep_plan.h"

using namespace smat;

#define SMAT_HIP(call)                                                                     \
    do {                                                                                   \
        hipError_t e_ = (call);                                                            \
        if (e_ != hipSuccess)                                                              \
            return set_error(SMAT_ERR_HIP, "%s failed: %s (%s:%d)", #call,                 \
                             hipGetErrorString(e_), __FILE__, __LINE__);                   \
    } while (0)

struct RowCuts { // of the row-wise kernel's list (rowwise_cuts)
    long above; // rows of more blocks are cut
    long piece; // blocks of a piece, at most
};
struct smat_plan {
    int kernel = SMAT_KERNEL_ROWWISE;
    int kernel_requested = SMAT_KERNEL_AUTO;
    size_t M = 0, K = 0, nnzb = 0, n_cap = 0;
    RowCuts cuts = {0, 0};
    int panel_tiles = 0;
    int n_items = 0, n_split_rows = 0, n_slots = 0;
    int max_item_blocks = 0; // blocks of the longest row-wise work item
    WorkItem *d_items = nullptr;
    SplitRow *d_split = nullptr;
    float *d_workspace = nullptr;
    size_t workspace_bytes = 0;
    uint16_t *d_bpack = nullptr; // slab-major copy of B, K * n_cap halves (row-wise kernel, when it pays)
    // sweep kernel work list (present when kernel == SMAT_KERNEL_SWEEP)
    struct SweepDev { // the work list of the sweep kernel in device memory
        int n_rg = 0, n_records = 0, n_ops = 0;
        int32_t *d_rg_chunk_ptr = nullptr, *d_chunk_ids = nullptr, *d_op_ptr = nullptr, *d_row_map = nullptr;
        SweepOp *d_ops = nullptr;
        SweepOp *d_ops_row_major = nullptr; // the streams for row-major B (plans made for SMAT_B_ROW_MAJOR)
        hipError_t upload(const SweepPlanHost &h, bool b_row_major);
        void release();
        void fill(SweepArgs &w, bool b_row_major) const
        {
            w.rg_chunk_ptr = d_rg_chunk_ptr; w.chunk_ids = d_chunk_ids; w.op_ptr = d_op_ptr;
            w.b_row_major = b_row_major; w.ops = b_row_major ? d_ops_row_major : d_ops;
            w.row_map = d_row_map; w.n_rg = n_rg;
        }
    };
    SweepDev sweep;       // all block rows (SMAT_KERNEL_SWEEP)
    bool sweep_few_tiles = false; // its row groups were chosen by sweep_estimate_us
    size_t sweep_chunks = 0;      // chunks its row groups list
    SweepDev sweep_dense; // mixed dispatch: the block rows with mostly full blocks, when they fill the device
    // mixed dispatch per block (rows that hold both kinds of blocks): the blocks with mostly nonzero columns, copied one
    // behind the other into d_vals_dense, go through the sweep kernel; the compact kernel adds the other blocks' columns
    SweepDev sweep_blocks;
    uint16_t *d_vals_dense = nullptr;
    int64_t n_blocks_split = 0;
    std::vector<int32_t> row_ptr_host; // the block row pointer the plan was made from: smat_plan_attach_values works from this copy
    std::vector<int32_t> col_idx_host; // kept for the split of a mixed plan (plans made with col_idx_host for AUTO / MIXED)
    uint64_t fingerprint = 0; // hash of row_ptr_host and, when given, col_idx_host
    bool fingerprint_has_cols = false;
    // compacted-column kernel (present after smat_plan_attach_values)
    CompactPlan *compact = nullptr;
    uint16_t *d_bt = nullptr; // copy of B in panels of rows, K * (n_cap rounded up to 256) halves (compact kernel)
    size_t bt_bytes() const { return K * ((n_cap + 255) / 256 * 256) * sizeof(uint16_t); }
    // mixed dispatch (after smat_plan_attach_values): row-wise work list of the block rows with mostly full blocks
    XcdDeal deal, deal_dense; // of d_items and d_items_dense; cost of an item: its pairs of blocks, and two more
    WorkItem *d_items_dense = nullptr;
    SplitRow *d_split_dense = nullptr;
    float *d_workspace_dense = nullptr;
    int n_items_dense = 0, n_split_dense = 0;
    int64_t n_blocks_dense = 0;
    WindowPlan *window = nullptr; // the row-wise kernel's place is taken by the one that multiplies from windows of B
    ResidentPlan *resident = nullptr; // or these, of the values as they were attached
    uint16_t *d_bcol = nullptr; // column-major copy of a row-major B, K * n_cap halves (plans made for SMAT_B_ROW_MAJOR)
};

hipError_t smat_plan::SweepDev::upload(const SweepPlanHost &h, bool b_row_major)
{
    release();
    n_rg = (int)h.rg_chunk_ptr.size() - 1;
    n_records = (int)h.chunk_ids.size() - SWEEP_CHUNK_PAD;
    n_ops = (int)(h.ops.size() - SWEEP_OP_PAD);
    hipError_t e = hipSuccess;
    auto up = [&](void **dst, const void *src, size_t bytes) {
        if (e != hipSuccess) return;
        e = dev_malloc(dst, std::max<size_t>(bytes, 16));
        if (e == hipSuccess && bytes) e = hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice);
    };
    up((void **)&d_rg_chunk_ptr, h.rg_chunk_ptr.data(), h.rg_chunk_ptr.size() * sizeof(int32_t));
    up((void **)&d_chunk_ids, h.chunk_ids.data(), h.chunk_ids.size() * sizeof(int32_t));
    up((void **)&d_op_ptr, h.op_ptr.data(), h.op_ptr.size() * sizeof(int32_t));
    up((void **)&d_row_map, h.row_map.data(), h.row_map.size() * sizeof(int32_t));
    std::vector<SweepOp> streams;
    encode_sweep_streams(h.rg_chunk_ptr, h.op_ptr, h.ops.data(), false, streams, h.light);
    up((void **)&d_ops, streams.data(), streams.size() * sizeof(SweepOp));
    if (b_row_major) {
        encode_sweep_streams(h.rg_chunk_ptr, h.op_ptr, h.ops.data(), true, streams, h.light);
        up((void **)&d_ops_row_major, streams.data(), streams.size() * sizeof(SweepOp));
    }
    if (e != hipSuccess) release();
    return e;
}
void smat_plan::SweepDev::release()
{
    for (void *q : {(void *)d_rg_chunk_ptr, (void *)d_chunk_ids, (void *)d_op_ptr, (void *)d_row_map, (void *)d_ops, (void *)d_ops_row_major})
        if (q) (void)dev_free(q);
    d_rg_chunk_ptr = d_chunk_ids = d_op_ptr = d_row_map = nullptr;
    d_ops = d_ops_row_major = nullptr;
    n_rg = n_records = n_ops = 0;
}

// Test hook (not part of smat.h): device allocations and releases made by the library since it was loaded.
extern "C" void smat_internal_alloc_counts(int64_t *out)
{
    out[0] = g_dev_mallocs.load();
    out[1] = g_dev_frees.load();
}

// Test hook (not part of smat.h): the library's n-th device allocation from now on (0 = the next) fails; < 0: none does.
extern "C" void smat_internal_fail_alloc(int64_t n) { g_dev_fail_in.store(n); }

// Test hook (not part of smat.h): block rows that the compact kernel's list of this plan splits, -1 without a list.
extern "C" int smat_internal_compact_split_rows(const smat_plan *p) { return p->compact ? p->compact->n_split_rows : -1; }

// Test hook (not part of smat.h): whether the plan's products hold columns of B in LDS.
extern "C" int smat_internal_plan_resident(const smat_plan *p) { return p->resident != nullptr; }
// Test hook (not part of smat.h): block rows of a group whose window the plan's products multiply from, 0 without windows.
extern "C" int smat_internal_plan_window_rows(const smat_plan *p) { return p->window ? p->window->rows : 0; }

// Test hook (not part of smat.h): rows of B that the compact kernel's copy holds, 0 where it holds all or there is no list.
extern "C" int64_t smat_internal_compact_placed_rows(const smat_plan *p) { return p->compact ? p->compact->n_placed : 0; }

extern "C" const char *smat_version(void) { return "smat-amd 0.1 gfx950"; }

static int check_shapes(const void *vals, const void *row_ptr, const void *col_idx, const void *B,
                        const void *C, size_t M, size_t N, size_t K, size_t nnzb)
{
    if (!row_ptr || !B || !C) return set_error(SMAT_ERR_INVALID, "row_ptr, B and C must not be NULL");
    if (nnzb && (!vals || !col_idx))
        return set_error(SMAT_ERR_INVALID, "vals and col_idx must not be NULL when nnzb > 0");
    if (M == 0 || N == 0 || K == 0) return set_error(SMAT_ERR_INVALID, "M, N, K must be positive");
    if (M % 16 || K % 16)
        return set_error(SMAT_ERR_INVALID, "M (%zu) and K (%zu) must be multiples of 16", M, K);
    if (N % 8) return set_error(SMAT_ERR_INVALID, "N (%zu) must be a multiple of 8", N);
    if (M / 16 > 0x7ffffff0u || N > 0x7ffffff0u || nnzb > 0x7ffffff0u)
        return set_error(SMAT_ERR_INVALID, "dimension exceeds the int32 index range of BCSR");
    if ((reinterpret_cast<uintptr_t>(vals) | reinterpret_cast<uintptr_t>(B) |
         reinterpret_cast<uintptr_t>(C)) & 15)
        return set_error(SMAT_ERR_INVALID, "vals, B and C must be 16-byte aligned");
    return SMAT_OK;
}

// The sweep kernel runs one workgroup per (group of SWEEP_G block rows, panel of 64 columns),
// one workgroup per CU at a time.
static bool sweep_fills_device(size_t mb, size_t n)
{
    const size_t n_rg = (mb + SWEEP_G - 1) / SWEEP_G, n_panels = (n + 16 * SWEEP_TN - 1) / (16 * SWEEP_TN);
    return n_rg * n_panels >= 256;
}

// Light streams (sweep_format.h) where a wavefront has few blocks in a chunk: a chunk is then as long as the copies of the one after the next take to come, which
// may be two chunks' time, at the price of pairs of blocks two chunks apart and of a choice between three chunks to run an op in.  All other streams -> light, us, by the blocks of
// a wavefront in a chunk: 2.7 (1216 x 13840, 9 %, N = 1888) 47.1 -> 38.3, 3.5 (4544 x 9520, 3 %, N = 4088) 86.6 -> 75.4, 4.3 (3088 x 4112, 15 %, N = 1000, fp32) 22.6 -> 21.0, 4.8 (4544 x 15056, 15 %,
// N = 768) 52.3 -> 44.3, 6.4 (8192^2, 10 %, N = 640) 27.5 -> 26.0; 6 to 8, 18 products, 0.99 to 1.06 of the time saved; 9 (9312 x 11360, 8 %, N = 1384) 47.3 -> 48.0, 13 (8192^2, 10 %, N = 4096) 94.8 -> 97.3.
static int g_force_light = 0; // test hook: 1 = all streams are light, -1 = none
static bool sweep_light(size_t listed_chunks, size_t nnzb)
{
    if (g_force_light) return g_force_light > 0;
    return (double)nnzb <= 8.0 * (double)listed_chunks * SWEEP_WAVES;
}

// Time of a product with fp16 results through the sweep kernel, from the tiles (row groups x panels of 64 columns, one
// workgroup of a compute unit each), the chunks that the row groups list together and the blocks of a wavefront per chunk: a
// tile costs 0.65 us, a chunk 0.74 us, which it takes however few blocks it has, or 0.35 us and 0.058 per block where a
// wavefront has more than six, C 0.66 us per 10^6 elements.  Against 1166 products (400 matrices, random blocks 768^2 to 16384^2 at 3 to 36 % and
// bands, N = 64 to 4096, on row groups of 16, 32 and 64, three on their own inputs in turn): 10 % standard deviation, none in the mean, 57 of them
// more than 25 % off.  The same terms fitted to these products anew: 9.5 %, and a choice between the kernels that is no better (1.2 % from the best
// in the mean, 1.1 with these).  Estimate (measured) on row groups of 16 / 32 / 64, us:
//   3088 x 4112, 15 %, N = 1000:  18.1 (19.1) / 19.3 (19.5) / 25.1 (25.7)
//   8192 x 8192, 10 %, N = 640:   55.2 (49.6) / 30.8 (28.7) / 42.3 (36.2); N = 1536: 84.5 (77.7) / 60.1 (55.8) / 47.1 (43.2)
//   768 x 3072, 10 %, N = 4096:   14.6 (13.7) / 14.6 (14.9) / 16.7 (16.7)
// Light streams, measured since: a chunk takes 0.61 to 0.65 us however few blocks it has.
static double sweep_estimate_us(size_t n_rg, size_t listed_chunks, size_t nnzb, size_t M, size_t N, bool may_be_light = true)
{
    if (n_rg == 0 || listed_chunks == 0) return 1e30;
    const size_t tiles = n_rg * ((N + 16 * SWEEP_TN - 1) / (16 * SWEEP_TN)), rounds = (tiles + 255) / 256;
    const double blocks = (double)nnzb / ((double)listed_chunks * SWEEP_WAVES);
    const double chunk = std::max(may_be_light && sweep_light(listed_chunks, nnzb) ? 0.63 : 0.7418, 0.3533 + 0.058275 * blocks);
    return 3.0 + (double)rounds * (0.65 + (double)listed_chunks / (double)n_rg * chunk) + 0.66e-6 * (double)M * (double)N;
}
// The same through the row-wise kernel, fitted to those of 239 products that it can lose: the rounds of 1024 wavefronts that
// rowwise_panel_tiles counts and the blocks of an item, or the blocks of all where four wavefronts share an item, behind the
// repack of B.  Standard deviation 7 % on repacked B, 12 % in place, 20 % with shared items.  Estimate (measured), us: 8192^2, 10 %,
// N = 640 40.1 (41.7); 5008 x 3008, 20 %, N = 800 25.9 (25.2); 1040 x 16384, 35 %, N = 1000 83.4 (78.4); 768 x 3072, 10 %,
// N = 4096, in place 21.7 (20.7); shared items in place, since they load no operands twice, 1472 x 9888, 18 %, N = 328 28.7 (25.7), 768 x 10912, 15 %, N = 240 10.6 (10.2); too high for narrow bands, whose rows share B (16384, 64, N = 1024: 55, measured 44.6).
// beside_sweep: in place, a last round of few wavefronts counts half (1472 x 9888, 18 %, N = 328 28.9, whole 36.6 (25.7); 3328 x 12192, 5 %, N = 352 20, 24 (17.6); 928 x 13648, 13 %, N = 1304 55, 68 (42.5)).
static double rowwise_estimate_us(size_t M, size_t K, size_t N, size_t nnzb, size_t n_items, RowLengths lengths, bool packed, bool beside_sweep = false)
{
    n_items = std::max<size_t>(n_items, 1);
    const size_t avg = nnzb / n_items;
    const double start = 0.6e-6 * (double)M * (double)N + (packed ? 5.6 + 0.6e-6 * (double)K * (double)N : 2.7);
    if (rowwise_shares_items(N, n_items, avg))
        return start + (double)nnzb * (double)((N + 63) / 64) / 256.0 * (packed ? 0.047 : 0.105);
    const size_t tiles = (size_t)rowwise_panel_tiles(N, n_items, avg, lengths, packed);
    const size_t wavefronts = n_items * ((N + 16 * tiles - 1) / (16 * tiles));
    double rounds = (double)((wavefronts + 1023) / 1024);
    if (beside_sweep && !packed) rounds = 0.5 * rounds + 0.5 * (double)wavefronts / 1024.0;
    const double column = !packed || tiles <= 4 ? 1.0 : tiles == 8 ? 0.83 : 0.8;
    return start + rounds * (double)tiles * (double)nnzb / (double)n_items * (packed ? 0.0274 * column : 0.074);
}
// The same on B in place up to 14 us, with what neighbouring block rows find of each other's rows of B in the caches: share4, block columns of a group of four
// rows per block.  Fitted to 1,600 products (bands, stencils and random patterns, N = 24 to 4,096): 7 to 8 % standard deviation, where the estimate above is 20 % too high
// in the mean for longer rows, 30 to 40 for bands, and 21 % off either way for shorter ones.  Columns of B a multiple of a cache line apart (K % 64 == 0) are slower to
// gather: bands of 11 blocks a row, 1 to 5 panels 4.5 us, 5.4 with such a K.
static double rowwise_in_place_us(size_t M, size_t K, size_t N, size_t nnzb, size_t n_items, int most_blocks, double share4)
{
    const double mn = 1e-6 * (double)M * (double)N, aligned = K % 64 == 0 ? 1.0 : 0.0;
    if (rowwise_takes_short_rows(N, n_items, most_blocks))
        return 2.62 + 1.56 * mn + 0.49e-6 * (double)K * (double)N + 4.26e-6 * share4 * (double)nnzb * (double)N + 0.435 * aligned;
    const double avg = (double)nnzb / (double)n_items;
    const size_t tiles = (size_t)rowwise_panel_tiles(N, n_items, (size_t)avg, RowLengths::EVEN, false), wavefronts = n_items * ((N + 16 * tiles - 1) / (16 * tiles));
    return 2.48 + 0.56 * mn + (double)tiles * avg * ((double)((wavefronts + 1023) / 1024) * (0.038 + 0.0189 * aligned) + (double)wavefronts / 1024.0 * 0.0338 * share4);
}
// The row-wise kernel on a row-major B in place: the rows of B under the blocks of every panel and the blocks, 17.5 TB/s, and C.  215 products (random blocks, bands, N = 8 to
// 4096, 5 to 1,000 us): 11 % standard deviation, 1 % low in the mean.
static double rowwise_row_major_us(size_t M, size_t N, size_t nnzb)
{
    const size_t width = rowwise_row_major_width(N), panels = (N + width - 1) / width;
    return 4.8 + 0.33e-6 * (double)M * (double)N + 0.057e-6 * (double)nnzb * (double)panels * (double)(32 * width + 512);
}
// A row-major B into column-major order, for the kernels that do not read it in place (8192 x 4096 23 us, 4112 x 504 3 us beside
// the launch that follows); and what the sweep kernel takes longer on a row-major B in place (8192^2, 10 %, N = 4096 103 against 97 us,
// with N = 2040, rows that straddle cache lines, 50 against 43).
static double to_col_major_us(size_t K, size_t N) { return 2.0 + 0.6e-6 * (double)K * (double)N; }
static double sweep_in_place_factor(size_t N) { return N % 64 == 0 ? 1.05 : 1.13; }
// The compact kernel and the pass over a column-major B before it: gathers of whole panels of 16, 32 or 64 columns, B, and the bytes of
// all (B three times) beyond what is found in the caches.  80 stencils and uniform random matrices, N = 8 to 816: 9.5 % standard deviation.
static double compact_estimate_us(double cols, double list_bytes, size_t M, size_t K, size_t N)
{
    const double b = 2.0 * (double)K * (double)N, gathered = cols * (double)(N <= 16 ? 16 : N <= 32 ? 32 : (N + 63) / 64 * 64) * 2.0;
    return 7.8 + gathered / 16.1e6 + b / 4.5e6 + std::max(0.0, 3.0 * b + 2.0 * (double)M * (double)N + list_bytes - 28e6) / 8.25e6;
}
static double compact_estimate_us(const CompactPlan &c, size_t M, size_t K, size_t N)
{
    // 3 us where the parts of split rows are added up (R-MAT scales 12 to 15)
    return compact_estimate_us((double)c.n_cols, c.d_acol ? 36.0 * (double)c.n_cols : 4.25 * (double)c.n_cols + 4.0 * (double)c.n_entries, M, K, N) + (c.n_split_rows ? 3.0 : 0.0);
}
static size_t sweep_listed_chunks(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t group_rows)
{
    std::vector<size_t> seen((kb + SWEEP_S - 1) / SWEEP_S, 0); // the last row group that listed the chunk, from 1
    size_t n = 0;
    for (size_t i = 0; i < mb; i++)
        for (int32_t q = row_ptr[i]; q < row_ptr[i + 1]; q++) {
            size_t &s = seen[(size_t)col_idx[q] / (16 * SWEEP_S)];
            if (s != i / group_rows + 1) s = i / group_rows + 1, n++;
        }
    return n;
}

// Block rows of a row group for a product of N columns whose tiles fill the device: 64, or fewer where the tiles of 64 would
// leave the last round of 256 workgroups nearly empty and the estimate gains 10 %.  (An emptier round is also a faster one, which
// the estimate does not know: of 28 products it promised 20 % in the mean and gave 12; where it promised less than 10 %, 8 % to be
// lost was among it, and one that it takes loses 7: 11456 x 7904, 9 %, N = 2912 122.6 -> 131.3 us.)  Rows of a group, us: 8192^2, 10 %, N = 2304: 64 80.5, 37 69.5; N = 3072:
// 64 93.9, 52 88.5; 30 %, N = 2296: 64 168, 37 135; 16384 x 4096, 10 %, N = 1200: 64 45.3, 40 43.6; 12304 x 7936, 21 %, N = 1360: 64 119, 34 96; 12000 x 6000, 7 %, N = 2000:
// 64 57.0, 47 (estimate 9 % less) 53 to 56 against 52.2.
static size_t sweep_even_rounds(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t N, bool b_row_major)
{
    const size_t nnzb = (size_t)row_ptr[mb], n64 = (mb + SWEEP_G - 1) / SWEEP_G;
    if (nnzb == 0 || n64 == 0) return SWEEP_G;
    const size_t listed = sweep_listed_chunks(row_ptr, col_idx, mb, kb, SWEEP_G);
    const double whole = sweep_estimate_us(n64, listed, nnzb, 16 * mb, N, false); // light streams gain either way
    double best = 0.9 * whole;
    size_t rows = SWEEP_G;
    for (size_t n_rg = n64 + 1; n_rg <= 2 * n64; n_rg++) {
        const size_t g = (mb + n_rg - 1) / n_rg;
        if ((mb + g - 1) / g != n_rg) continue;
        if (b_row_major && sweep_takes_row_major(N, 16 * kb, (int)n64) && !sweep_takes_row_major(N, 16 * kb, (int)n_rg)) break; // stays in place
        const double t = sweep_estimate_us(n_rg, (listed * n_rg + n64 - 1) / n64, nnzb, 16 * mb, N, false);
        if (t < best) best = t, rows = g;
    }
    return rows;
}

// The launch from windows of a plan that has them, or none: for another width than the plan's where the estimate is not below 0.9 of the other
// kernel's, which an estimate below 0.9 of the least that windows are ever estimated to take settles without a look at them (bands and stencils of 4 to 5.5 us
// at another width, 141 launches without this rule: 3 % slower in the mean than before there were windows, 13 % at most).
template <class Other> static WindowLaunch window_or_not(const SpmmArgs &a, const smat_plan &p, Other &&other_us)
{
    if (a.N == p.n_cap || window_forced()) return window_launch(a, *p.window);
    const double bar = 0.9 * other_us();
    if (bar <= window_least_us(*p.window)) return WindowLaunch();
    const WindowLaunch l = window_launch(a, *p.window);
    return l.us < bar ? l : WindowLaunch();
}

// Windows of whole blocks in the place of the row-wise kernel on B in place, for products of less than 14 us: not where what is fitted to such products says that they
// are slower, or, of patterns that share little, less than 5 % faster.  The estimates behind the choice so far know little of these, nor of narrow bands of few block rows: 31 of 60
// random patterns that windows were chosen for were up to 52 % slower for it, 45 of 260 bands up to 25 % (random 1664 x 2064, 4 %, N = 1560 8.2 -> 12.5 us; band of 1248 rows and 75,
// N = 832 4.48 -> 5.58).
constexpr double SHORT_US = 14.0;
static double rowwise_in_place_us(const smat_plan &p, size_t N, double share4)
{
    if (N < 24) return SHORT_US; // not fitted to these
    return rowwise_in_place_us(p.M, p.K, N, p.nnzb, (size_t)p.n_items, p.max_item_blocks, share4);
}
static bool windows_beat(const smat_plan &p, const WindowPlan &shape, const WindowLaunch &l, size_t N, double in_place)
{
    return l.tiles && window_short_us(shape, l, p.M, p.K, N, p.nnzb) < (shape.share > 0.6 ? 0.95 : 1.0) * in_place;
}

// Whether a launch of the row-wise kernel reads a row-major B in place: always but for large products on a repacked B, which are 5 to 35 % slower for it (13696 x 6768, 19 %,
// N = 2384 287 -> 391 us, 8160 x 9536, 24 %, N = 336 61 -> 72; 120 drawn products otherwise 0.44 to 0.93 of the time: a launch less, and loads of whole lines instead of 32
// pieces).  Windows are decided on before (rowwise_windows).
static bool rowwise_stays_row_major(size_t M, size_t K, size_t N, size_t nnzb, size_t n_items, RowLengths lengths, bool packed)
{
    // from 128 columns on a column-major launch takes wider panels, on B in place as well as repacked, and fits where this one does not
    if (N >= 128 && !rowwise_row_major_fits(n_items, N)) return false;
    return !packed || rowwise_row_major_us(M, N, nnzb) <= rowwise_estimate_us(M, K, N, nnzb, n_items, lengths, true) + to_col_major_us(K, N);
}
static bool rowwise_stays_row_major(const smat_plan &p, const SpmmArgs &a)
{
    return rowwise_stays_row_major(a.M, a.K, a.N, a.nnzb, (size_t)p.n_items, p.n_split_rows ? RowLengths::SPLIT : RowLengths::EVEN, a.b_packed != nullptr);
}
// Test hook (not part of smat.h): whether a launch over whole block rows reads a row-major B in place, windows aside.
extern "C" int smat_internal_rowwise_stays_row_major(size_t M, size_t K, size_t N, size_t nnzb, size_t n_items, int packed)
{
    return rowwise_stays_row_major(M, K, N, nnzb, n_items, RowLengths::EVEN, packed != 0);
}

// The launch from windows in the place of the row-wise kernel, or none, where the choice is the plan's; on a row-major B where they are faster than that kernel on B in place, the
// pass over B before them included.
static WindowLaunch rowwise_windows(const smat_plan &p, const SpmmArgs &a, bool b_row_major)
{
    const bool shares = rowwise_shares_items(a.N, (size_t)p.n_items, p.nnzb / (size_t)p.n_items);
    const double in_place = a.N == p.n_cap || window_forced() || shares || a.b_packed ? SHORT_US : rowwise_in_place_us(p, a.N, p.window->share4);
    WindowLaunch l;
    if (in_place < SHORT_US) {
        l = window_launch(a, *p.window);
        if (!windows_beat(p, *p.window, l, a.N, in_place)) return WindowLaunch();
    } else {
        l = window_or_not(a, p, [&] { return shares ? 0.0 : rowwise_estimate_us(a.M, a.K, a.N, a.nnzb, (size_t)p.n_items, RowLengths::EVEN, a.b_packed != nullptr); });
    }
    if (b_row_major && rowwise_row_major_fits((size_t)a.n_items, a.N) && rowwise_row_major_us(a.M, a.N, a.nnzb) <= l.us + to_col_major_us(a.K, a.N)) return WindowLaunch();
    return l;
}

static std::atomic<int64_t> g_turned{0}; // test hook: launches that brought a row-major B into column-major order
extern "C" int64_t smat_internal_turned_launches(void) { return g_turned.load(std::memory_order_relaxed); }

extern "C" int smat_spmm_bcsr_f16_ex(const uint16_t *vals, const int32_t *row_ptr,
                                      const int32_t *col_idx, const uint16_t *B, void *C, size_t M,
                                      size_t N, size_t K, size_t nnzb, const smat_spmm_opts *opts,
                                      const smat_plan *plan)
{
    int rc = check_shapes(vals, row_ptr, col_idx, B, C, M, N, K, nnzb);
    if (rc) return rc;
    smat_spmm_opts o = {SMAT_B_COL_MAJOR, SMAT_C_F16, SMAT_KERNEL_AUTO, 0, nullptr};
    if (opts) o = *opts;
    if (o.b_layout != SMAT_B_COL_MAJOR && o.b_layout != SMAT_B_ROW_MAJOR)
        return set_error(SMAT_ERR_INVALID, "b_layout must be SMAT_B_COL_MAJOR or SMAT_B_ROW_MAJOR");
    if (o.c_dtype != SMAT_C_F16 && o.c_dtype != SMAT_C_F32)
        return set_error(SMAT_ERR_INVALID, "c_dtype must be SMAT_C_F16 or SMAT_C_F32");
    if (o.c_dtype == SMAT_C_F32 && (reinterpret_cast<uintptr_t>(C) & 15))
        return set_error(SMAT_ERR_INVALID, "C must be 16-byte aligned");

    SpmmArgs a{};
    a.vals = vals; a.row_ptr = row_ptr; a.col_idx = col_idx; a.B = B; a.C = C;
    a.M = M; a.N = N; a.K = K; a.nnzb = nnzb;
    a.c_f32 = o.c_dtype == SMAT_C_F32;
    a.n_items = a.rule_items = (int)(M / 16);
    if (plan) {
        if (plan->M != M || plan->K != K || plan->nnzb != nnzb)
            return set_error(SMAT_ERR_INVALID, "plan was built for another matrix (M/K/nnzb differ)");
        if (plan->n_split_rows && N > plan->n_cap)
            return set_error(SMAT_ERR_INVALID,
                             "N (%zu) exceeds the plan's workspace width (%zu): rebuild with n_hint >= N",
                             N, plan->n_cap);
        a.items = plan->d_items; a.n_items = plan->n_items;
        a.split_rows = plan->d_split; a.n_split_rows = plan->n_split_rows;
        a.workspace = plan->d_workspace;
        a.rule_items = plan->n_items;
        a.max_item_blocks = plan->max_item_blocks;
        a.deal = &plan->deal;
        if (plan->d_bpack && N <= plan->n_cap && o.kernel != SMAT_KERNEL_ROWWISE_DIRECT) a.b_packed = plan->d_bpack;
    }
    int kernel = o.kernel;
    if (kernel == SMAT_KERNEL_AUTO) kernel = plan ? plan->kernel : SMAT_KERNEL_ROWWISE;
    if (kernel == SMAT_KERNEL_ROWWISE_PACKED && !a.b_packed)
        return set_error(SMAT_ERR_INVALID, "SMAT_KERNEL_ROWWISE_PACKED needs a plan built for it with n_hint >= N");
    if (kernel == SMAT_KERNEL_ROWWISE_DIRECT || kernel == SMAT_KERNEL_ROWWISE_PACKED) kernel = SMAT_KERNEL_ROWWISE;
    if (kernel != SMAT_KERNEL_ROWWISE && kernel != SMAT_KERNEL_SWEEP && kernel != SMAT_KERNEL_COMPACT && kernel != SMAT_KERNEL_MIXED)
        return set_error(SMAT_ERR_INVALID, "unknown kernel id %d", kernel);
    hipError_t e;
    if (kernel == SMAT_KERNEL_SWEEP && K >= ((size_t)1 << 28)) { // its B copies use 32-bit offsets inside four columns
        if (o.kernel == SMAT_KERNEL_SWEEP)
            return set_error(SMAT_ERR_UNSUPPORTED, "SMAT_KERNEL_SWEEP takes K below 2^28");
        kernel = SMAT_KERNEL_ROWWISE;
    }
    // a plan made for a wide N, used with a narrow one: too few workgroups for the sweep kernel
    if (kernel == SMAT_KERNEL_SWEEP && o.kernel == SMAT_KERNEL_AUTO) {
        // whatever the layout of this launch: both give the same bits through one plan
        const bool in_place = plan->sweep.d_ops_row_major && sweep_takes_row_major(N, K, plan->sweep.n_rg);
        double row_wise = rowwise_estimate_us(M, K, N, nnzb, (size_t)plan->n_items, plan->n_split_rows ? RowLengths::SPLIT : RowLengths::EVEN,
                                              a.b_packed != nullptr) + (in_place ? to_col_major_us(K, N) : 0.0);
        if (plan->d_bcol) row_wise = std::min(row_wise, rowwise_row_major_us(M, N, nnzb));
        const double factor = in_place ? sweep_in_place_factor(N) : 1.0;
        if (plan->sweep_few_tiles ? factor * sweep_estimate_us((size_t)plan->sweep.n_rg, plan->sweep_chunks, nnzb, M, N) > row_wise
                                  : !sweep_fills_device(M / 16, N))
            kernel = SMAT_KERNEL_ROWWISE;
    }
    const uint16_t *B_as_given = B;
    bool sweep_row_major = false;
    // Launches that leave the choice to the plan: windows of B or columns of B in LDS, which were weighed when the plan was made, or, for another width than
    // its own, where they are estimated to be faster.
    WindowLaunch windows;
    ResidentLaunch columns;
    const bool plans_choice = plan && o.kernel == SMAT_KERNEL_AUTO, column_major = o.b_layout == SMAT_B_COL_MAJOR;
    if (kernel == SMAT_KERNEL_MIXED && (!plan || !plan->compact || (!plan->d_items_dense && !plan->sweep_dense.d_ops && !plan->sweep_blocks.d_ops) || !plan->d_bt || N > plan->n_cap))
        return set_error(SMAT_ERR_INVALID, "SMAT_KERNEL_MIXED needs a plan that split the block rows when the values were "
                                           "attached (smat_plan_attach_values) and n_hint >= N");
    if (o.b_layout == SMAT_B_ROW_MAJOR && kernel != SMAT_KERNEL_COMPACT) {
        // The row-wise and the sweep kernel read B in place, or it is first brought into the reference layout in plan scratch, and they run as for
        // column-major B (same bits in C either way).
        if (!plan || !plan->d_bcol || N > plan->n_cap)
            return set_error(SMAT_ERR_UNSUPPORTED,
                             "row-major B (B[k*N+n]) with the row-wise or sweep kernel needs a plan created with "
                             "b_layout = SMAT_B_ROW_MAJOR and n_hint >= N; the compact kernel reads it in place");
        const smat_plan::SweepDev *sweep = kernel == SMAT_KERNEL_SWEEP ? &plan->sweep
                                         : kernel != SMAT_KERNEL_MIXED ? nullptr
                                         : plan->sweep_blocks.d_ops    ? &plan->sweep_blocks
                                         : plan->sweep_dense.d_ops     ? &plan->sweep_dense
                                                                       : nullptr;
        sweep_row_major = sweep && sweep->d_ops_row_major && sweep_takes_row_major(N, K, sweep->n_rg);
        if (kernel == SMAT_KERNEL_ROWWISE && plans_choice && plan->window) windows = rowwise_windows(*plan, a, true);
        a.b_row_major = !sweep && !windows.tiles && rowwise_stays_row_major(*plan, a);
        if (!sweep_row_major && !a.b_row_major) {
            g_turned.fetch_add(1, std::memory_order_relaxed);
            e = launch_b_to_col_major(B, plan->d_bcol, N, K, static_cast<hipStream_t>(o.stream));
            if (e != hipSuccess) return set_error(SMAT_ERR_HIP, "SpMM launch failed: %s", hipGetErrorString(e));
            a.B = B = plan->d_bcol;
        }
    }
    if (plans_choice && column_major && (plan->window || plan->resident)) {
        if (kernel == SMAT_KERNEL_ROWWISE && plan->window) {
            windows = rowwise_windows(*plan, a, false);
        } else if (kernel == SMAT_KERNEL_SWEEP && plan->window) {
            windows = window_or_not(a, *plan, [&] { return sweep_estimate_us((size_t)plan->sweep.n_rg, plan->sweep_chunks, nnzb, M, N); });
        } else if (kernel == SMAT_KERNEL_COMPACT && plan->window && N <= plan->n_cap) {
            windows = window_or_not(a, *plan, [&] { return compact_estimate_us(*plan->compact, M, K, N); });
        } else if (kernel == SMAT_KERNEL_COMPACT && plan->resident && N <= plan->n_cap) {
            columns = resident_launch(*plan->resident, K, N);
            if (N != plan->n_cap && !resident_forced() && columns.us >= 0.9 * compact_estimate_us(*plan->compact, M, K, N)) columns = ResidentLaunch();
        }
    }
    if (kernel == SMAT_KERNEL_MIXED) {
        // the block rows with mostly full blocks through the row-wise kernel, the others (and the empty ones) through
        // the compact kernel: disjoint rows of C, one after the other on the stream
        if (plan->sweep_blocks.d_ops) {
            // per-block split: the plan's copy of the mostly full blocks through the sweep kernel (every row of C is
            // written), then the compact kernel adds the columns of the other blocks
            SweepArgs w{};
            w.vals = plan->d_vals_dense; w.B = B; w.C = C; w.M = M; w.N = N; w.K = K; w.nnzb = (size_t)plan->n_blocks_split; w.c_f32 = a.c_f32;
            plan->sweep_blocks.fill(w, sweep_row_major);
            e = launch_sweep(w, static_cast<hipStream_t>(o.stream));
        } else if (plan->sweep_dense.d_ops) {
            SweepArgs w{};
            w.vals = vals; w.B = B; w.C = C; w.M = M; w.N = N; w.K = K; w.nnzb = nnzb; w.c_f32 = a.c_f32;
            plan->sweep_dense.fill(w, sweep_row_major);
            w.whole = false;
            e = launch_sweep(w, static_cast<hipStream_t>(o.stream));
        } else {
            SpmmArgs d = a; // a row-major B in place, or turned by now
            d.items = plan->d_items_dense; d.n_items = plan->n_items_dense;
            d.split_rows = plan->d_split_dense; d.n_split_rows = plan->n_split_dense;
            d.workspace = plan->d_workspace_dense;
            d.max_item_blocks = 0; // describes the whole matrix's list, not this one
            d.deal = &plan->deal_dense;
            e = d.n_items ? launch_rowwise(d, static_cast<hipStream_t>(o.stream)) : hipSuccess;
        }
        if (e == hipSuccess) {
            CompactArgs c{};
            c.B = B_as_given; c.Bt = plan->d_bt; c.b_row_major = o.b_layout == SMAT_B_ROW_MAJOR; c.C = C; c.M = M; c.N = N; c.K = K;
            c.c_f32 = a.c_f32;
            c.plan = plan->compact;
            c.accumulate = plan->sweep_blocks.d_ops != nullptr;
            e = launch_compact(c, static_cast<hipStream_t>(o.stream));
        }
    } else if (windows.tiles) {
        e = launch_window(a, *plan->window, windows, static_cast<hipStream_t>(o.stream));
    } else if (columns.columns) {
        e = launch_resident(a, *plan->resident, columns, static_cast<hipStream_t>(o.stream));
    } else if (kernel == SMAT_KERNEL_COMPACT) {
        if (!plan || !plan->compact || !plan->d_bt || N > plan->n_cap)
            return set_error(SMAT_ERR_INVALID,
                             "SMAT_KERNEL_COMPACT needs a plan with attached values (smat_plan_attach_values) and n_hint >= N");
        CompactArgs c{};
        c.B = B; c.Bt = plan->d_bt; c.b_row_major = o.b_layout == SMAT_B_ROW_MAJOR; c.C = C; c.M = M; c.N = N; c.K = K; c.c_f32 = a.c_f32;
        c.plan = plan->compact;
        e = launch_compact(c, static_cast<hipStream_t>(o.stream));
    } else if (kernel == SMAT_KERNEL_SWEEP) {
        if (!plan || !plan->sweep.d_ops)
            return set_error(SMAT_ERR_INVALID, "SMAT_KERNEL_SWEEP needs a plan built for it (with col_idx_host)");
        SweepArgs w{};
        w.vals = vals; w.B = B; w.C = C; w.M = M; w.N = N; w.K = K; w.nnzb = nnzb; w.c_f32 = a.c_f32;
        plan->sweep.fill(w, sweep_row_major);
        e = launch_sweep(w, static_cast<hipStream_t>(o.stream));
    } else {
        e = launch_rowwise(a, static_cast<hipStream_t>(o.stream));
    }
    if (e != hipSuccess)
        return set_error(SMAT_ERR_HIP, "SpMM launch failed: %s", hipGetErrorString(e));
    return SMAT_OK;
}

// The drop-in entry point smat_spmm_bcsr_f16 lives in plan_cache.hip.

// ---- SpMM without any allocation ------------------------------------------------
// For callers that cannot allocate (HIP graph capture, serving loops, harnesses that forbid hipMalloc): the
// row-wise kernel on a slab-major copy of B, like a SMAT_KERNEL_ROWWISE_PACKED plan, with the copy in a
// fixed array of the library instead of plan-owned memory.  One array per GPU, held until the process ends.
static __device__ __align__(256) unsigned char scratch[SMAT_STATIC_SCRATCH_BYTES];

#include <mutex>
namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[MAX_DEVICES] = {nullptr}; // device address of `scratch` on each GPU (the name is no device address)
} // namespace

extern "C" int smat_spmm_bcsr_f16_static(const uint16_t *vals, const int32_t *row_ptr, const int32_t *col_idx,
                                          const uint16_t *B, uint16_t *C, size_t M, size_t N, size_t K, size_t nnzb,
                                          void *stream)
{
    int rc = check_shapes(vals, row_ptr, col_idx, B, C, M, N, K, nnzb);
    if (rc) return rc;
    if (K * N * sizeof(uint16_t) > (size_t)SMAT_STATIC_SCRATCH_BYTES || K * N / N != K)
        return set_error(SMAT_ERR_UNSUPPORTED,
                         "smat_spmm_bcsr_f16_static: B (%zu x %zu fp16) exceeds the fixed scratch of %zu bytes", K, N,
                         (size_t)SMAT_STATIC_SCRATCH_BYTES);
    int dev = 0;
    SMAT_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) return set_error(SMAT_ERR_UNSUPPORTED, "device ordinal %d out of range", dev);
    void *ptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        if (!g_scratch_ptr[dev]) { // once per device, with that device current
            void *p = nullptr;
            SMAT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            g_scratch_ptr[dev] = p;
        }
        ptr = g_scratch_ptr[dev];
    }
    SpmmArgs a{};
    a.vals = vals; a.row_ptr = row_ptr; a.col_idx = col_idx; a.B = B; a.C = C;
    a.M = M; a.N = N; a.K = K; a.nnzb = nnzb;
    a.c_f32 = false;
    a.n_items = a.rule_items = (int)(M / 16); // whole block rows: no work list, no partial tiles
    a.b_packed = static_cast<uint16_t *>(ptr); // every element the kernel reads is rewritten by the repack first
    hipError_t e = launch_rowwise(a, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return set_error(SMAT_ERR_HIP, "SpMM launch failed: %s", hipGetErrorString(e));
    return SMAT_OK;
}

// ---- plans -----------------------------------------------------------------

// 64-bit hash of the index arrays, eight bytes at a time in four independent chains: 0.1 ms for the 0.95 MB of
// 237 k blocks, where FNV-1a, one byte after the other, takes 0.95 ms.
static uint64_t mix_word(uint64_t h, uint64_t v)
{
    h = (h ^ v) * 0x9e3779b97f4a7c15ull;
    return h ^ (h >> 29);
}
struct Hash { // of bytes that come in pieces, all but the last of whole 32 bytes
    uint64_t lane[4], bytes = 0;
    explicit Hash(uint64_t h) : lane{h, h ^ 0xbf58476d1ce4e5b9ull, h ^ 0x94d049bb133111ebull, h ^ 0xd6e8feb86659fd93ull} {}
    void add(const void *data, size_t n)
    {
        const unsigned char *p = static_cast<const unsigned char *>(data);
        bytes += n;
        size_t i = 0;
        for (; i + 32 <= n; i += 32) {
            uint64_t v[4];
            memcpy(v, p + i, 32);
            for (int l = 0; l < 4; l++) lane[l] = mix_word(lane[l], v[l]);
        }
        rest_bytes = n - i;
        memcpy(rest, p + i, rest_bytes);
    }
    uint64_t end()
    {
        uint64_t v[4] = {0, 0, 0, 0};
        memcpy(v, rest, rest_bytes);
        for (int l = 0; l < 4; l++) lane[l] = mix_word(lane[l], v[l]);
        return mix_word(mix_word(mix_word(mix_word(bytes, lane[0]), lane[1]), lane[2]), lane[3]);
    }
    unsigned char rest[32];
    size_t rest_bytes = 0;
};
static uint64_t hash_bytes(uint64_t h, const void *data, size_t bytes)
{
    Hash s(h);
    s.add(data, bytes);
    return s.end();
}
static uint64_t pattern_fingerprint(const int32_t *row_ptr_host, const int32_t *col_idx_host, size_t mb, size_t nnzb)
{
    uint64_t h = hash_bytes(0xcbf29ce484222325ull, row_ptr_host, (mb + 1) * sizeof(int32_t));
    if (col_idx_host) h = hash_bytes(h, col_idx_host, nnzb * sizeof(int32_t));
    return h;
}

static void rowwise_costs(const std::vector<WorkItem> &items, XcdDeal &deal)
{
    std::vector<uint64_t> prefix(items.size() + 1, 0);
    for (size_t i = 0; i < items.size(); i++)
        prefix[i + 1] = prefix[i] + (uint64_t)((items[i].end - items[i].begin + 1) / 2) + 2;
    deal.set_costs(std::move(prefix));
}

// Which block rows are cut, and into what: where one has more than four times the average and 64 blocks, pieces of at most 32 blocks and 0.4 of what one of 4,096 wavefronts has to
// do in a launch of the plan's width, since the longest item is as long as a small launch.  Pieces of four times the average -> these, us (R-MAT, row-wise): scale 12, 16 a row,
// N = 128 27.1 -> 16.2; 13, 16, N = 24 29.7 -> 12.7; 14, 20, N = 104 54 -> 38; 15, 16, N = 200 146 -> 119; 16, 16, N = 16 75 -> 52; 17, 16, N = 72 396 -> 367.
// Rows of more than twice the average are cut, and all rows longer than a piece where the launch has no more than a wavefront a SIMD (512 rows of 100 blocks and one of 570, N = 64
// 43.7 -> 18.6 us).  Of the others those from the length on from which their partial tiles, 4 blocks' time each, take up to 5 % of the time of all blocks: the few long rows of a power law, not
// the ordinary ones of a list with an outlier.  Whole / cut, us: R-MAT 14, 20 a row, N = 104 40.7 / 38.0, 16, 16, N = 16 58.4 / 51.5, 13, 24, N = 200 38.8 / 34.0; 1024 rows of 60 and one of 400, N = 128
// 25.2 / 30.6, 128 of 200 and one of 1070, N = 1024 (6 %) 74 / 83, 3000 of 50, N = 32 19.4 / 23.9; 1024 rows each of 10 and 80, N = 256 56 / 64.
static RowCuts rowwise_cuts(const int32_t *row_ptr_host, size_t mb, size_t n_hint)
{
    const auto even = [](double blocks) { return ((long)(blocks + 0.5) + 1) & ~1L; }; // pairs stay aligned with the MFMA's K = 32
    const double nnzb = (double)row_ptr_host[mb], panels = (double)((n_hint + 63) / 64);
    size_t nonempty = 0;
    long most = 0;
    for (size_t i = 0; i < mb; i++) {
        const long len = row_ptr_host[i + 1] - row_ptr_host[i];
        nonempty += len > 0;
        most = std::max(most, len);
    }
    const double avg = nonempty ? nnzb / (double)nonempty : 0.0;
    const long longest = std::max(even(4.0 * avg), 64L);
    if (most <= longest) return {longest, longest};
    const long piece = std::min(longest, even(32.0 + 0.4 * nnzb * panels / 4096.0));
    if ((double)nonempty * panels <= 1024.0) return {piece, piece};
    long above = std::max(piece, (long)(2.0 * avg));
    std::vector<int64_t> tiles((size_t)(above - piece), 0); // partial ones, of the rows of piece + 1, piece + 2, .. blocks
    for (size_t i = 0; i < mb; i++) {
        const long len = row_ptr_host[i + 1] - row_ptr_host[i];
        if (len > piece && len <= above) tiles[(size_t)(len - piece - 1)] += (len + piece - 1) / piece;
    }
    for (double left = 0.05 * nnzb / 4.0; above > piece && (left -= (double)tiles[(size_t)(above - piece - 1)]) >= 0.0;) above--;
    return {above, piece};
}
// The items of a list with cut rows in the order that the compact kernel's tasks have (spmm_compact.hip): pieces by where they begin in their rows, whole rows by octaves of
// length; whole rows that are longer than the pieces before them.  Pieces of one row after the other -> this, us
// (R-MAT, row-wise): scale 14, 12 a row, N = 256 60.2 -> 56.6; 16, 16, N = 184 304 -> 287; 16, 20, N = 256 509 -> 482; 18, 12, N = 128 1031 -> 852; 19, 16, N = 8 531 -> 485; scale 12 and 13 equal.
static void order_split_items(const int32_t *row_ptr_host, long piece, std::vector<WorkItem> &items)
{
    std::vector<uint16_t> keys(items.size());
    for (size_t i = 0; i < items.size(); i++) {
        const WorkItem &w = items[i];
        const int octave = 31 - octave_of((uint32_t)(w.end - w.begin));
        keys[i] = (uint16_t)(w.dst >= 0                ? 32 + begin_key(w.begin, row_ptr_host[w.block_row], row_ptr_host[w.block_row + 1])
                             : w.end - w.begin > piece ? octave
                                                       : 32 + BEGIN_KEYS + octave);
    }
    const std::vector<uint32_t> order = ordered_by(keys, BEGIN_KEYS + 64);
    std::vector<WorkItem> ordered(items.size());
    for (size_t i = 0; i < items.size(); i++) ordered[i] = items[order[i]];
    items.swap(ordered);
}

// Row-wise work list: whole block rows, cut ones in pieces with a partial-sum slot each, before the others.  only != NULL: just the block rows it flags.  Returns the slots.
static int rowwise_work_list(const int32_t *row_ptr_host, size_t mb, RowCuts cuts, const uint8_t *only,
                             std::vector<WorkItem> &items, std::vector<SplitRow> &split)
{
    items.clear();
    split.clear();
    items.reserve(mb + 16);
    int slot = 0;
    for (size_t i = 0; i < mb; i++) {
        const long len = row_ptr_host[i + 1] - row_ptr_host[i];
        if (len <= cuts.above || (only && !only[i])) continue;
        SplitRow sr{(int32_t)i, slot, slot, 0};
        for (long b = row_ptr_host[i]; b < row_ptr_host[i + 1]; b += cuts.piece) {
            const long e = std::min<long>(b + cuts.piece, row_ptr_host[i + 1]);
            items.push_back(WorkItem{(int32_t)i, (int32_t)b, (int32_t)e, slot++});
        }
        sr.slot_end = slot;
        split.push_back(sr);
    }
    for (size_t i = 0; i < mb; i++) {
        const long len = row_ptr_host[i + 1] - row_ptr_host[i];
        if (len > cuts.above || (only && !only[i])) continue;
        items.push_back(WorkItem{(int32_t)i, row_ptr_host[i], row_ptr_host[i + 1], -1});
    }
    return slot;
}
// The list of a plan of n_hint columns.
static int rowwise_plan_list(const int32_t *row_ptr_host, size_t mb, RowCuts cuts, std::vector<WorkItem> &items, std::vector<SplitRow> &split)
{
    const int slots = rowwise_work_list(row_ptr_host, mb, cuts, nullptr, items, split);
    if (!split.empty()) order_split_items(row_ptr_host, cuts.piece, items);
    return slots;
}
// Test hook (not part of smat.h, host only): that list, items[4 i ..] = {block row, first block, end, slot or -1} of up to `room` items; counts[0..2] = items, cut rows, slots.
extern "C" int smat_internal_rowwise_list(const int32_t *row_ptr_host, size_t mb, size_t n_hint, int32_t *out, size_t room, int64_t *counts)
{
    return smat::guarded("smat_internal_rowwise_list", [&] {
        std::vector<WorkItem> items;
        std::vector<SplitRow> split;
        counts[2] = rowwise_plan_list(row_ptr_host, mb, rowwise_cuts(row_ptr_host, mb, n_hint), items, split);
        counts[0] = (int64_t)items.size();
        counts[1] = (int64_t)split.size();
        memcpy(out, items.data(), std::min(room, items.size()) * sizeof(WorkItem));
        return (int)SMAT_OK;
    });
}

namespace {
struct PlanHolder { // frees a half-built plan on every way out but the good one
    smat_plan *p;
    ~PlanHolder() { if (p) smat_plan_destroy(p); }
};
} // namespace

// Row-wise kernel: repacking B slab-major costs a launch plus one read and one write of B
// per SpMM (about 3 us + 4*K*N bytes at 4 TB/s) and lets the operand gather, nnzb*16*N*2
// bytes, run at about 20 TB/s instead of 7.6 TB/s (measured on the row-wise kernel).
static bool repack_pays(size_t K, size_t N, size_t nnzb)
{
    const double gather_bytes = (double)nnzb * 16.0 * (double)N * 2.0;
    return gather_bytes * (1.0 / 7.6e6 - 1.0 / 20e6) > 1.5 * (3.0 + 4.0 * (double)K * (double)N / 4e6);
}
// The sweep kernel's work list is made with the plan, for M = 16 mb and N = n_hint.
static bool sweep_from_the_start(size_t mb, size_t kb, size_t N, size_t nnzb)
{
    return sweep_fills_device(mb, N) && (double)nnzb >= 0.05 * (double)mb * (double)kb && nnzb < (size_t)1 << 23 && nnzb >= 2;
}

static int smat_plan_create_impl(smat_plan **out, const int32_t *row_ptr_host,
                                 const int32_t *col_idx_host, size_t M, size_t K, size_t nnzb,
                                 size_t n_hint, const smat_spmm_opts *opts)
{
    if (!out || !row_ptr_host) return set_error(SMAT_ERR_INVALID, "plan and row_ptr_host must not be NULL");
    if (M == 0 || M % 16 || K % 16) return set_error(SMAT_ERR_INVALID, "M and K must be positive multiples of 16");
    if (n_hint == 0 || n_hint % 8) return set_error(SMAT_ERR_INVALID, "n_hint must be a positive multiple of 8");
    const size_t mb = M / 16;
    if (row_ptr_host[0] != 0 || (size_t)row_ptr_host[mb] != nnzb)
        return set_error(SMAT_ERR_INVALID, "row_ptr_host[0] must be 0 and row_ptr_host[M/16] == nnzb");
    for (size_t i = 0; i < mb; i++)
        if (row_ptr_host[i + 1] < row_ptr_host[i])
            return set_error(SMAT_ERR_INVALID, "row_ptr_host must be non-decreasing");
    const int want = opts ? opts->kernel : SMAT_KERNEL_AUTO;
    if (want == SMAT_KERNEL_SWEEP && !col_idx_host)
        return set_error(SMAT_ERR_INVALID, "SMAT_KERNEL_SWEEP needs col_idx_host");
    const size_t kb = K / 16;
    // The sweep kernel pairs neighbouring blocks of a block row and schedules them by the K chunk they sit in:
    // it needs the columns of a block row strictly ascending, as csrToBcsr emits them (matrix.h:441-463).  The
    // row-wise kernel does not care about the order (like mmaCBT.cu:44-66).
    bool cols_ascending = true;
    uint64_t fingerprint = pattern_fingerprint(row_ptr_host, nullptr, mb, nnzb);
    if (col_idx_host) {
        // One pass over the columns, 16 KiB at a time while they are in the first level cache, without a branch per block; what is wrong is looked
        // up after.  Bits of either word that matter: a column is negative, above limit or no multiple of 16.
        const int32_t limit = (int32_t)std::min<size_t>(K - 1, 0x7fffffff);
        int32_t low_bits = 0, signs = 0;
        size_t descents = 0, allowed = 0; // where a column does not exceed the one before: only between block rows
        Hash columns(fingerprint);
        for (size_t from = 0; from < nnzb; from += 4096) {
            const size_t n = std::min<size_t>(4096, nnzb - from);
            const int32_t *const c = col_idx_host + from;
            uint32_t here = from > 0 && c[0] <= c[-1];
            for (size_t i = 0; i < n; i++) {
                low_bits |= c[i];
                signs |= c[i] | (int32_t)((uint32_t)limit - (uint32_t)c[i]);
            }
            for (size_t i = 1; i < n; i++) here += c[i] <= c[i - 1];
            descents += here;
            columns.add(c, n * sizeof(int32_t));
        }
        fingerprint = columns.end();
        if (nnzb && ((low_bits & 15) || signs < 0 || K == 0))
            for (size_t p = 0; p < nnzb; p++)
                if (col_idx_host[p] < 0 || col_idx_host[p] % 16 || (size_t)col_idx_host[p] >= K)
                    return set_error(SMAT_ERR_INVALID, "col_idx_host[%zu] = %d is not a block column of K = %zu",
                                     p, col_idx_host[p], K);
        for (size_t i = 1; i < mb; i++) {
            const int32_t p = row_ptr_host[i];
            if (p > 0 && (size_t)p < nnzb && p != row_ptr_host[i - 1]) allowed += col_idx_host[p] <= col_idx_host[p - 1];
        }
        cols_ascending = descents == allowed;
        if (!cols_ascending && (want == SMAT_KERNEL_SWEEP || want == SMAT_KERNEL_MIXED))
            return set_error(SMAT_ERR_INVALID, "col_idx_host must be strictly ascending inside every block row for "
                                               "SMAT_KERNEL_SWEEP / SMAT_KERNEL_MIXED");
    }

    smat_plan *p = new (std::nothrow) smat_plan();
    if (!p) return set_error(SMAT_ERR_NOMEM, "out of host memory");
    PlanHolder holder{p};
    p->M = M; p->K = K; p->nnzb = nnzb; p->n_cap = n_hint;
    p->kernel_requested = want;
    p->fingerprint = fingerprint;
    p->fingerprint_has_cols = col_idx_host != nullptr;
    p->row_ptr_host.assign(row_ptr_host, row_ptr_host + mb + 1);
    if (col_idx_host && cols_ascending && (want == SMAT_KERNEL_AUTO || want == SMAT_KERNEL_MIXED)) p->col_idx_host.assign(col_idx_host, col_idx_host + nnzb);

    p->cuts = rowwise_cuts(row_ptr_host, mb, n_hint);

    std::vector<WorkItem> items;
    std::vector<SplitRow> split;
    const int slot = rowwise_plan_list(row_ptr_host, mb, p->cuts, items, split);
    p->n_items = (int)items.size();
    rowwise_costs(items, p->deal);
    for (const WorkItem &wi : items) p->max_item_blocks = std::max(p->max_item_blocks, wi.end - wi.begin);
    p->n_split_rows = (int)split.size();
    p->n_slots = slot;

    hipError_t e = dev_malloc(&p->d_items, std::max<size_t>(items.size(), 1) * sizeof(WorkItem));
    if (e == hipSuccess && !items.empty())
        e = hipMemcpy(p->d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice);
    if (e == hipSuccess && !split.empty()) {
        e = dev_malloc(&p->d_split, split.size() * sizeof(SplitRow));
        if (e == hipSuccess)
            e = hipMemcpy(p->d_split, split.data(), split.size() * sizeof(SplitRow), hipMemcpyHostToDevice);
        p->workspace_bytes = (size_t)slot * 16 * n_hint * sizeof(float);
        if (e == hipSuccess) e = dev_malloc(&p->d_workspace, p->workspace_bytes);
    }
    if (e == hipSuccess && want != SMAT_KERNEL_ROWWISE_DIRECT && (repack_pays(K, n_hint, nnzb) || want == SMAT_KERNEL_ROWWISE_PACKED))
        e = dev_malloc(&p->d_bpack, K * n_hint * sizeof(uint16_t));
    p->panel_tiles = rowwise_panel_tiles(n_hint, items.size(), items.empty() ? 0 : nnzb / items.size(),
                                         split.empty() ? RowLengths::EVEN : RowLengths::SPLIT, p->d_bpack != nullptr);
    // The sweep kernel pays one pass over the B panel per group of 32 block rows,
    // whatever the sparsity, and shares each staged slab between the blocks of the group
    // that sit in that block column.  Measured against the row-wise kernel on repacked B for
    // M = K in {4096, 8192, 16384}, N in {512 .. 4096} and 5% .. 25% of the blocks present: it
    // wins (by 1.02x at 5% up to 1.6x at 25%) whenever its workgroups (groups of 32 block
    // rows x panels of 128 columns) fill the 256 CUs, and loses (0.3x .. 0.9x) when they do not.
    if (e == hipSuccess && opts && opts->b_layout == SMAT_B_ROW_MAJOR) e = dev_malloc(&p->d_bcol, K * n_hint * sizeof(uint16_t));
    bool sweep = want == SMAT_KERNEL_SWEEP;
    if (want == SMAT_KERNEL_AUTO && col_idx_host && cols_ascending && sweep_from_the_start(mb, kb, n_hint, nnzb)) sweep = true;
    if (sweep && (nnzb >= (size_t)1 << 23 || nnzb < 2)) { // blocks are addressed in pairs, with 32-bit byte offsets
        if (want == SMAT_KERNEL_SWEEP)
            return set_error(SMAT_ERR_UNSUPPORTED, "SMAT_KERNEL_SWEEP takes between 2 and 2^23 - 1 nonzero blocks");
        sweep = false;
    }
    if (e == hipSuccess && sweep) {
        SweepPlanHost h;
        const size_t group_rows = want == SMAT_KERNEL_AUTO ? sweep_even_rounds(row_ptr_host, col_idx_host, mb, kb, n_hint, p->d_bcol != nullptr) : SWEEP_G;
        build_sweep_plan(row_ptr_host, col_idx_host, mb, kb, h, nullptr, 0, group_rows, 2e8, sweep_light(sweep_listed_chunks(row_ptr_host, col_idx_host, mb, kb, group_rows), nnzb));
        p->kernel = SMAT_KERNEL_SWEEP;
        static_assert(sizeof(SweepOpHost) == sizeof(SweepOp), "host and device op layouts");
        e = p->sweep.upload(h, p->d_bcol != nullptr);
        if (p->d_bpack && want != SMAT_KERNEL_ROWWISE_PACKED) { // the sweep kernel reads B in place
            (void)dev_free(p->d_bpack);
            p->d_bpack = nullptr;
        }
    }
    if (e != hipSuccess) return set_error(SMAT_ERR_HIP, "plan allocation failed: %s", hipGetErrorString(e));
    holder.p = nullptr;
    *out = p;
    return SMAT_OK;
}

extern "C" int smat_plan_create(smat_plan **out, const int32_t *row_ptr_host,
                                 const int32_t *col_idx_host, size_t M, size_t K, size_t nnzb,
                                 size_t n_hint, const smat_spmm_opts *opts)
{
    return smat::guarded("smat_plan_create", [&] { return smat_plan_create_impl(out, row_ptr_host, col_idx_host, M, K, nnzb, n_hint, opts); });
}

// A matrix of mostly full blocks that plan creation left with the row-wise kernel, because its tiles of 64 block rows x 64
// columns are fewer than the compute units or because fewer than 5 % of its blocks exist: the sweep kernel all the same, on
// row groups of 64, 32 or 16 block rows, where
//   * the estimate is below that of the row-wise kernel by more than the two are off, 10 % on repacked B and 20 % in place.  Of
//     239 products that creation leaves to the choice (random blocks 768^2 to 16384^2 at 3 to 36 %, bands; N = 64 to 4096) it
//     takes 96, all but a band of 8192 rows (8.7 -> 9.1 us) faster than row-wise with fp16 results (by up to 60 %; what the rule
//     leaves would gain another 1.7 % in the mean), seven up to 10 % slower with fp32 ones, whose stores cost the sweep kernel more;
//   * a thousand products (1,500 on a row-major B) make up for the building, 0.11 us a block (one core).  The products that it took to do so, as
//     measured: 109 in the middle, 958 for 2336 x 2192, 20 %, N = 896 (12.9 -> 12.4 us), 1,740 for a band of 16384 rows and 250,
//     N = 128 (12.4 -> 10.3), and that band of 8192 rows never does.
// Measured, us, before and after: 8192^2, 10 %, N = 640: 41.7 -> 28.9, N = 1536: 71.4 -> 41.9; 3088 x 4112, 15 %, N = 2000:
// 40.0 -> 22.1, N = 1000 24.5 -> 19.9; 768 x 3072, 30 %, N = 4096: 29.6 -> 15.4; bands, whose row groups list few chunks: 16384 rows,
// bandwidth 64, N = 1024 44.6 -> 19.4; 65536, 256, N = 512 146 -> 78.  A K of one or two chunks, less than the entry fetches, stays
// with the row-wise kernel.  Returns the block rows of a group, 0 = row-wise.
// As many block rows in every group (1056 x 7856, 5 %, N = 2176, fp32, groups of 64 and 2 rows 35.5 us, of 33 28.5, row-wise 23.4).
static size_t even_rows(size_t mb, size_t group_rows)
{
    const size_t n_rg = (mb + group_rows - 1) / group_rows;
    return (mb + n_rg - 1) / n_rg;
}
// The row groups that the plan builds for candidates of up to `rows` block rows: as many in each where the streams are light, others take as long or longer for it (2768 x 8000, 20 %,
// N = 3488, fp32 75.6 -> 76.9).
struct SweepGroups {
    size_t rows, listed; // block rows of a group; chunks that the groups list together
    bool light;
};
static SweepGroups sweep_groups(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, size_t rows)
{
    const size_t even = even_rows(mb, rows), listed = sweep_listed_chunks(row_ptr, col_idx, mb, kb, even);
    if (sweep_light(listed, nnzb)) return {even, listed, true};
    return {rows, even == rows ? listed : sweep_listed_chunks(row_ptr, col_idx, mb, kb, rows), false};
}
// Test hook (not part of smat.h): out[0..2] = block rows of a group, chunks listed, light.
extern "C" void smat_internal_sweep_groups(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t nnzb, size_t rows, int64_t *out)
{
    const SweepGroups g = sweep_groups(row_ptr, col_idx, M / 16, K / 16, nnzb, rows);
    out[0] = (int64_t)g.rows; out[1] = (int64_t)g.listed; out[2] = g.light;
}
static int g_force_group_rows = 0; // test hook: 64, 32 or 16 whatever the estimates say
static size_t sweep_group_rows(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t nnzb, size_t N, size_t n_items,
                               RowLengths lengths, bool packed, bool b_row_major, double *us = nullptr)
{
    const size_t mb = M / 16, kb = K / 16;
    if (nnzb < 2 || nnzb >= (size_t)1 << 23 || K >= (size_t)1 << 28 || kb <= 2 * SWEEP_S) return 0;
    if (g_force_group_rows) return (size_t)g_force_group_rows;
    const double to_col_major = b_row_major ? to_col_major_us(K, N) : 0.0;
    double row_wise = rowwise_estimate_us(M, K, N, nnzb, n_items, lengths, packed, true) + to_col_major;
    if (b_row_major) row_wise = std::min(row_wise, rowwise_row_major_us(M, N, nnzb));
    // On a row-major B in place, whose estimate errs to either side, 1,500 products have to pay.  With a thousand, long bands of few columns, which the
    // sweep kernel takes 5 to 20 % less time for, went row-wise for what is left of the gain without the pass over B (rows, bandwidth, N, row-wise and sweep,
    // us: 53232, 172, 40 13.5 and 11.3; 63760, 173, 48 15.3 and 12.8; 12672, 225, 88 11.4 and 9.8).  Of 640 products (bands, random blocks) that moves seven:
    // five gain, two lose 3 and 4 %; 2,000 move five more: one gains 8 %, one loses 8.
    const double build = 0.11e-3 * (double)nnzb / (b_row_major ? 1.5 : 1.0);
    double best = std::min(row_wise / (b_row_major ? 1.05 : packed ? 1.1 : 1.2), row_wise - build);
    size_t group_rows = 0;
    for (size_t rows : {(size_t)SWEEP_G, (size_t)SWEEP_G / 2, (size_t)SWEEP_G / 4}) {
        const size_t n_rg = (mb + rows - 1) / rows;
        const double sweep = sweep_estimate_us(n_rg, sweep_groups(row_ptr, col_idx, mb, kb, nnzb, rows).listed, nnzb, M, N);
        const bool in_place = b_row_major && sweep_takes_row_major(N, K, (int)n_rg);
        const double t = in_place ? sweep_in_place_factor(N) * sweep : sweep + to_col_major;
        if (t < best) best = t, group_rows = rows;
    }
    if (us) *us = best;
    return group_rows;
}
// Test hook (not part of smat.h): sweep_even_rounds.
extern "C" int smat_internal_sweep_even_rounds(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t N, int b_row_major)
{
    return (int)sweep_even_rounds(row_ptr, col_idx, M / 16, K / 16, N, b_row_major != 0);
}
// Test hooks (not part of smat.h): row groups of 64, 32 or 16 wherever the sweep kernel may be taken at all (0 = the
// choice, the default), and the choice itself.
extern "C" void smat_internal_sweep_force_groups(int rows) { g_force_group_rows = rows; }
extern "C" void smat_internal_sweep_force_light(int what) { g_force_light = what; }
extern "C" int smat_internal_sweep_group_rows(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t nnzb, size_t N, int packed)
{
    return (int)sweep_group_rows(row_ptr, col_idx, M, K, nnzb, N, M / 16, RowLengths::EVEN, packed != 0, false);
}
// Test hook (not part of smat.h): the same for plans made for a row-major B.
extern "C" int smat_internal_sweep_group_rows_row_major(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t nnzb, size_t N)
{
    return (int)sweep_group_rows(row_ptr, col_idx, M, K, nnzb, N, M / 16, RowLengths::EVEN, true, true);
}

// The streams are built once the values are known to be dense.  The search for a better deal of the rows to the wavefronts
// takes a tenth of the time (16 counter updates a block: 3088 x 4112, 15 % 0.84 ms for all, without the search 0.75, with a
// million updates, 0.5 % fewer ops in the busiest wavefronts, 1.8; same kernel times).
static hipError_t sweep_small_groups(smat_plan &p, size_t group_rows)
{
    const size_t mb = p.M / 16, kb = p.K / 16, nnzb = p.nnzb;
    const int32_t *row_ptr = p.row_ptr_host.data(), *col_idx = p.col_idx_host.data();
    SweepPlanHost h;
    const SweepGroups groups = sweep_groups(row_ptr, col_idx, mb, kb, nnzb, group_rows);
    build_sweep_plan(row_ptr, col_idx, mb, kb, h, nullptr, 0, groups.rows, 16.0 * (double)nnzb, groups.light);
    const hipError_t e = p.sweep.upload(h, p.d_bcol != nullptr);
    if (e != hipSuccess) {
        p.sweep.release();
        return e;
    }
    p.sweep_chunks = (size_t)h.rg_chunk_ptr.back();
    p.sweep_few_tiles = true;
    p.kernel = SMAT_KERNEL_SWEEP;
    return hipSuccess;
}

// A plan that plan creation left with the row-wise kernel: windows instead, where the block rows are short enough, none is split
// and none shared by wavefronts (which sums in another order: plans with and without windows give the same bits), and the
// estimate is below 0.9 of the row-wise kernel's and of other_us, the time of what else there is; both are off by 10 %.  Row-wise
// -> windows, us: 27-point stencil 64^3, N = 64 90 -> 56, 48^3, N = 256 111 -> 59, 48 x 25 x 48, N = 56 20.4 -> 12.7; bands of
// 14224 rows and 182, N = 544 33 -> 17, of 65536 and 20, N = 256 30 -> 15, of 8960 and 120, N = 48 7.4 -> 5.
// census: of the values, where the compact kernel would multiply: the window kernel then multiplies what it would, the values as attached.
// Whole blocks: does not wait for the lists, which launches on other streams than the default one may read.
// Not where wavefronts share items, nor for narrow products: 18 -> 17, 10.4 -> 9.2, but 8.2 -> 9, 6.6 -> 7.
static bool beside_rowwise(size_t N, size_t n_items, size_t nnzb)
{
    return window_forced() || (N > 16 && !rowwise_shares_items(N, n_items, nnzb / std::max<size_t>(n_items, 1)));
}
static double bytes_once_us(size_t M, size_t K, size_t N, double a_bytes) { return (a_bytes + 2.0 * (double)(K + M) * (double)N) / 5e6; }
// The estimate of the row-wise kernel knows nothing of the bytes that come from memory, A above all and three times B where that is repacked: 64^3 64 us and
// 64 us of bytes, measured 90; 73 x 61 x 62, N = 88 104 and 72, 125; 44 x 47 x 66, N = 40 31 and 26, 38.
static double rowwise_from_memory_us(size_t M, size_t K, size_t N, size_t nnzb, size_t n_items, bool packed)
{
    return std::hypot(rowwise_estimate_us(M, K, N, nnzb, n_items, RowLengths::EVEN, packed),
                      bytes_once_us(M, K, N, 512.0 * (double)nnzb) + (packed ? 4.0 * (double)K * (double)N / 5e6 : 0.0));
}
// Windows take a launch, or the bytes that they do not save.
static double least_bar_us(double once) { return std::max(4.7, 2.0 + once); }
// What take_window asks before it looks at the widths, of a drop-in call, before there is a plan.  (Counted all the same, first calls with random patterns, few of which get that
// far, took 3 % longer in the mean.)
bool smat::drop_in_may_take_window(size_t M, size_t K, size_t N, size_t nnzb, int most_blocks)
{
    const size_t mb = M / 16;
    if (!window_takes_rows(most_blocks) || !beside_rowwise(N, mb, nnzb)) return false;
    return window_forced() || (!sweep_from_the_start(mb, K / 16, N, nnzb) && 0.9 * rowwise_from_memory_us(M, K, N, nnzb, mb, repack_pays(K, N, nnzb)) >=
                                                                                 least_bar_us(bytes_once_us(M, K, N, 512.0 * (double)nnzb)));
}
// Test hook (not part of smat.h): the same.
extern "C" int smat_internal_drop_in_may_take_window(size_t M, size_t K, size_t N, size_t nnzb, int most_blocks)
{
    return drop_in_may_take_window(M, K, N, nnzb, most_blocks);
}
static bool may_take_window(const smat_plan &p) { return p.kernel_requested == SMAT_KERNEL_AUTO && !p.n_split_rows && window_takes_rows(p.max_item_blocks); }
static hipError_t take_window(smat_plan &p, const int32_t *row_ptr, const int32_t *col_idx, WindowCount &count, double other_us, const uint16_t *vals, const CompactCensus *census)
{
    const size_t mb = p.M / 16, kb = p.K / 16;
    if ((p.kernel != SMAT_KERNEL_ROWWISE && !(p.kernel == SMAT_KERNEL_SWEEP && p.sweep_few_tiles)) || !may_take_window(p)) return hipSuccess;
    if (!census && !beside_rowwise(p.n_cap, (size_t)p.n_items, p.nnzb)) return hipSuccess;
    const double once = bytes_once_us(p.M, p.K, p.n_cap, census ? 4.0 * (double)census->nnz + 12.0 * (double)p.nnzb : 512.0 * (double)p.nnzb);
    const double copy = p.d_bcol ? to_col_major_us(p.K, p.n_cap) : 0.0; // before either
    double bar = 0.9 * (census ? other_us - copy : std::min(rowwise_from_memory_us(p.M, p.K, p.n_cap, p.nnzb, (size_t)p.n_items, p.d_bpack != nullptr), other_us));
    if (p.d_bcol) bar = std::min(bar, 0.9 * (rowwise_row_major_us(p.M, p.n_cap, p.nnzb) - copy)); // which does without it
    if (!window_forced() && bar < least_bar_us(once)) return hipSuccess;
    hipError_t e = hipSuccess;
    if (!count.there && !count.begun && p.nnzb <= WindowCount::FEW && p.col_idx_host.size() == p.nnzb) count.on_host(p.row_ptr_host.data(), p.col_idx_host.data(), mb, kb);
    else e = count.end(row_ptr, col_idx, mb, kb, p.nnzb);
    if (e != hipSuccess) return e;
    const WindowWidths &widths = count.widths;
    int size;
    const double us = window_choose(widths, WindowProduct{p.M, p.K, p.n_cap, p.nnzb, census ? census->nnz : -1, p.max_item_blocks, false}, &size);
    // The sweep kernel brings all block columns in turn, and multiplies faster: not where the windows are most of them too (2448 x 1280, 16 %,
    // N = 552 7.9 -> 8.7 us).
    const bool most_of_b = size >= 0 && !census && other_us < 1e30 && (double)widths.sum[size] > 0.5 * (double)kb * (double)mb / (4 << size);
    if (size < 0 || (!window_forced() && (us >= bar || most_of_b))) return hipSuccess;
    if (!census && !p.d_bpack && (vals || other_us > 1e29) && !window_forced()) { // beside the row-wise kernel, not the sweep kernel
        WindowPlan shape;
        const WindowLaunch l = window_launch_of(widths, size, WindowProduct{p.M, p.K, p.n_cap, p.nnzb, -1, p.max_item_blocks, false}, shape);
        const double in_place = rowwise_in_place_us(p, p.n_cap, shape.share4);
        if (in_place < SHORT_US && !windows_beat(p, shape, l, p.n_cap, in_place)) return hipSuccess;
    }
    e = window_build(widths, size, row_ptr, col_idx, mb, kb, p.nnzb, p.max_item_blocks, &p.window);
    if (e == hipSuccess && !census) window_settle(*p.window, p.M, p.K, p.n_cap, p.nnzb);
    if (e != hipSuccess || !census) return e;
    bool taken;
    e = window_attach_entries(*p.window, vals, row_ptr, (const unsigned long long *)census->offset.p, mb, p.nnzb, census->nnz, &taken);
    if (e != hipSuccess || !taken) {
        window_destroy(p.window);
        p.window = nullptr;
    } else {
        window_settle(*p.window, p.M, p.K, p.n_cap, p.nnzb);
    }
    return e;
}
// No memory for the windows is not an error of the plan.
static hipError_t take_window_if_room(smat_plan &p, const int32_t *row_ptr, const int32_t *col_idx, WindowCount &count, double other_us, const uint16_t *vals, const CompactCensus *census)
{
    const hipError_t e = take_window(p, row_ptr, col_idx, count, other_us, vals, census);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    return hipSuccess;
}
hipError_t smat::plan_take_window(smat_plan *p, const int32_t *row_ptr, const int32_t *col_idx, WindowCount &count) {
    return take_window_if_room(*p, row_ptr, col_idx, count, 1e30, nullptr, nullptr); // a plan of the cache, which launches on the default stream alone
}

static int smat_plan_attach_values_impl(smat_plan *p, const uint16_t *vals, const int32_t *row_ptr,
                                        const int32_t *col_idx, const int32_t *row_ptr_host)
{
    if (!p || !row_ptr || !row_ptr_host) return set_error(SMAT_ERR_INVALID, "plan, row_ptr and row_ptr_host must not be NULL");
    if (p->nnzb && (!vals || !col_idx)) return set_error(SMAT_ERR_INVALID, "vals and col_idx must not be NULL");
    // the work lists below index the plan's copy of col_idx_host through the row pointer: it has to be the one the
    // plan was made from, not a stale or foreign array of the caller
    if (memcmp(row_ptr_host, p->row_ptr_host.data(), p->row_ptr_host.size() * sizeof(int32_t)) != 0)
        return set_error(SMAT_ERR_INVALID, "row_ptr_host differs from the block row pointer the plan was created with");
    row_ptr_host = p->row_ptr_host.data();
    // The new list is built before the old one goes.  Whatever happens below, the old list describes values
    // that have changed, so it is dropped, and a plan left without a list goes back to a dense kernel.
    const size_t mb = p->M / 16;
    const int want = p->kernel_requested;
    const bool may_mix = want == SMAT_KERNEL_AUTO || want == SMAT_KERNEL_MIXED;
    const int dense_kernel = p->sweep.d_ops ? SMAT_KERNEL_SWEEP : SMAT_KERNEL_ROWWISE;
    auto drop_mixed = [&] {
        p->sweep_dense.release();
        p->sweep_blocks.release();
        if (p->d_vals_dense) { (void)dev_free(p->d_vals_dense); p->d_vals_dense = nullptr; }
        p->n_blocks_split = 0;
        if (p->d_items_dense) { (void)dev_free(p->d_items_dense); p->d_items_dense = nullptr; }
        if (p->d_split_dense) { (void)dev_free(p->d_split_dense); p->d_split_dense = nullptr; }
        if (p->d_workspace_dense) { (void)dev_free(p->d_workspace_dense); p->d_workspace_dense = nullptr; }
        p->n_items_dense = p->n_split_dense = 0;
        p->n_blocks_dense = 0;
        window_destroy(p->window);
        p->window = nullptr;
        resident_destroy(p->resident);
        p->resident = nullptr;
    };
    auto fail = [&](hipError_t err) {
        if (p->compact) { compact_destroy(p->compact); p->compact = nullptr; }
        drop_mixed();
        if (p->kernel == SMAT_KERNEL_COMPACT || p->kernel == SMAT_KERNEL_MIXED) p->kernel = dense_kernel;
        return set_error(SMAT_ERR_HIP, "attaching values failed: %s", hipGetErrorString(err));
    };
    // Block rows with at least 60% of their 16 x blocks columns nonzero are the dense kernels' business: they
    // gather 16 rows of B per block, the compact kernel one row per nonzero column.  Measured: 7 nonzero columns
    // per block (27-point stencil) 53 us compact against 86 us row-wise; 16 per block (dense blocks, N = 4096)
    // 326 us against 180 us.  This is the per-block classification of the reference (matrix.h:400-419: blocks
    // without / with 2:4 / with dense rows) put to use per block row.
    CompactCensus census;
    CompactPlan *c = nullptr;
    // The widths of windows beside it, where the host would not count them sooner once they are asked for.
    WindowCount count;
    hipError_t e = compact_census(vals, row_ptr, mb, p->nnzb, census, col_idx, p->K / 16,
                                  may_take_window(*p) && (p->nnzb > WindowCount::FEW || p->col_idx_host.size() != p->nnzb) ? &count : nullptr);
    if (e != hipSuccess) return fail(e);
    std::vector<uint8_t> dense(mb, 0);
    int64_t dense_cols_all = 0;
    for (size_t i = 0; may_mix && i < mb; i++) {
        const int64_t blocks = row_ptr_host[i + 1] - row_ptr_host[i], cols = census.cols_of_row(i);
        if (blocks > 0 && (double)cols >= 0.6 * 16.0 * (double)blocks) {
            dense[i] = 1;
            dense_cols_all += cols;
        }
    }
    int64_t blocks_dense = 0;
    for (size_t i = 0; may_mix && i < mb; i++)
        if (dense[i]) blocks_dense += row_ptr_host[i + 1] - row_ptr_host[i];
    const int64_t blocks_sparse = (int64_t)p->nnzb - blocks_dense;
    // both kinds of rows matter (a tenth of the blocks each): mixed dispatch.  Otherwise one kernel for everything.
    bool mixed = may_mix && blocks_dense * 10 >= (int64_t)p->nnzb && blocks_sparse * 10 >= (int64_t)p->nnzb;
    // the dense rows through the sweep kernel when their row groups of 64 fill the device, else row-wise
    size_t n_dense_rows = 0;
    for (size_t i = 0; may_mix && i < mb; i++) n_dense_rows += dense[i] != 0;
    const bool dense_sweep_possible = !p->col_idx_host.empty() && blocks_dense >= 2 && p->nnzb < ((size_t)1 << 23) &&
                                      p->K < ((size_t)1 << 28) && sweep_fills_device(n_dense_rows, p->n_cap);
    bool dense_packed = p->d_bpack != nullptr; // row-wise route: B repacked slab-major first?
    if (mixed && !dense_sweep_possible && want != SMAT_KERNEL_MIXED) {
        // Row-wise route for the dense rows: it has to beat the compact kernel on those very rows, launch and (when B
        // is repacked for it) the extra pass over B included.  Rates as measured: the compact kernel gathers about 10 TB/s of
        // operand bytes, the row-wise kernel on B in place 7.6 TB/s, the row-wise kernel on repacked B 20 TB/s; a
        // pass over B moves 4*K*N bytes at 4 TB/s; a launch costs 3 us.  (27-point stencil on 64^3 after the reorder,
        // N = 64: a sixth of the blocks sit in dense rows, 10 us of compact kernel against 20 us for the repack alone.)
        const double dense_cols = (double)dense_cols_all;
        const double t_compact = dense_cols * (double)p->n_cap * 2.0 / 10e6;
        const double gather = (double)blocks_dense * 16.0 * (double)p->n_cap * 2.0;
        const double t_direct = gather / 7.6e6 + 3.0;
        const double t_packed = gather / 20e6 + 6.0 + 4.0 * (double)p->K * (double)p->n_cap / 4e6;
        dense_packed = t_packed < t_direct;
        if (std::min(t_direct, t_packed) >= 0.8 * t_compact) mixed = false;
    }
    // Per-block split, where the rows do not sort into two kinds but the blocks do (the reference's classification,
    // matrix.h:400-419, taken at its word): blocks with at least 10 of their 16 columns nonzero are copied one behind
    // the other and go through the sweep kernel, which writes every row of C; the compact kernel then ADDS the
    // columns of the other blocks (fp16 C: one more rounding of the partial result, well inside the tolerance).
    // Taken when both kinds hold a tenth of the blocks, the sweep kernel's workgroups fill the device, and an
    // estimate says it beats the better single kernel by 5 % - or when it is asked for (SMAT_KERNEL_MIXED) and the
    // rows do not split.  Rates as measured on 8192^2, N = 4096: the sweep kernel moves its panels of B into LDS once
    // per group of 64 block rows at 13.4 TB/s and multiplies at 1.04 Pflop/s on top of that (26,214 blocks 93 us, 79,540
    // blocks 201 us), the compact kernel gathers 10 TB/s of rows of B, a pass over B moves 4 K N bytes at 4 TB/s + 3 us
    // (10 % dense blocks with as many blocks again of one nonzero: estimate 179 us, measured 180; sweep kernel alone
    // 201 us, compact kernel alone 252 us).
    bool block_split = false;
    const int64_t n_split_blocks = census.full_blocks;
    const double n_est = (double)p->n_cap, n_rg_est = (double)((mb + SWEEP_G - 1) / SWEEP_G);
    auto t_sweep = [&](double blocks) { return n_rg_est * (double)p->K * n_est * 2.0 / 13.4e6 + blocks * n_est * 512.0 / 1.04e9; };
    auto t_compact = [&](double cols) { return cols * n_est * 2.0 / 10e6; };
    const double t_pass = 3.0 + (double)p->K * n_est / 1e6;
    // one kernel for everything: the sweep kernel (when the plan has its work list) or the compact kernel
    const double t_sweep_all = !p->sweep.d_ops ? 1e30
                               : p->sweep_few_tiles ? sweep_estimate_us((size_t)p->sweep.n_rg, p->sweep_chunks, p->nnzb, p->M, p->n_cap)
                                                    : t_sweep((double)p->nnzb);
    const double t_compact_all = t_compact((double)census.n_cols_all) + t_pass;
    if (may_mix && !mixed && !p->col_idx_host.empty() && p->nnzb < ((size_t)1 << 23) &&
        p->K < ((size_t)1 << 28) && sweep_fills_device(mb, p->n_cap)) {
        const int64_t n_rest = (int64_t)p->nnzb - n_split_blocks;
        if (n_split_blocks >= 2 && n_split_blocks * 10 >= (int64_t)p->nnzb && n_rest * 10 >= (int64_t)p->nnzb) {
            const double t_split = t_sweep((double)n_split_blocks) + t_compact((double)census.cols_rest) + t_pass;
            block_split = want == SMAT_KERNEL_MIXED || t_split < 0.95 * std::min(t_sweep_all, t_compact_all);
        }
    }
    std::vector<uint8_t> skip; // the blocks that the sweep kernel takes
    if (block_split) { // the list without them
        e = compact_full_blocks(census, skip);
        if (e == hipSuccess) e = compact_build(census, vals, row_ptr, col_idx, p->K, p->n_cap, p->d_bcol != nullptr, nullptr, true, &c);
        if (e != hipSuccess) return fail(e);
        if (c->n_split_rows > 0) { // partial tiles through the workspace cannot be added to C: one kernel for everything
            block_split = false;
            compact_destroy(c);
            c = nullptr;
            e = compact_census(vals, row_ptr, mb, p->nnzb, census);
            if (e != hipSuccess) return fail(e);
        }
    }
    if (want == SMAT_KERNEL_MIXED && !block_split) mixed = true;
    if (p->compact) { compact_destroy(p->compact); p->compact = nullptr; }
    drop_mixed();
    // the compact kernel for everything: few nonzero columns per block - unless the plan has the sweep kernel's work
    // list and the same estimate says that one is faster (blocks of both kinds in a matrix that is dense enough)
    bool take = mixed || block_split || want == SMAT_KERNEL_COMPACT ||
                (want == SMAT_KERNEL_AUTO && (double)census.n_cols_all < 0.6 * 16.0 * (double)p->nnzb &&
                 !(dense_kernel == SMAT_KERNEL_SWEEP && t_sweep_all < t_compact_all));
    if (p->kernel == SMAT_KERNEL_COMPACT || p->kernel == SMAT_KERNEL_MIXED) p->kernel = dense_kernel;
    if (want == SMAT_KERNEL_AUTO && dense_kernel == SMAT_KERNEL_ROWWISE && !mixed && !block_split) {
        // Windows against the compact kernel (whole panels of 16, 32 or 64 columns; row-major B in place), or against the row-wise one where the
        // sweep kernel's rule leaves a matrix to it.
        size_t group_rows = 0;
        double sweep_us = 1e30;
        if (!take && p->col_idx_host.size() == p->nnzb)
            group_rows = sweep_group_rows(row_ptr_host, p->col_idx_host.data(), p->M, p->K, p->nnzb, p->n_cap, (size_t)p->n_items,
                                          p->n_split_rows ? RowLengths::SPLIT : RowLengths::EVEN, p->d_bpack != nullptr, p->d_bcol != nullptr, &sweep_us);
        if (group_rows) {
            // Windows against the sweep kernel, whose streams are made all the same: the plan says that kernel, and launches that ask for it
            // get it.  us: bands of 13296 rows and 30, N = 304 9.6 -> 7.5, 8320 and 25, N = 576 10.4 -> 8.7, 39584 and 18, N = 904 55 -> 48; 21 x 14 x 52,
            // N = 88 8.4 -> 6.2, 21 x 76 x 25, N = 224 22.6 -> 20.1.
            if (!p->d_bcol && !g_force_group_rows) e = take_window_if_room(*p, row_ptr, col_idx, count, sweep_us, nullptr, nullptr);
            if (e == hipSuccess) e = sweep_small_groups(*p, group_rows);
        } else if (!take || !p->d_bcol)
            e = take_window_if_room(*p, row_ptr, col_idx, count, compact_estimate_us((double)census.n_cols_all, std::min(36.0 * (double)census.n_cols_all, 4.25 * (double)census.n_cols_all + 4.0 * (double)census.nnz), p->M, p->K,
                                                p->n_cap), vals, take ? &census : nullptr);
        if (e != hipSuccess) return fail(e);
    }
    if (want == SMAT_KERNEL_AUTO && dense_kernel == SMAT_KERNEL_SWEEP && p->sweep_few_tiles && !take && !p->d_bcol) { // attached before
        e = take_window_if_room(*p, row_ptr, col_idx, count, sweep_estimate_us((size_t)p->sweep.n_rg, p->sweep_chunks, p->nnzb, p->M, p->n_cap), nullptr, nullptr);
        if (e != hipSuccess) return fail(e);
    }
    if (!take) { // nothing would use the list: the plan keeps (or goes back to) a dense kernel
        if (p->window) e = hipStreamSynchronize(nullptr); // launches on other streams read its lists
        return e == hipSuccess ? SMAT_OK : fail(e);
    }
    if (!c) e = compact_build(census, vals, row_ptr, col_idx, p->K, p->n_cap, p->d_bcol != nullptr, mixed ? &dense : nullptr, false, &c);
    if (e != hipSuccess) return fail(e);
    if (!p->d_bt) e = dev_malloc(&p->d_bt, p->bt_bytes());
    std::vector<int32_t> dense_list;
    for (size_t i = 0; mixed && i < mb; i++)
        if (dense[i]) dense_list.push_back((int32_t)i);
    const bool dense_sweep = mixed && dense_sweep_possible;
    if (mixed && !dense_sweep) { // the scratch for the repacked B follows the choice made for the dense rows
        if (dense_packed && !p->d_bpack && e == hipSuccess) e = dev_malloc(&p->d_bpack, p->K * p->n_cap * sizeof(uint16_t));
        if (!dense_packed && p->d_bpack && want == SMAT_KERNEL_AUTO) { (void)dev_free(p->d_bpack); p->d_bpack = nullptr; }
    }
    if (e == hipSuccess && block_split) {
        // the sub-matrix of the copied blocks: same block rows, the copies numbered in row-major order
        std::vector<int32_t> rp_d(mb + 1, 0), ci_d, ids;
        ci_d.reserve((size_t)n_split_blocks);
        ids.reserve((size_t)n_split_blocks);
        for (size_t i = 0; i < mb; i++) {
            for (int32_t q = row_ptr_host[i]; q < row_ptr_host[i + 1]; q++)
                if (skip[(size_t)q]) { ci_d.push_back(p->col_idx_host[(size_t)q]); ids.push_back(q); }
            rp_d[i + 1] = (int32_t)ci_d.size();
        }
        e = dev_malloc(&p->d_vals_dense, ids.size() * 256 * sizeof(uint16_t));
        if (e == hipSuccess) e = copy_blocks(vals, ids.data(), ids.size(), p->d_vals_dense);
        if (e == hipSuccess) {
            try { // the list and the copies made so far are released by fail() below
                SweepPlanHost h;
                build_sweep_plan(rp_d.data(), ci_d.data(), mb, p->K / 16, h, nullptr, 0,
                                 want == SMAT_KERNEL_AUTO ? sweep_even_rounds(rp_d.data(), ci_d.data(), mb, p->K / 16, p->n_cap, p->d_bcol != nullptr) : SWEEP_G);
                e = p->sweep_blocks.upload(h, p->d_bcol != nullptr);
            } catch (...) {
                e = hipErrorOutOfMemory;
            }
        }
        p->n_blocks_split = n_split_blocks;
        p->n_blocks_dense = n_split_blocks;
    } else if (e == hipSuccess && dense_sweep) {
        try {
            SweepPlanHost h;
            build_sweep_plan(row_ptr_host, p->col_idx_host.data(), mb, p->K / 16, h, dense_list.data(), dense_list.size());
            e = p->sweep_dense.upload(h, p->d_bcol != nullptr);
        } catch (...) {
            e = hipErrorOutOfMemory;
        }
        p->n_blocks_dense = blocks_dense;
    } else if (e == hipSuccess && mixed) {
        std::vector<WorkItem> items;
        std::vector<SplitRow> split;
        const int slots = rowwise_work_list(row_ptr_host, mb, p->cuts, dense.data(), items, split);
        p->n_items_dense = (int)items.size();
        rowwise_costs(items, p->deal_dense);
        p->n_split_dense = (int)split.size();
        p->n_blocks_dense = blocks_dense;
        e = dev_malloc(&p->d_items_dense, std::max<size_t>(items.size(), 1) * sizeof(WorkItem));
        if (e == hipSuccess && !items.empty())
            e = hipMemcpy(p->d_items_dense, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice);
        if (e == hipSuccess && !split.empty()) {
            e = dev_malloc(&p->d_split_dense, split.size() * sizeof(SplitRow));
            if (e == hipSuccess) e = hipMemcpy(p->d_split_dense, split.data(), split.size() * sizeof(SplitRow), hipMemcpyHostToDevice);
            if (e == hipSuccess) e = dev_malloc(&p->d_workspace_dense, (size_t)slots * 16 * p->n_cap * sizeof(float));
        }
    }
    if (e != hipSuccess) {
        compact_destroy(c);
        return fail(e);
    }
    census.waited();
    p->compact = c;
    c->by_name = want != SMAT_KERNEL_AUTO;
    p->kernel = mixed || block_split ? SMAT_KERNEL_MIXED : SMAT_KERNEL_COMPACT;
    // the deal of the compact kernel's work items to the XCDs, measured on this list at the plan's width (B in the
    // layout the plan was made for: d_bcol is the scratch of a plan for row-major B)
    // Columns of B in LDS against the compact kernel; no memory for their lists is not an error of the plan.
    if (want == SMAT_KERNEL_AUTO && !mixed && !block_split && !p->window && !p->d_bcol) {
        const double bar = 0.9 * compact_estimate_us(*c, p->M, p->K, p->n_cap);
        if (resident_forced() || resident_estimate_us(p->M, p->K, p->n_cap, census.nnz, c->n_split_rows > 0) < bar) {
            e = resident_build(*c, p->M, p->K, census.nnz, &p->resident);
            if (e == hipErrorOutOfMemory) e = hipSuccess, (void)hipGetLastError();
            if (e != hipSuccess) return fail(e);
        }
        if (p->resident) resident_settle(*p->resident, p->K, p->n_cap);
        if (p->resident && !resident_forced() && p->resident->own.us >= bar) {
            resident_destroy(p->resident);
            p->resident = nullptr;
        }
    }
    if (p->window) compact_deal_beside_windows(*c, p->n_cap, p->K);
    if (!p->window && !p->resident) e = compact_tune(*c, p->d_bt, p->M, p->n_cap, p->K, p->d_bcol != nullptr, block_split); // else its launches are not what the plan is for
    if (e != hipSuccess) return set_error(SMAT_ERR_HIP, "timing the compact kernel failed: %s", hipGetErrorString(e));
    if (p->d_bpack && want == SMAT_KERNEL_AUTO && !mixed) { // the row-wise kernel's scratch is not needed any more
        (void)dev_free(p->d_bpack);
        p->d_bpack = nullptr;
    }
    return SMAT_OK;
}

extern "C" int smat_plan_attach_values(smat_plan *p, const uint16_t *vals, const int32_t *row_ptr,
                                        const int32_t *col_idx, const int32_t *row_ptr_host)
{
    return smat::guarded("smat_plan_attach_values", [&] { return smat_plan_attach_values_impl(p, vals, row_ptr, col_idx, row_ptr_host); });
}

extern "C" int smat_plan_destroy(smat_plan *p)
{
    if (!p) return SMAT_OK;
    if (p->compact) compact_destroy(p->compact);
    if (p->d_bt) (void)dev_free(p->d_bt);
    window_destroy(p->window);
    resident_destroy(p->resident);
    if (p->d_bcol) (void)dev_free(p->d_bcol);
    if (p->d_items_dense) (void)dev_free(p->d_items_dense);
    if (p->d_split_dense) (void)dev_free(p->d_split_dense);
    if (p->d_workspace_dense) (void)dev_free(p->d_workspace_dense);
    if (p->d_items) (void)dev_free(p->d_items);
    if (p->d_split) (void)dev_free(p->d_split);
    if (p->d_workspace) (void)dev_free(p->d_workspace);
    if (p->d_bpack) (void)dev_free(p->d_bpack);
    p->sweep.release();
    p->sweep_dense.release();
    p->sweep_blocks.release();
    if (p->d_vals_dense) (void)dev_free(p->d_vals_dense);
    delete p;
    return SMAT_OK;
}

extern "C" int smat_plan_check(const smat_plan *p, const int32_t *row_ptr_host, const int32_t *col_idx_host,
                               size_t M, size_t K, size_t nnzb)
{
    if (!p || !row_ptr_host) return set_error(SMAT_ERR_INVALID, "plan and row_ptr_host must not be NULL");
    if (p->M != M || p->K != K || p->nnzb != nnzb)
        return set_error(SMAT_ERR_INVALID, "plan was built for another matrix (M/K/nnzb differ)");
    if (p->fingerprint_has_cols && !col_idx_host)
        return set_error(SMAT_ERR_INVALID, "the plan was built with col_idx_host: pass it to check the plan");
    const uint64_t h = pattern_fingerprint(row_ptr_host, p->fingerprint_has_cols ? col_idx_host : nullptr, M / 16, nnzb);
    if (h != p->fingerprint)
        return set_error(SMAT_ERR_INVALID, "plan was built for another block pattern (row_ptr / col_idx differ)");
    return SMAT_OK;
}

extern "C" int smat_plan_values_current(const smat_plan *p, const uint16_t *vals, int *current)
{
    if (!p || !current) return set_error(SMAT_ERR_INVALID, "plan and current must not be NULL");
    *current = 1;
    if (!p->compact) return SMAT_OK; // no kernel of this plan works from a copy of the values
    if (p->nnzb && !vals) return set_error(SMAT_ERR_INVALID, "vals must not be NULL");
    uint64_t h = 0;
    hipError_t e = values_checksum(vals, p->nnzb, &h);
    if (e != hipSuccess) return set_error(SMAT_ERR_HIP, "checksum of the block values failed: %s", hipGetErrorString(e));
    *current = h == p->compact->values_checksum;
    return SMAT_OK;
}

extern "C" int smat_plan_info(const smat_plan *p, int64_t *info)
{
    if (!p || !info) return set_error(SMAT_ERR_INVALID, "plan and info must not be NULL");
    info[0] = p->kernel; info[1] = p->n_items; info[2] = p->n_split_rows; info[3] = p->cuts.piece;
    info[4] = (int64_t)p->workspace_bytes;
    info[5] = p->kernel == SMAT_KERNEL_SWEEP ? 16 * SWEEP_TN : 16 * p->panel_tiles;
    info[6] = p->sweep.n_ops + p->sweep_dense.n_ops + p->sweep_blocks.n_ops;
    info[7] = p->sweep.n_records + p->sweep_dense.n_records + p->sweep_blocks.n_records;
    info[8] = (p->d_bpack ? (int64_t)(p->K * p->n_cap * sizeof(uint16_t)) : 0) +
              (p->d_bt ? (int64_t)p->bt_bytes() : 0) +
              (p->d_bcol ? (int64_t)(p->K * p->n_cap * sizeof(uint16_t)) : 0);
    info[9] = p->compact ? p->compact->n_cols : 0;
    info[10] = p->sweep_blocks.d_ops ? -1 : p->n_items_dense; // -1: the mixed plan splits per block, not per block row
    info[11] = p->n_blocks_dense;
    return SMAT_OK;
}

// ---- runtime wrappers --------------------------------------------------------

extern "C" int smat_device_count(int *n)
{
    if (!n) return set_error(SMAT_ERR_INVALID, "n must not be NULL");
    SMAT_HIP(hipGetDeviceCount(n));
    return SMAT_OK;
}
extern "C" int smat_set_device(int dev) { SMAT_HIP(hipSetDevice(dev)); return SMAT_OK; }
extern "C" int smat_device_name(int dev, char *buf, size_t len)
{
    if (!buf || !len) return set_error(SMAT_ERR_INVALID, "buf must not be NULL");
    hipDeviceProp_t prop;
    SMAT_HIP(hipGetDeviceProperties(&prop, dev));
    snprintf(buf, len, "%s (%s)", prop.name, prop.gcnArchName);
    return SMAT_OK;
}
extern "C" int smat_device_attr(int dev, int64_t *cus, int64_t *lds_bytes, int64_t *mem_bytes,
                                 int64_t *clock_khz)
{
    hipDeviceProp_t prop;
    SMAT_HIP(hipGetDeviceProperties(&prop, dev));
    if (cus) *cus = prop.multiProcessorCount;
    if (lds_bytes) *lds_bytes = (int64_t)prop.maxSharedMemoryPerMultiProcessor;
    if (mem_bytes) *mem_bytes = (int64_t)prop.totalGlobalMem;
    if (clock_khz) *clock_khz = prop.clockRate;
    return SMAT_OK;
}
extern "C" int smat_malloc(void **dptr, size_t bytes)
{
    if (!dptr) return set_error(SMAT_ERR_INVALID, "dptr must not be NULL");
    SMAT_HIP(dev_malloc(dptr, bytes ? bytes : 1));
    return SMAT_OK;
}
extern "C" int smat_free(void *dptr) { if (dptr) SMAT_HIP(dev_free(dptr)); return SMAT_OK; }
extern "C" int smat_memcpy_h2d(void *d, const void *s, size_t n) { if (n) SMAT_HIP(hipMemcpy(d, s, n, hipMemcpyHostToDevice)); return SMAT_OK; }
extern "C" int smat_memcpy_d2h(void *d, const void *s, size_t n) { if (n) SMAT_HIP(hipMemcpy(d, s, n, hipMemcpyDeviceToHost)); return SMAT_OK; }
extern "C" int smat_memcpy_d2d(void *d, const void *s, size_t n) { if (n) SMAT_HIP(hipMemcpy(d, s, n, hipMemcpyDeviceToDevice)); return SMAT_OK; }
extern "C" int smat_memset(void *d, int byte, size_t n) { if (n) SMAT_HIP(hipMemset(d, byte, n)); return SMAT_OK; }
extern "C" int smat_device_synchronize(void) { SMAT_HIP(hipDeviceSynchronize()); return SMAT_OK; }
extern "C" int smat_stream_create(void **s)
{
    if (!s) return set_error(SMAT_ERR_INVALID, "stream must not be NULL");
    hipStream_t st;
    SMAT_HIP(hipStreamCreate(&st)); // default priority
    *s = st;
    return SMAT_OK;
}
extern "C" int smat_stream_destroy(void *s) { if (s) SMAT_HIP(hipStreamDestroy((hipStream_t)s)); return SMAT_OK; }
extern "C" int smat_stream_synchronize(void *s) { SMAT_HIP(hipStreamSynchronize((hipStream_t)s)); return SMAT_OK; }
extern "C" int smat_event_create(void **ev)
{
    if (!ev) return set_error(SMAT_ERR_INVALID, "event must not be NULL");
    hipEvent_t e;
    SMAT_HIP(hipEventCreate(&e));
    *ev = e;
    return SMAT_OK;
}
extern "C" int smat_event_destroy(void *ev) { if (ev) SMAT_HIP(hipEventDestroy((hipEvent_t)ev)); return SMAT_OK; }
extern "C" int smat_event_record(void *ev, void *s) { SMAT_HIP(hipEventRecord((hipEvent_t)ev, (hipStream_t)s)); return SMAT_OK; }
extern "C" int smat_event_synchronize(void *ev) { SMAT_HIP(hipEventSynchronize((hipEvent_t)ev)); return SMAT_OK; }
extern "C" int smat_event_elapsed_ms(void *a, void *b, float *ms)
{
    if (!ms) return set_error(SMAT_ERR_INVALID, "ms must not be NULL");
    SMAT_HIP(hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b));
    return SMAT_OK;
}

// ---- what the MFMA pipes of this device deliver --------------------------------
// A kernel of nothing but v_mfma_f32_16x16x32_f16 on registers: 8 wavefronts per workgroup, 8 independent
// accumulators each, one workgroup per CU and launch slot.  The rate it reaches is the ceiling any fp16 kernel
// on this device and clock can approach; benchmarks quote it next to the published peak.
namespace {
typedef _Float16 peak_f16x8 __attribute__((ext_vector_type(8)));
typedef float peak_f32x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(512) void mfma_peak_kernel(float *out, int iters)
{
    peak_f32x4 acc[8];
    for (int t = 0; t < 8; t++) acc[t] = (peak_f32x4){0, 0, 0, 0};
    const _Float16 x = (_Float16)(0.001f * (threadIdx.x & 7)), y = (_Float16)(threadIdx.x & 3);
    peak_f16x8 a = {x, x, x, x, x, x, x, x}, b = {y, y, y, y, y, y, y, y};
    for (int i = 0; i < iters; i += 8) { // 64 MFMAs per trip: the loop control disappears behind them
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int t = 0; t < 8; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[t], 0, 0, 0);
    }
    float s = 0;
    for (int t = 0; t < 8; t++) s += acc[t][0] + acc[t][1] + acc[t][2] + acc[t][3];
    if (s == 12345.678f) out[0] = s; // keeps the loop alive, never true for these operands
}
} // namespace

extern "C" int smat_bench_mfma_peak(double *tflops)
{
    if (!tflops) return set_error(SMAT_ERR_INVALID, "tflops must not be NULL");
    hipDeviceProp_t prop;
    int dev = 0;
    SMAT_HIP(hipGetDevice(&dev));
    SMAT_HIP(hipGetDeviceProperties(&prop, dev));
    const int cus = prop.multiProcessorCount, iters = 16384;
    float *out = nullptr;
    SMAT_HIP(dev_malloc(&out, sizeof(float)));
    hipEvent_t e0, e1;
    SMAT_HIP(hipEventCreate(&e0));
    SMAT_HIP(hipEventCreate(&e1));
    double best = 0;
    for (int rep = 0; rep < 8; rep++) { // the first passes warm the clocks
        SMAT_HIP(hipEventRecord(e0, nullptr));
        hipLaunchKernelGGL(mfma_peak_kernel, dim3(cus), dim3(512), 0, nullptr, out, iters);
        SMAT_HIP(hipEventRecord(e1, nullptr));
        SMAT_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SMAT_HIP(hipEventElapsedTime(&ms, e0, e1));
        const double flops = (double)cus * 8 * iters * 8 * 2.0 * 16 * 16 * 32;
        if (rep && ms > 0) best = std::max(best, flops / (ms * 1e-3) / 1e12);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)dev_free(out);
    SMAT_HIP(hipGetLastError());
    *tflops = best;
    return SMAT_OK;
}
