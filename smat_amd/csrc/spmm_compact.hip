// SpMM for block matrices whose 16x16 blocks hold only a few nonzero COLUMNS (random sparse
// matrices blocked without much clustering: about one nonzero per block).  The dense kernels
// gather 16 rows of B for every block; here only the rows of B that meet a nonzero column of A
// are touched, and 32 such columns of one block row are multiplied per MFMA step.
//
// Same product as the reference kernel (src/cuda_hgemm/src/mma/mmaCBT.cu:13-88): an all-zero
// column of a block contributes nothing to C, so leaving it out changes no result (with finite B).
//
//  * compact_build (once per matrix, from the block values):
//      colmask_kernel   16-bit mask of the nonzero columns of every block (two blocks per
//                       wavefront step, OR over the 16 rows with cross-lane shuffles);
//      exclusive scan   of the popcounts; the per-block-row totals go to the host, which pads
//                       every block row to a multiple of 32 columns (zero columns) and cuts the
//                       list into work items (whole block rows, long ones in chunks whose fp32
//                       partial tiles are summed afterwards);
//      gather_kernel    writes, for every nonzero column, its row of B (absolute column index)
//                       and a COPY of its values: either all 16 in MFMA operand order,
//                       acol[((step*4 + g)*16 + m)*8 + j] = A[m][column 32*step + 8*g + j],
//                       so that the A operand of a step is one coalesced 16-byte load per lane; or, where
//                       columns hold few nonzeros, the nonzeros alone with their places in that operand.
//    The SpMM then does not read the block values any more: they must be attached again when
//    they change.
//  * transpose_b_kernel: column-major B (B[n*K + k]) -> Bt at the start of every launch, so that
//    the row of B under a nonzero column is contiguous.  Bt holds the panels of W columns one
//    after the other, each a row-major K x W matrix: the pass over a panel gathers from one
//    contiguous K * 2*W bytes.
//  * spmm_compact_kernel<W>: one wavefront per (run of work items, panel of W columns).  A step takes
//    32 columns = K of one v_mfma_f32_16x16x32_f16.  The product is formed as C^T = B^T * A^T like in the other
//    kernels; every gather is 16 bytes per lane (a CU keeps a limited number of vector memory instructions and of
//    cache lines in flight, so an instruction should bring as much as it can).  The index list keeps, inside every
//    group of 8, the even entries first and then the odd ones: the four indices a lane needs are 16 contiguous bytes.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <type_traits>
#include <vector>

#include "devmem.h"
#include "spmm_kernels.h"

namespace smat {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

int g_force_run = 0;
int g_tune = 1; // test hook: 0 = attaching values measures nothing, the estimate decides the deal
std::atomic<int> g_last_share{1}, g_last_run{0}; // test hooks: wavefronts a task and the run length of the latest launch, of any thread
int g_force_list = 0; // test hook: 1 = lists of whole columns, 2 = of nonzeros, 0 = compact_build decides
int g_force_staged = 0; // test hook: 1 = entries go through LDS in blocks wherever they may, 2 = nowhere, 0 = the launcher decides
int g_force_order = 0; // test hook: 1 = tasks of lists with split rows in the order of their items, 2 = as order_tasks says, 0 = orders_tasks decides
int g_force_share = 0; // test hook: 1, 2 or 4 = wavefronts that share a task where they may, 0 = the launcher decides
int g_force_tq = 0; // test hook: 1 or 2 = panels of 64 or 128 columns whatever the sizes say, 0 = the launcher decides

constexpr int FULL_BLOCK_COLS = 10; // nonzero columns from which a block counts as full (of 16)
constexpr int TASK_STEPS = 12;     // short items are put together up to this many steps (8 to 24: level; one item each: 9 % slower on R-MAT)
constexpr int LONG_ROW_STEPS = 56; // steps from which a block row is split where a launch has few wavefronts
// Bytes of B that its copy has to leave out, and an eighth of B.  The place of every row, which the transposition has to read, costs 0.2 to 0.9 us
// where nothing else changes; what is left out is not written (1 us for about 6 MB where B comes from HBM) and not between the gathered
// rows, which counts from some 20 MB on.  70 products (uniform rows and R-MAT, K 8,192 to 1,048,576, N 16 to 1,008), copy of all rows -> of the used ones: from
// 11 MB on none is slower in any mode, with inputs taking turns from equal (3792 x 46784, 8 a row, N = 280, 14 MB 16.7 -> 16.7 us) over 20.8 -> 17.9
// (1264 x 35568, 10 a row, N = 480, 24 MB) to 213 -> 163 (17392 x 150672, 5 a row, N = 912, 148 MB).  Between 5 and 11 MB 14.6 -> 15.4 (13680 x 110544, 5 a
// row, N = 72, 9 MB) to 55.2 -> 51.1 (R-MAT scale 17, N = 72, 8 MB); below 5 MB 17.5 -> 18.4 (5888 x 76192, 27 a row, N = 112, 2 MB) to 35.8 -> 35.2.
constexpr size_t PLACE_MIN_BYTES = (size_t)21 << 19;
// Entries are staged where a wavefront's place on the device has many steps to do (before the longer way of the first entries of a task
// counts: 16384^2, 16 a row, N = 128 10.9 -> 11.5 us), where the lists are longer than the L2s hold, and where the product touches
// nearly half of the memory-side cache of 256 MiB or more.  Whether A is still in that cache when it is multiplied again follows
// from what the program does in between, which nothing here can know.  What is taken: products below the third line, two of which
// fit side by side, find their lists there again as a rule, larger ones do not.  In the figures beside the kernel a
// larger product gains 7 to 10 % where its lists do come from HBM and loses 0 to 4 % where they do not (row-major B 6 and 6 %); a smaller one would gain 2 to 7 and
// lose 0 to 7.
constexpr double STAGED_STEPS = 20.0;
constexpr int64_t STAGED_BYTES = 4 << 20;
constexpr int64_t STAGED_TOUCHED = 112 << 20, STAGED_TOUCHED_IN_PLACE = 100 << 20; // with a copy of B, which is touched too, and without
constexpr int ENTRY_PAD = 1024; // entries readable past the last one (blocks of 256, one ahead, another for the steps past the end of a task)
constexpr int LIST_PAD = 2304; // entries readable past the end of the list (the index loads of the 64-column panel run up to 16 steps ahead)

// ---- census of nonzero block columns ----

// Sums over a whole pass: a workgroup adds its part to one of SUM_SLOTS groups of words, 128 bytes apart.  Additions to
// one word queue up at 12 ns each, which for one word and every wavefront of a pass over 121 MB is 200 us of a 25 us pass.
constexpr int SUM_SLOTS = 32, SUM_STRIDE = 16;
constexpr size_t SUM_BYTES = SUM_SLOTS * SUM_STRIDE * sizeof(unsigned long long);
template <int N>
__device__ __forceinline__ void add_totals(const unsigned long long (&mine)[N], unsigned long long *__restrict__ sums)
{
    __shared__ unsigned long long part[4][N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        unsigned long long v = mine[i];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][i] = v;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        const unsigned long long v = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
        if (v) atomicAdd(&sums[(blockIdx.x % SUM_SLOTS) * SUM_STRIDE + threadIdx.x], v);
    }
}
// sums[i] of the pass, from the words that add_totals added to
void add_up_totals(const unsigned long long *all, unsigned long long *out, int n)
{
    for (int i = 0; i < n; i++) {
        out[i] = 0;
        for (int s = 0; s < SUM_SLOTS; s++) out[i] += all[s * SUM_STRIDE + i];
    }
}
// Order-independent 64-bit checksum of the block values: sum over all dwords of value * (2 * index + 1).
__device__ __forceinline__ unsigned long long checksum_term(uint32_t v, long i)
{
    return (unsigned long long)v * (2ull * (unsigned long long)i + 1ull);
}

// What a pass over the blocks counts besides the masks, summed over all blocks (add_totals): the checksum of the values,
// blocks with at least FULL_BLOCK_COLS nonzero columns, nonzero columns of the others, nonzeros.
enum { SUM_CHECK, SUM_FULL, SUM_COLS_REST, SUM_NNZ, N_SUMS };

// combined over the 16 lanes of a DPP row, in all of them
__device__ __forceinline__ uint32_t row_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false); // row_ror:8
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false);
    return v;
}
__device__ __forceinline__ uint32_t row_sum(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false);
    return v;
}

// Per block: mask of its nonzero columns; their number in the lower half of count, the number of nonzeros in the upper.
// Bound by the read of the values.  A lane holds one row of one half of a block, a DPP row of 16 lanes that half: its eight bits
// are or-ed and counted in the VALU, where exchanging the values through LDS was most of the time (237 k blocks, 121 MB:
// 40 -> 24 us).  The only nonzero of a block is put beside the mask, 4 bytes that spare the lists a second look at the 512 of the block.
__global__ __launch_bounds__(256) void colmask_kernel(const uint16_t *__restrict__ vals, long nnzb,
                                                      uint16_t *__restrict__ mask, uint32_t *__restrict__ single,
                                                      unsigned long long *__restrict__ count, unsigned long long *__restrict__ sums)
{
    unsigned long long total[N_SUMS] = {0, 0, 0, 0};
    const int lane = threadIdx.x & 63;
    const int at = (lane & 15) * 16 + ((lane >> 4) & 1) * 8; // row lane % 16, half lane / 16 % 2: 8 values
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const long n_waves = ((long)gridDim.x * blockDim.x) >> 6;
    auto load = [&](long pb) {
        const long blk = pb + (lane >> 5);
        return blk < nnzb ? *reinterpret_cast<const u32x4 *>(vals + blk * 256 + at) : (u32x4){0u, 0u, 0u, 0u};
    };
    u32x4 next = load(wave * 2);
    for (long pb = wave * 2; pb < nnzb; pb += n_waves * 2) {
        const u32x4 w = next;
        next = load(pb + n_waves * 2);
        const long blk = pb + (lane >> 5);
        // the checksum of four dwords from dword i on: (2 i + 1) sum of w[q] + 2 sum of q w[q]
        const unsigned long long plain = ((unsigned long long)w[0] + w[1]) + ((unsigned long long)w[2] + w[3]);
        const unsigned long long weighted = (unsigned long long)w[1] + 2ull * w[2] + 3ull * w[3];
        total[SUM_CHECK] += checksum_term(1, blk * 128 + at / 2) * plain + 2ull * weighted;
        uint32_t bits = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) { // -0.0 is a zero
            if (w[q] & 0x7fffu) bits |= 1u << (2 * q);
            if (w[q] & 0x7fff0000u) bits |= 2u << (2 * q);
        }
        const uint32_t mine = bits, nz_half = row_sum(__popc(bits));
        bits = row_or(bits);
        // lanes 0 and 32 put the halves of their blocks together
        const uint32_t other = __shfl(bits, (lane & 32) | 16), nz = nz_half + __shfl_xor(nz_half, 16);
        if (nz == 1 && mine && blk < nnzb) {
            const uint32_t i = (uint32_t)__ffs((int)mine) - 1, pair = i & 4 ? (i & 2 ? w[3] : w[2]) : (i & 2 ? w[1] : w[0]);
            single[blk] = (i & 1 ? pair & 0xffff0000u : pair << 16) | (uint32_t)(lane & 15);
        }
        if ((lane & 31) == 0 && blk < nnzb) {
            const uint32_t m = bits | (other << 8);
            const int cols = __popc(m);
            mask[blk] = (uint16_t)m;
            if (nz != 1) single[blk] = 0;
            count[blk] = (unsigned long long)nz << 32 | (unsigned)cols;
            total[SUM_NNZ] += nz;
            if (cols >= FULL_BLOCK_COLS) total[SUM_FULL]++;
            else total[SUM_COLS_REST] += cols;
        }
    }
    add_totals<N_SUMS>(total, sums);
}

__global__ __launch_bounds__(256) void values_checksum_kernel(const u32x4 *__restrict__ vals, long n_quads, unsigned long long *__restrict__ sums)
{
    unsigned long long sum = 0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n_quads; i += (long)gridDim.x * blockDim.x) {
        const u32x4 v = vals[i];
#pragma unroll
        for (int q = 0; q < 4; q++) sum += checksum_term(v[q], 4 * i + q);
    }
    const unsigned long long total[1] = {sum};
    add_totals<1>(total, sums);
}

// The block row that block p belongs to, the largest br with row_ptr[br] <= p, by all lanes of a wavefront together (p the
// same in all): every step looks at 64 rows.
__device__ __forceinline__ long row_of_block(const int32_t *__restrict__ row_ptr, long mb, long p, int lane)
{
    long lo = 0, n = mb; // br is one of lo .. lo + n - 1
    while (n > 1) {
        const long step = (n + 63) / 64;
        const long probe = lo + lane * step;
        const unsigned long long at_most = __ballot(lane * step < n && row_ptr[probe] <= p); // a run of low bits: row_ptr ascends
        const int last = 63 - __clzll((long long)at_most); // row_ptr[lo] <= p always
        n = n - last * step < step ? n - last * step : step;
        lo += last * step;
    }
    return lo;
}

// The nonzero columns of a block go to positions padded_start[br] + (columns of the block row in the blocks before it) .. of
// the padded list, and
//   acol != NULL: their 16 values each to acol, in MFMA operand order;
//   else: their nonzeros to entries from entry_start[br] + (nonzeros of the block row before) on, column by column,
//         each with its place in the operand of its step, and the range of entries of every step to step_range;
//   used != NULL: used[row] = 1 for the rows of B that the list names.
// A wavefront takes GATHER_BLOCKS consecutive blocks.  A lane looks one up and, where it holds one nonzero, writes that; the others follow four at a
// time: lane (g = lane / 16, r = lane % 16) holds row r of one.  Bound by loads that need each other (row, its start, values) and by the
// second read of the values of those others.  (Looking the blocks up four at a time, all 16 lanes alike, took 36 us for 16384^2, 16 a row, 98 % of the
// blocks of one nonzero; now 16.  64 blocks a wavefront 17.)
constexpr int GATHER_BLOCKS = 16;
__global__ __launch_bounds__(256) void gather_kernel(const uint16_t *__restrict__ vals, const uint16_t *__restrict__ mask, const uint32_t *__restrict__ single,
                              const unsigned long long *__restrict__ offset, const int32_t *__restrict__ row_ptr,
                              const int32_t *__restrict__ col_idx, const unsigned long long *__restrict__ raw,
                              const int2 *__restrict__ start, long mb, long nnzb, bool drop_full, int32_t *__restrict__ cols,
                              uint16_t *__restrict__ acol, uint32_t *__restrict__ entries, int2 *__restrict__ step_range, uint8_t *__restrict__ used)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const long p_first = (((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * GATHER_BLOCKS;
    if (p_first >= nnzb) return;
    // A lane looks its block up: the row, which is that of the first block or a little further on (past a run of empty rows the rest is halved).
    const bool live = lane < GATHER_BLOCKS && p_first + lane < nnzb;
    const long p_mine = live ? p_first + lane : p_first;
    long br = row_of_block(row_ptr, mb, p_first, lane);
    int ahead = 0;
    while (ahead < 8 && row_ptr[br + 1] <= p_mine) br++, ahead++;
    if (ahead == 8) {
        long lo = br, hi = mb;
        while (hi - lo > 1) {
            const long mid = (lo + hi) >> 1;
            if (row_ptr[mid] <= p_mine) lo = mid; else hi = mid;
        }
        br = lo;
    }
    uint32_t m_mine = live ? mask[p_mine] : 0;
    const uint32_t only = single[p_mine];
    const int2 first = start[br]; // of the columns and of the entries
    if (first.x < 0 || (drop_full && __popc(m_mine) >= FULL_BLOCK_COLS)) m_mine = 0; // another kernel multiplies the row or the block
    const unsigned long long before = offset[p_mine] - raw[br]; // no borrow: both halves of offset[p] are at least those of raw
    const int o_mine = first.x + (int)(uint32_t)before, end_mine = first.x + (int)(uint32_t)(raw[br + 1] - raw[br]);
    const int at_mine = first.y + (int)(before >> 32), c_mine = col_idx[p_mine];
    if (m_mine && only) { // acol holds zeros
        const int o = o_mine, c = c_mine + __ffs((int)m_mine) - 1;
        cols[(o & ~7) + ((o & 1) << 2) + ((o & 7) >> 1)] = c; // their order: below
        if (used) used[c] = 1;
        if (acol) {
            acol[((long)(o >> 3) * 16 + (only & 15)) * 8 + (o & 7)] = (uint16_t)(only >> 16);
        } else {
            entries[at_mine] = (only & 0xffff0000u) | (((uint32_t)((o & 31) >> 3) * 128u + (uint32_t)(o & 7) + (only & 15) * 8u) * 2u);
            if ((o & 31) == 0) step_range[o >> 5].x = at_mine;
            if ((o & 31) == 31 || o + 1 == end_mine) step_range[o >> 5].y = at_mine + 1;
        }
    }
    // The others four at a time, 16 lanes a block.
    for (unsigned long long left = __ballot(m_mine != 0 && !only); left;) {
        unsigned long long l = left;
        for (int i = 0; i < 4; i++) {
            if (i < g) l &= l - 1;
            left &= left - 1;
        }
        const int of = l ? __ffsll((long long)l) - 1 : 0;
        const uint32_t m_of = __shfl(m_mine, of), m = l ? m_of : 0; // all lanes take part
        const long p = p_first + of, row_end = __shfl(end_mine, of);
        u32x4 w[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
        if (m) w[0] = reinterpret_cast<const u32x4 *>(vals + p * 256 + r * 16)[0], w[1] = reinterpret_cast<const u32x4 *>(vals + p * 256 + r * 16)[1];
        long o = __shfl(o_mine, of);
        int32_t at = __shfl(at_mine, of);
        const int32_t c0 = __shfl(c_mine, of);
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const bool has = (m >> k) & 1;
            if (!__any(has)) continue;
            const uint32_t v = k & 1 ? w[k / 8][k % 8 / 2] >> 16 : w[k / 8][k % 8 / 2] & 0xffffu;
            const uint32_t nonzero = (uint32_t)(__ballot(has && (v & 0x7fffu)) >> (16 * g)) & 0xffffu; // rows of the lane's block
            if (!has) continue;
            // inside its group of 8 the even entries come first, then the odd ones: the lanes of the product kernel that
            // gather the even (odd) entries of a group read their four indices with one 16-byte load
            if (r == 0) {
                cols[(o & ~7L) + ((o & 1) << 2) + ((o & 7) >> 1)] = c0 + k;
                if (used) used[c0 + k] = 1;
            }
            if (acol) {
                acol[((o >> 3) * 16 + r) * 8 + (o & 7)] = (uint16_t)v; // (step*4 + g) = o / 8
            } else {
                if (r == 0 && (o & 31) == 0) step_range[o >> 5].x = at;
                const uint32_t place = (uint32_t)((o & 31) >> 3) * 128u + (uint32_t)(o & 7); // half of the step's operand, row 0; the entry holds it in bytes
                if ((nonzero >> r) & 1) entries[at + __popc(nonzero & ((1u << r) - 1u))] = v << 16 | (place + r * 8) * 2;
                at += __popc(nonzero);
                if (r == 0 && ((o & 31) == 31 || o + 1 == row_end)) step_range[o >> 5].y = at;
            }
            o++;
        }
    }
}

// Steps of every group of 32 listed columns: one for each `most` of its entries, at least one; none behind the last group.
__global__ void count_steps_kernel(const int2 *__restrict__ group_range, int n_groups, int most, int32_t *__restrict__ steps)
{
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (g > n_groups) return;
    const int n = g < n_groups ? group_range[g].y - group_range[g].x : 0;
    steps[g] = g == n_groups ? 0 : n > most ? (n + most - 1) / most : 1;
}
// The groups that take several steps are listed once for each, with another part of their entries.  32 threads a group.
__global__ __launch_bounds__(256) void expand_steps_kernel(const int2 *__restrict__ group_range, const int32_t *__restrict__ group_cols,
                                                           const int32_t *__restrict__ steps, const int32_t *__restrict__ first_step, int n_groups,
                                                           int most, int2 *__restrict__ step_range, int32_t *__restrict__ cols)
{
    const int g = (int)(blockIdx.x * 8 + threadIdx.x / 32), i = threadIdx.x & 31;
    if (g >= n_groups) return;
    const int2 r = group_range[g];
    const int32_t col = group_cols[(long)g * 32 + i];
    for (int k = 0; k < steps[g]; k++) {
        const int s = first_step[g] + k;
        cols[(long)s * 32 + i] = col;
        if (i == 0) step_range[s] = int2{r.x + k * most, min(r.x + (k + 1) * most, r.y)};
    }
}
// first_step of the first group of every block row (starts: its first listed column, and the end)
__global__ void row_steps_kernel(const int32_t *__restrict__ starts, const int32_t *__restrict__ first_step, long n, int32_t *__restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = first_step[starts[i] / 32];
}

// *count = how many of the K rows of B are used, row 0, which padding names, among them.  used: K bytes and zeros up to a multiple of 16.  One workgroup:
// a few loads a lane up to 10^5 rows, and nothing to clear or to add up behind it.
__global__ __launch_bounds__(1024) void count_rows_kernel(uint8_t *__restrict__ used, long K, int32_t *__restrict__ count)
{
    __shared__ int32_t part[16];
    int32_t n = 0;
    for (long i = threadIdx.x; i < (K + 15) / 16; i += 1024) {
        u32x4 v = reinterpret_cast<const u32x4 *>(used)[i];
        if (i == 0) v[0] |= 1u;
#pragma unroll
        for (int q = 0; q < 4; q++) n += __popc(v[q]); // every byte is 0 or 1
    }
    if (threadIdx.x == 0) used[0] = 1;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) n += part[w];
        *count = n;
    }
}
// place of a used row among the used ones, -1 for the others
__global__ __launch_bounds__(256) void place_rows_kernel(const uint8_t *__restrict__ used, const int32_t *__restrict__ before, long K, int32_t *__restrict__ place)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < K) place[k] = used[k] ? before[k] : -1;
}
__global__ __launch_bounds__(256) void place_cols_kernel(const int32_t *__restrict__ cols, const int32_t *__restrict__ place, long n, int32_t *__restrict__ out)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) out[i] = max(place[cols[i]], 0);
}

// raw[br] = what the blocks before block row br hold: columns in the lower, nonzeros in the upper half; raw[mb] = total
__global__ void row_offsets_kernel(const int32_t *__restrict__ row_ptr, const unsigned long long *__restrict__ offset,
                                   const unsigned long long *__restrict__ count, long mb, long nnzb, unsigned long long *__restrict__ raw)
{
    const long br = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (br > mb) return;
    const long p = row_ptr[br];
    raw[br] = p < nnzb ? offset[p] : (nnzb ? offset[nnzb - 1] + count[nnzb - 1] : 0);
}

// Blocks that another kernel multiplies (per-block split of a mixed plan): nothing of theirs is listed.
__global__ void drop_full_kernel(const uint16_t *__restrict__ mask, long nnzb, unsigned long long *__restrict__ count)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < nnzb && __popc((uint32_t)mask[p]) >= FULL_BLOCK_COLS) count[p] = 0;
}

// out[j] = block ids[j] of vals (512 bytes each; 32 lanes x 16 bytes per block).
__global__ __launch_bounds__(256) void copy_blocks_kernel(const uint16_t *__restrict__ vals, const int32_t *__restrict__ ids, long n,
                                                          uint16_t *__restrict__ out)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long j = t >> 5;
    if (j >= n) return;
    const int piece = (int)(t & 31);
    reinterpret_cast<u32x4 *>(out + j * 256)[piece] = reinterpret_cast<const u32x4 *>(vals + (long)ids[j] * 256)[piece];
}

// ---- B: column-major -> row-major ----
// Tile of COLS n x 4096 / COLS k through LDS.  A thread reads 16 bytes (8 k) of two neighbouring columns, pairs
// the values of equal k into dwords and writes them to the transposed tile; then every thread
// reads 8 n of one k back (two 8-byte LDS reads) and stores 16 bytes.  COLS = 64; 16 and 32 for a B of no more columns.
// The output is split into panels of `panel` columns, each a K x panel row-major matrix of leading
// dimension ld, the last one last_ld, one panel after the other (panel >= N and ld = N: plain row-major K x N).
// place != NULL: row k goes to row place[k] of a copy of `rows` rows, or nowhere (-1).
// STREAM: B does not stay in the caches behind the loads, which leaves them to the copy (launch_transpose).
template <int COLS, bool STREAM>
__global__ __launch_bounds__(256) void transpose_b_kernel(const uint16_t *__restrict__ B, uint16_t *__restrict__ Bt,
                                                          int N, long K, int panel, long ld, long last_ld, long rows, const int32_t *__restrict__ place)
{
    constexpr int KT = 4096 / COLS; // k of a tile
    constexpr int LD = COLS + 4; // halfs per LDS row (k): 8-byte aligned rows, dword writes spread over the banks
    __shared__ __align__(16) uint16_t tile[KT * LD];
    const int t = threadIdx.x;
    const long k0 = (long)blockIdx.x * KT;
    const int n0 = blockIdx.y * COLS;
    const int a = t / (KT / 8), seg = t % (KT / 8);
    u32x4 v0 = {0u, 0u, 0u, 0u}, v1 = {0u, 0u, 0u, 0u}; // columns 2a, 2a+1; k = 8seg .. 8seg+7
    if (k0 + seg * 8 < K) {
        const u32x4 *p0 = reinterpret_cast<const u32x4 *>(B + (long)(n0 + 2 * a) * K + k0 + seg * 8);
        const u32x4 *p1 = reinterpret_cast<const u32x4 *>(B + (long)(n0 + 2 * a + 1) * K + k0 + seg * 8);
        if (n0 + 2 * a < N) v0 = STREAM ? __builtin_nontemporal_load(p0) : *p0;
        if (n0 + 2 * a + 1 < N) v1 = STREAM ? __builtin_nontemporal_load(p1) : *p1;
    }
    const int row = t / (COLS / 8), piece = t % (COLS / 8); // stored by this thread: rows row, row + KT / 2
    long to[2]; // where they go, asked for beside the values (behind the barrier: 94 instead of 87 us for 256 MiB)
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const long k = k0 + row + KT / 2 * half;
        to[half] = k >= K ? -1 : place ? (long)place[k] : k;
    }
#pragma unroll
    for (int w = 0; w < 4; w++) {
        uint32_t *at = reinterpret_cast<uint32_t *>(tile + (seg * 8 + 2 * w) * LD + 2 * a);
        at[0] = __builtin_amdgcn_perm(v1[w], v0[w], 0x05040100u);      // k = 8seg + 2w
        at[LD / 2] = __builtin_amdgcn_perm(v1[w], v0[w], 0x07060302u); // k = 8seg + 2w + 1
    }
    __syncthreads();
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int k = row + KT / 2 * half;
        if (to[half] >= 0 && n0 + piece * 8 < N) {
            const uint2 lo = *reinterpret_cast<const uint2 *>(tile + k * LD + piece * 8);
            const uint2 hi = *reinterpret_cast<const uint2 *>(tile + k * LD + piece * 8 + 4);
            uint16_t *out = Bt + (long)(n0 / panel) * rows * panel + to[half] * (n0 / panel == (N - 1) / panel ? last_ld : ld) + n0 % panel + piece * 8;
            *reinterpret_cast<u32x4 *>(out) = (u32x4){lo.x, lo.y, hi.x, hi.y};
        }
    }
}

// A B of half of the memory-side cache and more is not there any more when the next launch reads it, so it need not displace
// the copy and the lists on its way through (R-MAT scale 20, N = 128, 256 MiB: 485 -> 472 us).  A smaller one may be
// (27-point stencil 64^3, N = 64, 33 MB, the same B again: 41.0 us, past the caches 44.3).
static hipError_t launch_transpose(const uint16_t *B, uint16_t *Bt, size_t N, size_t K, int panel, long ld, long last_ld, long rows, const int32_t *place, hipStream_t st)
{
    auto launch = [&](auto cols, auto stream) {
        constexpr int COLS = decltype(cols)::value;
        const dim3 grid((unsigned)((K + 4096 / COLS - 1) / (4096 / COLS)), (unsigned)((N + COLS - 1) / COLS));
        hipLaunchKernelGGL((transpose_b_kernel<COLS, decltype(stream)::value>), grid, dim3(256), 0, st, B, Bt, (int)N, (long)K, panel, ld, last_ld, rows, place);
    };
    using std::false_type;
    using std::integral_constant;
    if (N * K * sizeof(uint16_t) >= (size_t)128 << 20) launch(integral_constant<int, 64>{}, std::true_type{});
    else if (N <= 16) launch(integral_constant<int, 16>{}, false_type{});
    else if (N <= 32) launch(integral_constant<int, 32>{}, false_type{});
    else launch(integral_constant<int, 64>{}, false_type{});
    return hipGetLastError();
}

// ---- the product ----

// A wavefront takes a task x a panel of W = 16, 32, 64 or 128 columns.  A task is a run of items of the list, worked off as one stream of
// steps, so that the loads of the next step are under way across the end of an item.  In short launches the wavefronts of a workgroup share a task
// of one item (`shared`, compact_share).
//
// What a step of 32 columns x 64 columns of C waits for is the vector memory path: 4 KiB of rows of B and 0.15 to 1 KiB of A.
// Counted on R-MAT scale 20 (stencil 64^3), entries by blocks: its data unit is busy 91 (65) % of the time, the vector L1 waits for the L2 54
// (26) %, LDS is active 40 (39) %, and a step has 22 (36) VALU instructions, 18 (21) of LDS and 4.7 (5.3) loads.  Operands merged in
// the VALU took 130 VALU instructions a step, of which 56 exchanged and merged halves between lanes.  Hence:
//   * Rows of B go from the registers they were gathered into through 4 KiB of LDS, [entry][64 columns], and come back as
//     MFMA operands through transposing reads (ds_read_b64_tr_b16): no VALU work.  With W >= 64 lane (octet o = lane / 8, c = lane & 7)
//     gathers columns 8c .. 8c + 7 of the entries k = 8 (o / 2) + 2j + (o & 1), j = 0 .. 3; the 16-byte pieces of the rows k
//     with k & 2 are swapped in pairs, which leaves 16 of the 71 clocks that a step keeps LDS active to bank conflicts (AF = 0,
//     counted).  In lane (i = lane % 16, g = lane / 16) n-tile t of the
//     operand reads columns 16 (i & 3) + 4t .. + 3 of the rows 8g + i / 4 and + 4; the lane ends up with the 16
//     consecutive columns 16g .. of row i of the tile of C.
//   * The address of a gathered row is one multiply-add of 32 bits from its index (BIG: 64 bits, for copies of B of 4 GiB
//     and more).
//   * The A operand (AF): 0: acol, 1 KiB a step.  1, 2: entries, 4 bytes per nonzero; the at most 64 * AF of a step are put
//     to their places in 1 KiB of LDS that is zero otherwise, read back as the operand and cleared again (LDS operations
//     of a wavefront complete in order: nothing is waited for in between).
//   * Every load of a step (but a new block of indices or entries) is unconditional and nothing in the loop uses scalar loads, so that what is in flight can be
//     counted; the gathers asked for past the end of the task read row 0.
// Whole products with all of it (before: operands merged in the VALU, A in whole columns, an item per wavefront): R-MAT
// scale 20, N = 128, 703 -> 590 us; Erdos-Renyi 16384^2, 0.1 %, N = 256, 17.3 -> 16.0 us.  A third copy of the step's code
// costs more than it saves: kernels of 10 us wait for their instructions.
//
// C_ACC: the result is added to what C holds (the per-block split of a mixed plan: a dense kernel has written the
// part of the blocks it multiplies); work items that go through the workspace are not made for such plans.
//
// What the compiler has to be told (over 110 drawn random matrices 2.8 % in the mean, 4096 x 512, 64 a row, N = 1024: 19.5 -> 17.9 us):
//   * __launch_bounds__(256, 2): with one wavefront per SIMD allowed, the accumulators go to accumulation registers and W / 4 of
//     them are moved there and back every two steps.
//   * The loop ends at its bottom only.  A way out of its middle is turned into one that seems to lead from the first step
//     back to the first, where the registers of the second still seem to be waited for: every other step waited for operands
//     before it asked for the next ones.  A task that ends with the first step ends there with s_endpgm.
//
// Entries (AF > 0) come from memory in the step before they are needed, 256 bytes a load, or, STAGED, 256 at a time ahead of
// that, one load of 1 KiB to LDS: a load of 256 bytes takes the vector memory path as long as one of 1 KiB, and a list that
// comes from HBM arrives early enough.  A list that the memory-side cache still holds comes early enough either way, and
// then the trip through LDS costs a few percent where columns hold several nonzeros.  Direct / staged, us: with everything
// flushed before every launch; three matrices in turn; the same A with another B and C; the same everything:
//   stencil 64^3, N = 64           74.7/68.4   57.5/52.8   40.6/42.3   37.8/39.5
//   64^3, N = 64, row-major B                  38.1/35.7   26.5/28.2   26.8/28.0
//   64^3, N = 128                              103.5/94.3  77.5/79.5   68.9/71.7
//   R-MAT scale 18, N = 64                     72.3/67.5   57.5/57.0   57.3/56.8
//   scale 20, N = 128                          474/458     474/457     474/457
//   65536^2, 16 a row, N = 192     64.4/61.3   53.6/52.4   55.4/55.1   55.5/55.0
//   stencil 48^3, N = 128          55.9/52.4   40.1/39.9   34.6/37.1   34.7/37.1
//   8192 x 32768, 60 a row, N = 512 56.5/54.8  40.3/41.0   41.5/43.1   41.6/43.1
// The launcher's rule is at STAGED_STEPS.  A block asked for on every second step, which makes all waits exact, is slower than one
// asked for when it is needed (R-MAT scale 20 461 -> 477).
// LDS of a wavefront.  W = 64: for sixteen a CU; with more the gathers of R-MAT scale 20 lose 0.6 % and 16384^2 2 % (twelve: 16384^2 11 %).
constexpr int compact_lds_bytes(int W, bool staged) { return W == 64 ? 10240 : 1024 + 64 * W + 2048 + (staged ? 2048 : 0); }
template <int W, bool C_F32, bool C_ACC, int AF, bool STAGED, bool BIG>
__global__ __launch_bounds__(256, 2) void spmm_compact_kernel(
    const uint16_t *__restrict__ acol, const uint32_t *__restrict__ entries, const int2 *__restrict__ step_range, const int32_t *__restrict__ cols,
    const uint16_t *__restrict__ Bt, void *__restrict__ Cout, float *__restrict__ workspace, const WorkItem *__restrict__ items,
    const int4 *__restrict__ tasks, int n_tasks, int N, int n_panels, long panel_stride, long row_stride_of_most, long last_row_stride, unsigned xcd_run, int tasks_of_workgroup, int share_log2)
{
    constexpr int TQ = W > 64 ? 2 : 1, PW = W / TQ, T = PW / 16; // a row of PW columns is gathered by PW / 8 lanes, 32 rows by T instructions
    constexpr int A_BYTES = 1024, B_BYTES = 64 * W, I_BYTES = 2048;
    static_assert(compact_lds_bytes(W, STAGED) >= A_BYTES + B_BYTES + I_BYTES + (STAGED ? 2048 : 0), "the tiles of a wavefront");
    static_assert(compact_lds_bytes(W, STAGED) % 1024 == 0, "entries hold offsets that are or-ed to the address of the A tile");
    extern __shared__ __align__(1024) unsigned char lds_of_workgroup[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char *const lds = lds_of_workgroup + wave * compact_lds_bytes(W, STAGED);
    // Panel-major order of the (panel, task) space.  An XCD gets the workgroup ids that are equal modulo 8, whatever
    // their work costs; here the XCDs take runs of xcd_run consecutive workgroups of that order in turn (gridDim.x is a
    // multiple of 8 * xcd_run).  One run per XCD keeps neighbouring block rows, which share rows of B, on one L2;
    // short runs even out a list whose cost per task changes along it (R-MAT: 60 to 70 % of the steps are in the first
    // quarter of the items, and the launch took as long as the XCD that got them).
    const long total = (long)n_tasks * n_panels;
    const unsigned slot = blockIdx.x >> 3;
    const unsigned run = __builtin_amdgcn_readfirstlane(slot / xcd_run);
    const long wg = ((long)run * 8 + (blockIdx.x & 7)) * xcd_run + (slot - run * xcd_run);
    const bool shared = share_log2 > 0; // a task of one workgroup, between 2 or 4 wavefronts; else 1 or 4 tasks, one each
    const long w = wg * tasks_of_workgroup + (wave & (tasks_of_workgroup - 1));
    if (w >= total) return;
    const int panel = __builtin_amdgcn_readfirstlane((int)(w / n_tasks));
    const int task = __builtin_amdgcn_readfirstlane((int)(w - (long)panel * n_tasks));
    asm volatile("" ::"s"(items), "s"(step_range), "s"(cols), "s"(Bt)); // here with the arguments above, not one wait after the other below
    const int4 tk = tasks[task]; // first item, items (at most 64), first and last column of the stream
    int e = tk.z, e_last = tk.w;
    if (shared) { // tasks of one item: this wavefront's steps of it
        const int steps = (((e_last - e) >> 5) + (1 << share_log2) - 1) >> share_log2;
        e = min(e + wave * steps * 32, e_last);
        e_last = min(e + steps * 32, e_last);
    }
    const int begin = e;
    // Scalar loads share a counter with the LDS operations below, which would wait for them at every step: the items of
    // the task and the entry ranges of its steps come in through vector loads, one per lane, and are read from the lanes.
    // Both are asked for before one is waited for, which the shortest launches notice (16384^2, 16 a row, N = 16, row-major 4.11 -> 4.00 us, 64 6.99 -> 6.88; stencil 40 x 49 x 32,
    // N = 16, fp32 5.85 -> 5.73).
    const WorkItem mine = items[tk.x + min(lane, max(tk.y, 1) - 1)];
    const int first_step = e >> 5;
    int range_from = first_step;
    int2 ranges = {0, 0}; // AF > 0: entries of the step range_from + lane
    if constexpr (AF > 0) ranges = step_range[range_from + lane];
    int tasks_items = tk.y;
    asm volatile("" : "+s"(tasks_items)::"memory"); // the loads above stay above
    if (tasks_items == 0) return;                   // a place that order_tasks left empty
    int it = 0, item_end, br, dst;
    auto enter = [&] {
        br = __builtin_amdgcn_readlane(mine.block_row, it);
        const int own_end = __builtin_amdgcn_readlane(mine.end, it);
        item_end = shared ? e_last : own_end;
        dst = __builtin_amdgcn_readlane(mine.dst, it);
    };
    enter();

    const int i16 = lane & 15, g = lane >> 4;
    const int n0 = panel * W;
    // Row `col` of this panel of B starts at Bp + col * row_stride (B in place: panel_stride = W, row_stride = N; the
    // transposed copy: panels one after the other, row_stride = W, in the last one no more than it needs).
    const long row_stride = panel == n_panels - 1 ? last_row_stride : row_stride_of_most;
    const uint16_t *Bp = Bt + (long)panel * panel_stride;
    int boff[TQ]; // N % 8 == 0: all of the lane's columns or none (then its column 0)
#pragma unroll
    for (int q = 0; q < TQ; q++) boff[q] = n0 + 64 * q + 8 * (lane % (PW / 8)) < N ? 64 * q + 8 * (lane % (PW / 8)) : 0;

    unsigned char *const a_tile = lds, *const b_tile = lds + A_BYTES;
    const uint32_t a_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)a_tile; // a multiple of 1024
    // lane -> places first_place + j, j < T, of the step's 32 in the list, which are entries 8 (place / 8) + 2 (place % 4) + (place / 4) % 2
    const int c8 = lane % (PW / 8), first_place = T * (lane / (PW / 8));
    const int row0 = (8 * (first_place >> 3) + 2 * (first_place & 3) + ((first_place >> 2) & 1)) * (2 * PW);
    unsigned char *const put_even = b_tile + row0 + c8 * 16, *const put_odd = b_tile + row0 + (PW == 64 ? c8 ^ 1 : c8) * 16; // entry j: + j * 4 * PW
    const int swap = PW == 64 ? (i16 >> 3) & 1 : 0;
    const unsigned char *const get = b_tile + (8 * g + (i16 >> 2)) * (2 * PW) + (i16 & 3) * (PW / 2);
    const unsigned char *const get01 = get + 16 * swap, *const get23 = get - 16 * swap; // tiles 0, 1 and 2, 3: + t * 8

    f32x4 acc[TQ][T];
    auto clear_acc = [&] {
#pragma unroll
        for (int q = 0; q < TQ; q++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[q][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };
    clear_acc();

    struct Operands {
        u32x4 aw;                  // AF = 0
        uint32_t ent[AF ? AF : 1]; // AF > 0
        int n;                     // the step's entries
        u32x4 L[TQ][T];
    };
    if constexpr (AF > 0) *reinterpret_cast<u32x4 *>(a_tile + lane * 16) = (u32x4){0u, 0u, 0u, 0u};
    // The indices of 8 steps are 1 KiB, one load, and go to one half of 2 KiB of LDS, from where each lane takes the four of
    // its octet (an instruction that brings 128 bytes costs the vector memory path as much as one that brings 1 KiB).
    unsigned char *const i_tile = lds + A_BYTES + B_BYTES;
    auto load_block = [&](int s) { return reinterpret_cast<const u32x4 *>(cols + s)[lane]; };
    auto put_block = [&](int s, u32x4 x) { *reinterpret_cast<u32x4 *>(i_tile + (((s >> 5) - first_step) & 8) * 128 + lane * 16) = x; };
    typedef uint32_t Indices __attribute__((ext_vector_type(T)));
    auto indices = [&](int s) { return *reinterpret_cast<const Indices *>(i_tile + (((s >> 5) - first_step) & 15) * 128 + first_place * 4); };
    // Entries the same way: 256 of them, 1 KiB, a load, to one half of 2 KiB of LDS.  A block goes there when the first step that
    // needs it is asked for, and the one after it is loaded into the same registers then.  (Two blocks in registers, the further one moved
    // down, was every load in flight waited for at each move: the compiler's count of what is younger than a load that only some
    // steps make is zero where its registers are copied.  Waited for so -> as here: stencil 64^3, N = 64 53.3 -> 52.8 us with inputs from
    // HBM, 40.6 -> 39.5 with the same ones again; N = 128 97 -> 94; 48^3, N = 256 78 -> 74; R-MAT scale 20, N = 128 461.7 -> 458.4;
    // 65536^2, 40 a row, N = 192 101.7 -> 102.9.)
    unsigned char *const e_tile = lds + A_BYTES + B_BYTES + I_BYTES;
    u32x4 e_next = {0u, 0u, 0u, 0u};
    int e_block = 0, e_end = 0; // of 256 entries: the one in e_next, and the last of the task as far as its ranges are here
    auto load_entries = [&](int b) { return reinterpret_cast<const u32x4 *>(entries)[(long)b * 64 + lane]; };
    auto put_entries = [&](int b, u32x4 x) { *reinterpret_cast<u32x4 *>(e_tile + (b & 1) * 1024 + lane * 16) = x; };
    u32x4 e_first = {0u, 0u, 0u, 0u}, e_second = {0u, 0u, 0u, 0u};
    if constexpr (STAGED) {
        const int b = __builtin_amdgcn_readlane(ranges.x, 0) >> 8;
        const int steps = (e_last >> 5) - first_step;
        e_end = steps > 64 ? 0x7fffffff : (__builtin_amdgcn_readlane(ranges.y, steps > 0 ? steps - 1 : 0) - 1) >> 8;
        e_first = load_entries(b);
        e_second = load_entries(b + 1);
        e_block = b + 2;
        if (e_block <= e_end) e_next = load_entries(e_block);
    }
    auto request = [&](int s, const Indices x, Operands &o) {
        if constexpr (AF == 0) {
            o.aw = *reinterpret_cast<const u32x4 *>(acol + ((long)(s >> 3) + g) * 128 + i16 * 8);
        } else if constexpr (!STAGED) {
            const int first = __builtin_amdgcn_readlane(ranges.x, (s >> 5) - range_from);
            o.n = __builtin_amdgcn_readlane(ranges.y, (s >> 5) - range_from) - first;
#pragma unroll
            for (int u = 0; u < AF; u++) o.ent[u] = (entries + (long)first + 64 * u)[lane]; // past the step's end: the next step's, unused
        }
        if constexpr (BIG) {
            const long stride = s < e_last ? row_stride : 0;
#pragma unroll
            for (int q = 0; q < TQ; q++)
#pragma unroll
                for (int j = 0; j < T; j++) o.L[q][j] = *reinterpret_cast<const u32x4 *>(Bp + (long)x[j] * stride + boff[q]);
        } else {
            const uint32_t stride = s < e_last ? (uint32_t)row_stride * 2u : 0u;
#pragma unroll
            for (int q = 0; q < TQ; q++)
#pragma unroll
                for (int j = 0; j < T; j++)
                    o.L[q][j] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const unsigned char *>(Bp) +
                                                                 (size_t)(uint32_t)(__umul24(x[j], stride) + (uint32_t)boff[q] * 2u));
        }
        if constexpr (STAGED) {
            const int first = __builtin_amdgcn_readlane(ranges.x, (s >> 5) - range_from);
            o.n = __builtin_amdgcn_readlane(ranges.y, (s >> 5) - range_from) - first;
            // a step has at most 128 entries, which lie in the last block that is in LDS or reach into the one in e_next
            if ((first + o.n - 1) >> 8 >= e_block) {
                put_entries(e_block, e_next);
                e_block++;
                if (e_block <= e_end) e_next = load_entries(e_block);
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int u = 0; u < AF; u++) o.ent[u] = *reinterpret_cast<const uint32_t *>(e_tile + ((first + lane + 64 * u) & 511) * 4); // past the step's end: unused
        }
    };
    auto a_operand = [&](const Operands &o) {
        if constexpr (AF == 0) return __builtin_bit_cast(f16x8, o.aw);
        typedef __attribute__((address_space(3))) uint16_t lds_half;
        auto put = [&](bool clear) {
#pragma unroll
            for (int u = 0; u < AF; u++)
                if (64 * u + lane < o.n) *(lds_half *)(uintptr_t)((o.ent[u] & 0x3ffu) | a_base) = clear ? (uint16_t)0 : (uint16_t)(o.ent[u] >> 16);
        };
        put(false);
        asm volatile("" ::: "memory");
        const f16x8 av = *reinterpret_cast<const f16x8 *>(a_tile + lane * 16);
        asm volatile("" ::: "memory");
        put(true);
        return av;
    };
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    auto multiply = [&](const Operands &o) {
        const f16x8 av = a_operand(o);
#pragma unroll
        for (int q = 0; q < TQ; q++)
#pragma unroll
            for (int j = 0; j < T; j++) *reinterpret_cast<u32x4 *>((j & 1 ? put_odd : put_even) + q * 4096 + j * 4 * PW) = o.L[q][j];
        asm volatile("" ::: "memory");
        f16x8 b[TQ][T];
#pragma unroll
        for (int q = 0; q < TQ; q++)
#pragma unroll
            for (int t = 0; t < T; t++) {
                const unsigned char *p = (t < 2 ? get01 : get23) + q * 4096 + t * 8;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p + 8 * PW));
                b[q][t] = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < TQ; q++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[q][t], av, acc[q][t], 0, 0, 0);
    };
    // The tile of item `it` goes out (acc[q][t][r] = C[16 br + i16][n0 + 64 q + 16 g + 4 t + r]); the next item that has
    // steps is the current one afterwards.
    auto finish = [&] {
        if (shared) { // the parts of the others are added in their order by the first wavefront
            constexpr int OWN = compact_lds_bytes(W, STAGED);
            static_assert(OWN >= TQ * T * 1024, "a tile of sums");
            asm volatile("" ::: "memory");
            if (wave > 0) {
#pragma unroll
                for (int t = 0; t < TQ * T; t++) *reinterpret_cast<f32x4 *>(lds + t * 1024 + lane * 16) = acc[t / T][t % T];
            }
            __syncthreads();
            if (wave > 0) {
                it = tk.y;
                return;
            }
            // Not unrolled: the parts of several wavefronts in registers at once were 30 to 60 more of them for all launches, and panels of 16 and 32 columns ran four to six wavefronts a SIMD
            // instead of eight and seven (stencil 59 x 32 x 62, N = 8, row-major 9.42 -> 8.05 us, N = 32 11.9 -> 10.8, 64^3, N = 16 21.4 -> 19.8).
#pragma unroll 1
            for (int v = 1; v < 1 << share_log2; v++)
#pragma unroll
                for (int t = 0; t < TQ * T; t++) acc[t / T][t % T] += *reinterpret_cast<const f32x4 *>(lds_of_workgroup + v * OWN + t * 1024 + lane * 16);
        }
        do {
            const long m = (long)br * 16 + i16;
#pragma unroll
            for (int q = 0; q < TQ; q++) {
                const int c0 = n0 + 64 * q + PW / 4 * g;
                if (dst >= 0 || C_F32) {
                    float *row = dst >= 0 ? workspace + ((long)dst * 16 + i16) * (long)N
                                          : reinterpret_cast<float *>(Cout) + m * (long)N;
#pragma unroll
                    for (int t = 0; t < T; t++)
                        if (c0 + 4 * t < N) {
                            f32x4 v = acc[q][t];
                            if (C_ACC && dst < 0) v += *reinterpret_cast<const f32x4 *>(row + c0 + 4 * t);
                            *reinterpret_cast<f32x4 *>(row + c0 + 4 * t) = v;
                        }
                } else {
                    uint16_t *row = reinterpret_cast<uint16_t *>(Cout) + m * (long)N;
                    if constexpr (T == 1) {
                        static_assert(!C_ACC, "narrow panels are not accumulated");
                        if (c0 < N) *reinterpret_cast<f16x4 *>(row + c0) = __builtin_convertvector(acc[q][0], f16x4);
                    } else {
#pragma unroll
                        for (int h = 0; h < T / 2; h++) {
                            if (c0 + 8 * h >= N) continue;
                            f16x8 v;
                            if (C_ACC) {
                                const f16x8 old = *reinterpret_cast<const f16x8 *>(row + c0 + 8 * h);
#pragma unroll
                                for (int j = 0; j < 8; j++) v[j] = (_Float16)(acc[q][2 * h + j / 4][j % 4] + (float)old[j]);
                            } else {
#pragma unroll
                                for (int j = 0; j < 8; j++) v[j] = (_Float16)acc[q][2 * h + j / 4][j % 4];
                            }
                            *reinterpret_cast<f16x8 *>(row + c0 + 8 * h) = v;
                        }
                    }
                }
            }
            clear_acc();
            if (++it < tk.y) enter();
        } while (it < tk.y && item_end == e);
    };
    if (item_end == e) finish(); // block rows without a step: zeros
    if (it >= tk.y) return;

    Operands op_a, op_b;
    u32x4 block = load_block(e); // of the 8 steps after those in LDS
    put_block(e, block);
    block = load_block(e + 256);
    if constexpr (STAGED) {
        put_entries(e_block, e_first); // blocks e_block - 2
        put_entries(e_block + 1, e_second); // and e_block - 1
    }
    asm volatile("" ::: "memory");
    request(e, indices(e), op_a);
    int next = e + 32; // the step whose operands are asked for
    Indices x = indices(next); // read from LDS a step before they are used
    // Before the first step that `ranges` does not reach (every 64 steps): the ranges of 64 steps from there on.  The wait for
    // them is inside, so that no other step has one; a task of up to 62 steps never gets here.
    auto more_ranges = [&] {
        if (AF > 0 && (next >> 5) - range_from >= 60) {
            range_from = next >> 5;
            ranges = step_range[range_from + lane];
            asm volatile("" : "+v"(ranges.x), "+v"(ranges.y));
        }
    };
    // the bottom of the loop for a task that ends with the first of its two steps
    auto end_if_done = [&] { asm volatile("s_cmp_lt_i32 %0, %1\n\ts_cbranch_scc1 1f\n\ts_endpgm\n1:" ::"s"(it), "s"(tk.y) : "scc", "memory"); };
    do {
#define SMAT_STEP_OF(CUR, NEW, DONE)                                                                        \
        if (((next + 32 - begin) & 255) == 0) {                                                         \
            put_block(next + 32, block);                                                               \
            block = load_block(next + 288);                                                            \
            more_ranges();                                                                             \
        }                                                                                              \
        asm volatile("" ::: "memory");                                                                 \
        request(next, x, NEW);                                                                         \
        x = indices(next + 32);                                                                        \
        multiply(CUR);                                                                                 \
        e = next;                                                                                      \
        next += 32;                                                                                    \
        if (e == item_end) {                                                                           \
            finish();                                                                                  \
            DONE;                                                                                      \
        }
        SMAT_STEP_OF(op_a, op_b, end_if_done())
        SMAT_STEP_OF(op_b, op_a, )
#undef SMAT_STEP_OF
    } while (it < tk.y);
}

// Wavefronts that share a task.  A launch of less than a wavefront a SIMD takes as long as one of them goes from step to step, 0.3 us each; with the steps of a task between
// two or four of a workgroup, whose sums meet in LDS (1 us), it is shorter as long as there is room for them, and longer (up to 10 %) where a task has few steps or the
// wavefronts are enough.  Alone / two / four, us, the copy of B among them: 3584 x 4112, 8 % of full blocks and 10 more a row, N = 96 (448 tasks and panels of 15 steps) 10.5 / 8.7 / 8.6,
// 4416 x 8160, 8 % and 3, N = 72 (552 of 22) 13.4 / 11.0 / 11.4, 2832 x 2144, 32 a row, N = 48 (177 of 14) 5.65 / 4.37 / 4.07, 6992 x 7616, 7 % and 4, N = 80 (874 of 18) 12.7 / 11.4 / 12.0;
// 5776 x 6752, 5 % and 3, N = 192 (1083 of 12) 12.2 / 12.2 / 12.5, 4288 x 1088, 8 a row, N = 48 (268 of 4) 3.88 / 4.06 / 4.11.
int compact_share(bool by_name, int64_t n_steps, int64_t n_tasks, long total)
{
    if (by_name || total > 900 || n_steps < 6 * n_tasks) return 1;
    return total > 400 || n_steps < 12 * n_tasks ? 2 : 4;
}

// Halves from row to row of the copy's last panel: 8, 16, 32, .. as many as hold the columns that are left, so that what is gathered at random lies on as few lines as may be.
// A panel of 8 columns on rows of 128 bytes fills eight times the lines of the L2s.  Rows of the panel's width -> these, us: R-MAT scale 17, 10 a row, N = 72 42.3 -> 39.9; 18, 13, N = 136
// 140.6 -> 133.5; 19, 14, N = 200 425 -> 396; 19, 12, N = 8 51.6 -> 44.0; where the columns fill the panel equal.
long last_panel_width(size_t N, int panel)
{
    long width = 8;
    while (width < (long)((N - 1) % (size_t)panel) + 1) width *= 2;
    return width;
}

template <int W>
hipError_t launch_compact_as(const CompactArgs &a, hipStream_t st)
{
    const CompactPlan &p = *a.plan;
    constexpr int PANEL = W;
    const int n_panels = (int)((a.N + PANEL - 1) / PANEL);
    long panel_stride = PANEL, row_stride = (long)a.N, last_row_stride = row_stride;
    const int32_t *cols = p.d_cols;
    if (!a.b_row_major) {
        const long rows = p.d_place ? (long)p.n_placed : (long)a.K; // of the copy
        if (p.d_place) cols = p.d_cols_placed;
        last_row_stride = last_panel_width(a.N, PANEL);
        const hipError_t e = launch_transpose(a.B, a.Bt, a.N, a.K, PANEL, PANEL, last_row_stride, rows, p.d_place, st);
        if (e != hipSuccess) return e;
        panel_stride = rows * PANEL;
        row_stride = PANEL;
    }
    const long total = (long)p.n_tasks * n_panels;
    long wgs = (total + 3) / 4;
    if (wgs == 0) return hipSuccess;
    long xcd_run = p.deal.run((size_t)p.n_tasks, n_panels);
    if (p.tuned_run > 0 && p.tuned_n == a.N) xcd_run = p.tuned_run;
    if (p.ordered) xcd_run = 1;
    if (a.xcd_run > 0) xcd_run = a.xcd_run;
    if (g_force_run > 0) xcd_run = g_force_run;
    xcd_run = std::min<long>((wgs + 7) / 8, xcd_run);
    g_last_run.store((int)xcd_run, std::memory_order_relaxed);
    // A workgroup of four tasks keeps its place until the longest is done; one task each is up to 12 % faster (4864 x 6496, 12 % of full blocks and 15 more a row, N =
    // 400 30.5 -> 26.6 us, 40000 x 60000, 10 a row, N = 64, row-major 9.7 -> 9.3, R-MAT scale 18, N = 64 63.9 -> 62.7).  Where a place has many steps to do the end of a launch
    // matters less than the lines that neighbouring tasks find of each other's in their L1: four (R-MAT scale 20, N = 128, row-major 366, one each 378; 19, N = 256 362 and 365, 40000 x 60000, 30 a row, N = 256 73.8 and 74.6).
    const int share = !p.may_share ? 1 : g_force_share ? g_force_share : compact_share(p.by_name, p.n_steps, p.n_tasks, total);
    g_last_share.store(share, std::memory_order_relaxed);
    const int waves = share > 1 ? share : (double)p.n_steps * n_panels >= 32.0 * 16.0 * 256.0 ? 4 : 1;
    xcd_run *= share > 1 ? 4 : 4 / waves;
    wgs = share > 1 ? total : (total + waves - 1) / waves;
    wgs = (wgs + 8 * xcd_run - 1) / (8 * xcd_run) * (8 * xcd_run);
    if (wgs > 0x7fffffffL) return hipErrorInvalidValue;
    if (a.accumulate && p.n_split_rows > 0) return hipErrorInvalidValue; // partial tiles through the workspace overwrite C
    // 32-bit byte offsets from indices of 24 bits
    const bool big = a.K > ((size_t)1 << 24) || a.K * (size_t)row_stride * 2 >= ((size_t)1 << 32) || row_stride >= (1L << 23);
    auto launch = [&](auto af, auto staged, auto f32, auto acc, auto wide) {
        hipLaunchKernelGGL((spmm_compact_kernel<W, decltype(f32)::value, decltype(acc)::value, decltype(af)::value, decltype(staged)::value, decltype(wide)::value>),
                           dim3((unsigned)wgs), dim3(64 * waves), (size_t)(waves * compact_lds_bytes(W, decltype(staged)::value)), st, p.d_acol, p.d_entries, p.d_step_range, cols, a.Bt, a.C, p.d_workspace,
                           p.d_items, p.d_tasks, p.n_tasks, (int)a.N, n_panels, panel_stride, row_stride, last_row_stride, (unsigned)xcd_run, share > 1 ? 1 : waves, share == 4 ? 2 : share - 1);
    };
    using std::false_type;
    using std::true_type;
    auto by_output = [&](auto af, auto staged, auto wide) {
        if constexpr (W >= 64) if (a.accumulate) { // never staged
            if (a.c_f32) launch(af, false_type{}, true_type{}, true_type{}, wide); else launch(af, false_type{}, false_type{}, true_type{}, wide);
            return;
        }
        {
            if (a.c_f32) launch(af, staged, true_type{}, false_type{}, wide); else launch(af, staged, false_type{}, false_type{}, wide);
        }
    };
    const int64_t list_bytes = p.n_steps * 128 + p.n_entries * 4, b_bytes = (int64_t)a.K * a.N * 2, c_bytes = (int64_t)a.M * a.N * (a.c_f32 ? 4 : 2);
    const bool staged = g_force_staged ? g_force_staged == 1
                                       : (double)p.n_steps * n_panels >= STAGED_STEPS * 16.0 * 256.0 && list_bytes >= STAGED_BYTES &&
                                             list_bytes + c_bytes + (a.b_row_major ? b_bytes : 2 * b_bytes) >= (a.b_row_major ? STAGED_TOUCHED_IN_PLACE : STAGED_TOUCHED);
    auto by_entries = [&](auto wide) {
        if (p.d_acol) by_output(std::integral_constant<int, 0>{}, false_type{}, wide);
        else if (p.entries_ahead == 1) staged ? by_output(std::integral_constant<int, 1>{}, true_type{}, wide) : by_output(std::integral_constant<int, 1>{}, false_type{}, wide);
        else staged ? by_output(std::integral_constant<int, 2>{}, true_type{}, wide) : by_output(std::integral_constant<int, 2>{}, false_type{}, wide);
    };
    if (big) by_entries(true_type{}); else by_entries(false_type{});
    return hipGetLastError();
}

using Scratch = DevScratch;

} // namespace

// Row-major B (B[k*N + n]) -> column-major out[n*K + k]: the same tile transposition with the roles of the
// two dimensions swapped (N % 8 == 0 and K % 16 == 0 keep every 16-byte access aligned).
hipError_t launch_b_to_col_major(const uint16_t *B_row_major, uint16_t *out, size_t N, size_t K, hipStream_t st)
{
    return launch_transpose(B_row_major, out, K, N, 0x7fffffff, (long)K, (long)K, (long)N, nullptr, st);
}

// The columns of a panel of a launch.  A product of up to 16 or 32 columns takes panels of that many: a row of B is then 32 or 64 bytes, a step
// gathers its 32 rows in one or two instructions instead of four, and brings as many lines less (same order of sums, same bits).  Panels of
// 64 columns -> 16 or 32, us: R-MAT scale 18, 22 a row, N = 8 61 -> 45, N = 16 in fp32 68 -> 47, N = 32 72 -> 61; 27-point stencil 64^3, N = 16 37.4 -> 19.8, N = 32
// 43.4 -> 30.0; 61648 x 25136, 13 a row, N = 16 13.6 -> 10.9; 16384^2, 16 a row, N = 32, row-major B 6.1 -> 5.8.
static int compact_panel_width(const CompactPlan &p, size_t N, size_t K, bool accumulate)
{
    const long items = p.n_items;
    if (g_force_tq == 0 && N <= 32 && !accumulate) return N <= 16 ? 16 : 32;
    int tq = 1;
    if (N >= 128 && items * (long)(N / 128) >= 2048 && p.n_cols >= (int64_t)items * 384) tq = 2;
    if (g_force_tq == 1 || g_force_tq == 2) tq = g_force_tq;
    while (tq > 1 && K * (size_t)(64 * tq) * sizeof(uint16_t) > ((size_t)128 << 20)) tq >>= 1;
    return 64 * tq;
}

hipError_t launch_compact(const CompactArgs &a_in, hipStream_t st)
{
    CompactArgs a = a_in;
    hipError_t e = hipSuccess;
    if (a.b_row_major) a.Bt = const_cast<uint16_t *>(a.B); // read in place, never written
    // Panels of 128 columns read the A operand and the indices half as often as panels of 64; those of 64 give twice
    // the wavefronts.  Measured (N = 256 .. 4096): 128 wins where the items are long (dense blocks, 25 steps per
    // block row: 218 against 244 us), 64 where they are short (one nonzero per block, 4 to 8 steps: 21.7 against
    // 22.5 us, 94 against 97 us); panels of 256 columns never won.  The panels are swept one after the other, so the
    // rows of B that the gathers hit at random come from one panel at a time: a panel is kept under half of the
    // 256 MiB memory-side cache (the lists of A and the rows of C stream through it too).  On a 2^20-row B at
    // N = 128 the panel of 64 columns (128 MiB) takes 0.74 x the time of the panel of 128.
    switch (compact_panel_width(*a.plan, a.N, a.K, a.accumulate)) {
    case 128: e = launch_compact_as<128>(a, st); break;
    case 32: e = launch_compact_as<32>(a, st); break;
    case 16: e = launch_compact_as<16>(a, st); break;
    default: e = launch_compact_as<64>(a, st);
    }
    if (e != hipSuccess) return e;
    if (a.plan->n_split_rows > 0)
        e = launch_reduce(a.plan->d_workspace, a.plan->d_split, a.plan->n_split_rows, a.C, a.N, a.c_f32, st);
    return e;
}

hipError_t compact_tune(CompactPlan &p, uint16_t *Bt, size_t M, size_t N, size_t K, bool b_row_major, bool accumulate)
{
    p.tuned_n = 0;
    p.tuned_run = 0;
    if (!g_tune || p.n_items == 0 || N == 0 || !Bt || p.ordered) return hipSuccess;
    // Timed as a program launches it, the transposition of a column-major B included: the copy is written over what the
    // launch before left in the L2s, and how many of them hold a line of it follows from the deal (16384^2, 0.1 %, N = 256: the
    // product kernel alone is fastest in runs of 128, 10.9 against 11.9 us; launch after launch it is 64, 19.8 against 21.4.
    // 8192 x 16384, 24 a row, N = 512: 24.2 against 27.1 in runs of 32 and 128).
    const int width = compact_panel_width(p, N, K, accumulate);
    const int n_panels = (int)((N + width - 1) / width);
    const long wgs = ((long)p.n_tasks * n_panels + 3) / 4;
    const unsigned eighth = (unsigned)std::max<long>((wgs + 7) / 8, 1);
    // the run length of an untuned launch, as launch_compact_as computes it for this N
    const unsigned base = std::min(eighth, p.deal.run((size_t)p.n_tasks, n_panels));
    constexpr int MAX_RUNS = 4;
    unsigned runs[MAX_RUNS] = {base};
    int n = 1;
    if (base * 4 >= eighth) // a list that the estimate finds even: the longer runs are worth a try
        for (unsigned r : {eighth, eighth / 2, eighth / 4})
            if (r >= 4 && std::find(runs, runs + n, r) == runs + n) runs[n++] = r;
    // R-MAT scale 20 has 10^6 steps and takes 0.5 ms: a launch of over 20 ms is not worth trying several times
    if (n == 1 || p.n_steps * n_panels > 40000000) return hipSuccess;
    Scratch B, C;
    if (B.alloc(K * N * sizeof(uint16_t)) != hipSuccess || C.alloc(M * N * sizeof(uint16_t)) != hipSuccess) {
        (void)hipGetLastError(); // no room for the trial: not an error of the plan
        return hipSuccess;
    }
    hipError_t e = hipMemset(B.p, 0, K * N * sizeof(uint16_t));
    if (e == hipSuccess) e = hipMemset(C.p, 0, M * N * sizeof(uint16_t));
    hipEvent_t mark[MAX_RUNS + 1] = {};
    for (int i = 0; i <= MAX_RUNS && e == hipSuccess; i++) e = hipEventCreate(&mark[i]);
    CompactArgs a{};
    a.B = static_cast<const uint16_t *>(B.p); a.b_row_major = b_row_major; a.Bt = Bt; a.C = C.p;
    a.M = M; a.N = N; a.K = K; a.c_f32 = false; a.plan = &p; a.accumulate = accumulate;
    // one after the other without a gap between them, three launches each, the first after one more (the choice is the same twelve times out of
    // twelve on these matrices)
    constexpr int LAUNCHES = 3;
    a.xcd_run = runs[0];
    if (e == hipSuccess) e = launch_compact(a, nullptr);
    if (e == hipSuccess) e = hipEventRecord(mark[0], nullptr);
    for (int k = 0; k < n; k++) {
        a.xcd_run = runs[k];
        for (int i = 0; i < LAUNCHES && e == hipSuccess; i++) e = launch_compact(a, nullptr);
        if (e == hipSuccess) e = hipEventRecord(mark[k + 1], nullptr);
    }
    if (e == hipSuccess) e = hipEventSynchronize(mark[n]);
    float ms[MAX_RUNS] = {};
    for (int k = 0; k < n && e == hipSuccess; k++) e = hipEventElapsedTime(&ms[k], mark[k], mark[k + 1]);
    if (e == hipSuccess) {
        p.tuned_n = N;
        p.tuned_run = base;
        float best = ms[0] * 0.97f; // another run length has to be 3 % faster than the estimate's choice
        for (int k = 1; k < n; k++)
            if (ms[k] < best) best = ms[k], p.tuned_run = runs[k];
    }
    for (hipEvent_t m : mark)
        if (m) (void)hipEventDestroy(m);
    return e;
}

// Of 36 such launches of two panels and more (stencils, N = 72 to 256, column- and row-major B) in one run an XCD 4.3 % slower in the mean than the best of the
// runs that are tried, 21 % at most (45 x 15 x 54, N = 72, row-major 11.3 against 9.4 us); in halves 0.9 and 10, in quarters 2.6 and 12.  One panel, 66
// launches: 0.7, 1.8, 3.6 %.  Where the panels are a multiple of four, a quarter of an eighth is whole panels again: 41 stencils, N = 200 to 256 and
// 456 to 512, against the runs that were timed, halves 1 % slower column-major and 2.4 row-major, 25 at most (56 x 14 x 25, N = 240, row-major
// 10.9 us, 12.9 in halves), quarters 0 and 2.5 % faster, 9 slower at most; of five to seven panels quarters are 1 to 3 % slower than halves.  (Beside columns in LDS, uniform random matrices: 1.3, 2.0 and 4.9 %, left as they are.)
void compact_deal_beside_windows(CompactPlan &p, size_t N, size_t K)
{
    const int width = compact_panel_width(p, N, K, false), n_panels = (int)((N + width - 1) / width);
    const unsigned eighth = (unsigned)((((long)p.n_tasks * n_panels + 3) / 4 + 7) / 8);
    if (p.ordered || n_panels < 2 || eighth < 8 || p.deal.run((size_t)p.n_tasks, n_panels) < eighth) return;
    p.tuned_n = N;
    p.tuned_run = eighth / (n_panels % 4 ? 2 : 4);
}

hipError_t values_checksum(const uint16_t *vals, size_t nnzb, uint64_t *out)
{
    *out = 0;
    if (!nnzb) return hipSuccess;
    DevScratch d;
    hipError_t e = d.alloc(SUM_BYTES);
    if (e == hipSuccess) e = hipMemsetAsync(d.p, 0, SUM_BYTES, nullptr);
    if (e != hipSuccess) return e;
    const long n_quads = (long)nnzb * 32;
    const unsigned blocks = (unsigned)std::min<long>((n_quads + 255) / 256, 256L * 8);
    hipLaunchKernelGGL(values_checksum_kernel, dim3(blocks), dim3(256), 0, 0, reinterpret_cast<const u32x4 *>(vals), n_quads, (unsigned long long *)d.p);
    e = hipGetLastError();
    unsigned long long sum = 0, all[SUM_BYTES / 8] = {0};
    if (e == hipSuccess) e = hipMemcpy(all, d.p, SUM_BYTES, hipMemcpyDeviceToHost);
    add_up_totals(all, &sum, 1);
    if (e == hipSuccess) *out = sum;
    return e;
}

void compact_destroy(CompactPlan *p)
{
    if (!p) return;
    if (p->d_cols) (void)dev_free(p->d_cols);
    if (p->d_place) (void)dev_free(p->d_place);
    if (p->d_cols_placed) (void)dev_free(p->d_cols_placed);
    if (p->d_acol) (void)dev_free(p->d_acol);
    if (p->d_entries) (void)dev_free(p->d_entries);
    if (p->d_step_range) (void)dev_free(p->d_step_range);
    if (p->d_items) (void)dev_free(p->d_items);
    if (p->d_split) (void)dev_free(p->d_split);
    if (p->d_workspace) (void)dev_free(p->d_workspace);
    delete p;
}

hipError_t copy_blocks(const uint16_t *vals, const int32_t *ids_host, size_t n, uint16_t *out)
{
    if (!n) return hipSuccess;
    Scratch ids;
    hipError_t e = ids.alloc(n * sizeof(int32_t));
    if (e == hipSuccess) e = hipMemcpy(ids.p, ids_host, n * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(copy_blocks_kernel, dim3((unsigned)((n * 32 + 255) / 256)), dim3(256), 0, 0, vals, (const int32_t *)ids.p, (long)n, out);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize(); // ids goes out of scope
    return e;
}

#define SMAT_STEP(call)                                                                            \
    do {                                                                                           \
        if (e == hipSuccess) e = (call);                                                           \
    } while (0)

// count -> offset (exclusive sums), rows (what the blocks before every block row hold) and raw, its copy on the host
// more: bytes behind the rows' sums that come along to `to`.
static hipError_t census_offsets(CompactCensus &s, const int32_t *row_ptr, size_t more = 0, unsigned long long *to = nullptr)
{
    hipError_t e = hipSuccess;
    Scratch tmp;
    size_t bytes = 0;
    auto *count = static_cast<unsigned long long *>(s.count.p), *offset = static_cast<unsigned long long *>(s.offset.p);
    SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, count, offset, (int)s.nnzb));
    SMAT_STEP(tmp.alloc(bytes));
    SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, count, offset, (int)s.nnzb));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(row_offsets_kernel, dim3((unsigned)((s.mb + 1 + 255) / 256)), dim3(256), 0, 0, row_ptr, offset, count, (long)s.mb,
                           (long)s.nnzb, (unsigned long long *)s.rows.p);
        e = hipGetLastError();
    }
    s.raw.resize(s.mb + 1 + more / 8);
    SMAT_STEP(hipMemcpy(s.raw.data(), s.rows.p, (s.mb + 1) * 8 + more, hipMemcpyDeviceToHost));
    std::copy(s.raw.begin() + (long)s.mb + 1, s.raw.end(), to);
    s.raw.resize(s.mb + 1);
    tmp.idle = e == hipSuccess;
    return e;
}

hipError_t compact_census(const uint16_t *vals, const int32_t *row_ptr, size_t mb, size_t nnzb, CompactCensus &s, const int32_t *col_idx, size_t kb, WindowCount *widths)
{
    hipError_t e = hipSuccess;
    s.mb = mb;
    s.nnzb = nnzb;
    s.raw.assign(mb + 1, 0);
    if (!nnzb) return e;
    for (Scratch *q : {&s.mask, &s.single, &s.count, &s.offset, &s.rows}) q->release();
    s.dropped = false;
    SMAT_STEP(s.mask.alloc(nnzb * 2));
    SMAT_STEP(s.single.alloc(nnzb * 4));
    SMAT_STEP(s.count.alloc(nnzb * 8));
    SMAT_STEP(s.offset.alloc(nnzb * 8));
    SMAT_STEP(s.rows.alloc((mb + 1) * 8 + SUM_BYTES + WindowCount::BYTES)); // the totals behind the rows' sums: one copy to the host, 13 us a copy
    unsigned long long *const sums = static_cast<unsigned long long *>(s.rows.p) + mb + 1;
    SMAT_STEP(hipMemsetAsync(sums, 0, SUM_BYTES, nullptr));
    if (e == hipSuccess && widths && !widths->launch(row_ptr, col_idx, mb, kb, nnzb, sums + SUM_BYTES / 8)) widths = nullptr;
    if (e == hipSuccess) {
        const long waves = std::min<long>((long)(nnzb + 1) / 2, 256L * 32);
        hipLaunchKernelGGL(colmask_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, 0, vals, (long)nnzb,
                           (uint16_t *)s.mask.p, (uint32_t *)s.single.p, (unsigned long long *)s.count.p, sums);
        e = hipGetLastError();
    }
    std::vector<unsigned long long> all((SUM_BYTES + (widths ? WindowCount::BYTES : 0)) / 8);
    SMAT_STEP(census_offsets(s, row_ptr, all.size() * 8, all.data()));
    if (e != hipSuccess) return e;
    unsigned long long total[N_SUMS];
    add_up_totals(all.data(), total, N_SUMS);
    if (widths) widths->take(all.data() + SUM_BYTES / 8);
    s.values_checksum = total[SUM_CHECK];
    s.full_blocks = (int64_t)total[SUM_FULL];
    s.cols_rest = (int64_t)total[SUM_COLS_REST];
    s.nnz = (int64_t)total[SUM_NNZ];
    s.n_cols_all = (int64_t)(uint32_t)s.raw[mb];
    return e;
}

hipError_t compact_full_blocks(const CompactCensus &s, std::vector<uint8_t> &full)
{
    std::vector<uint16_t> mask(s.nnzb);
    full.assign(s.nnzb, 0);
    if (!s.nnzb) return hipSuccess;
    const hipError_t e = hipMemcpy(mask.data(), s.mask.p, s.nnzb * 2, hipMemcpyDeviceToHost);
    for (size_t i = 0; i < s.nnzb; i++) full[i] = __builtin_popcount(mask[i]) >= FULL_BLOCK_COLS;
    return e;
}

// Whether the nonzeros are listed one by one (4 bytes each, and 8 per step) instead of whole columns (32 bytes each): a step of
// random sparse columns, one nonzero each, is then 152 bytes of A instead of 1024, of the 4 to 5 KiB that the vector L1
// returns for it, but its operand takes two trips through LDS.  Over 260 drawn matrices (random, R-MAT, 27-point stencils; rows
// 1,024 to 262,144, N 8 to 1,024, either layout of B, three products on their own inputs in turn) this rule is 0.8 % from the
// better of the two in the mean, always listing nonzeros 3.3 %, a rule by K alone (>= 4096) 3.2 %:
//   * the trips through LDS are what a wavefront waits for where there are fewer than five on a CU (whole columns / nonzeros, us:
//     8192 x 4096, 40 a row, N = 128 10.4 / 11.6; R-MAT scale 12, N = 64 11.5 / 13.5);
//   * with more, the nonzeros win while they are few per column (65536 x 512, 8 a row, N = 512 43.4 / 38.9; 59328 x 27344, 17.5 a
//     row, N = 288 76 / 55; at 2.3 per column 4096 x 512, 64 a row, N = 1024 they lose, 15.2 / 17.0);
//   * whole columns with more nonzeros pay while their list takes no more than half of the eight L2s of 4 MiB (27-point stencil,
//     2.8 per column: 32^3, 300 k columns, N = 256 22.5 / 23.9; 48^3, 1.05 M, 70.8 / 62.8; 64^3, 2.5 M, N = 64 47.8 / 42.5).
static bool lists_nonzeros(int64_t nnz, int64_t n_cols, size_t n_rows, size_t N)
{
    if (n_rows * ((N + 63) / 64) < 5 * 256) return false;
    return 2 * nnz <= 3 * n_cols || (n_cols >= 500000 && nnz <= 4 * n_cols);
}

struct ByteToInt {
    __host__ __device__ int32_t operator()(uint8_t v) const { return v; }
};
// The copy of B without the rows that no listed column names, where those are an eighth or more.  R-MAT scale 20, 16 a row: 48 % of
// the columns are empty, and the rows of B under the others fill 67 of 128 MiB a panel, which the memory-side cache holds for
// the gathers: N = 128 transposition 101 -> 94 us, product 469 -> 401; scale 18, N = 256 226 -> 211, both together; scale 16 equal.
// With the rows that most columns meet in front the gathers take as long.  The list is marked and counted on the way (gather_kernel,
// count_rows_kernel), and the number comes to the host where it waits anyway, since most matrices use all rows of B: with a pass over
// the list, a scan and a copy of their own attaching took 35 to 50 us longer for nothing (stencil 64^3 942 us, so 916; 54336^2, 16 a row, N = 256
// 1053 and 1032; 16384^2, N = 512 631 and 604).
static hipError_t place_rows(CompactPlan &p, const uint8_t *used, int32_t n_used, size_t K, long total)
{
    hipError_t e = hipSuccess;
    Scratch before, tmp;
    size_t bytes = 0;
    const long padded = total + LIST_PAD;
    const hipcub::TransformInputIterator<int32_t, ByteToInt, const uint8_t *> flags(used, ByteToInt{});
    SMAT_STEP(before.alloc(K * sizeof(int32_t)));
    SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, flags, (int32_t *)before.p, (int)K));
    SMAT_STEP(tmp.alloc(bytes));
    SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, flags, (int32_t *)before.p, (int)K));
    SMAT_STEP(dev_malloc(&p.d_place, K * sizeof(int32_t)));
    SMAT_STEP(dev_malloc(&p.d_cols_placed, (size_t)padded * sizeof(int32_t)));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(place_rows_kernel, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, 0, used, (const int32_t *)before.p, (long)K, p.d_place);
        hipLaunchKernelGGL(place_cols_kernel, dim3((unsigned)std::min<long>((padded + 255) / 256, 256L * 8)), dim3(256), 0, 0, (const int32_t *)p.d_cols,
                           (const int32_t *)p.d_place, padded, p.d_cols_placed);
        e = hipGetLastError();
    }
    p.n_placed = n_used;
    return e;
}

// Steps of the chunks that long block rows are cut into, for a list of `steps` steps in `rows` block rows, the longest of `longest`
// steps, and products of n_cap columns.
//
// What a wavefront's place on the device does in a launch (steps and panels over 16 places a CU) bounds the time that one chunk may
// take, and the partial tiles ask for long ones.  Chunks are the first items of a panel, so one that takes as long as its panel
// ends with it, and where several panels follow each other it may take longer.  Steps of a chunk, us (R-MAT, 16 a row, avg 7 steps):
//   scale 20, N = 128, 240 steps a place:  14 607, 28 512, 56 486, 112 458, 224 480
//   scale 19, N = 128, 120:                14 268, 28 236, 56 221, 112 225, 224 234
//   scale 18, N = 256, 120:                14 248, 28 207, 56 196, 112 211
//   scale 18, N = 64, 30:                  14 79.0, 28 68.7, 56 65.3, 112 80.0
//   scale 17, N = 1024, 240:               14 477, 28 385, 56 359, 112 378
//   scale 16, N = 128, 15:                 14 35.5, 28 33.0, 56 42.2
//   scale 14, N = 128, 4:                  14 17.8, 28 20.5, 56 32.0
// Taken: 16 steps and those that a place has in one panel, or 0.38 of what it has in all, whichever is more; with 0.38 alone two panels take longer
// (scale 20, N = 128 461 against 457, scale 19 217 against 213), with those of one panel alone many do (scale 17, N = 1024 377 against 359).
// Whether a list is split at all, which costs a launch: where its longest row has more than four times the average, and more than 16
// steps, and more than a chunk.
static long split_chunk_steps(long steps, size_t rows, long longest, size_t n_cap)
{
    const size_t panels = (n_cap + 63) / 64;
    const double avg = rows ? (double)steps / (double)rows : 0.0, one_panel = (double)steps / (16.0 * 256.0);
    long chunk = (long)(std::max(16.0 + std::max(one_panel, 0.38 * one_panel * (double)panels), 2.5 * avg) + 0.5);
    const long from = std::max((long)(128.0 * avg + 0.5), 512L) / 32; // four times the average, rounded to a column
    if (longest <= from) chunk = std::max(chunk, from);
    if (rows * panels < 1024) chunk = std::min(chunk, (long)LONG_ROW_STEPS);
    return chunk;
}

// The order of the tasks of a list with split rows, which is skewed, and the XCD of each: workgroup i, tasks 4 i .. 4 i + 3, runs on XCD i % 8.
//
// Bound by the lines that the L2s miss: 128-byte rows at random out of 67 MiB come at 7.2 TB/s however many wavefronts ask (220 lines per us and CU, with
// 2 MiB 750), and in the order of the block rows a product of R-MAT scale 20 moved 6.6 TB/s.  Long rows list their columns in ascending order, so
//   * a chunk of a split row goes to the XCD of the eighth of its row that it begins in: an XCD gathers from an eighth of B for the chunks of all rows, and those
//     that run at the same time from about the same part of it;
//   * whole rows come by classes of length, the longest first: what runs at the same time advances through B at about the same pace.  256 tasks of a class,
//     or what is a 256th of the launch, go to the XCD that has least to do so far, which makes the XCDs even where runs of the deal left up to 4 %.  Inside
//     a class rows keep their order.
// Counted on R-MAT scale 20, N = 128: 58.5 % of the requests to the L2s found, 53.0 in the order before, and 1.85 GB fetched from beyond them, 2.17.  (A model of the gathers alone finds 67 and 55 %, 61
// with exact lengths in runs of 16 tasks, 73 with rows from 1000 columns on cut in eighths too, whose partial tiles would be ten times as many.)  In the order of the block rows -> so, us: R-MAT scale 20, 16 a row, N = 128 456 -> 428, row-major 449 -> 377, N =
// 64 228 -> 190; 18, 22 a row, N = 64, row-major 63 -> 55; 18, 16, N = 128 111 -> 107; 15, 16, N = 256 33.6 -> 31.3; 15, N = 24, 14, 13 and 12 within 1 %.
// Classes are octaves; two of them where a column-major B has more than two panels (18, 10 a row, N = 256 159.1, with octaves 161.9, with two 157.9; 19, 22 a row, N = 200 513, 513,
// 517; with two panels or fewer two octaves are 1 to 5 % slower).
// Not where a row-major B has more than two panels and an eighth to a half of the memory-side cache's 256 MiB; in the order of the block rows -> ordered, us: 17, 16 a row, N = 184 96.0 -> 99.9, N =
// 256 98.4 -> 103.3; 17, 20, N = 160 79.3 -> 81.3; 18, 16, N = 256 186.4 -> 190.6; smaller and larger ones gain: 16, 20, N = 256 52.2 -> 51.4, 16, 9, N = 184 32.9 -> 31.0; 19, 16, N = 136, fp32 397 -> 380,
// 19, 10, N = 200 358 -> 337; two panels: 17, 16, N = 128 46.0 -> 43.9.  Nor where one panel of it is less than an L2's 4 MiB, which all XCDs hold whole: 15, 17 a row, N = 16 10.0 -> 11.1, N = 32 11.7 -> 12.3;
// 16, 20, N = 8 13.8 -> 14.3; 42 such products 1.6 % in the mean (14, 20, N = 32 9.6 -> 9.3); from 4 MiB on 18, 12, N = 8 25.1 -> 23.7; several panels 12, 16, N = 256 9.9 -> 9.2.
static bool orders_tasks(size_t K, size_t n_cap, bool b_row_major)
{
    const size_t b = 2 * K * n_cap;
    if (!b_row_major) return true;
    return n_cap <= 64 ? b >= ((size_t)4 << 20) : n_cap <= 128 || b <= ((size_t)32 << 20) || b > ((size_t)128 << 20);
}
static void order_tasks(std::vector<int4> &tasks, std::vector<uint32_t> &costs, const std::vector<WorkItem> &items, const std::vector<int32_t> &row_first, int octaves)
{
    uint64_t total = 0, total_chunks = 0;
    std::vector<uint16_t> keys(tasks.size());
    for (size_t i = 0; i < tasks.size(); i++) {
        const WorkItem &w = items[(size_t)tasks[i].x];
        total += costs[i];
        if (w.dst >= 0) total_chunks += costs[i];
        keys[i] = w.dst >= 0 ? begin_key(w.begin, row_first[(size_t)w.block_row], row_first[(size_t)w.block_row + 1])
                             : (uint16_t)(BEGIN_KEYS + 31 - octave_of(costs[i]) / octaves);
    }
    const std::vector<uint32_t> order = ordered_by(keys, BEGIN_KEYS + 32);
    std::vector<uint32_t> queue[8];
    for (auto &q : queue) q.reserve(tasks.size() / 4);
    uint64_t load[8] = {};
    auto put = [&](int x, uint32_t i) { queue[x].push_back(i); load[x] += costs[i]; };
    uint64_t before = 0;
    size_t at = 0;
    for (; at < order.size() && keys[order[at]] < BEGIN_KEYS; at++) { // the chunks
        put((int)std::min<uint64_t>(7, before * 8 / total_chunks), order[at]);
        before += costs[order[at]];
    }
    while (at < order.size()) {
        const int x = (int)(std::min_element(load, load + 8) - load);
        uint64_t piece = 0;
        for (size_t n = 0; at < order.size() && n < 256 && (n % 4 || n == 0 || piece * 256 < total); n++, at++) {
            piece += costs[order[at]];
            put(x, order[at]);
        }
    }
    size_t rounds = 0; // of four tasks an XCD; places past the end of a queue stay empty
    for (const auto &q : queue) rounds = std::max(rounds, (q.size() + 3) / 4);
    std::vector<int4> placed(rounds * 32, int4{0, 0, 0, 0});
    std::vector<uint32_t> placed_costs(rounds * 32, 0);
    for (int x = 0; x < 8; x++)
        for (size_t i = 0; i < queue[x].size(); i++) {
            const size_t to = (i / 4 * 8 + (size_t)x) * 4 + i % 4;
            placed[to] = tasks[queue[x][i]];
            placed_costs[to] = costs[queue[x][i]];
        }
    tasks.swap(placed);
    costs.swap(placed_costs);
}

hipError_t compact_build(CompactCensus &s, const uint16_t *vals, const int32_t *row_ptr, const int32_t *col_idx, size_t K, size_t n_cap,
                         bool b_row_major, const std::vector<uint8_t> *leave_rows, bool drop_full, CompactPlan **out)
{
    *out = nullptr;
    const size_t mb = s.mb, nnzb = s.nnzb;
    CompactPlan *p = new (std::nothrow) CompactPlan();
    if (!p) return hipErrorOutOfMemory;
    hipError_t e = hipSuccess;
    if (drop_full && nnzb && !s.dropped) {
        hipLaunchKernelGGL(drop_full_kernel, dim3((unsigned)((nnzb + 255) / 256)), dim3(256), 0, 0, (const uint16_t *)s.mask.p, (long)nnzb,
                           (unsigned long long *)s.count.p);
        e = hipGetLastError();
        SMAT_STEP(census_offsets(s, row_ptr));
        s.dropped = true;
    }
    p->values_checksum = s.values_checksum;
    p->n_cols_all = s.n_cols_all;
    std::vector<uint8_t> none;
    const std::vector<uint8_t> &dense = leave_rows ? *leave_rows : (none.assign(mb, 0), none);
    // Block rows left to a dense kernel get no list and no work item here; the others are padded to a multiple of 32
    // columns (one MFMA step) with zero columns.
    int64_t total = 0, n_cols = 0, nnz = 0;
    size_t n_rows = 0; // block rows with listed columns
    std::vector<int32_t> padded(mb + 1, 0);
    std::vector<int2> start(mb + 1); // what the gather kernel sees: list and entries of the row, -1 for rows without a list
    for (size_t i = 0; i < mb; i++) {
        padded[i] = (int32_t)total;
        start[i] = dense[i] ? int2{-1, 0} : int2{(int32_t)total, (int32_t)nnz};
        if (!dense[i]) {
            const uint64_t d = s.raw[i + 1] - s.raw[i];
            total += ((int64_t)(uint32_t)d + 31) / 32 * 32;
            n_cols += (int64_t)(uint32_t)d;
            n_rows += (uint32_t)d != 0;
            nnz += (int64_t)(d >> 32);
        }
        if (total > 0x7fffff00) e = hipErrorInvalidValue;
    }
    padded[mb] = (int32_t)total;
    start[mb] = int2{(int32_t)total, (int32_t)nnz};
    p->n_cols = n_cols;
    const bool by_entry = s.nnz < 0x7fffff00 && (g_force_list ? g_force_list == 2 : lists_nonzeros(nnz, n_cols, n_rows, n_cap));
    const size_t cap = (size_t)total + LIST_PAD;
    SMAT_STEP(dev_malloc(&p->d_cols, cap * sizeof(int32_t)));
    SMAT_STEP(hipMemsetAsync(p->d_cols, 0, cap * sizeof(int32_t), nullptr)); // padding: row 0 of B
    if (by_entry) {
        const size_t steps = cap / 32;
        p->n_entries = nnz;
        p->entries_ahead = nnz <= 48 * (total / 32) ? 1 : 2; // most steps have no more than 64 a load
        SMAT_STEP(dev_malloc(&p->d_entries, ((size_t)nnz + ENTRY_PAD) * sizeof(uint32_t)));
        SMAT_STEP(dev_malloc(&p->d_step_range, steps * sizeof(int2)));
        SMAT_STEP(hipMemsetAsync(p->d_step_range, 0, steps * sizeof(int2), nullptr)); // the steps read ahead of the last one have no entries
    } else {
        SMAT_STEP(dev_malloc(&p->d_acol, cap * 16 * sizeof(uint16_t)));
        SMAT_STEP(hipMemsetAsync(p->d_acol, 0, cap * 16 * sizeof(uint16_t), nullptr));
    }
    // Rows of B that the list names, looked for where the copy might do without others: not below PLACE_MIN_BYTES of B, nor where the
    // plan is made for row-major B, which is read in place.
    const bool look = total > 0 && !b_row_major && K * n_cap * sizeof(uint16_t) >= PLACE_MIN_BYTES;
    const size_t used_bytes = (K + 15) / 16 * 16;
    Scratch used; // a byte a row, and their number
    int32_t n_used = 0;
    if (look) {
        SMAT_STEP(used.alloc(used_bytes + sizeof(int32_t)));
        SMAT_STEP(hipMemsetAsync(used.p, 0, used_bytes, nullptr));
    }
    auto count_used = [&](int32_t *to) {
        hipLaunchKernelGGL(count_rows_kernel, dim3(1), dim3(1024), 0, 0, (uint8_t *)used.p, (long)K, to);
        return hipGetLastError();
    };
    Scratch starts;
    SMAT_STEP(starts.alloc((mb + 1) * sizeof(int2)));
    if (e == hipSuccess && nnzb) {
        SMAT_STEP(hipMemcpy(starts.p, start.data(), (mb + 1) * sizeof(int2), hipMemcpyHostToDevice));
        if (e == hipSuccess) {
            hipLaunchKernelGGL(gather_kernel, dim3((unsigned)((nnzb + 4 * GATHER_BLOCKS - 1) / (4 * GATHER_BLOCKS))), dim3(256), 0, 0, vals, (const uint16_t *)s.mask.p, (const uint32_t *)s.single.p,
                               (const unsigned long long *)s.offset.p, row_ptr, col_idx, (const unsigned long long *)s.rows.p, (const int2 *)starts.p,
                               (long)mb, (long)nnzb, drop_full, p->d_cols, p->d_acol, p->d_entries, p->d_step_range, (uint8_t *)used.p);
            e = hipGetLastError();
        }
    }
    if (by_entry && total > 0) { // no step with more entries than the product kernel asks for
        const int n_groups = (int)(total / 32), most = 64 * p->entries_ahead;
        const size_t padded_groups = cap / 32;
        Scratch steps, first, tmp, starts_dev, row_first;
        size_t bytes = 0;
        SMAT_STEP(steps.alloc(((size_t)n_groups + 1) * sizeof(int32_t)));
        SMAT_STEP(first.alloc(((size_t)n_groups + 2) * sizeof(int32_t))); // one more for the rows that are used
        if (e == hipSuccess) {
            hipLaunchKernelGGL(count_steps_kernel, dim3((unsigned)((n_groups + 256) / 256)), dim3(256), 0, 0, p->d_step_range, n_groups, most, (int32_t *)steps.p);
            e = hipGetLastError();
        }
        SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (int32_t *)steps.p, (int32_t *)first.p, n_groups + 1));
        SMAT_STEP(tmp.alloc(bytes));
        SMAT_STEP(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, (int32_t *)steps.p, (int32_t *)first.p, n_groups + 1));
        if (look) SMAT_STEP(count_used((int32_t *)first.p + n_groups + 1));
        int32_t numbers[2] = {0, 0};
        SMAT_STEP(hipMemcpy(numbers, (int32_t *)first.p + n_groups, (look ? 2 : 1) * sizeof(int32_t), hipMemcpyDeviceToHost));
        const int32_t n_steps = numbers[0];
        n_used = numbers[1];
        if (e == hipSuccess && n_steps > n_groups) {
            if ((int64_t)n_steps * 32 > 0x7fffff00) e = hipErrorInvalidValue;
            const size_t step_cap = (size_t)n_steps + (padded_groups - (size_t)n_groups);
            int32_t *cols = nullptr;
            int2 *range = nullptr;
            SMAT_STEP(dev_malloc(&cols, step_cap * 32 * sizeof(int32_t)));
            SMAT_STEP(dev_malloc(&range, step_cap * sizeof(int2)));
            SMAT_STEP(hipMemsetAsync(cols + (size_t)n_steps * 32, 0, (step_cap - (size_t)n_steps) * 32 * sizeof(int32_t), nullptr));
            SMAT_STEP(hipMemsetAsync(range + n_steps, 0, (step_cap - (size_t)n_steps) * sizeof(int2), nullptr));
            SMAT_STEP(starts_dev.alloc((mb + 1) * sizeof(int32_t)));
            SMAT_STEP(row_first.alloc((mb + 1) * sizeof(int32_t)));
            SMAT_STEP(hipMemcpy(starts_dev.p, padded.data(), (mb + 1) * sizeof(int32_t), hipMemcpyHostToDevice));
            if (e == hipSuccess) {
                hipLaunchKernelGGL(expand_steps_kernel, dim3((unsigned)((n_groups + 7) / 8)), dim3(256), 0, 0, p->d_step_range, p->d_cols,
                                   (const int32_t *)steps.p, (const int32_t *)first.p, n_groups, most, range, cols);
                hipLaunchKernelGGL(row_steps_kernel, dim3((unsigned)((mb + 1 + 255) / 256)), dim3(256), 0, 0, (const int32_t *)starts_dev.p,
                                   (const int32_t *)first.p, (long)mb + 1, (int32_t *)row_first.p);
                e = hipGetLastError();
            }
            SMAT_STEP(hipMemcpy(padded.data(), row_first.p, (mb + 1) * sizeof(int32_t), hipMemcpyDeviceToHost));
            if (e == hipSuccess) { // the copy back has waited for the kernels, so the old lists are idle
                for (int32_t &v : padded) v *= 32;
                total = (int64_t)n_steps * 32;
                std::swap(p->d_cols, cols);
                std::swap(p->d_step_range, range);
                (void)dev_free_idle(cols);
                (void)dev_free_idle(range);
            } else { // kernels may still be at work on either
                if (cols) (void)dev_free(cols);
                if (range) (void)dev_free(range);
            }
        }
        for (Scratch *q : {&steps, &first, &tmp, &starts_dev, &row_first}) q->idle = e == hipSuccess; // a copy to the host came last
    }
    auto place_if_it_pays = [&] {
        if (e == hipSuccess && (size_t)n_used <= K / 8 * 7 && (K - (size_t)n_used) * n_cap * sizeof(uint16_t) >= PLACE_MIN_BYTES)
            e = place_rows(*p, (const uint8_t *)used.p, n_used, K, (long)total);
    };
    int32_t *const count = reinterpret_cast<int32_t *>(static_cast<uint8_t *>(used.p) + used_bytes);
    if (look && by_entry) place_if_it_pays();
    else if (look) SMAT_STEP(count_used(count));
    // Work items: whole block rows; rows much longer than the average in chunks of 32-column steps, all of a row's about
    // as long.  Long rows that are all alike stay whole: their partial tiles are 2 * 16 * N floats to write and read again
    // for each (32768 x 65536, 131 a row, N = 256: 138 us whole, 191 in chunks of 1792 columns; 8192 x 65536, 140 a row,
    // N = 1024: 175 against 241) - except where whole rows would be fewer than four wavefronts a CU (2048 x 65536, 140 a row,
    // N = 256, 512 wavefronts: 43 us whole, 34 in halves; 512 x 65536, 300 a row, N = 1024, 512 of them: 96 against 75).
    const std::vector<int32_t> &cc_host = padded;
    size_t nonempty = 0;
    long longest = 0;
    for (size_t i = 0; i < mb; i++) {
        const long len = cc_host[i + 1] - cc_host[i];
        nonempty += len > 0;
        if (!dense[i]) longest = std::max(longest, len);
    }
    const long chunk = 32 * split_chunk_steps((long)(total / 32), nonempty, longest / 32, n_cap);
    std::vector<WorkItem> items;
    std::vector<SplitRow> split;
    int slot = 0;
    for (size_t i = 0; i < mb; i++) {
        const long len = cc_host[i + 1] - cc_host[i];
        if (len <= chunk || dense[i]) continue;
        SplitRow sr{(int32_t)i, slot, slot, 0};
        const long pieces = (len + chunk - 1) / chunk, piece = (len / 32 + pieces - 1) / pieces * 32;
        for (long b = cc_host[i]; b < cc_host[i + 1]; b += piece)
            items.push_back(WorkItem{(int32_t)i, (int32_t)b, (int32_t)std::min<long>(b + piece, cc_host[i + 1]), slot++});
        sr.slot_end = slot;
        split.push_back(sr);
    }
    for (size_t i = 0; i < mb; i++) {
        const long len = cc_host[i + 1] - cc_host[i];
        if (len > chunk || dense[i]) continue;
        items.push_back(WorkItem{(int32_t)i, cc_host[i], cc_host[i + 1], -1});
    }
    // Tasks: whole items that follow each other in the list, TASK_STEPS steps together at most and fewer where that leaves
    // less than 28 wavefronts a CU (65536 x 4096, 8 a row, N = 96: 16.0 us, with 16 a CU 17.8; chunks of split rows and longer
    // items are a task each).  Their costs, for the deal to the XCDs: the steps, two more for what is fetched first,
    // and one per item for the stores of its tile.
    const long task_steps = std::min<long>(TASK_STEPS, (long)(total / 32 * (int64_t)((n_cap + 63) / 64) / 7168));
    std::vector<int4> tasks;
    std::vector<uint32_t> costs;
    for (size_t i = 0; i < items.size();) {
        size_t j = i + 1;
        long steps = (items[i].end - items[i].begin) / 32;
        while (j < items.size() && j - i < 64 && items[i].dst < 0 && items[j].begin == items[j - 1].end &&
               steps + (items[j].end - items[j].begin) / 32 <= task_steps) {
            steps += (items[j].end - items[j].begin) / 32;
            j++;
        }
        tasks.push_back(int4{(int)i, (int)(j - i), items[i].begin, items[j - 1].end});
        costs.push_back((uint32_t)steps + 2 + (uint32_t)(j - i));
        i = j;
    }
    p->ordered = !split.empty() && g_force_order != 1 && (g_force_order == 2 || orders_tasks(K, n_cap, b_row_major));
    if (p->ordered) order_tasks(tasks, costs, items, cc_host, n_cap > 128 && !b_row_major ? 2 : 1);
    std::vector<uint64_t> cost_prefix(costs.size() + 1, 0);
    for (size_t i = 0; i < costs.size(); i++) cost_prefix[i + 1] = cost_prefix[i] + costs[i];
    p->deal.set_costs(std::move(cost_prefix));
    // Not where columns of B may be held in LDS (few nonzeros a column, column-major), whose sums are to be as close to the exact ones as this kernel's: 60 a row 6.4e-7 root
    // mean square error, this kernel's 9.0e-7 in one sum and 5.6e-7 in two.
    p->may_share = (nnz >= 2 * n_cols || b_row_major || !resident_holds(K)) && std::all_of(tasks.begin(), tasks.end(), [](const int4 &t) { return t.y <= 1; });
    p->n_items = (int)items.size();
    p->n_tasks = (int)tasks.size();
    p->n_steps = total / 32;
    p->n_split_rows = (int)split.size();
    p->n_slots = slot;
    static_assert(sizeof(WorkItem) == sizeof(int4), "the tasks lie behind the items");
    SMAT_STEP(dev_malloc(&p->d_items, (items.size() + tasks.size() + 1) * sizeof(WorkItem)));
    p->d_tasks = reinterpret_cast<int4 *>(p->d_items + items.size());
    const size_t n_items = items.size();
    items.resize(n_items + tasks.size());
    if (!tasks.empty()) memcpy(static_cast<void *>(items.data() + n_items), tasks.data(), tasks.size() * sizeof(int4));
    if (!items.empty()) SMAT_STEP(hipMemcpy(p->d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice));
    if (!split.empty()) {
        SMAT_STEP(dev_malloc(&p->d_split, split.size() * sizeof(SplitRow)));
        SMAT_STEP(hipMemcpy(p->d_split, split.data(), split.size() * sizeof(SplitRow), hipMemcpyHostToDevice));
        SMAT_STEP(dev_malloc(&p->d_workspace, (size_t)slot * 16 * n_cap * sizeof(float)));
    }
    if (look && !by_entry) { // the number is there when everything else is
        SMAT_STEP(hipMemcpy(&n_used, count, sizeof n_used, hipMemcpyDeviceToHost));
        place_if_it_pays();
    }
    SMAT_STEP(hipStreamSynchronize(nullptr)); // launches on other streams read the lists
#undef SMAT_STEP
    starts.idle = used.idle = e == hipSuccess;
    if (e != hipSuccess) {
        compact_destroy(p);
        return e;
    }
    *out = p;
    return hipSuccess;
}

} // namespace smat

// Test hook (not part of smat.h): 1 or 2 = the compact kernel works on panels of 64 or 128 columns whatever the sizes
// say (each width has its own way of gathering the rows of B), 0 = the launcher decides (the default).
extern "C" void smat_internal_compact_panel(int tq) { smat::g_force_tq = tq; }
// Test hook: 1 = lists of whole columns, 2 = of nonzeros (where their number allows it), 0 = as the sizes say (the default).
extern "C" void smat_internal_compact_list(int what) { smat::g_force_list = what; }
// Test hook: 1 = entries go through LDS in blocks of 256 wherever they may, 2 = nowhere, 0 = as the sizes say (the default).
extern "C" void smat_internal_compact_staged(int what) { smat::g_force_staged = what; }
// Test hooks: 1 = tasks of lists with split rows in the order of their items, 2 = as order_tasks says, 0 = as the sizes say (the default); and the rule (host only).
extern "C" int smat_internal_compact_orders(size_t K, size_t n_cap, int b_row_major) { return smat::orders_tasks(K, n_cap, b_row_major != 0); }
extern "C" void smat_internal_compact_order(int what) { smat::g_force_order = what; }
// Test hook: 1, 2 or 4 = wavefronts of a launch that share a task, where tasks are of one item, 0 = as the sizes say (the default).
extern "C" void smat_internal_compact_share(int what) { smat::g_force_share = what; }
// Test hook: registers of a product from entries, panels of 16, 32, 64 or 128 columns; 0 = not known.
extern "C" int smat_internal_compact_registers(int width, int c_f32)
{
    using namespace smat;
    const auto of = [](auto kernel) {
        hipFuncAttributes a = {};
        return hipFuncGetAttributes(&a, reinterpret_cast<const void *>(kernel)) == hipSuccess ? a.numRegs : 0;
    };
    switch (width) {
    case 16: return c_f32 ? of(spmm_compact_kernel<16, true, false, 2, false, false>) : of(spmm_compact_kernel<16, false, false, 2, false, false>);
    case 32: return c_f32 ? of(spmm_compact_kernel<32, true, false, 2, false, false>) : of(spmm_compact_kernel<32, false, false, 2, false, false>);
    case 64: return c_f32 ? of(spmm_compact_kernel<64, true, false, 2, false, false>) : of(spmm_compact_kernel<64, false, false, 2, false, false>);
    default: return c_f32 ? of(spmm_compact_kernel<128, true, false, 2, false, false>) : of(spmm_compact_kernel<128, false, false, 2, false, false>);
    }
}
// Test hook (host only): the rule for such a list, total tasks x panels.
extern "C" int smat_internal_compact_share_rule(int by_name, int64_t n_steps, int64_t n_tasks, int64_t total) { return smat::compact_share(by_name != 0, n_steps, n_tasks, total); }
extern "C" int smat_internal_compact_last_share(void) { return smat::g_last_share.load(); }
// Test hook (host only): steps of the chunks of split rows.
extern "C" long smat_internal_compact_chunk(long steps, size_t rows, long longest, size_t n_cap) { return smat::split_chunk_steps(steps, rows, longest, n_cap); }
// Test hooks for the deal of the compact kernel's workgroups to the XCDs: a run length that every launch uses
// (0 = chosen per plan and number of panels), the run length of the latest launch, and the choice itself for a list
// of item costs (host only).
extern "C" void smat_internal_compact_run(int run) { smat::g_force_run = run; }
extern "C" int smat_internal_compact_last_run(void) { return smat::g_last_run.load(); }
extern "C" void smat_internal_compact_tune(int on) { smat::g_tune = on; }
extern "C" unsigned smat_internal_choose_xcd_run(const uint64_t *cost_prefix, uint64_t n_items, int n_panels)
{
    return smat::choose_xcd_run(cost_prefix, n_items, n_panels);
}
