// CSR -> 16x16 blocked CSR on the GPU: same arrays, bit for bit, as the host
// smat_csr_to_bcsr (and therefore as SparseMatrix::csrToBcsr,
// src/cuda_hgemm/src/common/matrix.h:376-502), without the host pass over the matrix.
//
//   1. count_blocks: one workgroup per block row marks the block columns of its entries in a bitmap in LDS and
//      counts the bits.  The set bits in ascending order ARE the blocks in the row-major order in which the reference
//      numbers them (matrix.h:425-431), so nothing is sorted.  Block rows of more than HEAVY_ROW entries are put on a
//      list and counted by workgroups of 1024 threads afterwards;
//   2. scan_counts: row_ptr from the counts (one workgroup).  The number of blocks goes to the host, which allocates;
//   3. emit_blocks: the bitmap again; col_idx from its set bits, and every entry to block (blocks of the rows before +
//      set bits before its own), row % 16, col % 16.  Blocks are put together in LDS (emit_held); a block row of over
//      8192 entries is filled with zeros and gets its entries from the same workgroup afterwards (emit_row);
//   4. the "dense"/"sparse" counters of the reference's log line (matrix.h:176, 400-419): a
//      block is "dense" when some entry (r, c) with c % 4 in {2, 3} directly follows entries
//      (r, c-1) and (r, c-2) in storage order.  Such a triple lies in one block and its last
//      entry is never the first entry of the block, so the test is independent per entry.
//   Rows whose columns do not ascend strictly (step 1 sees that) can hold an element twice, and a later duplicate of
//   the same (row, col) overwrites the earlier one exactly as the serial loop does (matrix.h:470-487): such a matrix
//   gets its values from scatter_rows / scatter_long_rows, which keep the storage order inside a row (one thread per
//   row; a wavefront per row of more than LONG_ROW entries, 64 entries per step).
// Bound: writing the blocks (512 bytes each).  Radix sort and unique of one key per entry, a memset of the values and
// a scatter by row, with an allocation for each array, took 1.41 ms on 16384^2 with 0.1 % (237 k blocks, 121 MB) and
// 21.8 ms on R-MAT scale 20.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/smat.h"
#include "devmem.h"
#include "errors.h"

using namespace smat;

namespace {

constexpr int LONG_ROW = 512;

constexpr int HELD = 8;               // entries that a thread of emit_held keeps in registers
// Block columns per pass over the entries: three words of LDS per 32 of them beside the blocks that are put together, in
// the 64 KiB that a launch may ask for without more ado (12 KiB a bitmap; K above 1.5 * 2^20 takes more passes).
constexpr int BITMAP_COLS = 3 << 15;
constexpr int LIGHT_THREADS = 256, HEAVY_THREADS = 1024, HEAVY_GRID = 256;
constexpr int HEAVY_ROW = HELD * LIGHT_THREADS; // entries of a block row above which it goes to the workgroups of 1024
constexpr int CHUNK = 32;             // blocks that emit_held puts together in LDS at a time (16 KiB)
constexpr int STATIC_LDS = 256;       // at most: row_ptr of a block row and one word per wavefront
static_assert(BITMAP_COLS % 32 == 0 && BITMAP_COLS / 32 * 12 + CHUNK * 512 + STATIC_LDS <= 65536, "LDS of the emitting kernels");

struct State { // zeroed before the first kernel
    int32_t bad;      // a column index is outside the matrix
    int32_t unsorted; // some row does not ascend strictly
    int32_t n_heavy;  // block rows on the list
    int32_t nnzb;
    int32_t dense; // blocks with a run of three
};

// row (0..15) of entry j inside its block row; rs = row_ptr of the 16 rows and the end
__device__ __forceinline__ int row_in_block(const int32_t *rs, int32_t j)
{
    int r = 0;
#pragma unroll
    for (int step = 8; step; step >>= 1)
        if (rs[r + step] <= j) r += step;
    return r;
}

// exclusive prefix of v over the workgroup and its total; scratch: one word per wavefront
template <int THREADS>
__device__ __forceinline__ int block_scan(int v, int *scratch, int &total)
{
    constexpr int WAVES = THREADS / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(inc, d);
        if (lane >= d) inc += up;
    }
    if (lane == 63) scratch[wave] = inc;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        if (w < wave) before += scratch[w];
        total += scratch[w];
    }
    __syncthreads();
    return before + inc - v;
}

// Marks the block columns [base, base + range) of the entries [begin, end).
template <int THREADS>
__device__ __forceinline__ void mark_columns(const int32_t *__restrict__ col_idx, int32_t begin, int32_t end, int64_t K,
                                             int32_t base, int32_t range, uint32_t *bits)
{
    for (int w = threadIdx.x; w < (range + 31) / 32; w += THREADS) bits[w] = 0;
    __syncthreads();
    for (int32_t j = begin + (int32_t)threadIdx.x; j < end; j += THREADS) {
        const int32_t col = col_idx[j];
        const int32_t bc = (col >> 4) - base;
        if (col >= 0 && col < K && bc >= 0 && bc < range) atomicOr(&bits[bc >> 5], 1u << (bc & 31));
    }
    __syncthreads();
}

template <int THREADS>
__device__ void count_row(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, int64_t br, int64_t K,
                          int32_t kb, uint32_t *bits, int32_t *rs, int *scratch, State *st, int32_t *__restrict__ count)
{
    if (threadIdx.x < 17) rs[threadIdx.x] = row_ptr[br * 16 + threadIdx.x];
    __syncthreads();
    const int32_t begin = rs[0], end = rs[16];
    int total = 0;
    bool bad = false, unsorted = false;
    for (int32_t base = 0; base < kb; base += BITMAP_COLS) {
        const int32_t range = kb - base < BITMAP_COLS ? kb - base : BITMAP_COLS;
        mark_columns<THREADS>(col_idx, begin, end, K, base, range, bits);
        int mine = 0;
        for (int w = threadIdx.x; w < (range + 31) / 32; w += THREADS) mine += __popc(bits[w]);
        int sum;
        (void)block_scan<THREADS>(mine, scratch, sum);
        total += sum;
    }
    for (int32_t j = begin + (int32_t)threadIdx.x; j < end; j += THREADS) {
        const int32_t col = col_idx[j];
        bad |= col < 0 || col >= K;
        if (j > begin && col <= col_idx[j - 1]) unsorted |= j != rs[row_in_block(rs, j)];
    }
    if (bad) st->bad = 1;
    if (unsorted) st->unsorted = 1;
    if (threadIdx.x == 0) count[br] = total;
    __syncthreads();
}

__global__ __launch_bounds__(LIGHT_THREADS) void count_blocks_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
                                                                     int64_t K, int32_t kb, State *st, int32_t *__restrict__ heavy,
                                                                     int32_t *__restrict__ count)
{
    extern __shared__ uint32_t lds[];
    __shared__ int32_t rs[17];
    __shared__ int scratch[LIGHT_THREADS / 64];
    const int64_t br = blockIdx.x;
    if (row_ptr[br * 16 + 16] - row_ptr[br * 16] > HEAVY_ROW) {
        if (threadIdx.x == 0) heavy[atomicAdd(&st->n_heavy, 1)] = (int32_t)br;
        return;
    }
    count_row<LIGHT_THREADS>(row_ptr, col_idx, br, K, kb, lds, rs, scratch, st, count);
}
__global__ __launch_bounds__(HEAVY_THREADS) void count_heavy_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
                                                                    int64_t K, int32_t kb, State *st, const int32_t *__restrict__ heavy,
                                                                    int32_t *__restrict__ count)
{
    extern __shared__ uint32_t lds[];
    __shared__ int32_t rs[17];
    __shared__ int scratch[HEAVY_THREADS / 64];
    const int n = st->n_heavy;
    for (int i = blockIdx.x; i < n; i += gridDim.x)
        count_row<HEAVY_THREADS>(row_ptr, col_idx, heavy[i], K, kb, lds, rs, scratch, st, count);
}

// b_row_ptr[0 .. mb] = exclusive prefix of count: one workgroup, 8192 counts a step, the next ones on their way
__global__ __launch_bounds__(1024) void scan_counts_kernel(const int32_t *__restrict__ count, int64_t mb, int32_t *__restrict__ b_row_ptr, State *st)
{
    __shared__ int scratch[16];
    int carry = 0;
    auto fetch = [&](int64_t first, int (&v)[8]) {
        if (first + 8 <= mb) {
            const int4 lo = *reinterpret_cast<const int4 *>(count + first), hi = *reinterpret_cast<const int4 *>(count + first + 4);
            v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = first + i < mb ? count[first + i] : 0;
        }
    };
    int v[8];
    fetch(threadIdx.x * 8, v);
    for (int64_t base = 0; base < mb; base += 8192) {
        const int64_t first = base + threadIdx.x * 8;
        int next[8], sum = 0;
        fetch(first + 8192, next);
#pragma unroll
        for (int i = 0; i < 8; i++) sum += v[i];
        int total;
        int at = carry + block_scan<1024>(sum, scratch, total);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (first + i < mb) b_row_ptr[first + i] = at;
            at += v[i];
            v[i] = next[i];
        }
        carry += total;
    }
    if (threadIdx.x == 0) {
        b_row_ptr[mb] = carry;
        st->nnzb = carry;
    }
}

// st->dense = sum of count (blocks with a run of three per block row, as the emitting kernels leave them): added to
// one word by every workgroup itself, the counts of 16384 block rows queue up behind it for 800 us
__global__ __launch_bounds__(256) void sum_dense_kernel(const int32_t *__restrict__ count, int64_t mb, State *st)
{
    int mine = 0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < mb; i += (int64_t)gridDim.x * 256) mine += count[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) mine += __shfl_xor(mine, d);
    if ((threadIdx.x & 63) == 0 && mine) atomicAdd(&st->dense, mine);
}

// Set bits of the words before each word, col_idx of the set bits, dense flags cleared.  Returns the set bits of all words.
template <int THREADS>
__device__ __forceinline__ int32_t number_blocks(const uint32_t *bits, uint32_t *dense, int32_t *before, int n_words, int32_t base,
                                                 int *scratch, int32_t *__restrict__ b_col_idx)
{
    // a thread owns the words [w0, w1): their set bits follow those of the threads before it
    const int per = (n_words + THREADS - 1) / THREADS;
    const int w0 = min((int)threadIdx.x * per, n_words), w1 = min(w0 + per, n_words);
    int mine = 0;
    for (int w = w0; w < w1; w++) {
        dense[w] = 0;
        mine += __popc(bits[w]);
    }
    int total;
    int32_t at = block_scan<THREADS>(mine, scratch, total);
    for (int w = w0; w < w1; w++) {
        uint32_t b = bits[w];
        before[w] = at;
        while (b) {
            const int k = __ffs(b) - 1;
            b &= b - 1;
            b_col_idx[at++] = (base + w * 32 + k) * 16;
        }
    }
    __syncthreads();
    return total;
}
template <int THREADS>
__device__ __forceinline__ int count_bits(const uint32_t *words, int n_words)
{
    int n = 0;
    for (int w = threadIdx.x; w < n_words; w += THREADS) n += __popc(words[w]);
    return n;
}
// *out = sum of n over the workgroup
template <int THREADS>
__device__ __forceinline__ void leave_sum(int n, int *scratch, int32_t *out)
{
    int total;
    (void)block_scan<THREADS>(n, scratch, total);
    if (threadIdx.x == 0) *out = total;
}
__device__ __forceinline__ int32_t rank_of(const uint32_t *bits, const int32_t *before, int32_t bc)
{
    return before[bc >> 5] + __popc(bits[bc >> 5] & ((1u << (bc & 31)) - 1u));
}

// A block row of at most HELD * THREADS entries whose rows ascend: every thread keeps its entries in registers and the
// blocks are put together in LDS, CHUNK at a time, so that their 512 bytes are written once and whole.  (Zeros first
// and the entries into them as 2-byte stores, as emit_row below does it, takes four times as long: the lines have left
// the L2 by then, and each comes back for two bytes.)
template <int THREADS>
__device__ void emit_held(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ val,
                          int64_t br, int32_t kb, int32_t words, uint32_t *lds, int32_t *rs, int *scratch, int32_t *__restrict__ n_dense,
                          const int32_t *__restrict__ b_row_ptr, int32_t *__restrict__ b_col_idx, uint16_t *__restrict__ b_val)
{
    uint4 *tile = reinterpret_cast<uint4 *>(lds);
    uint32_t *bits = lds + CHUNK * 128, *dense = bits + words;
    int32_t *before = reinterpret_cast<int32_t *>(dense + words);
    if (threadIdx.x < 17) rs[threadIdx.x] = row_ptr[br * 16 + threadIdx.x];
    const int32_t first = b_row_ptr[br], n_blocks = b_row_ptr[br + 1] - first;
    __syncthreads();
    const int32_t begin = rs[0], n = rs[16] - begin;
    int32_t col[HELD], rank[HELD];
    uint32_t what[HELD]; // place in the block, value, whether it ends a run of three
#pragma unroll
    for (int i = 0; i < HELD; i++) {
        const int32_t e = i * THREADS + (int32_t)threadIdx.x;
        col[i] = -1;
        rank[i] = -1;
        if (e < n) {
            const int32_t j = begin + e, c = col_idx[j];
            const int r = row_in_block(rs, j);
            col[i] = c;
            what[i] = (uint32_t)val[j] << 16 | (uint32_t)(r * 16 + (c & 15));
            if ((c & 2) && j >= rs[r] + 2 && col_idx[j - 1] == c - 1 && col_idx[j - 2] == c - 2) what[i] |= 1u << 8;
        }
    }
    int flagged = 0, done = 0;
    for (int32_t base = 0; base < kb; base += BITMAP_COLS) {
        const int32_t range = kb - base < BITMAP_COLS ? kb - base : BITMAP_COLS;
        const int n_words = (range + 31) / 32;
        for (int w = threadIdx.x; w < n_words; w += THREADS) bits[w] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < HELD; i++) {
            const int32_t bc = (col[i] >> 4) - base;
            if (col[i] >= 0 && bc >= 0 && bc < range) atomicOr(&bits[bc >> 5], 1u << (bc & 31));
        }
        __syncthreads();
        const int32_t total = number_blocks<THREADS>(bits, dense, before, n_words, base, scratch, b_col_idx + first + done);
#pragma unroll
        for (int i = 0; i < HELD; i++) {
            const int32_t bc = (col[i] >> 4) - base;
            if (col[i] < 0 || bc < 0 || bc >= range) continue;
            rank[i] = done + rank_of(bits, before, bc);
            if (what[i] >> 8 & 1) atomicOr(&dense[bc >> 5], 1u << (bc & 31));
        }
        done += total;
        __syncthreads();
        flagged += count_bits<THREADS>(dense, n_words);
        __syncthreads();
    }
    leave_sum<THREADS>(flagged, scratch, n_dense);
    uint16_t *halves = reinterpret_cast<uint16_t *>(tile);
    for (int32_t c0 = 0; c0 < n_blocks; c0 += CHUNK) {
        const int pieces = min(CHUNK, n_blocks - c0) * 32;
        for (int p = threadIdx.x; p < pieces; p += THREADS) tile[p] = uint4{0, 0, 0, 0};
        __syncthreads();
#pragma unroll
        for (int i = 0; i < HELD; i++) {
            const int32_t at = rank[i] - c0;
            if (rank[i] >= 0 && at >= 0 && at < CHUNK) halves[at * 256 + (what[i] & 255)] = (uint16_t)(what[i] >> 16);
        }
        __syncthreads();
        uint4 *out = reinterpret_cast<uint4 *>(b_val + ((int64_t)first + c0) * 256);
        for (int p = threadIdx.x; p < pieces; p += THREADS) out[p] = tile[p];
        __syncthreads();
    }
}

// Any block row: zeros into its values, then its entries (with scatter; without, scatter_rows writes them).
template <int THREADS>
__device__ void emit_row(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ val,
                         int64_t br, int64_t K, int32_t kb, int32_t words, uint32_t *lds, int32_t *rs, int *scratch, bool scatter,
                         int32_t *__restrict__ n_dense, const int32_t *__restrict__ b_row_ptr, int32_t *__restrict__ b_col_idx,
                         uint16_t *__restrict__ b_val)
{
    uint32_t *bits = lds, *dense = lds + words;
    int32_t *before = reinterpret_cast<int32_t *>(lds + 2 * words);
    if (threadIdx.x < 17) rs[threadIdx.x] = row_ptr[br * 16 + threadIdx.x];
    int32_t first = b_row_ptr[br]; // block of the first set bit of this pass
    const int32_t last = b_row_ptr[br + 1];
    {
        uint4 *z = reinterpret_cast<uint4 *>(b_val + (int64_t)first * 256);
        for (int64_t i = threadIdx.x; i < (int64_t)(last - first) * 32; i += THREADS) z[i] = uint4{0, 0, 0, 0};
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // in place before the barriers below let the entries in
    }
    __syncthreads();
    const int32_t begin = rs[0], end = rs[16];
    int flagged = 0;
    for (int32_t base = 0; base < kb; base += BITMAP_COLS) {
        const int32_t range = kb - base < BITMAP_COLS ? kb - base : BITMAP_COLS;
        const int n_words = (range + 31) / 32;
        mark_columns<THREADS>(col_idx, begin, end, K, base, range, bits);
        const int32_t total = number_blocks<THREADS>(bits, dense, before, n_words, base, scratch, b_col_idx + first);
        if (scatter) {
            for (int32_t j = begin + (int32_t)threadIdx.x; j < end; j += THREADS) {
                const int32_t col = col_idx[j];
                const int32_t bc = (col >> 4) - base;
                if (bc < 0 || bc >= range) continue;
                const int r = row_in_block(rs, j);
                const int64_t p = first + rank_of(bits, before, bc);
                b_val[p * 256 + r * 16 + (col & 15)] = val[j];
                if ((col & 2) && j >= rs[r] + 2 && col_idx[j - 1] == col - 1 && col_idx[j - 2] == col - 2)
                    atomicOr(&dense[bc >> 5], 1u << (bc & 31));
            }
            __syncthreads();
            flagged += count_bits<THREADS>(dense, n_words);
        }
        first += total;
        __syncthreads();
    }
    leave_sum<THREADS>(flagged, scratch, n_dense);
}

__global__ __launch_bounds__(LIGHT_THREADS) void emit_blocks_kernel(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ val, int64_t K, int32_t kb, int32_t words,
    bool scatter, int32_t *__restrict__ n_dense, const int32_t *__restrict__ b_row_ptr, int32_t *__restrict__ b_col_idx, uint16_t *__restrict__ b_val)
{
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int32_t rs[17];
    __shared__ int scratch[LIGHT_THREADS / 64];
    const int64_t br = blockIdx.x;
    const int32_t n = row_ptr[br * 16 + 16] - row_ptr[br * 16];
    if (n > HEAVY_ROW) return;
    if (n == 0) {
        if (threadIdx.x == 0) n_dense[br] = 0;
        return;
    }
    if (scatter) emit_held<LIGHT_THREADS>(row_ptr, col_idx, val, br, kb, words, lds, rs, scratch, n_dense + br, b_row_ptr, b_col_idx, b_val);
    else emit_row<LIGHT_THREADS>(row_ptr, col_idx, val, br, K, kb, words, lds, rs, scratch, false, n_dense + br, b_row_ptr, b_col_idx, b_val);
}
__global__ __launch_bounds__(HEAVY_THREADS) void emit_heavy_kernel(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ val, int64_t K, int32_t kb, int32_t words,
    const State *st, bool scatter, int32_t *__restrict__ n_dense, const int32_t *__restrict__ heavy, const int32_t *__restrict__ b_row_ptr,
    int32_t *__restrict__ b_col_idx, uint16_t *__restrict__ b_val)
{
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int32_t rs[17];
    __shared__ int scratch[HEAVY_THREADS / 64];
    const int n_heavy = st->n_heavy;
    for (int i = blockIdx.x; i < n_heavy; i += gridDim.x) {
        const int64_t br = heavy[i];
        const int32_t n = row_ptr[br * 16 + 16] - row_ptr[br * 16];
        if (scatter && n <= HELD * HEAVY_THREADS)
            emit_held<HEAVY_THREADS>(row_ptr, col_idx, val, br, kb, words, lds, rs, scratch, n_dense + br, b_row_ptr, b_col_idx, b_val);
        else
            emit_row<HEAVY_THREADS>(row_ptr, col_idx, val, br, K, kb, words, lds, rs, scratch, scatter, n_dense + br, b_row_ptr, b_col_idx, b_val);
        __syncthreads();
    }
}

// position of block column `bc` inside block row [lo, hi) of b_col_idx (it is always present)
__device__ __forceinline__ int32_t find_block(const int32_t *__restrict__ b_col_idx, int32_t lo, int32_t hi, int32_t col16)
{
    while (hi - lo > 1) {
        const int32_t mid = (lo + hi) >> 1;
        if (b_col_idx[mid] <= col16) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ bool promotes(const int32_t *__restrict__ col_idx, int64_t j, int64_t row_start, int32_t col)
{
    const int r = col & 3;
    return (r == 2 || r == 3) && j >= row_start + 2 && col_idx[j - 1] == col - 1 && col_idx[j - 2] == col - 2;
}

// one thread per CSR row of at most LONG_ROW entries
__global__ void scatter_rows_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
                                    const uint16_t *__restrict__ val, int64_t M,
                                    const int32_t *__restrict__ b_row_ptr, const int32_t *__restrict__ b_col_idx,
                                    uint16_t *__restrict__ b_val, uint8_t *__restrict__ dense_flag)
{
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= M) return;
    const int64_t begin = row_ptr[row], end = row_ptr[row + 1];
    if (end - begin > LONG_ROW) return;
    const int32_t lo = b_row_ptr[row >> 4], hi = b_row_ptr[(row >> 4) + 1];
    int32_t last_c16 = -1, p = 0;
    for (int64_t j = begin; j < end; j++) {
        const int32_t col = col_idx[j];
        const int32_t c16 = col & ~15;
        if (c16 != last_c16) { p = find_block(b_col_idx, lo, hi, c16); last_c16 = c16; }
        b_val[(int64_t)p * 256 + (row & 15) * 16 + (col & 15)] = val[j];
        if (promotes(col_idx, j, begin, col)) dense_flag[p] = 1;
    }
}

// one wavefront per CSR row with more than LONG_ROW entries
__global__ __launch_bounds__(256) void scatter_long_rows_kernel(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ val,
    int64_t M, const int32_t *__restrict__ b_row_ptr, const int32_t *__restrict__ b_col_idx,
    uint16_t *__restrict__ b_val, uint8_t *__restrict__ dense_flag)
{
    const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (row >= M) return;
    const int64_t begin = row_ptr[row], end = row_ptr[row + 1];
    if (end - begin <= LONG_ROW) return; // wave-uniform
    const int32_t lo = b_row_ptr[row >> 4], hi = b_row_ptr[(row >> 4) + 1];
    for (int64_t base = begin; base < end; base += 64) {
        const int64_t j = base + lane;
        const bool live = j < end;
        const int32_t col = live ? col_idx[j] : -1;
        // a later entry of this step with the same column wins: drop this one
        bool shadowed = false;
        for (int d = 1; d < 64; d++) {
            const int32_t other = __shfl_down(col, d);
            if (lane + d < 64 && other == col) shadowed = true;
        }
        if (live) {
            const int32_t p = find_block(b_col_idx, lo, hi, col & ~15);
            if (!shadowed) b_val[(int64_t)p * 256 + (row & 15) * 16 + (col & 15)] = val[j];
            if (promotes(col_idx, j, begin, col)) dense_flag[p] = 1;
        }
        // stores of this step are complete before the next step may overwrite them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    }
}

// blocks flagged by the scatter kernels above
__global__ __launch_bounds__(256) void count_flags_kernel(const uint8_t *__restrict__ flags, int64_t n, int32_t *__restrict__ total)
{
    int mine = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) mine += flags[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) mine += __shfl_xor(mine, d);
    if ((threadIdx.x & 63) == 0 && mine) atomicAdd(total, mine);
}

} // namespace

static int smat_csr_to_bcsr_device_impl(size_t M, size_t K, const int32_t *row_ptr, const int32_t *col_idx,
                                        const uint16_t *val, size_t nnz, int64_t *counts,
                                        int32_t **b_row_ptr, int32_t **b_col_idx, uint16_t **b_val)
{
    if (!row_ptr || !b_row_ptr || !b_col_idx || !b_val)
        return set_error(SMAT_ERR_INVALID, "NULL argument");
    if (M == 0 || K == 0 || M % 16 || K % 16)
        return set_error(SMAT_ERR_INVALID, "M (%zu) and K (%zu) must be positive multiples of 16", M, K);
    if (nnz && (!col_idx || !val)) return set_error(SMAT_ERR_INVALID, "col_idx/val must not be NULL");
    if (nnz > 0x7fffffffu) return set_error(SMAT_ERR_INVALID, "more than 2^31-1 entries");
    const size_t mb = M / 16, kb = K / 16;
    if (mb > 0x7fffffffu || kb > 0x7fffffffu)
        return set_error(SMAT_ERR_INVALID, "dimension exceeds the int32 index range of BCSR");
    *b_row_ptr = nullptr; *b_col_idx = nullptr; *b_val = nullptr;

    int32_t *orp = nullptr, *oci = nullptr;
    uint16_t *ov = nullptr;
    DevScratch state, count, heavy, flags;
    State h{};
    hipError_t e = dev_malloc(&orp, (mb + 1) * sizeof(int32_t));
    auto step = [&](hipError_t r) { if (e == hipSuccess) e = r; };
    step(state.alloc(sizeof(State)));
    step(count.alloc(mb * sizeof(int32_t)));
    step(heavy.alloc((nnz / HEAVY_ROW + 1) * sizeof(int32_t)));
    State *st = static_cast<State *>(state.p);
    const int32_t words = (int32_t)((std::min<size_t>(kb, BITMAP_COLS) + 31) / 32);
    const int32_t kb32 = (int32_t)std::min<size_t>(kb, (size_t)1 << 27); // the block columns that an int32 column index can name
    if (e == hipSuccess) {
        step(hipMemsetAsync(st, 0, sizeof(State), nullptr));
        if (nnz) {
            hipLaunchKernelGGL(count_blocks_kernel, dim3((unsigned)mb), dim3(LIGHT_THREADS), words * 4, 0, row_ptr, col_idx, (int64_t)K,
                               kb32, st, (int32_t *)heavy.p, (int32_t *)count.p);
            hipLaunchKernelGGL(count_heavy_kernel, dim3(HEAVY_GRID), dim3(HEAVY_THREADS), words * 4, 0, row_ptr, col_idx, (int64_t)K,
                               kb32, st, (const int32_t *)heavy.p, (int32_t *)count.p);
        } else {
            step(hipMemsetAsync(count.p, 0, mb * sizeof(int32_t), nullptr));
        }
        hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(1024), 0, 0, (const int32_t *)count.p, (int64_t)mb, orp, st);
        step(hipGetLastError());
        step(hipMemcpy(&h, st, sizeof h, hipMemcpyDeviceToHost));
    }
    if (e == hipSuccess && h.bad) {
        (void)dev_free(orp);
        return set_error(SMAT_ERR_INVALID, "a column index is outside 0..%zu", K - 1);
    }
    const int64_t nnzb = h.nnzb;
    if (e == hipSuccess) e = dev_malloc(&oci, std::max<size_t>(nnzb, 1) * sizeof(int32_t));
    if (e == hipSuccess) e = dev_malloc(&ov, std::max<size_t>(nnzb, 1) * 512);
    if (e == hipSuccess && nnzb) {
        const unsigned lds = (unsigned)(words * 12 + CHUNK * 512);
        hipLaunchKernelGGL(emit_blocks_kernel, dim3((unsigned)mb), dim3(LIGHT_THREADS), lds, 0, row_ptr, col_idx, val, (int64_t)K,
                           kb32, words, !h.unsorted, (int32_t *)count.p, orp, oci, ov);
        if (h.n_heavy)
            hipLaunchKernelGGL(emit_heavy_kernel, dim3(HEAVY_GRID), dim3(HEAVY_THREADS), lds, 0, row_ptr, col_idx, val, (int64_t)K,
                               kb32, words, st, !h.unsorted, (int32_t *)count.p, (const int32_t *)heavy.p, orp, oci, ov);
        if (!h.unsorted && counts)
            hipLaunchKernelGGL(sum_dense_kernel, dim3((unsigned)std::min<size_t>((mb + 1023) / 1024, 64)), dim3(256), 0, 0,
                               (const int32_t *)count.p, (int64_t)mb, st);
        step(hipGetLastError());
        if (h.unsorted && e == hipSuccess) {
            step(flags.alloc(nnzb));
            if (e == hipSuccess) {
                step(hipMemsetAsync(flags.p, 0, nnzb, nullptr));
                hipLaunchKernelGGL(scatter_rows_kernel, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, 0, row_ptr,
                                   col_idx, val, (int64_t)M, orp, oci, ov, (uint8_t *)flags.p);
                hipLaunchKernelGGL(scatter_long_rows_kernel, dim3((unsigned)((M * 64 + 255) / 256)), dim3(256), 0, 0,
                                   row_ptr, col_idx, val, (int64_t)M, orp, oci, ov, (uint8_t *)flags.p);
                hipLaunchKernelGGL(count_flags_kernel, dim3((unsigned)std::min<int64_t>((nnzb + 255) / 256, 1024)), dim3(256), 0, 0,
                                   (const uint8_t *)flags.p, nnzb, &st->dense);
                step(hipGetLastError());
            }
        }
        step(hipMemcpy(&h, st, sizeof h, hipMemcpyDeviceToHost)); // the counter, and everything before it is done
    }
    if (e != hipSuccess) {
        for (void *q : {(void *)orp, (void *)oci, (void *)ov})
            if (q) (void)dev_free(q);
        return set_error(SMAT_ERR_HIP, "device blocking failed: %s", hipGetErrorString(e));
    }
    if (counts) {
        counts[0] = nnzb;
        counts[1] = h.dense;
        counts[2] = nnzb - h.dense;
    }
    *b_row_ptr = orp; *b_col_idx = oci; *b_val = ov;
    return SMAT_OK;
}

extern "C" int smat_csr_to_bcsr_device(size_t M, size_t K, const int32_t *row_ptr, const int32_t *col_idx,
                                        const uint16_t *val, size_t nnz, int64_t *counts,
                                        int32_t **b_row_ptr, int32_t **b_col_idx, uint16_t **b_val)
{
    return smat::guarded("smat_csr_to_bcsr_device", [&] { return smat_csr_to_bcsr_device_impl(M, K, row_ptr, col_idx, val, nnz, counts, b_row_ptr, b_col_idx, b_val); });
}
