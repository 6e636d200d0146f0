// Product of whole 16x16 blocks for matrices whose neighbouring block rows use the same block columns (bands, stencils).  The
// row-wise kernel fetches the rows of B under a block for every block anew, 924 MB for 33 MB of B on the 27-point stencil on
// 64^3 at N = 64, and repacks B first so that the caches can deliver that.  Here a group of 4, 8 or 16 consecutive block rows, a wavefront
// each, brings the block columns that any of them uses, its window, to LDS once, from column-major B as it lies in memory, and
// multiplies from there: 164 MB on that matrix, and no copy of B.
//
//  * window_count_kernel, window_list_kernel (once per pattern, on the device): how wide the windows of groups of each size
//    are; the columns of every window in ascending order, and for every block its place in its window.
//  * spmm_window_kernel: below.
//
// The order of the sums is that of the row-wise kernel (blocks of a row two by two from its first), the results have the same bits; with listed
// nonzeros the halves of blocks without one are left out (window_entries_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <new>
#include <type_traits>
#include <vector>

#include "devmem.h"
#include "row_tile.h"
#include "spmm_kernels.h"

namespace smat {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int COPIES = 7;               // KiB of a window that a wavefront copies at a time
constexpr int SLOT_BITS = 10;           // of a block's entry: its place in the window; above them its block column
constexpr int BITMAP_WORDS = 8192;      // block columns of the matrix / 32
constexpr uint32_t NO_SLOT = 0xffffffffu; // a block that has none, which no column matches
constexpr int MAX_LISTED = 128;         // block columns of a window with listed nonzeros: octets are named in 8 bits
constexpr size_t MAX_LDS = 160 * 1024;  // of a compute unit
constexpr int CU_WAVES = 16;            // wavefronts of 128 registers on a compute unit
constexpr int SIZES[WINDOW_SIZES] = {4, 8, 16}; // block rows of a group
// block pairs of a row that a wavefront holds
constexpr int MAX_PAIRS = 17;
template <int TN> constexpr int pairs_held = TN == 4 ? 12 : MAX_PAIRS;
// Listed nonzeros become operands a round of so many steps at a time (three: 3 to 7 % slower where every octet holds some).
constexpr int ROUND = 4, MAX_ROUNDS = (MAX_PAIRS + ROUND - 1) / ROUND;
static_assert(ROUND % 2 == 0, "the product takes two steps at a time: behind an odd number the next one of its round, zeros");
constexpr int LIST_BITS = 26; // of a round's list: the fours of entries before it; above them its own fours
constexpr int FILL_BITS = 4; // a round's places that are none: one at least is an octet
static_assert(4 * ROUND <= 1 << FILL_BITS && 8 + FILL_BITS * MAX_ROUNDS <= 32, "");
constexpr uint32_t MAX_LIST = 4 * ((1u << (32 - LIST_BITS)) - 1); // entries of a round: four a lane

// ---- which block columns a group uses ----

__device__ __forceinline__ void mark_columns(uint32_t *bitmap, int words, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
                                             int first, int last)
{
    for (int w = threadIdx.x; w < words; w += blockDim.x) bitmap[w] = 0;
    __syncthreads();
    for (long p = row_ptr[first] + (long)threadIdx.x; p < row_ptr[last]; p += blockDim.x) {
        const uint32_t c = (uint32_t)col_idx[p] >> 4;
        if (c < (uint32_t)words * 32u) atomicOr(&bitmap[c >> 5], 1u << (c & 31));
    }
    __syncthreads();
}

// A workgroup takes every gridDim.x-th group of one size; parts[size * WindowCount::PARTS + blockIdx.x]: the most block columns of one of its groups, and
// those of all its groups.  (Additions to one word queue up at 12 ns each, and need zeros first.)
__global__ __launch_bounds__(256) void window_count_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, int mb, int words,
                                                           uint2 *__restrict__ parts)
{
    extern __shared__ uint32_t bitmap[];
    __shared__ uint32_t part[4];
    const int rows = blockIdx.y == 0 ? SIZES[0] : blockIdx.y == 1 ? SIZES[1] : SIZES[2];
    uint32_t most = 0, sum = 0; // of blocks, which are fewer than 2^31
    for (long first = (long)blockIdx.x * rows; first < mb; first += (long)gridDim.x * rows) {
        mark_columns(bitmap, words, row_ptr, col_idx, (int)first, (int)min(first + rows, (long)mb));
        uint32_t n = 0;
        for (int w = threadIdx.x; w < words; w += 256) n += __popc(bitmap[w]);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = n;
        __syncthreads();
        n = part[0] + part[1] + part[2] + part[3];
        most = max(most, n);
        sum += n;
        __syncthreads();
    }
    if (threadIdx.x == 0) parts[blockIdx.y * WindowCount::PARTS + blockIdx.x] = uint2{most, sum};
}

// window[group * cap ..]: the first columns of the group's blocks, ascending, filled up to a multiple of 4; slot[p]: the place
// of block p's column in it.
__global__ __launch_bounds__(256) void window_list_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, int mb, int words,
                                                          int rows, int cap, int32_t *__restrict__ window, int32_t *__restrict__ count,
                                                          uint32_t *__restrict__ slot)
{
    extern __shared__ uint32_t bitmap[]; // words, and as many half words of ranks behind them
    uint16_t *const rank = reinterpret_cast<uint16_t *>(bitmap + words);
    __shared__ uint32_t part[4];
    const int first = (int)blockIdx.x * rows, last = min(first + rows, mb);
    mark_columns(bitmap, words, row_ptr, col_idx, first, last);
    const int per = (words + 255) / 256, w0 = min((int)threadIdx.x * per, words), w1 = min(w0 + per, words);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t n = 0;
    for (int w = w0; w < w1; w++) n += __popc(bitmap[w]);
    uint32_t before = n; // to the sum of the threads before this one
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t of = __shfl_up(before, d);
        before += lane >= d ? of : 0;
    }
    if (lane == 63) part[wave] = before;
    before -= n;
    __syncthreads();
    uint32_t all = 0;
    for (int w = 0; w < 4; w++) {
        before += w < wave ? part[w] : 0;
        all += part[w];
    }
    int32_t *const out = window + (long)blockIdx.x * cap;
    for (int w = w0; w < w1; w++) {
        rank[w] = (uint16_t)before;
        for (uint32_t b = bitmap[w]; b; b &= b - 1, before++)
            if ((int)before < cap) out[before] = (w * 32 + __ffs((int)b) - 1) * 16;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        all = min(all, (uint32_t)cap);
        count[blockIdx.x] = (int32_t)((all + 3) & ~3u);
        for (uint32_t i = all; i & 3; i++) out[i] = all ? out[all - 1] : 0;
    }
    for (long p = row_ptr[first] + (long)threadIdx.x; p < row_ptr[last]; p += 256) {
        const int32_t col = col_idx[p];
        const uint32_t c = (uint32_t)col >> 4;
        uint32_t of = NO_SLOT; // not a column, or, where the widths were counted in another pattern, one without a place
        if (c < (uint32_t)words * 32u && !(col & 15)) {
            const uint32_t at = (uint32_t)rank[c >> 5] + __popc(bitmap[c >> 5] & ((1u << (c & 31)) - 1u));
            if (at < (uint32_t)cap) of = c << SLOT_BITS | at;
        }
        slot[p] = of;
    }
}

// The nonzeros of the blocks.  Unit: an octet, 8 neighbouring columns of a block; the product multiplies four of them a step, and those without a
// nonzero are left out, a third of a 27-point stencil's (64^3, N = 64 36.0 -> 32.6 us).  ROUND steps of a block row after the other:
// value << 16 | byte in the MFMA operands of the round, which lie rows KiB apart, filled up to a multiple of four with the last one.  A round
// ends early where the next pair of blocks does not fit its list.  table: MAX_PAIRS pairs of words a block row, the places of the four octets of step j
// in the window (8 bits each, in octets; of those that are none that of the row's first) and the list of round j, the fours of
// entries before it and its own << LIST_BITS; behind the table of every row twice its steps and, FILL_BITS each from bit 8 on, the places of every round
// that are none, its last ones.  A wavefront takes a block
// row; offset[p]: nonzeros before block p in the upper half.  Bound by the read of the values.
__global__ __launch_bounds__(256) void window_entries_kernel(const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr,
                                                             const uint32_t *__restrict__ slot, const unsigned long long *__restrict__ offset, int mb, int rows, int held,
                                                             uint32_t *__restrict__ entries, uint32_t *__restrict__ table, uint32_t *__restrict__ most)
{
    const int lane = threadIdx.x & 63, br = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (br >= mb) return;
    const int p0 = row_ptr[br], blocks = row_ptr[br + 1] - p0;
    const int g = lane >> 4, sel = g >> 1, at = (lane & 15) * 16 + (g & 1) * 8; // octet g of two blocks
    auto load = [&](int d) {
        const int b = 2 * d + sel;
        return b < blocks ? *reinterpret_cast<const u32x4 *>(vals + (long)(p0 + b) * 256 + at) : (u32x4){0u, 0u, 0u, 0u};
    };
    u32x4 w = load(0);
    uint32_t first = blocks > 0 ? ((uint32_t)(offset[p0] >> 32) + 8u * (uint32_t)((p0 + br + 1) / 2)) & ~3u : 0; // of the round
    uint32_t octets = 0, n = 0, last = 0, longest = 0;   // of the row; entries of the round, the last one; of the longest round
    uint32_t none = 0; // places of the rounds that are no octets
    bool no_slot = false;
    uint32_t places = 0, list = 0, first_place = 0;       // places, list: of step and round `lane`
    auto close = [&](uint32_t round) {                    // fills the round up; the next one begins behind it
        const uint32_t end = (n + 3u) & ~3u;
        if (n + lane < end) entries[first + n + lane] = last;
        if (lane == (int)round) list = first / 4 | min(end, MAX_LIST) / 4 << LIST_BITS;
        longest = max(longest, end);
        first += end;
    };
    auto fill = [&](uint32_t from, uint32_t to) { // octets that are none
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((uint32_t)(lane * 4 + i) >= from && (uint32_t)(lane * 4 + i) < to) places |= first_place << (8 * i);
    };
    for (int d = 0; 2 * d < blocks; d++) {
        const u32x4 now = w;
        w = load(d + 1);
        const int b = min(2 * d + sel, blocks - 1);
        const uint32_t of_block = slot[p0 + b], place = (of_block & ((1u << SLOT_BITS) - 1u)) * 2u + (uint32_t)(g & 1);
        no_slot |= of_block == NO_SLOT;
        uint32_t bits = 0, before = 0, all = 0; // entries of the lanes before this one, and of all
        unsigned long long has_k[8];
#pragma unroll
        for (int k = 0; k < 8; k++) { // -0.0 is a zero
            const bool has = (now[k / 2] >> (k & 1 ? 16 : 0) & 0x7fffu) != 0;
            bits |= (uint32_t)has << k;
            has_k[k] = __ballot(has);
            all += __popcll(has_k[k]);
            before += __popcll(has_k[k] & ((1ull << lane) - 1ull));
        }
        const unsigned long long some = __ballot(bits != 0);
        uint32_t used = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) used |= (uint32_t)((some >> (16 * i) & 0xffffu) != 0) << i;
        uint32_t round = octets / (4 * ROUND), o = octets + __popc(used & ((1u << g) - 1u)), n_in = 0;
        bool now_in = o / (4 * ROUND) == round; // else in the next one
        unsigned long long in = __ballot(bits != 0 && now_in);
#pragma unroll
        for (int k = 0; k < 8; k++) n_in += __popcll(has_k[k] & in);
        if (n > 0 && n + n_in > MAX_LIST) { // all in the next one
            close(round);
            round++;
            fill(octets, round * (4 * ROUND));
            if (round <= MAX_ROUNDS) none |= (round * (4 * ROUND) - octets) << (FILL_BITS * (round - 1));
            o += round * (4 * ROUND) - octets;
            octets = round * (4 * ROUND);
            now_in = true;
            in = some;
            n = 0;
            n_in = all;
        }
        const uint32_t next = (first + n + n_in + 3u) & ~3u;
        uint32_t i = now_in ? first + n + before : next + before - n_in, e = 0;
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (bits >> k & 1) {
                e = (now[k / 2] >> (k & 1 ? 16 : 0)) << 16 | (o / 4 % ROUND * (uint32_t)rows * 1024u + (o & 3u) * 256u + (uint32_t)(lane & 15) * 16u + (uint32_t)k * 2u);
                entries[i++] = e;
            }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t of = __shfl(place, 16 * i), at = octets + __popc(used & ((1u << i) - 1u));
            if (used >> i & 1) {
                if (at == 0) first_place = of;
                if (lane == (int)(at / 4)) places |= of << (8 * (at & 3));
            }
        }
        octets += __popc(used);
        n += n_in;
        if (in) last = __shfl(e, 63 - __clzll((long long)in));
        if (octets / (4 * ROUND) != round) {
            close(round);
            n = all - n_in;
            if (n) last = __shfl(e, 63 - __clzll((long long)some));
        }
    }
    if (octets % (4 * ROUND)) {
        const uint32_t round = octets / (4 * ROUND);
        close(round);
        if (round < MAX_ROUNDS) none |= (4 * ROUND - octets % (4 * ROUND)) << (FILL_BITS * round);
    }
    no_slot = __any(no_slot);
    uint32_t *const to = table + (long)br * (2 * MAX_PAIRS);
    fill(octets, ~0u);
    if (lane < MAX_PAIRS) to[2 * lane] = places, to[2 * lane + 1] = list;
    if (lane == 0) {
        const uint32_t steps = min((octets + 3) / 4, (uint32_t)MAX_PAIRS);
        table[(long)mb * (2 * MAX_PAIRS) + br] = 2 * steps | none << 8;
        if (no_slot || longest > MAX_LIST || steps > (uint32_t)held || octets > 4 * MAX_PAIRS) atomicMax(most, max(longest, 1u)); // not for the windows
    }
}

// ---- the product ----

// Column c < 16 TN of a part's copy lies so many columns behind the panel's first, n0 < N.  Past N, where nothing is stored, the panel's first stands
// in: a whole part may lie past N (panels of two tiles and two parts, N % 64 = 8), so its own first column need not be one of B.
template <int TN, int PARTS>
__host__ __device__ __forceinline__ int copied_column(int n0, int part, int c, int N)
{
    constexpr int P = 16 * TN, PANEL = P * PARTS;
    const int col = part * (P / 4) + c / (P / 4) * (PANEL / 4) + c % (P / 4);
    return n0 + col < N ? col : 0;
}

// Waits until at most n of the wavefront's vector memory operations are under way (they end in order), or a few less.
__device__ __forceinline__ void wait_vector_memory(int n)
{
    if (n < 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (n < 4) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    else if (n < 6) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else if (n < 10) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if (n < 14) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(14)" ::: "memory");
}

template <int TN, int PARTS, bool C_F32, bool ENTRIES>
__global__ __launch_bounds__(1024) void spmm_window_kernel(const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr,
                                                           const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ B, void *__restrict__ Cout,
                                                           const int32_t *__restrict__ window, const int32_t *__restrict__ count,
                                                           const uint32_t *__restrict__ slot, const uint32_t *__restrict__ entries, int mb, int rows, int cap, int n_groups, int n_panels,
                                                           int panels_per_unit, int N, long K)
{
    constexpr int NP = pairs_held<TN>, U = TN == 4 ? 1 : 2, TILES = TN * PARTS;
    constexpr int P = 16 * TN, PANEL = P * PARTS, QUAD_BYTES = P * 128; // four blocks of a window: [column][8 pieces of 8 k]
    extern __shared__ __align__(16) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // An XCD takes an eighth of the groups, its workgroups neighbouring ones at a time, all at the same panel, so that what their
    // windows share is in its L2.  Unit: a run of panels of a group.  A panel is taken in parts, which hold the columns
    // PANEL / 4 * a + P / 4 * part + r with r < P / 4 and a < 4, so that a lane has 4 TILES consecutive columns of C in the end.
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3;
    const int group0 = (int)((long)n_groups * xcd / 8), my_groups = (int)((long)n_groups * (xcd + 1) / 8) - group0;
    const int my_units = my_groups * ((n_panels + panels_per_unit - 1) / panels_per_unit);
    struct Unit {
        int unit, group, end; // its panels: end - panels_per_unit .. min(end, n_panels) - 1
    };
    auto unit_after = [&](Unit p) {
        p.unit += per_xcd;
        p.group += per_xcd;
        while (p.group >= group0 + my_groups && p.unit < my_units) p.group -= my_groups, p.end += panels_per_unit;
        return p;
    };
    auto is_last = [&](const Unit &p, int panel) { return panel + 1 == p.end || panel + 1 == n_panels; };
    Unit here_unit{(int)(blockIdx.x >> 3) - per_xcd, group0 + (int)(blockIdx.x >> 3) - per_xcd, panels_per_unit};
    here_unit = unit_after(here_unit);
    if (here_unit.unit >= my_units) return;
    const int i16 = lane & 15, g = lane >> 4, sel = g >> 1, kh = g & 1;

    const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)lds;
    const uint32_t buffer = ENTRIES ? (uint32_t)max(cap * (P * 32), rows * (ROUND * 1024)) : (uint32_t)cap * (P * 32);
    // Piece o of column c of a quad lies at place o ^ swizzle(c) of its 128 bytes: the 16 columns that an operand takes lie in different banks.
    auto swizzle = [](uint32_t c) { return ((c >> 1) & 1u) | ((c / (P / 4)) & 3u) << 1; };
    // the lane, for addresses that are made anew where they are used instead of being kept in registers
    auto lane_here = [&] {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    // Loads that the compiler does not know of: what they bring may be used after the next meet().
    auto load_dword = [](uint32_t &x, const void *base, uint32_t at) { asm volatile("global_load_dword %0, %1, %2" : "+v"(x) : "v"(at), "s"(base)); };

    // The block row of a wavefront in a group: what is asked for, and what is made of it.
    struct Asked {
        int p0, blocks;
        uint32_t q0, q1, c0, c1; // lane j: blocks 2 j and 2 j + 1; ENTRIES: the places of step j in q0, the list of round j in q1
    };
    struct Row {
        int p0, blocks;  // blocks: 0 where the wavefront has none; ENTRIES: twice the steps
        uint32_t packed; // lane j: places of blocks 2 j and 2 j + 1 in the window, in 32 bytes; ENTRIES: of the octets of step j, 8 bits each
        bool known;
        uint32_t none;   // ENTRIES: places of round k that are no octets, FILL_BITS each
    };
    uint32_t list = 0; // ENTRIES: of the row taken last, lane j: the list of round j
    auto ask_row = [&](int gr, Asked &r) {
        const int br = gr * rows + wave, b = br < mb ? br : mb - 1;
        if constexpr (ENTRIES) { // a table of MAX_PAIRS pairs a block row, and twice the steps of every row behind it
            r.p0 = 0;
            r.blocks = br < mb ? __builtin_amdgcn_readfirstlane(row_ptr[b]) : 0;
            const uint32_t at = (uint32_t)min(lane_here(), MAX_PAIRS - 1) * 8u;
            load_dword(r.q0, slot + (long)b * (2 * MAX_PAIRS), at);
            load_dword(r.q1, slot + (long)b * (2 * MAX_PAIRS), at + 4u);
            return;
        }
        r.p0 = __builtin_amdgcn_readfirstlane(row_ptr[b]);
        r.blocks = br < mb ? __builtin_amdgcn_readfirstlane(row_ptr[b + 1]) - r.p0 : 0;
        if (r.blocks <= 0) r.blocks = 0, r.p0 = 0;
        const int l = lane_here(), last = r.blocks > 0 ? r.blocks - 1 : 0;
        const uint32_t a0 = (uint32_t)min(2 * l, last) * 4u, a1 = (uint32_t)min(2 * l + 1, last) * 4u;
        load_dword(r.q0, slot + r.p0, a0);
        load_dword(r.q1, slot + r.p0, a1);
        load_dword(r.c0, col_idx + r.p0, a0);
        load_dword(r.c1, col_idx + r.p0, a1);
    };
    auto place = [&](uint32_t q) { return (q & ((1u << SLOT_BITS) - 1u)) / 4 * (QUAD_BYTES / 32) + (q & 3u); };
    auto take_row = [&](Asked &r) {
        if constexpr (ENTRIES) {
            asm volatile("" : "+v"(r.q0), "+v"(r.q1));
            list = r.q1;
            return Row{0, r.blocks & 0xff, r.q0, true, (uint32_t)r.blocks >> 8};
        }
        asm volatile("" : "+v"(r.q0), "+v"(r.q1), "+v"(r.c0), "+v"(r.c1));
        const bool same = (r.q0 >> SLOT_BITS) * 16u == r.c0 && (r.q1 >> SLOT_BITS) * 16u == r.c1;
        return Row{r.p0, r.blocks, place(r.q0) | place(r.q1) << 16, r.blocks <= 2 * NP && (r.blocks == 0 || __all(same)), 0};
    };
    f16x8 a[NP];
#pragma unroll
    for (int d = 0; d < NP; d++) a[d] = (f16x8){0, 0, 0, 0, 0, 0, 0, 0};
    // Pair d of a row to a[d] where d < n: through a buffer that ends with the row, so that what is past its end is zero.
    // ENTRIES: the entries of round d, four a lane, until build_a makes operands of them.
    const uint32_t a_off = (uint32_t)(sel * 512 + i16 * 32 + kh * 16);
    auto load_a = [&](int d, const Row &r, int n) {
        if constexpr (ENTRIES) {
            // lanes past the list read past the end of the buffer: zeros, and no traffic
            const uint32_t part_of = (uint32_t)__builtin_amdgcn_readlane((int)list, d);
            const uint32_t l = (uint32_t)lane_here();
            const uint32_t at = l < part_of >> LIST_BITS ? (part_of + l) << (32 - LIST_BITS) >> (32 - LIST_BITS - 4) : ~0u;
            i32x4 all;
            all[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)entries);
            all[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uintptr_t)entries >> 32) & 0xffff);
            all[2] = (int)(16u << LIST_BITS);
            all[3] = 0x00020000;
            asm volatile("s_cmp_le_i32 %3, %4\n\ts_cbranch_scc1 .Lskip%=\n\tbuffer_load_dwordx4 %0, %1, %2, 0 offen\n.Lskip%=:"
                         : "+v"(a[d])
                         : "v"(at), "s"(all), "s"(n), "n"(d)
                         : "scc");
            return;
        }
        i32x4 row;
        const uint64_t base = (uint64_t)(uintptr_t)(vals + (long)r.p0 * 256);
        row[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)base);
        row[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32) & 0xffff);
        row[2] = __builtin_amdgcn_readfirstlane(min(r.blocks, 2 * NP) * 512);
        row[3] = 0x00020000;
        uint32_t tmp;
        asm volatile("s_cmp_le_i32 %4, %5\n\ts_cbranch_scc1 .Lskip%=\n\tv_add_u32 %1, %6, %2\n\t"
                     "buffer_load_dwordx4 %0, %1, %3, 0 offen\n.Lskip%=:"
                     : "+v"(a[d]), "=&v"(tmp)
                     : "v"(a_off), "s"(row), "s"(n), "n"(d), "s"(d * 1024)
                     : "scc");
    };
    // ENTRIES: the operands of the row from its entries, a round after the other, the last one first (the entries of the others lie in front of
    // its operands), through ROUND KiB of LDS that this wavefront's next copies will overwrite.
    auto build_a = [&](const Row &r, uint32_t tile) {
        typedef __attribute__((address_space(3))) uint16_t lds_half;
        typedef __attribute__((address_space(3))) u32x4 lds_quad;
        const uint32_t mine = tile + (uint32_t)lane_here() * 16u;
#pragma unroll
        for (int k = MAX_ROUNDS - 1; k >= 0; k--) {
            if (k * ROUND < NP && 2 * k * ROUND < r.blocks) {
                const uint32_t fours = (uint32_t)__builtin_amdgcn_readlane((int)list, k) >> LIST_BITS;
                const u32x4 e = __builtin_bit_cast(u32x4, a[k]);
#pragma unroll
                for (int j = 0; j < ROUND; j++)
                    if (k * ROUND + j < NP) *(lds_quad *)(uintptr_t)(mine + (uint32_t)(j * rows * 1024)) = (u32x4){0u, 0u, 0u, 0u};
                asm volatile("" ::: "memory");
                if ((uint32_t)lane_here() < fours) {
                    uint32_t x[4] = {e[0], e[1], e[2], e[3]};
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        uint32_t to;
                        asm("v_mad_u32_u16 %0, %1, 1, %2" : "=v"(to) : "v"(x[i]), "s"(tile)); // its low half
                        *(lds_half *)(uintptr_t)to = (uint16_t)(x[i] >> 16);
                    }
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < ROUND; j++)
                    if (k * ROUND + j < NP) a[k * ROUND + j < NP ? k * ROUND + j : 0] = __builtin_bit_cast(f16x8, *(lds_quad *)(uintptr_t)(mine + (uint32_t)(j * rows * 1024)));
                asm volatile("" ::: "memory");
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    // what is loaded: pairs, a multiple of U, the last ones zeros, or rounds
    auto loads_of = [&](const Row &r) { return ENTRIES ? (r.blocks + 2 * ROUND - 1) / (2 * ROUND) : min(((r.blocks + 1) / 2 + U - 1) / U * U, NP); };
    constexpr int LOADS = ENTRIES ? (NP + ROUND - 1) / ROUND : NP;
    auto wait_a = [&](int younger) {
        wait_vector_memory(younger);
#pragma unroll
        for (int d = 0; d < NP; d++) asm volatile("" : "+v"(a[d]));
    };
    // A copy instruction brings 8 columns x 128 bytes, part wave % (P / 8) of quads wave / (P / 8), + quads_apart, ...
    const int copy_part = wave % (P / 8), copy_quad = wave / (P / 8), quads_apart = rows / (P / 8);
    auto copy_col = [&](int lane) { return (uint32_t)(8 * copy_part + (lane >> 3)); };
    uint32_t from_k[COPIES] = {};
    int quads;
    auto ask_window = [&](int gr) {
        const int lane = lane_here();
        quads = __builtin_amdgcn_readfirstlane(count[gr]) >> 2;
        const uint32_t piece = (uint32_t)(lane & 7) ^ swizzle(copy_col(lane));
#pragma unroll
        for (int t = 0; t < COPIES; t++) {
            const int q = max(min(copy_quad + t * quads_apart, quads - 1), 0); // a group without blocks has none: what is there is not used
            load_dword(from_k[t], window + (long)gr * cap + q * 4, (piece >> 1) * 4u);
        }
    };
    auto take_window = [&] {
#pragma unroll
        for (int t = 0; t < COPIES; t++) asm volatile("" : "+v"(from_k[t]));
    };
    // a part's columns of the window to LDS; returns the instructions
    auto stage = [&](int pan, int part, uint32_t dst) {
        const int n0 = pan * PANEL;
        const uint64_t base = (uint64_t)(uintptr_t)(B + (long)n0 * K);
        const int lane = lane_here();
        const uint32_t c = copy_col(lane);
        const uint32_t from = (uint32_t)copied_column<TN, PARTS>(n0, part, (int)c, N) * (uint32_t)K * 2u + 16u * (((uint32_t)lane ^ swizzle(c)) & 1u);
        int n = 0;
#pragma unroll
        for (int t = 0; t < COPIES; t++) {
            const int q = copy_quad + t * quads_apart;
            if (q < quads) {
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(from + 2u * from_k[t]), "s"(base),
                             "s"(dst + (uint32_t)(q * QUAD_BYTES) + (uint32_t)copy_part * 1024u)
                             : "memory");
                n++;
            }
        }
        return n;
    };

    const uint32_t c0 = (uint32_t)ncol_of<TN>(0, i16); // tile t: 4 t columns on
    const uint32_t at = ENTRIES ? swizzle(c0) * 16u : c0 * 128u + (((uint32_t)kh ^ swizzle(c0)) * 16u);
    const uint32_t half = ENTRIES ? (uint32_t)g * 8 : (uint32_t)sel * 16; // of what readlane brings, the lane's first bit
    const f16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    f32x4 acc[TILES];
    Row row, next;
    int panel = here_unit.end - panels_per_unit;
    uint32_t buf = 0; // of the part that is multiplied next
    // The part's product from LDS; RELOAD: the pairs of the next row follow into a[] as its own are done with.
    auto multiply = [&](auto part, auto reload, int n_reload) {
        constexpr int T0 = decltype(part)::value * TN;
        constexpr bool RELOAD = decltype(reload)::value;
#pragma unroll
        for (int t = 0; t < TN; t++) acc[T0 + t] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (!row.known) { // the pattern is not the one that the windows were made of: operands from memory
            const int n0 = panel * PANEL + decltype(part)::value * (P / 4);
            const int lane = lane_here(), i16 = lane & 15, g = lane >> 4, sel = g >> 1, kh = g & 1;
            for (int j = 0; j < row.blocks; j += 2) {
                const bool live = j + sel < row.blocks;
                const int p = row.p0 + (live ? j + sel : j);
                const f16x8 av = live ? load_f16x8(vals + (long)p * 256 + i16 * 16 + kh * 8) : zero8;
                const long k = (long)col_idx[p] + kh * 8;
#pragma unroll
                for (int t = 0; t < TN; t++) {
                    const int n = n0 + (i16 >> 2) * (PANEL / 4) + 4 * t + (i16 & 3);
                    const f16x8 bv = live ? load_f16x8(B + (long)(n < N ? n : 0) * K + k) : zero8;
                    acc[T0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv, av, acc[T0 + t], 0, 0, 0);
                }
            }
        }
        const int blocks = row.known ? row.blocks : 0;
        const uint32_t b_at = lbase + buf + (ENTRIES ? c0 * 128u : 0u);
#pragma unroll
        for (int d0 = 0; d0 < NP; d0 += U) { // the operands of U pairs at a time
            if (2 * d0 < blocks) {
                f16x8 bv[U][TN];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (d0 + u >= NP) continue;
                    const uint32_t four = (uint32_t)__builtin_amdgcn_readlane((int)row.packed, d0 + u);
                    uint32_t b;
                    if constexpr (ENTRIES) { // octets lie in 16 bytes, 8 to a quad
                        b = ((__builtin_amdgcn_ubfe(four, half, 8) << 4) ^ at) + b_at;
                        b += __umul24(__builtin_amdgcn_ubfe(four, half + 3, 5), (uint32_t)QUAD_BYTES - 128u);
                    } else {
                        b = ((__builtin_amdgcn_ubfe(four, half, 16) << 5) ^ at) + b_at;
                    }
#pragma unroll
                    for (int t = 0; t < TN; t++) bv[u][t] = *(const __attribute__((address_space(3))) f16x8 *)(uintptr_t)(b + t * 512);
                }
                if constexpr (ENTRIES) // places that are no octets: zeros times zeros, whatever B holds under the octet that they name (64^3, N = 64 32.3 -> 32.6 us)
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        constexpr int LAST = 4 * (ROUND - 1);
                        const int j = (d0 + u) % ROUND, none = (int)(row.none >> (FILL_BITS * ((d0 + u) / ROUND)) & ((1u << FILL_BITS) - 1u));
                        if (d0 + u < NP && none > LAST - 4 * j) {
                            const bool octet = (lane_here() >> 4) + 4 * j < 4 * ROUND - none;
#pragma unroll
                            for (int t = 0; t < TN; t++) bv[u][t] = octet ? bv[u][t] : zero8;
                        }
                    }
                if (!ENTRIES && 2 * (d0 + U) > blocks) { // what is past the end of the row: zeros times zeros
                    const int sel = lane_here() >> 5;
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int t = 0; t < TN; t++) bv[u][t] = 2 * (d0 + u) + sel < blocks ? bv[u][t] : zero8;
                }
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int t = 0; t < TN; t++)
                        if (d0 + u < NP) acc[T0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[u][t], a[d0 + u < NP ? d0 + u : 0], acc[T0 + t], 0, 0, 0);
            }
            if constexpr (RELOAD)
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (d0 + u < LOADS) load_a(d0 + u < LOADS ? d0 + u : 0, next, n_reload);
        }
    };
    // Everybody has left the part's buffer, and the next part's copies, which all but `younger` operations are older than, have landed.
    auto meet = [&](int younger) {
        wait_vector_memory(younger);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        buf ^= buffer;
    };

    Asked asked{};
    ask_window(here_unit.group);
    ask_row(here_unit.group, asked);
    wait_vector_memory(0);
    take_window();
    row = next = take_row(asked);
    stage(panel, 0, lbase);
#pragma unroll
    for (int d = 0; d < LOADS; d++) load_a(d, row, loads_of(row));
    const uint32_t tile = lbase + (uint32_t)(copy_quad * QUAD_BYTES + copy_part * 1024); // of build_a, in either half
    if constexpr (ENTRIES) {
        wait_a(0);
        build_a(row, tile + buffer);
    }
    Unit soon = unit_after(here_unit);
    bool loaded = !ENTRIES, ahead = false; // a[] is under way; the row of the unit after next is
    if (PARTS == 1 && is_last(here_unit, panel) && soon.unit < my_units) {
        ask_window(soon.group);
        ask_row(soon.group, asked);
        ahead = true;
    }
    wait_vector_memory(0);
    if (ahead) {
        take_window();
        next = take_row(asked);
        ahead = false;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // A part's copies, and the operands of the row, where they are new: ENTRIES makes them in the place of its first copies.
    int stored = 0; // stores that are younger than the loads of the row
    auto stage_and_take_a = [&](int pan, int part, bool copy) {
        const uint32_t to = buf ^ buffer;
        if (ENTRIES && loaded) {
            wait_a(stored);
            build_a(row, tile + to);
        }
        const int copies = copy ? stage(pan, part, lbase + to) : 0;
        if (!ENTRIES && loaded) wait_a(copies);
    };
    for (;;) { // a panel
        const bool last = is_last(here_unit, panel), more = !last || soon.unit < my_units;
        if constexpr (PARTS == 2) {
            stage_and_take_a(panel, 1, true);
            if (last && more) { // the unit's last copies are on their way: the window and the row of the next
                ask_window(soon.group);
                ask_row(soon.group, asked);
            }
            multiply(std::integral_constant<int, 0>(), std::false_type(), 0);
            meet(0);
            loaded = false;
            if (last && more) {
                take_window();
                next = take_row(asked);
            }
        }
        const int staged = last ? soon.end - panels_per_unit : panel + 1;
        stage_and_take_a(staged, 0, more);
        if (PARTS == 1 && ahead) {
            next = take_row(asked);
            ahead = false;
        }
        loaded = last && more;
        if (PARTS == 1 && more && is_last(last ? soon : here_unit, staged)) {
            const Unit later = last ? unit_after(soon) : soon;
            ahead = later.unit < my_units;
            if (ahead) {
                ask_window(later.group);
                ask_row(later.group, asked);
            }
        }
        const int reload = loaded ? loads_of(next) : 0;
        if (loaded) multiply(std::integral_constant<int, PARTS - 1>(), std::true_type(), reload);
        else multiply(std::integral_constant<int, PARTS - 1>(), std::false_type(), 0);
        asm volatile("" ::: "memory");
        const int br = here_unit.group * rows + wave, n0 = panel * PANEL;
        if (br < mb) {
            const int l = lane_here();
            store_tile<TILES, C_F32>(acc, br, -1, n0, l & 15, l >> 4, Cout, nullptr, N);
        }
        asm volatile("" ::: "memory");
        if (!more) break;
        // store instructions: at least so many where no column is past N
        constexpr int STORES = C_F32 ? TILES : (TILES + 1) / 2;
        stored = br < mb && n0 + PANEL <= N ? STORES : 0;
        meet(reload + stored);
        if (last) {
            row = next;
            here_unit = soon;
            soon = unit_after(soon);
            panel = staged;
        } else panel++;
        if (ahead) take_window();
    }
}

int g_force_rows = 0, g_force_tiles = 0; // test hook
std::atomic<int64_t> g_launches{0};      // test hook

size_t lds_of(int rows, int cap, int tiles, bool entries) { return 2 * std::max((size_t)cap * tiles * 512, entries ? (size_t)rows * (ROUND * 1024) : 0); }
// Whether windows of `cap` block columns fit: twice in LDS, and COPIES KiB a wavefront.
bool fits(int rows, int cap, int tiles, bool entries)
{
    return (entries ? cap <= MAX_LISTED : cap < 1 << SLOT_BITS) && rows % (2 * tiles) == 0 && (size_t)cap * tiles * 512 <= (size_t)COPIES * 1024 * rows &&
           lds_of(rows, cap, tiles, entries) <= MAX_LDS;
}
// Parts of a panel: two where N is wider than one.
int parts_of(int tiles, size_t N) { return tiles < 4 && N > (size_t)16 * tiles ? 2 : 1; }

struct Launch {
    int n_panels, panels_per_unit, workgroups, rounds;
};
// The panels of a group are split into the units that leave the last round of workgroups fullest; half a panel more for every unit,
// whose A is read again.
Launch launch_of(int rows, int cap, int tiles, int n_groups, size_t N, bool entries)
{
    const size_t panel = (size_t)16 * tiles * parts_of(tiles, N);
    Launch l{(int)((N + panel - 1) / panel), 0, 0, 0};
    const int slots = 32 * std::max(1, std::min(CU_WAVES / rows, (int)(MAX_LDS / lds_of(rows, cap, tiles, entries)))); // workgroups of an XCD at a time
    const int my_groups = (n_groups + 7) / 8;
    double best = 1e30;
    for (int split = 1; split <= std::min(l.n_panels, 64); split++) {
        const int per = (l.n_panels + split - 1) / split, units = my_groups * ((l.n_panels + per - 1) / per), rounds = (units + slots - 1) / slots;
        if ((double)rounds * (per + 0.5) >= best) continue;
        best = (double)rounds * (per + 0.5);
        l.panels_per_unit = per; l.rounds = rounds; l.workgroups = 8 * std::min(slots, units);
    }
    return l;
}

// The kernel may have as much LDS as there is: said once on a device, when a plan is made, so that a captured launch says nothing.
template <int TN, int PARTS, bool C_F32, bool ENTRIES>
hipError_t prepare()
{
    static std::atomic<uint64_t> prepared{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || (dev < 64 && prepared.load(std::memory_order_relaxed) >> dev & 1)) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(spmm_window_kernel<TN, PARTS, C_F32, ENTRIES>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MAX_LDS);
    if (e == hipSuccess && dev < 64) prepared.fetch_or(1ull << dev, std::memory_order_relaxed);
    return e;
}
template <bool ENTRIES>
hipError_t prepare_all()
{
    for (auto f : {prepare<1, 1, false, ENTRIES>, prepare<1, 1, true, ENTRIES>, prepare<1, 2, false, ENTRIES>, prepare<1, 2, true, ENTRIES>, prepare<2, 1, false, ENTRIES>,
                   prepare<2, 1, true, ENTRIES>, prepare<2, 2, false, ENTRIES>, prepare<2, 2, true, ENTRIES>, prepare<4, 1, false, ENTRIES>, prepare<4, 1, true, ENTRIES>}) {
        const hipError_t e = f();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int TN, int PARTS, bool C_F32, bool ENTRIES>
hipError_t launch_as(const SpmmArgs &a, const WindowPlan &p, const WindowLaunch &l, hipStream_t st)
{
    const size_t lds = lds_of(p.rows, p.cap, TN, ENTRIES);
    const hipError_t e = prepare<TN, PARTS, C_F32, ENTRIES>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((spmm_window_kernel<TN, PARTS, C_F32, ENTRIES>), dim3((unsigned)l.workgroups), dim3((unsigned)(p.rows * 64)), lds, st, a.vals, ENTRIES ? p.d_blocks : a.row_ptr, a.col_idx, a.B,
                       a.C, p.d_window, p.d_count, ENTRIES ? p.d_table : p.d_slot, p.d_entries, (int)(a.M / 16), p.rows, p.cap, p.n_groups, l.n_panels, l.panels_per_unit, (int)a.N, (long)a.K);
    return hipGetLastError();
}

double least_us(bool entries) { return entries ? 4.7 : 5.5; } // of a product, as estimated

int best_tiles(const WindowPlan &p, const WindowProduct &w, double *us)
{
    int tiles = 0;
    *us = 1e30;
    for (int t : {1, 2, 4}) {
        const double e = window_estimate_us(p.rows, p.cap, p.sum, t, w);
        if (e < *us) *us = e, tiles = t;
    }
    return g_force_tiles && tiles ? g_force_tiles : tiles;
}

} // namespace

// Time of a product, from the steps that a workgroup takes one after the other (1.07 us and 0.0155 per block of a row and tile of
// 16 columns), the bytes that a compute unit's memory path moves (copies of windows, A once a unit, C: 8.7 TB/s on all), those
// that come from memory (5 TB/s), whichever is longest, and the start (1.6 us, and up to 2.2 for groups of 16).  Fitted to 311 products of 41 bands, stencils
// and pruned matrices, N = 8 to 1,000, three on their own inputs in turn: 10 % standard deviation, and the group and panel it picks are
// 4 % from the best in the mean; never below 5.5 us (4.6 to 5.5 measured), for the row-wise kernel is as fast there.  Estimate (measured), us: stencil 73 x 61 x 62, N = 88, groups of 8 80 (85); band of 52960 and 64, N = 472,
// groups of 16 34 (34.5); band of 2144 and 47, N = 808, groups of 4 5.5 (5.6).
// ENTRIES: the building of the operands besides, for every unit; fitted to 186 products of 39 stencils, N = 8 to 256: 8 %.  66 x 31 x 43,
// N = 120 25 (26); 41 x 35 x 30, N = 208 20.6 (21.1); 72 x 51 x 40, N = 144 48 (56).
double window_estimate_us(int rows, int cap, unsigned long long sum, int tiles, const WindowProduct &w)
{
    const bool entries = w.nnz >= 0;
    if (!fits(rows, cap, tiles, entries) || w.most_blocks > 2 * (tiles == 4 ? pairs_held<4> : pairs_held<1>)) return 1e30;
    const size_t mb = w.M / 16;
    const Launch l = launch_of(rows, cap, tiles, (int)((mb + rows - 1) / rows), w.N, entries);
    const double parts = parts_of(tiles, w.N), units = (l.n_panels + l.panels_per_unit - 1) / l.panels_per_unit;
    const double c_bytes = (double)w.M * (double)w.N * (w.c_f32 ? 4.0 : 2.0), a_bytes = entries ? 4.0 * (double)w.nnz + 12.0 * (double)w.nnzb : 512.0 * (double)w.nnzb;
    const double blocks = (double)w.nnzb / (double)mb * tiles, groups16 = rows / 16.0, copies = (double)sum * 512.0 * tiles * parts * l.n_panels + a_bytes * units + c_bytes;
    const double once = a_bytes + 2.0 * (double)w.K * (double)w.N + c_bytes;
    double steps, path, memory, start;
    if (entries) {
        steps = l.rounds * (l.panels_per_unit * parts * (0.96 + 0.014 * blocks) + 2.3 * groups16);
        path = copies / 11.9e6, memory = once / 2.7e6, start = 2.75;
    } else {
        steps = l.rounds * l.panels_per_unit * parts * (1.07 + 0.0155 * blocks);
        path = copies / 8.7e6, memory = once / 5.0e6, start = 1.6 + 2.2 * groups16;
    }
    return std::max(least_us(entries), start + std::pow(std::pow(steps, 4.0) + std::pow(path, 4.0) + std::pow(memory, 4.0), 0.25));
}

bool WindowCount::launch(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, void *to)
{
    const int words = (int)((kb + 31) / 32);
    if (nnzb == 0 || kb > (size_t)BITMAP_WORDS * 32) return false;
    static_assert(PARTS * WINDOW_SIZES * sizeof(uint2) == BYTES, "");
    hipLaunchKernelGGL(window_count_kernel, dim3(PARTS, WINDOW_SIZES), dim3(256), (size_t)words * 4, nullptr, row_ptr, col_idx, (int)mb, words, (uint2 *)to);
    return hipGetLastError() == hipSuccess;
}

void WindowCount::take(const void *from)
{
    const uint2 *of = static_cast<const uint2 *>(from);
    widths = WindowWidths{};
    for (int s = 0; s < WINDOW_SIZES; s++)
        for (int i = 0; i < PARTS; i++) {
            widths.most[s] = std::max(widths.most[s], of[s * PARTS + i].x);
            widths.sum[s] += of[s * PARTS + i].y;
        }
    there = true;
}

void WindowCount::begin(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb)
{
    parts.release();
    begun = parts.alloc(BYTES) == hipSuccess && launch(row_ptr, col_idx, mb, kb, nnzb, parts.p);
}

hipError_t WindowCount::end(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb)
{
    if (there) return hipSuccess;
    widths = WindowWidths{}; // none known
    if (!begun) begin(row_ptr, col_idx, mb, kb, nnzb);
    there = true;
    if (!begun) return parts.p ? hipSuccess : hipErrorOutOfMemory;
    uint2 of[WINDOW_SIZES * PARTS];
    const hipError_t e = hipMemcpy(of, parts.p, sizeof of, hipMemcpyDeviceToHost);
    parts.idle = e == hipSuccess;
    if (e == hipSuccess) take(of);
    return e;
}

void WindowCount::on_host(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb)
{
    static_assert(SIZES[0] == 4 && SIZES[1] == 8 && SIZES[2] == 16, "groups of one size are halves of those of the next");
    widths = WindowWidths{};
    there = true;
    std::vector<uint32_t> seen(kb, 0); // the last block row that used the column, from 1
    uint32_t n[WINDOW_SIZES] = {};
    for (size_t r = 0; r < mb; r++) {
        for (int32_t q = row_ptr[r]; q < row_ptr[r + 1]; q++) {
            uint32_t &last = seen[(size_t)col_idx[q] / 16];
            const uint32_t apart = (last - 1) ^ (uint32_t)r; // below the size of a group where both rows are in one
            last = (uint32_t)r + 1;
            for (int s = 0; s < WINDOW_SIZES; s++) n[s] += apart >= (uint32_t)SIZES[s];
        }
        for (int s = 0; s < WINDOW_SIZES; s++)
            if ((r + 1) % SIZES[s] == 0 || r + 1 == mb) {
                widths.most[s] = std::max(widths.most[s], n[s]);
                widths.sum[s] += n[s];
                n[s] = 0;
            }
    }
}

double window_choose(const WindowWidths &widths, const WindowProduct &w, int *size)
{
    double best = 1e30;
    *size = -1;
    for (int i = 0; i < WINDOW_SIZES; i++) {
        if (widths.most[i] == 0 || (g_force_rows && SIZES[i] != g_force_rows)) continue;
        for (int t : {1, 2, 4}) {
            double e = window_estimate_us(SIZES[i], (int)((widths.most[i] + 3) / 4 * 4), widths.sum[i], t, w);
            // Nothing shared: the pieces that the copies bring are single blocks, 32 bytes of a column, and from a B beyond an XCD's 4 MiB of L2 each
            // costs a cache line (928 x 4160, 3 %, N = 3472: estimate 12, 27 us, row-wise 15; 1376 x 5344, 4 %, N = 896 9.8, 13.6 and 11.4;
            // 12656 x 832, 6 %, N = 352 11.4 -> 8.4 all the same).
            if ((double)widths.sum[i] > 0.75 * (double)w.nnzb) {
                if (2 * w.K * w.N > (size_t)4 << 20) continue;
                e *= 1.25;
            }
            if (e < best) best = e, *size = i;
        }
    }
    return best;
}

static void shape_of(WindowPlan &p, const WindowWidths &w, int size, size_t mb, size_t nnzb, int most_blocks)
{
    p.rows = SIZES[size];
    p.cap = (int)((w.most[size] + 3) / 4 * 4);
    p.sum = w.sum[size];
    p.share = (double)w.sum[size] / (double)nnzb;
    p.share4 = (double)w.sum[0] / (double)nnzb;
    p.most_blocks = most_blocks;
    p.n_groups = (int)((mb + p.rows - 1) / p.rows);
}

hipError_t window_build(const WindowWidths &w, int size, const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, int most_blocks, WindowPlan **out)
{
    *out = nullptr;
    WindowPlan *p = new (std::nothrow) WindowPlan();
    if (!p) return hipErrorOutOfMemory;
    const int words = (int)((kb + 31) / 32);
    shape_of(*p, w, size, mb, nnzb, most_blocks);
    hipError_t e = dev_malloc(&p->d_slot, nnzb * sizeof(uint32_t));
    if (e == hipSuccess) e = dev_malloc(&p->d_window, (size_t)p->n_groups * (p->cap + 1) * sizeof(int32_t));
    p->d_count = p->d_window + (size_t)p->n_groups * p->cap;
    if (e == hipSuccess) {
        hipLaunchKernelGGL(window_list_kernel, dim3((unsigned)p->n_groups), dim3(256), (size_t)words * 6, nullptr, row_ptr, col_idx, (int)mb, words, p->rows, p->cap,
                           p->d_window, p->d_count, p->d_slot);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = prepare_all<false>();
    if (e != hipSuccess) {
        window_destroy(p);
        return e;
    }
    *out = p;
    return hipSuccess;
}

hipError_t window_attach_entries(WindowPlan &p, const uint16_t *vals, const int32_t *row_ptr, const unsigned long long *offset, size_t mb, size_t nnzb, int64_t nnz,
                                 bool *taken)
{
    *taken = false;
    if (p.cap > MAX_LISTED) return hipSuccess;
    const size_t room = (size_t)nnz + 8 * ((nnzb + mb + 1) / 2 + MAX_PAIRS) + 16;
    if (room / 4 >= (size_t)1 << LIST_BITS) return hipSuccess;
    const size_t table = mb * (2 * MAX_PAIRS + 1);
    hipError_t e = dev_malloc(&p.d_entries, (room + table + 1) * sizeof(uint32_t));
    if (e != hipSuccess) return e;
    p.d_table = p.d_entries + (room + 1) / 2 * 2; // pairs of words
    p.d_blocks = reinterpret_cast<int32_t *>(p.d_table + mb * (2 * MAX_PAIRS));
    p.nnz = nnz;
    DevScratch most;
    uint32_t too_many = 0;
    e = most.alloc(sizeof too_many);
    if (e == hipSuccess) e = hipMemsetAsync(most.p, 0, sizeof too_many, nullptr);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(window_entries_kernel, dim3((unsigned)((mb + 3) / 4)), dim3(256), 0, nullptr, vals, row_ptr, p.d_slot, offset, (int)mb, p.rows,
                           p.most_blocks <= 2 * pairs_held<4> ? pairs_held<4> : MAX_PAIRS, p.d_entries, p.d_table,
                           (uint32_t *)most.p);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = prepare_all<true>();
    if (e == hipSuccess) e = hipMemcpy(&too_many, most.p, sizeof too_many, hipMemcpyDeviceToHost);
    most.idle = e == hipSuccess;
    *taken = e == hipSuccess && too_many == 0;
    return e;
}

void window_destroy(WindowPlan *p)
{
    if (!p) return;
    for (void *q : {(void *)p->d_window, (void *)p->d_slot, (void *)p->d_entries})
        if (q) (void)dev_free(q);
    delete p;
}

bool window_forced() { return g_force_rows > 0; }
bool window_takes_rows(int most_blocks) { return most_blocks > 0 && most_blocks <= 2 * pairs_held<1>; }

double window_least_us(const WindowPlan &p) { return least_us(p.d_entries != nullptr); }

static WindowLaunch work_out(const WindowPlan &p, const WindowProduct &w)
{
    WindowLaunch r;
    r.tiles = best_tiles(p, w, &r.us);
    if (!r.tiles || !fits(p.rows, p.cap, r.tiles, p.d_entries != nullptr)) return WindowLaunch();
    const Launch l = launch_of(p.rows, p.cap, r.tiles, p.n_groups, w.N, p.d_entries != nullptr);
    r.n_panels = l.n_panels; r.panels_per_unit = l.panels_per_unit; r.workgroups = l.workgroups; r.rounds = l.rounds;
    return r;
}
WindowLaunch window_launch_of(const WindowWidths &widths, int size, const WindowProduct &w, WindowPlan &shape)
{
    shape_of(shape, widths, size, w.M / 16, w.nnzb, w.most_blocks);
    return work_out(shape, w);
}
// Below 5.5 us, and where little is shared, the estimate above says little: here the start, the steps one after the other, their blocks, the copies, B and C, and the parts of the
// panels; copies of single blocks of a B beyond half an XCD's L2, a cache line for 32 bytes of it, cost twice.  Fitted to 3,474 launches of less than 16 us of every size of group and
// panel (240 bands, 200 stencils, 200 random patterns, N = 24 to 2,048): 6 % standard deviation, 15 for the estimate above.
double window_short_us(const WindowPlan &p, const WindowLaunch &l, size_t M, size_t K, size_t N, size_t nnzb)
{
    const double parts = parts_of(l.tiles, N), steps = (double)l.rounds * l.panels_per_unit * parts, b = 2e-6 * (double)K * (double)N, c = 2e-6 * (double)M * (double)N;
    const double copies = 512e-6 * (double)p.sum * l.tiles * parts * l.n_panels;
    return 2.28 + 2.1 * p.rows / 16.0 + steps * (0.356 + 0.0102 * (double)nnzb * 16.0 / (double)M * l.tiles) + 0.143 * (b + c) +
           copies * (p.share > 0.6 && b > 2.0 ? 0.133 : 0.0666) + 0.0153 * parts * l.n_panels;
}
void window_settle(WindowPlan &p, size_t M, size_t K, size_t N, size_t nnzb)
{
    p.n = N;
    for (bool c_f32 : {false, true}) p.own[c_f32] = work_out(p, WindowProduct{M, K, N, nnzb, p.nnz, p.most_blocks, c_f32});
}
WindowLaunch window_launch(const SpmmArgs &a, const WindowPlan &p)
{
    if (a.N == p.n && !g_force_tiles) return p.own[a.c_f32];
    return work_out(p, WindowProduct{a.M, a.K, a.N, a.nnzb, p.nnz, p.most_blocks, a.c_f32});
}

hipError_t launch_window(const SpmmArgs &a, const WindowPlan &p, const WindowLaunch &l, hipStream_t st)
{
    const bool entries = p.d_entries != nullptr;
    auto as = [&](auto tn, auto parts) {
        constexpr int TN = decltype(tn)::value, PARTS = decltype(parts)::value;
        if (entries) return a.c_f32 ? launch_as<TN, PARTS, true, true>(a, p, l, st) : launch_as<TN, PARTS, false, true>(a, p, l, st);
        return a.c_f32 ? launch_as<TN, PARTS, true, false>(a, p, l, st) : launch_as<TN, PARTS, false, false>(a, p, l, st);
    };
    using std::integral_constant;
    const integral_constant<int, 1> one;
    const integral_constant<int, 2> two;
    if (l.tiles == 0) return hipErrorInvalidValue;
    g_launches.fetch_add(1, std::memory_order_relaxed);
    const bool halves = parts_of(l.tiles, a.N) == 2;
    if (l.tiles == 4) return as(integral_constant<int, 4>(), one);
    if (l.tiles == 2) return halves ? as(two, two) : as(two, one);
    return halves ? as(one, two) : as(one, one);
}

} // namespace smat

// Test hook (not part of smat.h): groups of 4, 8 or 16 block rows and panels of 1, 2 or 4 tiles wherever they fit, whatever the
// estimates say (0 = the choice); rows = -1: no windows.
extern "C" void smat_internal_window_force(int rows, int tiles) { smat::g_force_rows = rows; smat::g_force_tiles = tiles; }
// Test hook (not part of smat.h): products that were multiplied from windows so far.
extern "C" int64_t smat_internal_window_launches(void) { return smat::g_launches.load(); }

// Test hook (not part of smat.h): the widths of windows, most and sum of each size, from device arrays and from host arrays.
extern "C" int smat_internal_window_widths(const int32_t *row_ptr, const int32_t *col_idx, const int32_t *row_ptr_host, const int32_t *col_idx_host, size_t mb, size_t kb,
                                           size_t nnzb, int64_t *out)
{
    smat::WindowCount device, host;
    const hipError_t e = device.end(row_ptr, col_idx, mb, kb, nnzb);
    host.on_host(row_ptr_host, col_idx_host, mb, kb);
    for (int i = 0; i < smat::WINDOW_SIZES; i++) {
        *out++ = device.widths.most[i], *out++ = (int64_t)device.widths.sum[i];
        *out++ = host.widths.most[i], *out++ = (int64_t)host.widths.sum[i];
    }
    return (int)e;
}

// Test hook (not part of smat.h): the column of B that column c of a part's copy brings, of panel `panel` with `tiles` tiles a part; -1: no such panel.
extern "C" int64_t smat_internal_window_copied_column(int tiles, int64_t N, int panel, int part, int c)
{
    using namespace smat;
    const int parts = parts_of(tiles, (size_t)N), n0 = panel * 16 * tiles * parts;
    if (n0 >= N || part >= parts || c >= 16 * tiles) return -1;
    if (tiles == 4) return n0 + copied_column<4, 1>(n0, part, c, (int)N);
    if (tiles == 2) return n0 + (parts == 2 ? copied_column<2, 2>(n0, part, c, (int)N) : copied_column<2, 1>(n0, part, c, (int)N));
    return n0 + (parts == 2 ? copied_column<1, 2>(n0, part, c, (int)N) : copied_column<1, 1>(n0, part, c, (int)N));
}
