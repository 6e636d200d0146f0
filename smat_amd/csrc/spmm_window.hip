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
// The order of the sums is that of the row-wise kernel (blocks of a row two by two from its first), the results have the same bits.
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

constexpr int COPIES = 7;               // KiB of a window that a wavefront copies at a time
constexpr int SLOT_BITS = 10;           // of a block's entry: its place in the window; above them its block column
constexpr int BITMAP_WORDS = 8192;      // block columns of the matrix / 32
constexpr size_t MAX_LDS = 160 * 1024;  // of a compute unit
constexpr int CU_WAVES = 16;            // wavefronts of 128 registers on a compute unit
constexpr int SIZES[WINDOW_SIZES] = {4, 8, 16}; // block rows of a group

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

// A workgroup takes every gridDim.x-th group of one size: additions to one word queue up at 12 ns each (with a workgroup a group
// 170 us for 16384 block rows).
__global__ __launch_bounds__(256) void window_count_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, int mb, int words,
                                                           WindowWidths *__restrict__ stat)
{
    extern __shared__ uint32_t bitmap[];
    __shared__ uint32_t part[4];
    const int rows = blockIdx.y == 0 ? SIZES[0] : blockIdx.y == 1 ? SIZES[1] : SIZES[2];
    uint32_t most = 0;
    unsigned long long sum = 0;
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
    if (threadIdx.x == 0 && most) {
        atomicMax(&stat->most[blockIdx.y], most);
        atomicAdd(&stat->sum[blockIdx.y], sum);
    }
}

// window[group * cap ..]: the first columns of the group's blocks, ascending, filled up to a multiple of 4; slot[p]: the place
// of block p's column in it.
__global__ __launch_bounds__(256) void window_list_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, int mb, int words,
                                                          int rows, int cap, int32_t *__restrict__ window, int32_t *__restrict__ count,
                                                          uint32_t *__restrict__ slot)
{
    extern __shared__ uint32_t bitmap[]; // words, and as many half words of ranks behind them
    uint16_t *const rank = reinterpret_cast<uint16_t *>(bitmap + words);
    __shared__ uint32_t part[256];
    const int first = (int)blockIdx.x * rows, last = min(first + rows, mb);
    mark_columns(bitmap, words, row_ptr, col_idx, first, last);
    const int per = (words + 255) / 256, w0 = min((int)threadIdx.x * per, words), w1 = min(w0 + per, words);
    uint32_t n = 0;
    for (int w = w0; w < w1; w++) n += __popc(bitmap[w]);
    part[threadIdx.x] = n;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int t = 0; t < 256; t++) {
        if (t < (int)threadIdx.x) before += part[t];
        all += part[t];
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
        slot[p] = 0xffffffffu;
        if (c < (uint32_t)words * 32u && !(col & 15))
            slot[p] = c << SLOT_BITS | min((uint32_t)rank[c >> 5] + __popc(bitmap[c >> 5] & ((1u << (c & 31)) - 1u)), (uint32_t)cap - 1u);
    }
}

// ---- the product ----

// Waits until at most n of the wavefront's vector memory operations are under way (they end in order).
__device__ __forceinline__ void wait_vector_memory(int n)
{
#define SMAT_WAIT(I) case I: asm volatile("s_waitcnt vmcnt(" #I ")" ::: "memory"); break;
    switch (n) {
        SMAT_WAIT(1) SMAT_WAIT(2) SMAT_WAIT(3) SMAT_WAIT(4) SMAT_WAIT(5) SMAT_WAIT(6) SMAT_WAIT(7) SMAT_WAIT(8) SMAT_WAIT(9) SMAT_WAIT(10)
        SMAT_WAIT(11) SMAT_WAIT(12) SMAT_WAIT(13) SMAT_WAIT(14) SMAT_WAIT(15) SMAT_WAIT(16) SMAT_WAIT(17) SMAT_WAIT(18) SMAT_WAIT(19)
        SMAT_WAIT(20) SMAT_WAIT(21) SMAT_WAIT(22)
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#undef SMAT_WAIT
}

// A workgroup goes through steps: a part of a panel (16 TN columns) of a group.  While it multiplies one from one half of its
// LDS, the window of the next is copied to the other half; the A operands of a wavefront's block row stay in its registers for all
// panels of a unit and are replaced, pair by pair, by those of the next unit's row as the last part is done with them.
//
// Bound by what a step costs beside its work: with 16 wavefronts on a compute unit (128 registers each) a step of the 27-point
// stencil on 48^3, N = 256 takes 3 us, of which copies alone would be 1.9 and LDS reads and MFMAs alone 1.9 (timed with the rest
// taken out), and the two overlap by half; on 64^3 at N = 64 the read of A, 185 MB, from HBM is as long (49 us for all its bytes at
// the rate of a copy).  Us, row-wise kernel -> windows, step by step: 48^3, N = 256 111 -> one workgroup a group and panel, window and A asked
// for and waited for in turn 88 -> steps, two halves of LDS, A kept for all panels 68 -> parts unrolled, loads counted instead of all
// waited for, 128 bytes of a row of C at a time 59; 64^3, N = 64 90 -> 62 -> 66 -> 56; band of 65536 and 20, N = 256 30 -> 21 -> 16 -> 15.
// What the panel width costs: 16 columns instead of 32 on 48^3 66, on 64^3 63; groups of 8 instead of 16 66 and 58.
//
// The row-wise kernel reads the pattern where it lies, so this one does: it compares the block columns with those its windows were
// made of and takes a row that has other ones from memory.
//
// block pairs of a row that a wavefront holds
template <int TN> constexpr int pairs_held = TN == 4 ? 12 : 17;

template <int TN, int PARTS, bool C_F32>
__global__ __launch_bounds__(1024) void spmm_window_kernel(const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr,
                                                           const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ B, void *__restrict__ Cout,
                                                           const int32_t *__restrict__ window, const int32_t *__restrict__ count,
                                                           const uint32_t *__restrict__ slot, int mb, int rows, int cap, int n_groups, int n_panels,
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
    const uint32_t buffer = (uint32_t)cap * (P * 32);
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
        uint32_t q0, q1, c0, c1; // lane j: blocks 2 j and 2 j + 1
    };
    struct Row {
        int p0, blocks;  // blocks: 0 where the wavefront has none
        uint32_t packed; // lane j: places of blocks 2 j and 2 j + 1 in the window, in 32 bytes
        bool known;
    };
    auto ask_row = [&](int gr, Asked &r) {
        const int br = gr * rows + wave, b = br < mb ? br : mb - 1;
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
        asm volatile("" : "+v"(r.q0), "+v"(r.q1), "+v"(r.c0), "+v"(r.c1));
        const bool same = (r.q0 >> SLOT_BITS) * 16u == r.c0 && (r.q1 >> SLOT_BITS) * 16u == r.c1;
        return Row{r.p0, r.blocks, place(r.q0) | place(r.q1) << 16, r.blocks <= 2 * NP && (r.blocks == 0 || __all(same))};
    };
    f16x8 a[NP];
#pragma unroll
    for (int d = 0; d < NP; d++) a[d] = (f16x8){0, 0, 0, 0, 0, 0, 0, 0};
    // Pair d of a row to a[d] where d < n: through a buffer that ends with the row, so that what is past its end is zero.
    const uint32_t a_off = (uint32_t)(sel * 512 + i16 * 32 + kh * 16);
    auto load_a = [&](int d, const Row &r, int n) {
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
    // pairs to load: a multiple of U, the last ones zeros
    auto loads_of = [&](const Row &r) { return min(((r.blocks + 1) / 2 + U - 1) / U * U, NP); };
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
            const int q = min(copy_quad + t * quads_apart, quads - 1);
            load_dword(from_k[t], window + (long)gr * cap + q * 4, (piece >> 1) * 4u);
        }
    };
    auto take_window = [&] {
#pragma unroll
        for (int t = 0; t < COPIES; t++) asm volatile("" : "+v"(from_k[t]));
    };
    // a part's columns of the window to LDS; returns the instructions
    auto stage = [&](int pan, int part, uint32_t dst) {
        const int n0 = pan * PANEL + part * (P / 4);
        const uint64_t base = (uint64_t)(uintptr_t)(B + (long)n0 * K);
        const int lane = lane_here();
        const uint32_t c = copy_col(lane), col = c / (P / 4) * (PANEL / 4) + c % (P / 4);
        const uint32_t from = (n0 + (int)col < N ? col : 0u) * (uint32_t)K * 2u // past N: not stored
                              + 16u * (((uint32_t)lane ^ swizzle(c)) & 1u);
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
    const uint32_t at = c0 * 128u + (((uint32_t)kh ^ swizzle(c0)) * 16u);
    const uint32_t half = (uint32_t)sel * 16;
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
        const uint32_t b_at = lbase + buf;
#pragma unroll
        for (int d0 = 0; d0 < NP; d0 += U) { // the operands of U pairs at a time
            if (2 * d0 < blocks) {
                f16x8 bv[U][TN];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (d0 + u >= NP) continue;
                    const uint32_t v = __builtin_amdgcn_ubfe((uint32_t)__builtin_amdgcn_readlane((int)row.packed, d0 + u), half, 16);
                    const uint32_t b = ((v << 5) ^ at) + b_at;
#pragma unroll
                    for (int t = 0; t < TN; t++) bv[u][t] = *(const __attribute__((address_space(3))) f16x8 *)(uintptr_t)(b + t * 512);
                }
                if (2 * (d0 + U) > blocks) { // what is past the end of the row: zeros times zeros
                    asm volatile("");
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
                    if (d0 + u < NP) load_a(d0 + u < NP ? d0 + u : 0, next, n_reload);
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
    for (int d = 0; d < NP; d++) load_a(d, row, loads_of(row));
    Unit soon = unit_after(here_unit);
    bool loaded = true, ahead = false; // a[] is under way; the row of the unit after next is
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
    for (;;) { // a panel
        const bool last = is_last(here_unit, panel), more = !last || soon.unit < my_units;
        if constexpr (PARTS == 2) {
            const int copies = stage(panel, 1, lbase + (buf ^ buffer));
            if (loaded) wait_a(copies);
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
        const int copies = more ? stage(staged, 0, lbase + (buf ^ buffer)) : 0;
        if (loaded) wait_a(copies);
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
        if (br < mb) store_tile<TILES, C_F32>(acc, br, -1, n0, i16, g, Cout, nullptr, N);
        asm volatile("" ::: "memory");
        if (!more) break;
        // store instructions: at least so many where no column is past N
        constexpr int STORES = C_F32 ? TILES : (TILES + 1) / 2;
        meet(reload + (br < mb && n0 + PANEL <= N ? STORES : 0));
        if (last) {
            row = next;
            here_unit = soon;
            soon = unit_after(soon);
            panel = staged;
        } else panel++;
        if (ahead) {
            take_window();
            next = take_row(asked);
            ahead = false;
        }
    }
}

int g_force_rows = 0, g_force_tiles = 0; // test hook

// Whether windows of `cap` block columns fit: twice in LDS, and COPIES KiB a wavefront.
bool fits(int rows, int cap, int tiles)
{
    const size_t part = (size_t)cap * tiles * 512;
    return cap < 1 << SLOT_BITS && rows % (2 * tiles) == 0 && part <= (size_t)COPIES * 1024 * rows && 2 * part <= MAX_LDS;
}
// Parts of a panel: two where N is wider than one.
int parts_of(int tiles, size_t N) { return tiles < 4 && N > (size_t)16 * tiles ? 2 : 1; }

struct Launch {
    int n_panels, panels_per_unit, workgroups, rounds;
};
// The panels of a group are split into the units that leave the last round of workgroups fullest; half a panel more for every unit,
// whose A is read again.
Launch launch_of(int rows, int cap, int tiles, int n_groups, size_t N)
{
    const size_t panel = (size_t)16 * tiles * parts_of(tiles, N);
    Launch l{(int)((N + panel - 1) / panel), 0, 0, 0};
    const int slots = 32 * std::max(1, std::min(CU_WAVES / rows, (int)(MAX_LDS / ((size_t)cap * tiles * 1024)))); // workgroups of an XCD at a time
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

template <int TN, int PARTS, bool C_F32>
hipError_t launch_as(const SpmmArgs &a, const WindowPlan &p, const Launch &l, hipStream_t st)
{
    static std::atomic<uint64_t> prepared{0}; // devices on which the kernel may have that much LDS
    const size_t lds = (size_t)p.cap * TN * 1024;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 64 || !(prepared.load(std::memory_order_relaxed) >> dev & 1)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(spmm_window_kernel<TN, PARTS, C_F32>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MAX_LDS);
        if (e != hipSuccess) return e;
        if (dev < 64) prepared.fetch_or(1ull << dev, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((spmm_window_kernel<TN, PARTS, C_F32>), dim3((unsigned)l.workgroups), dim3((unsigned)(p.rows * 64)), lds, st, a.vals, a.row_ptr, a.col_idx, a.B,
                       a.C, p.d_window, p.d_count, p.d_slot, (int)(a.M / 16), p.rows, p.cap, p.n_groups, l.n_panels, l.panels_per_unit, (int)a.N, (long)a.K);
    return hipGetLastError();
}

int best_tiles(const WindowPlan &p, size_t M, size_t K, size_t N, size_t nnzb, bool c_f32, double *us)
{
    int tiles = 0;
    *us = 1e30;
    for (int t : {1, 2, 4}) {
        const double e = window_estimate_us(p.rows, p.cap, p.sum, t, M, K, N, nnzb, p.most_blocks, c_f32);
        if (e < *us) *us = e, tiles = t;
    }
    return g_force_tiles && tiles ? g_force_tiles : tiles;
}

} // namespace

// Time of a product, from the steps that a workgroup takes one after the other (1.07 us and 0.0155 per block of a row and tile of
// 16 columns), the bytes that a compute unit's memory path moves (copies of windows, A once a unit, C: 8.7 TB/s on all), those
// that come from memory (5 TB/s), whichever is longest, and the start (1.6 us, and up to 2.2 for groups of 16).  Fitted to 311 products of 41 bands, stencils
// and pruned matrices, N = 8 to 1,000, three on their own inputs in turn: 10 % standard deviation, and the group and panel it picks are
// 4 % from the best in the mean.  Estimate (measured), us: stencil 73 x 61 x 62, N = 88, groups of 8 80 (85); band of 52960 and 64, N = 472,
// groups of 16 34 (34.5); band of 2144 and 47, N = 808, groups of 4 5.5 (5.6).
double window_estimate_us(int rows, int cap, unsigned long long sum, int tiles, size_t M, size_t K, size_t N, size_t nnzb, int most_blocks, bool c_f32)
{
    if (!fits(rows, cap, tiles) || most_blocks > 2 * (tiles == 4 ? pairs_held<4> : pairs_held<1>)) return 1e30;
    const size_t mb = M / 16;
    const Launch l = launch_of(rows, cap, tiles, (int)((mb + rows - 1) / rows), N);
    const double parts = parts_of(tiles, N), units = (l.n_panels + l.panels_per_unit - 1) / l.panels_per_unit;
    const double c_bytes = (double)M * (double)N * (c_f32 ? 4.0 : 2.0), a_bytes = (double)nnzb * 512.0;
    const double steps = l.rounds * l.panels_per_unit * parts * (1.07 + 0.0155 * (double)nnzb / (double)mb * tiles);
    const double path = ((double)sum * 512.0 * tiles * parts * l.n_panels + a_bytes * units + c_bytes) / 8.7e6;
    const double memory = (a_bytes + 2.0 * (double)K * (double)N + c_bytes) / 5.0e6;
    return std::max(4.7, 1.6 + 2.2 * rows / 16.0 + std::pow(std::pow(steps, 4.0) + std::pow(path, 4.0) + std::pow(memory, 4.0), 0.25));
}

hipError_t window_widths(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, WindowWidths &out, void **slots)
{
    out = WindowWidths{};
    *slots = nullptr;
    const int words = (int)((kb + 31) / 32);
    if (nnzb == 0 || kb > (size_t)BITMAP_WORDS * 32) return hipSuccess; // none known
    hipError_t e = dev_malloc(slots, std::max(nnzb * sizeof(uint32_t), sizeof out));
    if (e != hipSuccess) return e;
    e = hipMemsetAsync(*slots, 0, sizeof out, nullptr);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(window_count_kernel, dim3((unsigned)std::min<size_t>((mb + SIZES[0] - 1) / SIZES[0], 512), WINDOW_SIZES), dim3(256), (size_t)words * 4, nullptr, row_ptr, col_idx,
                           (int)mb, words, (WindowWidths *)*slots);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&out, *slots, sizeof out, hipMemcpyDeviceToHost);
    if (e != hipSuccess) {
        (void)dev_free(*slots);
        *slots = nullptr;
    }
    return e;
}

void window_widths_host(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, WindowWidths &out)
{
    out = WindowWidths{};
    std::vector<uint32_t> seen(kb, 0); // the last group that used the column, counted over all sizes from 1
    uint32_t group = 0;
    for (int s = 0; s < WINDOW_SIZES; s++)
        for (size_t first = 0; first < mb; first += (size_t)SIZES[s]) {
            group++;
            uint32_t n = 0;
            for (int32_t q = row_ptr[first], end = row_ptr[std::min(first + (size_t)SIZES[s], mb)]; q < end; q++) {
                uint32_t &last = seen[(size_t)col_idx[q] / 16];
                n += last != group;
                last = group;
            }
            out.most[s] = std::max(out.most[s], n);
            out.sum[s] += n;
        }
}

double window_choose(const WindowWidths &w, size_t M, size_t K, size_t N, size_t nnzb, int most_blocks, int *size)
{
    double best = 1e30;
    *size = -1;
    for (int i = 0; i < WINDOW_SIZES; i++) {
        if (w.most[i] == 0 || (g_force_rows && SIZES[i] != g_force_rows)) continue;
        for (int t : {1, 2, 4}) {
            double e = window_estimate_us(SIZES[i], (int)((w.most[i] + 3) / 4 * 4), w.sum[i], t, M, K, N, nnzb, most_blocks, false);
            // Nothing shared: the pieces that the copies bring are single blocks, 32 bytes of a column (1376 x 5344, 4 %, N = 896: estimate 9.8,
            // 13.6 us, row-wise 11.4; 12656 x 832, 6 %, N = 352 11.4 -> 8.4 all the same).
            if ((double)w.sum[i] > 0.8 * (double)nnzb) e *= 1.25;
            if (e < best) best = e, *size = i;
        }
    }
    return best;
}

hipError_t window_build(const WindowWidths &w, int size, void *slots, const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, size_t nnzb, int most_blocks,
                        WindowPlan **out)
{
    *out = nullptr;
    WindowPlan *p = new (std::nothrow) WindowPlan();
    if (!p) {
        if (slots) (void)dev_free(slots);
        return hipErrorOutOfMemory;
    }
    p->d_slot = static_cast<uint32_t *>(slots);
    const int words = (int)((kb + 31) / 32);
    p->rows = SIZES[size];
    p->cap = (int)((w.most[size] + 3) / 4 * 4);
    p->sum = w.sum[size];
    p->most_blocks = most_blocks;
    p->n_groups = (int)((mb + p->rows - 1) / p->rows);
    hipError_t e = slots ? hipSuccess : dev_malloc(&p->d_slot, nnzb * sizeof(uint32_t));
    if (e == hipSuccess) e = dev_malloc(&p->d_window, (size_t)p->n_groups * (p->cap + 1) * sizeof(int32_t));
    p->d_count = p->d_window + (size_t)p->n_groups * p->cap;
    if (e == hipSuccess) {
        hipLaunchKernelGGL(window_list_kernel, dim3((unsigned)p->n_groups), dim3(256), (size_t)words * 6, nullptr, row_ptr, col_idx, (int)mb, words, p->rows, p->cap,
                           p->d_window, p->d_count, p->d_slot);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr); // launches on other streams read the lists
    if (e != hipSuccess) {
        window_destroy(p);
        return e;
    }
    *out = p;
    return hipSuccess;
}

void window_destroy(WindowPlan *p)
{
    if (!p) return;
    for (void *q : {(void *)p->d_window, (void *)p->d_slot})
        if (q) (void)dev_free(q);
    delete p;
}

bool window_forced() { return g_force_rows > 0; }
bool window_takes_rows(int most_blocks) { return most_blocks > 0 && most_blocks <= 2 * pairs_held<1>; }

double window_launch_us(const WindowPlan &p, size_t M, size_t K, size_t N, size_t nnzb, bool c_f32)
{
    double us;
    (void)best_tiles(p, M, K, N, nnzb, c_f32, &us);
    return us;
}

hipError_t launch_window(const SpmmArgs &a, const WindowPlan &p, hipStream_t st)
{
    double us;
    const int tiles = best_tiles(p, a.M, a.K, a.N, a.nnzb, a.c_f32, &us);
    if (tiles == 0 || !fits(p.rows, p.cap, tiles)) return hipErrorInvalidValue;
    const Launch l = launch_of(p.rows, p.cap, tiles, p.n_groups, a.N);
    const bool two = parts_of(tiles, a.N) == 2;
    if (tiles == 4) return a.c_f32 ? launch_as<4, 1, true>(a, p, l, st) : launch_as<4, 1, false>(a, p, l, st);
    if (tiles == 2 && two) return a.c_f32 ? launch_as<2, 2, true>(a, p, l, st) : launch_as<2, 2, false>(a, p, l, st);
    if (tiles == 2) return a.c_f32 ? launch_as<2, 1, true>(a, p, l, st) : launch_as<2, 1, false>(a, p, l, st);
    if (two) return a.c_f32 ? launch_as<1, 2, true>(a, p, l, st) : launch_as<1, 2, false>(a, p, l, st);
    return a.c_f32 ? launch_as<1, 1, true>(a, p, l, st) : launch_as<1, 1, false>(a, p, l, st);
}

} // namespace smat

// Test hook (not part of smat.h): groups of 4, 8 or 16 block rows and panels of 1, 2 or 4 tiles wherever they fit, whatever the
// estimates say (0 = the choice); rows = -1: no windows.
extern "C" void smat_internal_window_force(int rows, int tiles) { smat::g_force_rows = rows; smat::g_force_tiles = tiles; }
