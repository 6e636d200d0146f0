// Block-sparse SpMM kernels for gfx950 (MI355X): C = A_bcsr(16x16, fp16) * B(fp16),
// fp32 accumulation on v_mfma_f32_16x16x32_f16.
//
// Replaces the reference's live kernel mmaCBTKernelSparse and its launcher
// (src/cuda_hgemm/src/mma/mmaCBT.cu:13-88).  Same operands and semantics
// (absolute col_idx, column-major B, row-major C overwritten), different
// machine mapping:
//
//  * The product is formed transposed, C^T = B^T * A^T, so that a lane ends up
//    owning runs of consecutive C columns of one C row (wide stores) and both
//    MFMA operands are 16-byte, k-contiguous loads: B^T rows are the columns of
//    the column-major B, A^T columns are the rows of a row-major 16x16 block.
//  * One MFMA consumes two nonzero blocks of the same block row (K = 32 = 2x16):
//    lanes 0-31 feed block p, lanes 32-63 feed block p+1; a pair of blocks is one
//    contiguous, fully coalesced 1 KiB load.
//  * Work is a list of (block row, block range) items; block rows longer than
//    the chunk size are split and their fp32 partial tiles are summed in a fixed
//    order by a second kernel, so results do not depend on scheduling.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "row_tile.h"
#include "spmm_kernels.h"

#define SMAT_ORDER_FENCE()                      \
    do {                                        \
        asm volatile("" ::: "memory");          \
        __builtin_amdgcn_sched_barrier(0);      \
    } while (0)

namespace smat {

__device__ __forceinline__ f16x8 zero_f16x8()
{
    f16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    return z;
}

// One wavefront per work item x N panel, a workgroup of its own: workgroups of four kept their places until the longest of four items was done, and the last
// round of a launch had fewer of them than there are compute units.  Workgroups of four -> of one, us (120 products of random blocks, in place and repacked, are 10 and 4 % faster
// in the mean and 6 % slower at most, those of 6 us): 8272 x 4176, 32 %, N = 72 39.9 -> 28.4, 5680 x 9936, 15 %, N = 136 48.9 -> 34.8, repacked 23.8 -> 20.5; 8368 x
// 2736, 32 %, N = 48 15.8 -> 11.6; 27-point stencil of 78944 rows, N = 128 27.8 -> 23.8.  (The short-row kernel keeps workgroups of four: bands of few rows, N = 968 4.96, of one 6.20.)
//   items == nullptr : item w is the whole block row w (no work list)
//   items != nullptr : items[w] = {block row, first block, end block, dst}
//                      dst < 0  -> write the finished tile to C
//                      dst >= 0 -> write the fp32 partial tile to workspace slot dst
// Item index runs fastest inside a panel, so neighbouring workgroups share one B panel (K x 16*TN) in L2.  Workgroup
// ids are dealt round-robin to the 8 XCDs by the dispatcher; the remap below
// gives the XCDs runs of xcd_run consecutive workgroups of the (panel-major) item
// space in turn: an eighth of the launch each, so that an XCD's private L2 holds few
// distinct B panels, or shorter runs where the items' cost changes along the list
// (gridDim.x is a multiple of 8 * xcd_run).
// amdgpu_waves_per_eu(1, 4): at most 4 wavefronts per SIMD are asked for, which leaves the
// compiler 128 registers; with the default target of 8 it squeezes the kernel into 64 and
// gets there by loading each operand right before its MFMA, one memory latency apiece.
//
// PACKED: B is the slab-major copy made by pack_b_kernel, Bp[(bc/16 * N + n) * 16 + k % 16]:
// the 16 x 16 operand of one (block column, n-tile) is 512 contiguous bytes and a
// wavefront load touches 8 full cache lines instead of 32 quarter-used ones.
template <int TN, bool C_F32, bool PACKED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 4))) void spmm_rowwise_kernel(
    const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col_idx, const uint16_t *__restrict__ B, void *__restrict__ Cout,
    float *__restrict__ workspace, const WorkItem *__restrict__ items, int n_items, int N, long K,
    int n_panels, unsigned xcd_run)
{
    constexpr int PANEL = 16 * TN;
    const int lane = threadIdx.x;
    const long total = (long)n_items * n_panels;
    const unsigned slot = blockIdx.x >> 3;
    const unsigned run = __builtin_amdgcn_readfirstlane(slot / xcd_run); // wavefront-uniform values are forced into scalar registers
    const long w = ((long)run * 8 + (blockIdx.x & 7)) * xcd_run + (slot - run * xcd_run);
    if (w >= total) return;
    const int panel = (int)(w / n_items);
    const int it = (int)(w - (long)panel * n_items);

    int br, p0, p1, dst;
    if (items) {
        WorkItem wi = items[it];
        br = wi.block_row; p0 = wi.begin; p1 = wi.end; dst = wi.dst;
    } else {
        br = it; p0 = row_ptr[it]; p1 = row_ptr[it + 1]; dst = -1;
    }
    br = __builtin_amdgcn_readfirstlane(br);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    dst = __builtin_amdgcn_readfirstlane(dst);

    const int i16 = lane & 15; // A row m / B^T row (n within tile)
    const int g = lane >> 4;   // k group 0..3
    const int sel = g >> 1;    // which block of the pair
    const int kh = g & 1;      // which half (8 k) of the block
    const int n0 = panel * PANEL;

    f32x4 acc[TN];
    long boff[TN];
#pragma unroll
    for (int t = 0; t < TN; t++) {
        acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
        // columns past N read column 0 instead: what they produce is never stored
        const int n = n0 + ncol_of<TN>(t, i16);
        boff[t] = PACKED ? (long)(n < N ? n : 0) * 16 + kh * 8 : (long)(n < N ? n : 0) * K + kh * 8;
    }
    const uint16_t *abase = vals + i16 * 16 + kh * 8;
    const f16x8 zero8 = zero_f16x8();

    // Two register sets: the operands of pair j+1 are in flight while pair j is multiplied.  The loads of a
    // trip are without conditions: loads inside branches cannot be counted by the compiler's vmcnt bookkeeping,
    // which then waits for everything in flight and serialises load and MFMA phases.  The branch is behind the
    // loop, where one or two pairs are left.
    for (int pb = p0; pb < p1; pb += 64) {
        const int cnt = (p1 - pb) < 64 ? (p1 - pb) : 64;
        const int npair = (cnt + 1) >> 1;
        // one coalesced load of up to 64 column indices, then lane broadcasts
        const int myc = col_idx[pb + (lane < cnt ? lane : cnt - 1)];

        auto issue = [&](int j, f16x8 &a, f16x8 (&b)[TN]) {
            const int second = (2 * j + 1 < cnt) ? 2 * j + 1 : 2 * j; // a single block pairs with itself
            const int c0 = __builtin_amdgcn_readlane(myc, 2 * j);
            const int c1 = __builtin_amdgcn_readlane(myc, second);
            const int bc = sel ? c1 : c0;
            const long pp = (long)pb + (sel ? second : 2 * j);
            a = load_f16x8(abase + pp * 256);
            // column-major: + first column of the block; packed: + slab of the block column
            const long boffs = PACKED ? (long)bc * N : (long)bc;
#pragma unroll
            for (int t = 0; t < TN; t++) b[t] = load_f16x8(B + boff[t] + boffs);
        };
        auto multiply = [&](int j, f16x8 a, const f16x8 (&b)[TN]) {
            if (2 * j + 1 >= cnt) a = sel ? zero8 : a; // single block: the upper K half contributes nothing
#pragma unroll
            for (int t = 0; t < TN; t++)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[t], a, acc[t], 0, 0, 0);
        };

        // The main loop multiplies two pairs per trip with no branch around either of them:
        // a multiply inside a branch drags its loads into the branch with it (they sink to
        // their only use) and the prefetch distance collapses.  The fences pin the issue
        // order against the scheduler.
        f16x8 a0, a1, b0[TN], b1[TN];
        issue(0, a0, b0);
        SMAT_ORDER_FENCE();
        int j = 0;
        for (; j + 2 < npair; j += 2) {
            issue(j + 1, a1, b1);
            SMAT_ORDER_FENCE();
            multiply(j, a0, b0);
            SMAT_ORDER_FENCE();
            issue(j + 2, a0, b0);
            SMAT_ORDER_FENCE();
            multiply(j + 1, a1, b1);
            SMAT_ORDER_FENCE();
        }
        if (j + 1 < npair) { // two are left: nothing is asked for beyond them
            issue(j + 1, a1, b1);
            SMAT_ORDER_FENCE();
            multiply(j, a0, b0);
            SMAT_ORDER_FENCE();
            multiply(j + 1, a1, b1);
        } else {
            multiply(j, a0, b0);
        }
    }

    store_tile<TN, C_F32>(acc, br, dst, n0, i16, g, Cout, workspace, N);
}

// Launches of few (item, panel) pairs with long items: the four wavefronts of a workgroup share one, each takes a run of
// the item's block pairs, NP of them in flight, and the partial tiles are added in LDS in the order of the runs.
// Bound by the loads of B in place, whose 64 lanes ask for 32 pieces of 32 bytes: 53 clocks of a CU each, whatever is in flight (8192^2 with
// 10 % of the blocks, N = 16: 1.7 us a launch, 4.7 with the loads of A, 6.1 with those of B).  So no load is made for nothing: what is left of a run has code
// of its own length, where the last pair was asked for again up to NP times (same bits, us): that matrix 6.66 -> 6.1, 1184 x 5264, 27 %, N = 80 10.2 -> 8.2, 976 x
// 16096, 36 %, N = 32 17.8 -> 13.9, 2896 x 14064, 30 %, N = 32 15.2 -> 12.2.  Three to twelve pairs in flight are level, and so are eight wavefronts (5.9 to 6.1 us
// on the first); sixteen lose 20 to 40 % at N = 64.
template <int TN, bool C_F32, bool PACKED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void spmm_rowwise_split_kernel(
    const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
    const uint16_t *__restrict__ B, void *__restrict__ Cout, float *__restrict__ workspace, const WorkItem *__restrict__ items,
    int n_items, int N, long K, int n_panels)
{
    constexpr int SPLIT = 4, PANEL = 16 * TN;
    constexpr int NP = 4;
    __shared__ f32x4 part[SPLIT][TN][64];
    const int lane = threadIdx.x & 63;
    const int run = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // an XCD takes an eighth of the panel-major (panel, item) space: few panels of B in its L2
    const long total = (long)n_items * n_panels, per_xcd = (total + 7) / 8;
    const long w = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per_xcd || w >= total) return; // the whole workgroup
    const int panel = (int)(w / n_items);
    const int it = (int)(w - (long)panel * n_items);
    int br, p0, p1, dst;
    if (items) {
        const WorkItem wi = items[it];
        br = wi.block_row; p0 = wi.begin; p1 = wi.end; dst = wi.dst;
    } else {
        br = it; p0 = row_ptr[it]; p1 = row_ptr[it + 1]; dst = -1;
    }
    br = __builtin_amdgcn_readfirstlane(br);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    dst = __builtin_amdgcn_readfirstlane(dst);

    const int i16 = lane & 15, g = lane >> 4, sel = g >> 1, kh = g & 1;
    const int n0 = panel * PANEL;
    f32x4 acc[TN];
#pragma unroll
    for (int t = 0; t < TN; t++) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int npair = (p1 - p0 + 1) >> 1, per = (npair + SPLIT - 1) / SPLIT;
    const int j0 = run * per, j1 = j0 + per < npair ? j0 + per : npair;
    if (j0 < j1) { // uniform over the wavefront
        long boff[TN];
#pragma unroll
        for (int t = 0; t < TN; t++) {
            const int n = n0 + ncol_of<TN>(t, i16);
            boff[t] = PACKED ? (long)(n < N ? n : 0) * 16 + kh * 8 : (long)(n < N ? n : 0) * K + kh * 8; // past N: column 0, never stored
        }
        const uint16_t *abase = vals + i16 * 16 + kh * 8;
        const f16x8 zero8 = zero_f16x8();
        for (int jw = j0; jw < j1; jw += 32) { // a window of 64 column indices
            const int first = p0 + 2 * jw, last = p1 - 1;
            const int myc = col_idx[first + lane < last ? first + lane : last];
            const int jend = jw + 32 < j1 ? jw + 32 : j1;
            // the operands of R pairs at once, as many as there are
            auto pairs = [&](int j, auto count) {
                constexpr int R = decltype(count)::value;
                f16x8 a[R], b[R][TN];
#pragma unroll
                for (int u = 0; u < R; u++) { // the values first: they do not wait for the column indices
                    const int q0 = p0 + 2 * (j + u), q1 = q0 < last ? q0 + 1 : q0; // a single block pairs with itself
                    a[u] = load_f16x8(abase + (long)(sel ? q1 : q0) * 256);
                }
                SMAT_ORDER_FENCE();
#pragma unroll
                for (int u = 0; u < R; u++) {
                    const int q0 = p0 + 2 * (j + u), q1 = q0 < last ? q0 + 1 : q0;
                    const int c0 = __builtin_amdgcn_readlane(myc, q0 - first), c1 = __builtin_amdgcn_readlane(myc, q1 - first);
                    const int bc = sel ? c1 : c0;
                    const long boffs = PACKED ? (long)bc * N : (long)bc;
#pragma unroll
                    for (int t = 0; t < TN; t++) b[u][t] = load_f16x8(B + boff[t] + boffs);
                }
                SMAT_ORDER_FENCE();
#pragma unroll
                for (int u = 0; u < R; u++) {
                    const f16x8 au = sel && p0 + 2 * (j + u) >= last ? zero8 : a[u]; // single block: the upper K half contributes nothing
#pragma unroll
                    for (int t = 0; t < TN; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[u][t], au, acc[t], 0, 0, 0);
                }
            };
            using std::integral_constant;
            int j = jw;
            for (; j + NP <= jend; j += NP) pairs(j, integral_constant<int, NP>{});
            if (jend - j == 3) pairs(j, integral_constant<int, 3>{});
            else if (jend - j == 2) pairs(j, integral_constant<int, 2>{});
            else if (jend - j == 1) pairs(j, integral_constant<int, 1>{});
        }
    }
    if (run > 0)
#pragma unroll
        for (int t = 0; t < TN; t++) part[run][t][lane] = acc[t];
    __syncthreads();
    if (run > 0) return;
#pragma unroll
    for (int s = 1; s < SPLIT; s++)
#pragma unroll
        for (int t = 0; t < TN; t++) acc[t] += part[s][t][lane];
    store_tile<TN, C_F32>(acc, br, dst, n0, i16, g, Cout, workspace, N);
}

// Small problems with short block rows (a band matrix: 9 blocks per row, 256 rows): the kernel above keeps the
// operands of two block pairs in flight, so a row of five pairs costs four memory latencies one after the other
// and the launch is over before the chip is busy.  Here a wavefront asks for the operands of all its pairs
// (at most NP) at once: work item -> column indices -> operands, three latencies, then the MFMAs.  As in the kernel above the loads of B are what a CU does
// most of the time, so rows of fewer pairs have code of their own instead of loads for NP (band of 2208 rows and 12, N = 536: 6.13 -> 4.78 us, of 5328, N = 256
// 6.24 -> 5.05).  Whole block rows only (dst < 0), B in place.
template <int TN, bool C_F32, int NP>
__global__ __launch_bounds__(256) void spmm_rowwise_short_kernel(
    const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
    const uint16_t *__restrict__ B, void *__restrict__ Cout, const WorkItem *__restrict__ items, int n_items, int N,
    long K, int n_panels)
{
    static_assert(TN == 2 || TN == 4, "panels of 32 or 64 columns");
    constexpr int PANEL = 16 * TN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long w = (long)blockIdx.x * 4 + wave;
    if (w >= (long)n_items * n_panels) return;
    const int panel = (int)(w / n_items);
    const int it = (int)(w - (long)panel * n_items);
    int br, p0, p1;
    if (items) {
        const WorkItem wi = items[it];
        br = wi.block_row; p0 = wi.begin; p1 = wi.end;
    } else {
        br = it; p0 = row_ptr[it]; p1 = row_ptr[it + 1];
    }
    br = __builtin_amdgcn_readfirstlane(br);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    const int cnt = p1 - p0; // <= 2 * NP: the launcher has checked the work list
    const int npair = (cnt + 1) >> 1;

    const int i16 = lane & 15, g = lane >> 4, sel = g >> 1, kh = g & 1;
    const int n0 = panel * PANEL;
    f32x4 acc[TN];
#pragma unroll
    for (int t = 0; t < TN; t++) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (cnt > 0) { // uniform over the wavefront
        long boff[TN];
#pragma unroll
        for (int t = 0; t < TN; t++) {
            const int n = n0 + ncol_of<TN>(t, i16);
            boff[t] = (long)(n < N ? n : 0) * K + kh * 8; // columns past N read column 0: never stored
        }
        const uint16_t *abase = vals + i16 * 16 + kh * 8;
        const f16x8 zero8 = zero_f16x8();
        const int myc = col_idx[p0 + (lane < cnt ? lane : cnt - 1)];
        auto pairs = [&](auto count) {
            constexpr int R = decltype(count)::value;
            f16x8 a[R], b[R][TN];
            const int last = cnt - 1;
#pragma unroll
            for (int u = 0; u < R; u++) { // the values first: they do not wait for the column indices
                const int second = u < R - 1 ? 2 * u + 1 : last; // a single block pairs with itself
                a[u] = load_f16x8(abase + ((long)p0 + (sel ? second : 2 * u)) * 256);
            }
            SMAT_ORDER_FENCE();
#pragma unroll
            for (int u = 0; u < R; u++) {
                const int c0 = __builtin_amdgcn_readlane(myc, 2 * u), c1 = __builtin_amdgcn_readlane(myc, u < R - 1 ? 2 * u + 1 : last);
                const long bc = sel ? c1 : c0;
#pragma unroll
                for (int t = 0; t < TN; t++) b[u][t] = load_f16x8(B + boff[t] + bc);
            }
            SMAT_ORDER_FENCE();
#pragma unroll
            for (int u = 0; u < R; u++) {
                const f16x8 au = u == R - 1 && sel && 2 * u == last ? zero8 : a[u]; // single block: the upper K half contributes nothing
#pragma unroll
                for (int t = 0; t < TN; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[u][t], au, acc[t], 0, 0, 0);
            }
        };
        static_assert(NP == 5, "a case for each number of pairs");
        using std::integral_constant;
        switch (npair) { // uniform over the wavefront
        case 1: pairs(integral_constant<int, 1>{}); break;
        case 2: pairs(integral_constant<int, 2>{}); break;
        case 3: pairs(integral_constant<int, 3>{}); break;
        case 4: pairs(integral_constant<int, 4>{}); break;
        default: pairs(integral_constant<int, 5>{}); break;
        }
    }
    // acc[t][r] = C[br*16 + i16][n0 + ncol_of(t, 4*g + r)]: 4*TN consecutive columns per lane, as in the kernel above
    const long m = (long)br * 16 + i16;
    const int nbase = n0 + 4 * TN * g;
    if (C_F32) {
        float *crow = reinterpret_cast<float *>(Cout) + m * (long)N;
#pragma unroll
        for (int t = 0; t < TN; t++)
            if (nbase + 4 * t < N) *reinterpret_cast<f32x4 *>(crow + nbase + 4 * t) = acc[t];
    } else {
        uint16_t *crow = reinterpret_cast<uint16_t *>(Cout) + m * (long)N;
#pragma unroll
        for (int t = 0; t < TN; t += 2) {
            const f32x4 v0 = acc[t], v1 = acc[t + 1];
            const f16x8 h = {(_Float16)v0[0], (_Float16)v0[1], (_Float16)v0[2], (_Float16)v0[3],
                             (_Float16)v1[0], (_Float16)v1[1], (_Float16)v1[2], (_Float16)v1[3]};
            if (nbase + 4 * t < N) *reinterpret_cast<f16x8 *>(crow + nbase + 4 * t) = h;
        }
    }
}

// Row-major B (B[k * N + n]) in place: the 16 rows of B under a block are PW columns of it each, 2 * PW consecutive bytes, which go from the registers they
// were loaded into through LDS and come back as MFMA operands through transposing reads (ds_read_b64_tr_b16; layout and the swap of pieces against bank
// conflicts as in the compact kernel).  Pairs of blocks, their order and the shares of an item are those of the kernels above: same bits.
// SHARES = 4: four wavefronts share an item as in spmm_rowwise_split_kernel; 1: one wavefront, a workgroup of its own.
// Bound by the rows of B and the blocks that a wavefront brings over the L2, 17.5 TB/s of them in large launches: 64 lanes ask for 8 to 32 whole pieces of 128 to 32 bytes, 16
// clocks, where they ask for 32 pieces of 32 bytes of a column-major B, 53.  Before, B was turned in a launch of its own, 1.7 us and its bytes three times, and read as
// above.  That -> this, us: band of 5024 rows and 12, N = 240 8.0 -> 4.6; 2320 x 1328, 5 %, N = 632 9.2 -> 4.7; 960 x 11824, 6 %, N = 912, fp32 28 -> 12; band of 41472 and 64, N = 208
// 43 -> 22; stencil 49648, N = 8 9.2 -> 6.1; 2304 x 5840, 6 %, N = 2072 48 -> 24.
template <int PW, bool C_F32, int SHARES>
__global__ __launch_bounds__(64 * SHARES) __attribute__((amdgpu_waves_per_eu(1, 4))) void spmm_rowwise_row_major_kernel(
    const uint16_t *__restrict__ vals, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
    const uint16_t *__restrict__ B, void *__restrict__ Cout, float *__restrict__ workspace, const WorkItem *__restrict__ items,
    int n_items, int N, int n_panels, unsigned xcd_run)
{
    constexpr int T = PW / 16, NP = 4; // tiles of 16 columns, and loads that bring the 32 rows of B under a pair; pairs in flight
    constexpr int TILE = 64 * PW;      // bytes of 32 rows
    __shared__ __align__(1024) unsigned char tiles[SHARES][TILE];
    const int lane = threadIdx.x & 63;
    const int share = SHARES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long total = (long)n_items * n_panels;
    const unsigned slot = blockIdx.x >> 3, run = __builtin_amdgcn_readfirstlane(slot / xcd_run);
    const long w = ((long)run * 8 + (blockIdx.x & 7)) * xcd_run + (slot - run * xcd_run);
    if (w >= total) return; // the whole workgroup
    const int panel = (int)(w / n_items);
    const int it = (int)(w - (long)panel * n_items);
    int br, p0, p1, dst;
    if (items) {
        const WorkItem wi = items[it];
        br = wi.block_row; p0 = wi.begin; p1 = wi.end; dst = wi.dst;
    } else {
        br = it; p0 = row_ptr[it]; p1 = row_ptr[it + 1]; dst = -1;
    }
    br = __builtin_amdgcn_readfirstlane(br);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    dst = __builtin_amdgcn_readfirstlane(dst);

    const int i16 = lane & 15, g = lane >> 4, sel = g >> 1;
    const int n0 = panel * PW;
    // load j < T: 16 bytes of row k = row0 + 2 j of the pair's 32
    const int c8 = lane % (PW / 8), place = T * (lane / (PW / 8));
    const int row0 = 8 * (place >> 3) + 2 * (place & 3) + ((place >> 2) & 1);
    const bool second_block = row0 >= 16;
    const uint16_t *const from = B + (long)(row0 & 15) * N + (n0 + 8 * c8 < N ? n0 + 8 * c8 : 0); // N % 8 == 0: all of the lane's columns or none
    unsigned char *const tile = tiles[share];
    unsigned char *const put_even = tile + row0 * (2 * PW) + c8 * 16, *const put_odd = tile + row0 * (2 * PW) + (PW == 64 ? c8 ^ 1 : c8) * 16;
    const int swap = PW == 64 ? (i16 >> 3) & 1 : 0;
    const unsigned char *const get = tile + (8 * g + (i16 >> 2)) * (2 * PW) + (i16 & 3) * (PW / 2);
    const unsigned char *const get01 = get + 16 * swap, *const get23 = get - 16 * swap;
    const uint16_t *const abase = vals + i16 * 16 + (g & 1) * 8;
    const f16x8 zero8 = zero_f16x8();

    f32x4 acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int last = p1 - 1, npair = (p1 - p0 + 1) >> 1, per = (npair + SHARES - 1) / SHARES;
    const int j_first = share * per, j_last = SHARES == 1 ? npair : j_first + per < npair ? j_first + per : npair;
    for (int jw = j_first; jw < j_last; jw += 32) { // a window of 64 column indices
        const int first = p0 + 2 * jw;
        const int myc = col_idx[first + lane < last ? first + lane : last];
        const int j_end = jw + 32 < j_last ? jw + 32 : j_last;
        auto pairs = [&](int j, auto count) {
            constexpr int R = decltype(count)::value;
            f16x8 a[R], b[R][T];
#pragma unroll
            for (int u = 0; u < R; u++) { // the values first: they do not wait for the column indices
                const int q0 = p0 + 2 * (j + u), q1 = q0 < last ? q0 + 1 : q0; // a single block pairs with itself
                a[u] = load_f16x8(abase + (long)(sel ? q1 : q0) * 256);
            }
            SMAT_ORDER_FENCE();
#pragma unroll
            for (int u = 0; u < R; u++) {
                const int q0 = p0 + 2 * (j + u), q1 = q0 < last ? q0 + 1 : q0;
                const long o0 = (long)__builtin_amdgcn_readlane(myc, q0 - first) * N, o1 = (long)__builtin_amdgcn_readlane(myc, q1 - first) * N;
                const uint16_t *const p = from + (second_block ? o1 : o0);
#pragma unroll
                for (int l = 0; l < T; l++) b[u][l] = load_f16x8(p + (long)(2 * l) * N);
            }
            SMAT_ORDER_FENCE();
#pragma unroll
            for (int u = 0; u < R; u++) {
                const f16x8 au = sel && p0 + 2 * (j + u) >= last ? zero8 : a[u]; // single block: the upper K half contributes nothing
#pragma unroll
                for (int l = 0; l < T; l++) *reinterpret_cast<f16x8 *>((l & 1 ? put_odd : put_even) + l * 4 * PW) = b[u][l];
                asm volatile("" ::: "memory"); // LDS operations of a wavefront complete in order
                f16x8 op[T];
#pragma unroll
                for (int t = 0; t < T; t++) {
                    typedef short s16x4 __attribute__((ext_vector_type(4)));
                    const unsigned char *const q = (t < 2 ? get01 : get23) + t * 8;
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)q);
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(q + 8 * PW));
                    op[t] = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int t = 0; t < T; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[t], au, acc[t], 0, 0, 0);
            }
        };
        using std::integral_constant;
        int j = jw;
        for (; j + NP <= j_end; j += NP) pairs(j, integral_constant<int, NP>{});
        if (j_end - j == 3) pairs(j, integral_constant<int, 3>{});
        else if (j_end - j == 2) pairs(j, integral_constant<int, 2>{});
        else if (j_end - j == 1) pairs(j, integral_constant<int, 1>{});
    }
    if constexpr (SHARES > 1) {
        f32x4 *const part = reinterpret_cast<f32x4 *>(tile); // T KiB, the size of the tile
        asm volatile("" ::: "memory");
        if (share > 0)
#pragma unroll
            for (int t = 0; t < T; t++) part[t * 64 + lane] = acc[t];
        __syncthreads();
        if (share > 0) return;
#pragma unroll
        for (int s = 1; s < SHARES; s++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[t] += reinterpret_cast<const f32x4 *>(tiles[s])[t * 64 + lane];
    }
    // acc[t][r] = C[16 br + i16][n0 + PW / 4 * g + 4 t + r]
    const int c0 = n0 + PW / 4 * g;
    if (dst >= 0 || C_F32) {
        float *const row = dst >= 0 ? workspace + ((long)dst * 16 + i16) * (long)N : reinterpret_cast<float *>(Cout) + ((long)br * 16 + i16) * (long)N;
#pragma unroll
        for (int t = 0; t < T; t++)
            if (c0 + 4 * t < N) *reinterpret_cast<f32x4 *>(row + c0 + 4 * t) = acc[t];
    } else {
        uint16_t *const row = reinterpret_cast<uint16_t *>(Cout) + ((long)br * 16 + i16) * (long)N;
        if constexpr (T == 1) {
            if (c0 < N) *reinterpret_cast<f16x4 *>(row + c0) = __builtin_convertvector(acc[0], f16x4);
        } else {
#pragma unroll
            for (int t = 0; t < T; t += 2)
                if (c0 + 4 * t < N)
                    *reinterpret_cast<f16x8 *>(row + c0 + 4 * t) = __builtin_shufflevector(__builtin_convertvector(acc[t], f16x4), __builtin_convertvector(acc[t + 1], f16x4), 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }
}

// Sums the fp32 partial tiles of every split block row in slot order and writes
// the finished rows to C.  One thread per 4 consecutive columns of one row.
template <bool C_F32>
__global__ __launch_bounds__(256) void spmm_reduce_kernel(const float *__restrict__ workspace,
                                                         const SplitRow *__restrict__ rows,
                                                         int n_rows, void *__restrict__ Cout, int N)
{
    const int quads = N >> 2; // N % 8 == 0
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long per_row = (long)16 * quads;
    if (tid >= per_row * n_rows) return;
    const int r = (int)(tid / per_row);
    const long rem = tid - (long)r * per_row;
    const int i = (int)(rem / quads);
    const int q = (int)(rem - (long)i * quads);
    const SplitRow sr = rows[r];
    // Four running sums, slot k into sum k % 4 (a fixed order: the result does not depend on the launch): the loads of
    // four slots are under way at a time instead of one, which is what a block row of many slots waits for.
    const float *base = workspace + (long)i * (long)N + 4 * q;
    const long slot_stride = 16L * (long)N;
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0, s3 = s0;
    int slot = sr.slot_begin;
    for (; slot + 4 <= sr.slot_end; slot += 4) {
        const f32x4 v0 = *reinterpret_cast<const f32x4 *>(base + (long)slot * slot_stride);
        const f32x4 v1 = *reinterpret_cast<const f32x4 *>(base + (long)(slot + 1) * slot_stride);
        const f32x4 v2 = *reinterpret_cast<const f32x4 *>(base + (long)(slot + 2) * slot_stride);
        const f32x4 v3 = *reinterpret_cast<const f32x4 *>(base + (long)(slot + 3) * slot_stride);
        s0 += v0; s1 += v1; s2 += v2; s3 += v3;
    }
    if (slot < sr.slot_end) s0 += *reinterpret_cast<const f32x4 *>(base + (long)slot * slot_stride);
    if (slot + 1 < sr.slot_end) s1 += *reinterpret_cast<const f32x4 *>(base + (long)(slot + 1) * slot_stride);
    if (slot + 2 < sr.slot_end) s2 += *reinterpret_cast<const f32x4 *>(base + (long)(slot + 2) * slot_stride);
    const f32x4 s = (s0 + s1) + (s2 + s3);
    const long m = (long)sr.block_row * 16 + i;
    if (C_F32) {
        *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(Cout) + m * (long)N + 4 * q) = s;
    } else {
        f16x4 h = {(_Float16)s[0], (_Float16)s[1], (_Float16)s[2], (_Float16)s[3]};
        *reinterpret_cast<f16x4 *>(reinterpret_cast<uint16_t *>(Cout) + m * (long)N + 4 * q) = h;
    }
}

// Column-major B (B[n*K + k]) -> slab-major Bp[(k/16 * N + n) * 16 + k % 16].
// One workgroup moves a tile of 64 n x 64 k through LDS: reads are 128-byte runs along k,
// writes are 2 KiB runs (64 n x 32 B) per block column.
__global__ __launch_bounds__(256) void pack_b_kernel(const uint16_t *__restrict__ B,
                                                     uint16_t *__restrict__ Bp, int N, long K)
{
    __shared__ __align__(16) unsigned char tile[8192];
    const int t = threadIdx.x;
    const long k0 = (long)blockIdx.x * 64;
    const int n0 = blockIdx.y * 64;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int idx = i * 256 + t;
        const int nl = idx >> 3, seg = idx & 7; // seg: 8 k (16 bytes) along k
        f16x8 v = zero_f16x8();
        if (n0 + nl < N && k0 + seg * 8 < K) v = load_f16x8(B + (long)(n0 + nl) * K + k0 + seg * 8);
        *reinterpret_cast<f16x8 *>(tile + ((seg >> 1) * 64 + nl) * 32 + (seg & 1) * 16) = v;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int idx = i * 256 + t;
        const int bcl = idx >> 7, nl = (idx & 127) >> 1, half = idx & 1;
        if (n0 + nl < N && k0 + bcl * 16 < K)
            *reinterpret_cast<f16x8 *>(Bp + ((k0 / 16 + bcl) * N + n0 + nl) * 16 + half * 8) =
                *reinterpret_cast<const f16x8 *>(tile + (size_t)idx * 16);
    }
}

template <int TN>
static hipError_t launch_rowwise_tn(const SpmmArgs &a, hipStream_t st)
{
    const int panel = 16 * TN;
    const int n_panels = (int)((a.N + panel - 1) / panel);
    const long total = (long)a.n_items * n_panels;
    if (total == 0) return hipSuccess;
    const long xcd_run = 4 * (a.deal && a.items ? (long)a.deal->run((size_t)a.n_items, n_panels) : ((total + 3) / 4 + 7) / 8);
    const long wgs = (total + 8 * xcd_run - 1) / (8 * xcd_run) * (8 * xcd_run);
    if (wgs > 0x7fffffffL) return hipErrorInvalidValue;
    dim3 grid((unsigned)wgs), block(64);
#define SMAT_LAUNCH_ROWWISE(F32, PK)                                                              \
    hipLaunchKernelGGL((spmm_rowwise_kernel<TN, F32, PK>), grid, block, 0, st, a.vals, a.row_ptr, \
                       a.col_idx, a.b_packed ? a.b_packed : a.B, a.C, a.workspace, a.items,       \
                       a.n_items, (int)a.N, (long)a.K, n_panels, (unsigned)xcd_run)
    if (a.b_packed) {
        if (a.c_f32) SMAT_LAUNCH_ROWWISE(true, true);
        else SMAT_LAUNCH_ROWWISE(false, true);
    } else if constexpr (TN < 16) { // the rule takes 256 columns on repacked B only
        if (a.c_f32) SMAT_LAUNCH_ROWWISE(true, false);
        else SMAT_LAUNCH_ROWWISE(false, false);
    } else {
        return hipErrorInvalidValue;
    }
#undef SMAT_LAUNCH_ROWWISE
    return hipGetLastError();
}

unsigned choose_xcd_run(const uint64_t *P, uint64_t n, int n_panels)
{
    const uint64_t total = n * (uint64_t)n_panels;
    const uint64_t wgs = (total + 3) / 4;
    const uint64_t eighth = std::max<uint64_t>((wgs + 7) / 8, 1);
    if (n == 0 || P[n] == 0) return (unsigned)eighth;
    auto cost_before = [&](uint64_t wg) { // of the workgroups before wg in the panel-major item space
        const uint64_t w = std::min(wg * 4, total);
        return (w / n) * P[n] + P[w % n];
    };
    uint64_t best_run = eighth;
    double best = 1e30;
    for (uint64_t run : {eighth, (uint64_t)1024, (uint64_t)256, (uint64_t)64, (uint64_t)16, (uint64_t)4}) {
        if (run > eighth || (run == eighth && best < 1e30)) continue;
        if (wgs / run > ((uint64_t)1 << 26)) break; // a launch this large is not walked run by run on the host
        uint64_t load[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (uint64_t first = 0, x = 0; first < wgs; first += run, x = (x + 1) & 7)
            load[x] += cost_before(first + run) - cost_before(first);
        const uint64_t busiest = *std::max_element(load, load + 8);
        const double ratio = (double)busiest * 8.0 / (double)std::max<uint64_t>(cost_before(wgs), 1);
        if (ratio < best) best = ratio, best_run = run;
        if (ratio <= 1.04) break;
    }
    return (unsigned)best_run;
}

void XcdDeal::set_costs(std::vector<uint64_t> &&prefix)
{
    std::lock_guard<std::mutex> lock(mutex_);
    cost_prefix_ = std::move(prefix);
    known_.clear();
}

unsigned XcdDeal::run(size_t n_items, int n_panels) const
{
    const uint64_t n = n_items;
    std::lock_guard<std::mutex> lock(mutex_);
    if (n == 0 || cost_prefix_.size() != n + 1) // no costs for this list: an eighth of the launch each
        return (unsigned)std::max<uint64_t>(((n * (uint64_t)n_panels + 3) / 4 + 7) / 8, 1);
    for (const auto &k : known_)
        if (k.first == n_panels) return k.second;
    const unsigned r = choose_xcd_run(cost_prefix_.data(), n, n_panels);
    known_.emplace_back(n_panels, r);
    return r;
}

// Panel width of the row-wise kernel in tiles of 16 columns, from 842 timed products (random blocks 768^2 to 16384^2 at 3 to
// 36 %, bands; N = 96 to 4096, every width):
//   repacked B  the launch runs in rounds of 1024 wavefronts, one per SIMD, and a column of a round costs 0.83 in a panel of
//               128 and 0.8 in one of 256 of what it costs in one of 64, which reads the blocks more often: the width with the
//               lowest product.  Of 614 launches 0.5 % slower than the best width in the mean, at most 14 %.  64, 128, 256
//               columns, us: 640 items of 59 blocks, N = 384 39.4, 35.9, 54.6, N = 512 51.3, 48.2, 56.9; 512 of 113, N = 512
//               60.2, 51.3, 47.9; 284 of 122, N = 888 69.9, 60.5, 96.1; 651 of 155, N = 136 42.6, 62.2, -;
//   in place    64 columns, 128 where that still leaves 8000 wavefronts, or 2000 with items of 32 blocks and more.  Of 228
//               launches 1 % slower than the best width in the mean, at most 12 %; 256 columns win by 4 % at most.
//               120 items of 66 blocks, N = 2344 102.5, 121.1, 174.2; 2913 of 5, N = 2224 195.8, 168.0, 189.1; 1024 of 51, N = 384
//               100.8, 96.2, 133.6;
//   UNKNOWN     whole block rows without a plan, in place: the heaviest row may be many times the average and is one
//               wavefront per panel, so 64 columns below N = 512 (R-MAT scale 16, 16 a row: N = 256 1,595, 2,686, 3,315;
//               scale 14, N = 1024 730, 839, 986);
//   SPLIT       lists with split rows, uneven in more than their items' lengths: 64 columns (R-MAT scale 16, N = 512: 618
//               against 944 us; scale 20, N = 128: 13.8 against 18.2 ms).
int rowwise_panel_tiles(size_t N, size_t n_items, size_t avg_blocks, RowLengths lengths, bool packed)
{
    if (N < 32) return 1;
    if (N < 64) return 2;
    if (lengths == RowLengths::SPLIT || N < 128) return 4;
    if (!packed) {
        const size_t wavefronts = n_items * ((N + 127) / 128);
        return N >= (lengths == RowLengths::UNKNOWN ? 512 : 128) && wavefronts >= (avg_blocks < 32 ? 8000 : 2000) ? 8 : 4;
    }
    static const struct { int tiles; double column; } widths[] = {{4, 1.0}, {8, 0.83}, {16, 0.8}};
    int best_tiles = 4;
    double best = 1e30;
    for (const auto &w : widths) {
        if (N < (size_t)w.tiles * 16) break;
        const size_t panels = (N + 16 * w.tiles - 1) / (16 * w.tiles);
        const double cost = w.tiles * w.column * (double)((n_items * panels + 1023) / 1024);
        if (cost < best) best = cost, best_tiles = w.tiles;
    }
    return best_tiles;
}

// Four wavefronts per (item, panel of 64 columns): up to 512 of those, of 12 blocks and more.  (256 items of 26 blocks,
// N = 64: 6.0 against 9.7 us; 512 items of 51 blocks, N = 64: 11.7 against 17.0; with 1024 the two are level, with more
// the shared items lose.)  The rule knows nothing about the layout of B: in place and repacked give the same bits.
bool rowwise_shares_items(size_t N, size_t n_items, size_t avg_blocks)
{
    return n_items * ((N + 63) / 64) <= 512 && avg_blocks >= 12;
}

// The short-row kernel: rows of at most 2 * SHORT_NP blocks, no split rows, B in place, few wavefronts.
constexpr int SHORT_NP = 5;
constexpr size_t SHORT_MAX_WAVES = 8192;
bool rowwise_takes_short_rows(size_t N, size_t n_items, int most_blocks)
{
    return most_blocks > 0 && most_blocks <= 2 * SHORT_NP && N >= 32 && n_items * ((N + 31) / 32) <= SHORT_MAX_WAVES;
}

template <int TN>
static hipError_t launch_rowwise_short(const SpmmArgs &a, hipStream_t st)
{
    const int n_panels = (int)((a.N + 16 * TN - 1) / (16 * TN));
    const long total = (long)a.n_items * n_panels;
    if (total == 0) return hipSuccess;
    dim3 grid((unsigned)((total + 3) / 4)), block(256);
    if (a.c_f32)
        hipLaunchKernelGGL((spmm_rowwise_short_kernel<TN, true, SHORT_NP>), grid, block, 0, st, a.vals, a.row_ptr, a.col_idx,
                           a.B, a.C, a.items, a.n_items, (int)a.N, (long)a.K, n_panels);
    else
        hipLaunchKernelGGL((spmm_rowwise_short_kernel<TN, false, SHORT_NP>), grid, block, 0, st, a.vals, a.row_ptr, a.col_idx,
                           a.B, a.C, a.items, a.n_items, (int)a.N, (long)a.K, n_panels);
    return hipGetLastError();
}

template <int TN>
static hipError_t launch_rowwise_split(const SpmmArgs &a, hipStream_t st)
{
    const int n_panels = (int)((a.N + 16 * TN - 1) / (16 * TN));
    const long wgs = (long)a.n_items * n_panels;
    if (wgs == 0) return hipSuccess;
    dim3 grid((unsigned)((wgs + 7) / 8 * 8)), block(256);
#define SMAT_LAUNCH_SPLIT(F32, PK)                                                                                         \
    hipLaunchKernelGGL((spmm_rowwise_split_kernel<TN, F32, PK>), grid, block, 0, st, a.vals, a.row_ptr, a.col_idx, \
                       a.b_packed ? a.b_packed : a.B, a.C, a.workspace, a.items, a.n_items, (int)a.N, (long)a.K, n_panels)
    if (a.b_packed) {
        if (a.c_f32) SMAT_LAUNCH_SPLIT(true, true);
        else SMAT_LAUNCH_SPLIT(false, true);
    } else {
        if (a.c_f32) SMAT_LAUNCH_SPLIT(true, false);
        else SMAT_LAUNCH_SPLIT(false, false);
    }
#undef SMAT_LAUNCH_SPLIT
    return hipGetLastError();
}

size_t rowwise_row_major_width(size_t N) { return N <= 16 ? 16 : N <= 32 ? 32 : 64; }
// A launch has fewer than 2^32 threads, 64 of them for a panel of an item, and is rounded up to eight runs of at most 4096 items (deal) or of an eighth of it.
bool rowwise_row_major_fits(size_t n_items, size_t N)
{
    const size_t width = rowwise_row_major_width(N);
    return n_items * ((N + width - 1) / width) < ((size_t)1 << 26) - ((size_t)1 << 16);
}

template <int PW>
static hipError_t launch_rowwise_row_major(const SpmmArgs &a, bool shared, hipStream_t st)
{
    const int n_panels = (int)((a.N + PW - 1) / PW);
    const long total = (long)a.n_items * n_panels;
    if (total == 0) return hipSuccess;
    const long eighth = (total + 7) / 8;
    const long xcd_run = shared ? eighth : 4 * (a.deal && a.items ? (long)a.deal->run((size_t)a.n_items, n_panels) : ((total + 3) / 4 + 7) / 8);
    const long wgs = (total + 8 * xcd_run - 1) / (8 * xcd_run) * (8 * xcd_run);
    if (wgs * 64 * (shared ? 4 : 1) >= 1L << 32) return hipErrorInvalidValue;
#define SMAT_LAUNCH_ROW_MAJOR(F32, SHARES)                                                                                                   \
    hipLaunchKernelGGL((spmm_rowwise_row_major_kernel<PW, F32, SHARES>), dim3((unsigned)wgs), dim3(64 * SHARES), 0, st, a.vals, a.row_ptr,  \
                       a.col_idx, a.B, a.C, a.workspace, a.items, a.n_items, (int)a.N, n_panels, (unsigned)xcd_run)
    if (shared) {
        if (a.c_f32) SMAT_LAUNCH_ROW_MAJOR(true, 4);
        else SMAT_LAUNCH_ROW_MAJOR(false, 4);
    } else {
        if (a.c_f32) SMAT_LAUNCH_ROW_MAJOR(true, 1);
        else SMAT_LAUNCH_ROW_MAJOR(false, 1);
    }
#undef SMAT_LAUNCH_ROW_MAJOR
    return hipGetLastError();
}

hipError_t launch_rowwise(const SpmmArgs &a, hipStream_t st)
{
    hipError_t e;
    const size_t n_items = (size_t)a.rule_items, avg = n_items ? a.nnzb / n_items : 0;
    const bool shares = rowwise_shares_items(a.N, n_items, avg);
    if (a.b_row_major) {
        switch (rowwise_row_major_width(a.N)) {
        case 16: e = launch_rowwise_row_major<16>(a, shares, st); break;
        case 32: e = launch_rowwise_row_major<32>(a, shares, st); break;
        default: e = launch_rowwise_row_major<64>(a, shares, st); break;
        }
        if (e == hipSuccess && a.n_split_rows > 0) e = launch_reduce(a.workspace, a.split_rows, a.n_split_rows, a.C, a.N, a.c_f32, st);
        return e;
    }
    if (!a.b_packed && a.n_split_rows == 0 && rowwise_takes_short_rows(a.N, (size_t)a.n_items, a.max_item_blocks)) {
        // 32-column panels while that still leaves the chip short of wavefronts, else 64
        const bool narrow = (long)a.n_items * (long)((a.N + 63) / 64) < 2048;
        return narrow ? launch_rowwise_short<2>(a, st) : launch_rowwise_short<4>(a, st);
    }
    if (a.b_packed) {
        dim3 grid((unsigned)((a.K + 63) / 64), (unsigned)((a.N + 63) / 64));
        hipLaunchKernelGGL(pack_b_kernel, grid, dim3(256), 0, st, a.B, a.b_packed, (int)a.N, (long)a.K);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (shares) {
        if (a.N < 32) e = launch_rowwise_split<1>(a, st);
        else if (a.N < 64) e = launch_rowwise_split<2>(a, st);
        else e = launch_rowwise_split<4>(a, st);
    } else {
        const RowLengths lengths = a.n_split_rows > 0 ? RowLengths::SPLIT : a.items ? RowLengths::EVEN : RowLengths::UNKNOWN;
        switch (rowwise_panel_tiles(a.N, n_items, avg, lengths, a.b_packed != nullptr)) {
        case 16: e = launch_rowwise_tn<16>(a, st); break;
        case 8: e = launch_rowwise_tn<8>(a, st); break;
        case 4: e = launch_rowwise_tn<4>(a, st); break;
        case 2: e = launch_rowwise_tn<2>(a, st); break;
        default: e = launch_rowwise_tn<1>(a, st); break;
        }
    }
    if (e != hipSuccess) return e;
    if (a.n_split_rows > 0) e = launch_reduce(a.workspace, a.split_rows, a.n_split_rows, a.C, a.N, a.c_f32, st);
    return e;
}

hipError_t launch_reduce(const float *workspace, const SplitRow *split_rows, int n_split_rows, void *C, size_t N,
                         bool c_f32, hipStream_t st)
{
    const long threads = (long)n_split_rows * 16 * (long)(N / 4);
    const long blocks = (threads + 255) / 256;
    if (blocks <= 0) return hipSuccess;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    if (c_f32)
        hipLaunchKernelGGL((spmm_reduce_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, st, workspace,
                           split_rows, n_split_rows, C, (int)N);
    else
        hipLaunchKernelGGL((spmm_reduce_kernel<false>), dim3((unsigned)blocks), dim3(256), 0, st, workspace,
                           split_rows, n_split_rows, C, (int)N);
    return hipGetLastError();
}

} // namespace smat

// Test hook (not part of smat.h): the panel width of the row-wise kernel in tiles of 16 columns; lengths as in RowLengths.
extern "C" int smat_internal_rowwise_panel(size_t N, size_t n_items, size_t avg_blocks, int lengths, int packed)
{
    return smat::rowwise_panel_tiles(N, n_items, avg_blocks, static_cast<smat::RowLengths>(lengths), packed != 0);
}
