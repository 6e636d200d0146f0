// Products of matrices with few nonzeros a block and B narrow enough in K that whole columns of it stay in LDS.
//
// A workgroup holds T columns of B, K x T halves with the T of a row of B side by side, and walks the nonzeros of a share of the
// rows of A: a lane owns a row, reads its next nonzero (value << 16 | row of B, 64 rows side by side) and the T halves of that row
// of B from LDS, and adds their products in fp32.  B is read once for every share, column-major as it comes, and no copy of it is made first.
//
// 16384 x 16384, 16 a row, N = 256 16.0 -> 13.2 us against the compact kernel; 44832 x 8800, 35 a row, N = 152 48 -> 22; 3600 x 10064, 9 a row,
// N = 408 11.8 -> 7.8; 2496 x 3344, 27 a row, N = 192 9.8 -> 5.6.  The compact kernel's gathers of whole rows of B move 2 bytes a nonzero
// and column over a compute unit's memory path, behind a pass that writes B anew; here a nonzero costs that path 4 bytes for T columns.
// What bounds it, of those 13.2 us (4 columns, 4 shares): a launch and 1.3 for B into LDS; the vector unit 3.9, a nonzero and lane
// 1 instruction for its address, T to multiply and T / 4 to add; 1.4 more for the list; 3.4 for C, a million pieces of 8 bytes that the L2s take
// one a channel and cycle (none of it bank conflicts: as fast with all lanes at their own banks).  More columns cost less of all of it, so T is as large as LDS
// allows and the launch is still wide enough for.  Loads of the list four ahead, since 16 wavefronts wait for them together.
//
// Rows are put in order of their lengths and dealt 64 at a time, back and forth over the wavefronts, so that the lanes of one
// end together and the wavefronts have equally much.  A row of more than PART nonzeros is shared by 2 to 64 neighbouring lanes, whose sums
// are added in the end.  Lists are padded to fours of nonzeros by zeros that meet a row of zeros behind B.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <new>

#include "devmem.h"
#include "spmm_kernels.h"

namespace smat {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <int T> using halves = _Float16 __attribute__((ext_vector_type(T)));
template <int T> using floats = float __attribute__((ext_vector_type(T)));

constexpr int WAVES = 16;              // wavefronts of a workgroup
constexpr size_t MAX_LDS = 160 * 1024;
constexpr int AHEAD = 4;               // fours that a wavefront asks for ahead
constexpr int PART = 64;               // nonzeros of a lane
constexpr int SHARED = 6;              // a row is shared by 1 << SHARED lanes at most
constexpr int MAX_ROW = PART << SHARED;
constexpr uint32_t ROW_BITS = 28;      // of a lane's first word: its row; above them the logarithm of the lanes that share it
constexpr uint32_t PADDED = (1u << ROW_BITS) - 1; // the row of a lane that has none
// Kinds of rows, the longest first: those shared by 64, 32, .. 2 lanes, then those of PART, PART - 1, .. 0 nonzeros.
constexpr int KINDS = SHARED + PART + 1;
__host__ __device__ constexpr int lanes_log(int kind) { return kind < SHARED ? SHARED - kind : 0; }
__device__ __forceinline__ int kind_of(int n)
{
    if (n <= PART) return SHARED + PART - n;
    const int log = 32 - __clz((n + PART - 1) / PART - 1);
    return log < SHARED ? SHARED - log : 0; // longer ones than MAX_ROW: the lists are not taken
}
// Numbers of rows of every kind and the longest row, COUNTS times: additions to one word queue up at 12 ns each.
constexpr int COUNTS = 16;
struct ResidentTotals { // in front of ResidentPlan::d_first
    uint32_t n_slices, fours, longest, places;
    uint32_t rows_of[COUNTS][KINDS], longest_of[COUNTS];
};
constexpr size_t IN_FRONT = sizeof(ResidentTotals) / sizeof(uint32_t);

size_t lds_of(size_t K, int T) { return ((K + 1) * 2 * T + 15) / 16 * 16; }

// ---- the lists, from the compact kernel's ----

// The steps of 32 listed columns of an item one after the other: of each the 8 values of row `lane % 16` in columns 8 * (lane / 16) .., asked
// for a step ahead (a wavefront that asked when it needed them waited for three loads in turn every step: 16384 rows of 16 25 -> 15 us).  The
// wavefronts of a workgroup take an eighth of an item each.
constexpr int BUILD_WAVES = 8;
struct Steps {
    const uint16_t *acol;
    const uint32_t *entries;
    const int2 *range;
    uint16_t *tile; // 1 KiB of the wavefront's own
    int lane;
    long first, end, next;
    u32x4 values;
    uint32_t e[2];
    int n;
    int2 ranges; // of step next / 64 * 64 + lane from the first
    __device__ __forceinline__ Steps(const WorkItem &it, int eighth, const uint16_t *acol, const uint32_t *entries, const int2 *range, u32x4 *tile, int lane)
        : acol(acol), entries(entries), range(range), tile(reinterpret_cast<uint16_t *>(tile)), lane(lane)
    {
        const long each = (it.end - it.begin) / 32 / BUILD_WAVES + ((it.end - it.begin) / 32 % BUILD_WAVES != 0);
        end = min((long)it.begin / 32 + (eighth + 1) * each, (long)it.end / 32);
        next = first = min((long)it.begin / 32 + eighth * each, end);
        ask();
    }
    __device__ __forceinline__ void ask()
    {
        if (next >= end) return;
        if (acol) {
            values = reinterpret_cast<const u32x4 *>(acol)[next * 64 + lane];
        } else {
            const int i = (int)(next - first) & 63;
            if (i == 0) ranges = next + lane < end ? range[next + lane] : int2{0, 0};
            const int from = __builtin_amdgcn_readlane(ranges.x, i);
            n = __builtin_amdgcn_readlane(ranges.y, i) - from; // 128 at most
            e[0] = lane < n ? entries[from + lane] : 0;
            e[1] = lane + 64 < n ? entries[from + lane + 64] : 0;
        }
        next++;
    }
    __device__ __forceinline__ u32x4 take()
    {
        if (acol) {
            const u32x4 v = values;
            ask();
            return v;
        }
        asm volatile("" ::: "memory");
        reinterpret_cast<u32x4 *>(tile)[lane] = (u32x4){0, 0, 0, 0};
        asm volatile("" ::: "memory");
        if (lane < n) tile[(e[0] & 0xffffu) / 2] = (uint16_t)(e[0] >> 16);
        if (lane + 64 < n) tile[(e[1] & 0xffffu) / 2] = (uint16_t)(e[1] >> 16);
        asm volatile("" ::: "memory");
        ask();
        return reinterpret_cast<const u32x4 *>(tile)[lane];
    }
};
__device__ __forceinline__ uint32_t half_of(const u32x4 &v, int j) { return j & 1 ? v[j / 2] >> 16 : v[j / 2] & 0xffffu; }
// Nonzeros of the lane's 8 values
__device__ __forceinline__ int nonzeros(const u32x4 &v)
{
    int n = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) n += (half_of(v, j) & 0x7fffu) != 0;
    return n;
}

// Nonzeros of the rows of an item: of a block row that is one item to length, and to the numbers of rows of every kind; of a part of a block row to
// its own 16 in parts.  before: nonzeros of the eighths before every eighth of the item.  A workgroup takes an item.
__global__ __launch_bounds__(64 * BUILD_WAVES) void resident_lengths_kernel(const WorkItem *__restrict__ items, const uint16_t *__restrict__ acol,
                                                                            const uint32_t *__restrict__ entries, const int2 *__restrict__ range,
                                                                            int32_t *__restrict__ length, int32_t *__restrict__ parts, int32_t *__restrict__ before,
                                                                            ResidentTotals *__restrict__ totals)
{
    __shared__ u32x4 tiles[BUILD_WAVES][64];
    __shared__ int32_t of[BUILD_WAVES][16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const WorkItem it = items[blockIdx.x];
    int n = 0;
    Steps steps(it, w, acol, entries, range, tiles[w], lane);
    for (long s = steps.first; s < steps.end; s++) n += nonzeros(steps.take());
    n += __shfl_xor(n, 16);
    n += __shfl_xor(n, 32);
    if (lane < 16) of[w][lane] = n;
    __syncthreads();
    if (w) return;
    if (lane >= 16) return;
    const int m = lane; // row
    int all = 0;
#pragma unroll
    for (int k = 0; k < BUILD_WAVES; k++) {
        before[((size_t)blockIdx.x * BUILD_WAVES + k) * 16 + m] = all;
        all += of[k][m];
    }
    (it.dst < 0 ? length + it.block_row * 16 : parts + it.dst * 16)[m] = all;
    if (it.dst >= 0) return;
    // one addition for the rows of a kind
    const int copy = (int)blockIdx.x % COUNTS;
    const int kind = kind_of(all);
    int same = 0, first = 16, most = all;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int other = __shfl(kind, k);
        if (other == kind) same++, first = min(first, k);
        most = max(most, __shfl(all, k));
    }
    if (first == m) atomicAdd(&totals->rows_of[copy][kind], (uint32_t)same);
    if (m == 0) atomicMax(&totals->longest_of[copy], (uint32_t)most);
}

// parts of a split block row: from nonzeros of every part to those of the parts before it.  A wavefront takes a block row, four parts at a time.
__global__ __launch_bounds__(64) void resident_parts_kernel(const SplitRow *__restrict__ split, int32_t *__restrict__ length, int32_t *__restrict__ parts,
                                                            ResidentTotals *__restrict__ totals)
{
    const SplitRow row = split[blockIdx.x];
    const int lane = threadIdx.x, g = lane >> 4;
    int before = 0;
    for (int p = row.slot_begin; p < row.slot_end; p += 4) {
        const int n = p + g < row.slot_end ? parts[(p + g) * 16 + (lane & 15)] : 0;
        int mine = before;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int of = __shfl(n, (lane & 15) + 16 * k);
            mine += k < g ? of : 0;
            before += of;
        }
        if (p + g < row.slot_end) parts[(p + g) * 16 + (lane & 15)] = mine;
    }
    if (lane < 16) {
        length[row.block_row * 16 + lane] = before;
        atomicAdd(&totals->rows_of[blockIdx.x % COUNTS][kind_of(before)], 1u);
        atomicMax(&totals->longest_of[blockIdx.x % COUNTS], (uint32_t)before);
    }
}

// rows_of[0][kind] becomes the place of the first row of that kind; first[s] the fours before slice s (64 places), first[n_slices] those of all.  One workgroup.
__global__ __launch_bounds__(1024) void resident_slices_kernel(uint32_t *__restrict__ first, ResidentTotals *__restrict__ totals)
{
    __shared__ uint32_t place[KINDS + 1], part[1024], carry;
    const int t = (int)threadIdx.x;
    auto scan = [&](uint32_t v) { // exclusive sum over the workgroup; part[1023] holds the inclusive one of all
        part[t] = v;
        __syncthreads();
        for (int d = 1; d < 1024; d *= 2) {
            const uint32_t o = t >= d ? part[t - d] : 0;
            __syncthreads();
            part[t] += o;
            __syncthreads();
        }
        return part[t] - v;
    };
    uint32_t rows = 0;
    if (t < KINDS)
#pragma unroll
        for (int k = 0; k < COUNTS; k++) rows += totals->rows_of[k][t];
    const uint32_t before = scan(rows << lanes_log(t));
    const uint32_t places = part[1023];
    if (t < KINDS) place[t] = before, totals->rows_of[0][t] = before;
    if (t == 0) {
        place[KINDS] = 0xffffffffu, carry = 0;
        uint32_t longest = 0;
        for (int k = 0; k < COUNTS; k++) longest = max(longest, totals->longest_of[k]);
        totals->longest = longest;
    }
    __syncthreads();
    const int n_slices = (int)((places + 63) / 64);
    for (int s0 = 0; s0 < n_slices; s0 += 1024) {
        const int s = s0 + t;
        uint32_t fours = 0;
        if (s < n_slices) { // the last kind whose place is not behind the slice's first row
            int lo = 0, hi = KINDS;
            while (hi - lo > 1) {
                const int mid = (lo + hi) / 2;
                if (place[mid] <= (uint32_t)s * 64u) lo = mid; else hi = mid;
            }
            const uint32_t len = lo < SHARED ? PART : (uint32_t)(SHARED + PART - lo);
            fours = (len + 4) / 4; // the row's number first
        }
        const uint32_t at = scan(fours);
        if (s < n_slices) first[s] = carry + at;
        __syncthreads();
        if (t == 0) carry += part[1023];
        __syncthreads();
    }
    if (t == 0) first[n_slices] = carry, totals->n_slices = (uint32_t)n_slices, totals->fours = carry, totals->places = places;
}

// The place of every row among the sorted ones, and the first words of its lanes; the lists of lanes without a row, and a four of zeros behind all.
__global__ __launch_bounds__(1024) void resident_places_kernel(const int32_t *__restrict__ length, int M, uint32_t *__restrict__ place,
                                                               const uint32_t *__restrict__ first, ResidentTotals *__restrict__ totals, uint32_t K, uint32_t *__restrict__ list)
{
    __shared__ uint32_t mine[KINDS];
    for (int i = threadIdx.x; i < KINDS; i += 1024) mine[i] = 0;
    __syncthreads();
    const int row = (int)(blockIdx.x * 1024 + threadIdx.x);
    const int kind = row < M ? kind_of(length[row]) : 0, log = lanes_log(kind);
    uint32_t at = 0;
    // empty rows, of which there may be many, a wavefront at a time
    const bool none = row < M && kind == KINDS - 1;
    const unsigned long long nones = __ballot(none);
    if (none) {
        const int lead = __ffsll((long long)nones) - 1, lane = threadIdx.x & 63;
        if (lane == lead) at = atomicAdd(&mine[kind], (uint32_t)__popcll(nones));
        at = __shfl(at, lead) + __popcll(nones & ((1ull << lane) - 1));
    } else if (row < M) {
        at = atomicAdd(&mine[kind], 1u << log);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < KINDS; i += 1024)
        if (mine[i]) mine[i] = atomicAdd(&totals->rows_of[0][i], mine[i]);
    __syncthreads();
    auto word = [&](uint32_t at) -> uint32_t & { return list[(size_t)first[at / 64] * 256 + (at & 63) * 4]; };
    if (row < M) {
        at += mine[kind];
        place[row] = at;
        uint32_t *const to = &word(at);
        for (uint32_t k = 0; k < 1u << log; k++) to[k * 4] = (uint32_t)log << ROW_BITS | (uint32_t)row;
    }
    if (blockIdx.x == 0 && totals->places + threadIdx.x < totals->n_slices * 64) {
        uint32_t *const to = &word(totals->places + threadIdx.x);
        to[0] = PADDED;
        for (uint32_t w = 1; w < (totals->fours - first[totals->n_slices - 1]) * 4; w++) to[w / 4 * 256 + (w & 3)] = K;
    }
    if (blockIdx.x == 0 && threadIdx.x < 256) list[(size_t)totals->fours * 256 + threadIdx.x] = K;
}

// The nonzeros of every row in the order of their columns behind the first words, and zeros that meet the row of zeros behind B.  list: of slice s from 256 * first[s] on, four words after the other
// for each lane.
__global__ __launch_bounds__(64 * BUILD_WAVES) void resident_fill_kernel(const WorkItem *__restrict__ items, const uint16_t *__restrict__ acol,
                                                                         const uint32_t *__restrict__ entries, const int2 *__restrict__ range,
                                                                         const int32_t *__restrict__ cols, const int32_t *__restrict__ length,
                                                                         const int32_t *__restrict__ parts, const int32_t *__restrict__ before_eighth,
                                                                         const uint32_t *__restrict__ place,
                                                                         const uint32_t *__restrict__ first, uint32_t K, bool zeros_there, uint32_t *__restrict__ list)
{
    __shared__ u32x4 tiles[BUILD_WAVES][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4;
    const WorkItem it = items[blockIdx.x];
    const int row = it.block_row * 16 + (lane & 15), all_of_row = length[row], log = lanes_log(kind_of(all_of_row));
    const uint32_t at = place[row], slice = at / 64; // the lanes that share a row are in one slice
    uint32_t *const to = list + (size_t)first[slice] * 256 + (at & 63) * 4;
    const int room = (int)(first[slice + 1] - first[slice]) * 4, each = max((all_of_row + (1 << log) - 1) >> log, 1);
    const float per_each = 1.0f / (float)each; // for numbers below MAX_ROW: a product has the quotient's whole part
    int done = (it.dst < 0 ? 0 : parts[it.dst * 16 + (lane & 15)]) + before_eighth[((size_t)blockIdx.x * BUILD_WAVES + w) * 16 + (lane & 15)];
    Steps steps(it, w, acol, entries, range, tiles[w], lane);
    auto columns = [&](long s, int i) { return reinterpret_cast<const u32x4 *>(cols)[s * 8 + g * 2 + i]; };
    u32x4 here[2], soon[2];
    if (steps.first < steps.end) soon[0] = columns(steps.first, 0), soon[1] = columns(steps.first, 1);
    for (long s = steps.first; s < steps.end; s++) {
        here[0] = soon[0], here[1] = soon[1];
        if (s + 1 < steps.end) soon[0] = columns(s + 1, 0), soon[1] = columns(s + 1, 1);
        const u32x4 v = steps.take();
        const int n = nonzeros(v);
        int before = 0, all = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int of = __shfl(n, (lane & 15) + 16 * k);
            before += k < g ? of : 0;
            all += of;
        }
        int o = done + before;
#pragma unroll
        for (int j = 0; j < 8; j++) { // the even columns come first
            const uint32_t h = half_of(v, j);
            if (h & 0x7fffu) {
                const int share = log ? (int)(((float)o + 0.5f) * per_each) : 0, word = o - share * each + 1;
                if (word < room && share < 1 << log) to[(size_t)(word / 4) * 256 + (word & 3) + share * 4] = h << 16 | here[j & 1][j >> 1];
                o++;
            }
        }
        done += all;
    }
    if (!zeros_there && done == all_of_row) // behind the last of them
        for (int share = 0; share < 1 << log; share++)
            for (int word = min(max(all_of_row - share * each, 0), each) + 1 + g; word < room; word += 4) to[(size_t)(word / 4) * 256 + (word & 3) + share * 4] = K;
}

// ---- the product ----

template <int T, bool C_F32>
__global__ __launch_bounds__(1024) void spmm_resident_kernel(const u32x4 *__restrict__ list, const uint32_t *__restrict__ first, int n_slices, const uint16_t *__restrict__ B, void *__restrict__ C, int N, int K, int groups, int shares,
                                                             int by_group)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int units = groups * shares, per_xcd = (units + 7) / 8;
    const int u = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (u >= units) return;
    const int n0 = (by_group ? u / shares : u % groups) * T, share = by_group ? u % shares : u / groups;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int all = shares * WAVES, me = share * WAVES + w;
    auto slice_of = [&](int j) { return j * all + (j & 1 ? all - 1 - me : me); };

    // the fours of the wavefront's slices one after the other, AHEAD of the products
    int j_next = -1;
    uint32_t c_next = 0, c_end = 0;
    auto load = [&]() {
        if (c_next == c_end) {
            const int s = slice_of(++j_next);
            if (s < n_slices) c_next = first[s], c_end = first[s + 1];
            else c_next = first[n_slices], c_end = c_next + 1, j_next--; // past the end: zeros
        }
        return list[(size_t)(c_next++) * 64 + lane];
    };
    u32x4 q[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) q[i] = load();

    // two rows of B a lane at a time
    {
        const uint16_t *const b = B + (size_t)n0 * K;
        constexpr int U = 16 / T; // 16 loads a lane at a time
        const int last = K / 2 - 1;
        for (int k0 = (int)threadIdx.x; k0 <= last; k0 += 1024 * U) {
            uint32_t v[U][T];
#pragma unroll
            for (int i = 0; i < U; i++)
#pragma unroll
                for (int t = 0; t < T; t++) v[i][t] = *reinterpret_cast<const uint32_t *>(b + (size_t)t * K + 2 * min(k0 + 1024 * i, last));
#pragma unroll
            for (int i = 0; i < U; i++) {
                uint32_t o[T];
#pragma unroll
                for (int t = 0; t < T; t += 2) {
                    o[t / 2] = __builtin_amdgcn_perm(v[i][t + 1], v[i][t], 0x05040100u);
                    o[T / 2 + t / 2] = __builtin_amdgcn_perm(v[i][t + 1], v[i][t], 0x07060302u);
                }
                if (k0 + 1024 * i <= last)
#pragma unroll
                    for (int t = 0; t < T; t++) lds[(size_t)(k0 + 1024 * i) * T + t] = o[t];
            }
        }
        if (threadIdx.x < T / 2) lds[(size_t)K / 2 * T + threadIdx.x] = 0; // what padding names
    }
    __syncthreads();

    int j = 0, s = slice_of(0);
    uint32_t row = PADDED; // and the lanes that share it
    uint32_t left = 0;
    bool fresh;
    floats<T> acc;
    auto begin = [&] {
        left = first[s + 1] - first[s];
        acc = 0.0f;
        fresh = true;
    };
    auto store = [&] {
        const uint32_t log = row >> ROW_BITS, m = row & PADDED;
        if (__any(log != 0))
            for (uint32_t d = 1; d < 1u << SHARED; d *= 2)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const float other = __shfl_xor(acc[t], d);
                    if (d < 1u << log) acc[t] += other;
                }
        if (m == PADDED || (lane & ((1u << log) - 1))) return;
        if constexpr (C_F32) {
            constexpr int V = T < 4 ? T : 4;
            float *const c = static_cast<float *>(C) + (size_t)m * N + n0;
#pragma unroll
            for (int t = 0; t < T; t += V) {
                floats<V> v;
#pragma unroll
                for (int i = 0; i < V; i++) v[i] = acc[t + i];
                *reinterpret_cast<floats<V> *>(c + t) = v;
            }
        } else {
            *reinterpret_cast<halves<T> *>(static_cast<uint16_t *>(C) + (size_t)m * N + n0) = __builtin_convertvector(acc, halves<T>);
        }
    };
    if (s >= n_slices) return;
    begin();
    bool more = true;
    while (more) { // looked at once a round: the loads of the rounds would all be waited for where a round could end in the middle
#pragma unroll
        for (int k = 0; k < AHEAD; k++) {
            uint32_t e[4];
            halves<T> b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) e[i] = q[k][i];
            if (fresh) row = e[0], e[0] = (uint32_t)K, fresh = false;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t at;
                asm("v_mad_u32_u16 %0, %1, %2, 0" : "=v"(at) : "v"(e[i]), "n"(2 * T)); // its low half
                typedef __attribute__((address_space(3))) const halves<T> lds_row;
                b[i] = *(lds_row *)(uintptr_t)at;
            }
#pragma unroll
            for (int t = 0; t < T; t++) {
                float sum = 0.0f; // of four first: shorter chains of rounded sums
#pragma unroll
                for (int i = 0; i < 4; i++) sum = fmaf((float)__builtin_bit_cast(f16x2, e[i])[1], (float)b[i][t], sum);
                acc[t] += sum;
            }
            q[k] = load();
            if (--left == 0) {
                store();
                s = slice_of(++j);
                if (s < n_slices) begin();
                else more = false, left = AHEAD; // zeros for the rest of the round
            }
        }
    }
}

int g_force_columns = 0, g_force_shares = 0; // test hook

// Workgroups of the same columns on one XCD, whose L2 then reads those columns of B alone, or workgroups of the same rows, whose
// parts of a row of C meet in one L2.  16384 rows, 16 a row, rows together -> columns together, us: N = 64, K = 8192 6.4 -> 8.0; N = 128, K = 1040
// 6.9 -> 8.2, K = 8192 10.1 -> 9.5; N = 256, K = 8192 13.7 -> 10.9, K = 16384 16.8 -> 14.0.
bool columns_together(size_t K, size_t N) { return N >= 128 && N * K >= (size_t)1 << 20; }

// The shares of the rows that take the least time with T columns a workgroup.  Of a round of 256 workgroups: B into LDS (70 KB/us), the
// fours one after the other (12, 14 or 23 ns on 2, 4 or 8 columns) and the ends of slices; of all: the pieces of C of a row and T columns, which
// the L2s take one by one, and bytes.  Fitted to 259 products of 40 uniform random matrices and 7 stencils, M and K 1,040 to 63,760, N = 8 to 816: 11 %
// standard deviation, and what it picks is 0.6 % from the best tried in the mean.  Estimate (measured), us: 18736 x 18704, 38 a row, N = 88, 4 columns,
// 11 shares 12.7 (13.4); 2000 x 6448, 40 a row, N = 816, 8 and 2 10.6 (10.6); 32400 x 2096, 17 a row, N = 680, fp32, 8 and 3 38 (51).
ResidentLaunch launch_of(const ResidentPlan &p, size_t K, size_t N, int T)
{
    ResidentLaunch best{T, (int)(N / T), 1, 1e30};
    if (lds_of(K, T) > MAX_LDS || N % T) return best;
    const double four = T == 2 ? 0.0124 : T == 4 ? 0.014 : 0.0232, fill = 2.2 + 1.41e-5 * (double)K * 2.0 * T;
    const int most = std::max(1, std::min((p.n_slices + WAVES - 1) / WAVES, 512 / best.groups + 1));
    for (int shares = g_force_shares ? std::min(g_force_shares, most) : 1; shares <= (g_force_shares ? g_force_shares : most); shares++) {
        const int rounds = (best.groups * shares + 255) / 256;
        const double us = rounds * (fill + std::max((double)p.fours / shares * four + (double)p.n_slices / shares * 0.012, p.longest / 4 * 0.14));
        if (us < best.us) best.us = us, best.shares = shares;
    }
    const double b = 2e-6 * (double)K * (double)N, rows = 64.0 * p.n_slices;
    best.us += 1.4 + 2.4e-6 * rows * best.groups + ((columns_together(K, N) ? 1.0 : 8.0) * b + 2e-6 * rows * (double)N) / 16.0;
    return best;
}

std::atomic<int64_t> g_searches{0}; // test hook
ResidentLaunch best_launch(const ResidentPlan &p, size_t K, size_t N)
{
    g_searches.fetch_add(1, std::memory_order_relaxed);
    ResidentLaunch best;
    for (int T : {8, 4, 2}) {
        if (g_force_columns && T != g_force_columns) continue;
        const ResidentLaunch x = launch_of(p, K, N, T);
        if (x.us < best.us) best = x;
    }
    return best;
}

// The kernel may have as much LDS as there is: said once on a device, when a plan is made, so that a captured launch says nothing.
template <int T, bool C_F32>
hipError_t prepare()
{
    static std::atomic<uint64_t> prepared{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || (dev < 64 && prepared.load(std::memory_order_relaxed) >> dev & 1)) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(spmm_resident_kernel<T, C_F32>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MAX_LDS);
    if (e == hipSuccess && dev < 64) prepared.fetch_or(1ull << dev, std::memory_order_relaxed);
    return e;
}

template <int T, bool C_F32>
hipError_t launch_as(const SpmmArgs &a, const ResidentPlan &p, const ResidentLaunch &l, hipStream_t st)
{
    const hipError_t e = prepare<T, C_F32>();
    if (e != hipSuccess) return e;
    const int units = l.groups * l.shares;
    hipLaunchKernelGGL((spmm_resident_kernel<T, C_F32>), dim3((unsigned)((units + 7) / 8 * 8)), dim3(1024), lds_of(a.K, T), st, (const u32x4 *)p.d_list, p.d_first, p.n_slices,
                       a.B, a.C, (int)a.N, (int)a.K, l.groups, l.shares, (int)columns_together(a.K, a.N));
    return hipGetLastError();
}

} // namespace

double resident_estimate_us(size_t M, size_t K, size_t N, int64_t nnz, bool long_rows)
{
    ResidentPlan p;
    p.n_slices = (int)((M + 63) / 64);
    p.fours = nnz / 256 + (int64_t)p.n_slices * 3 / 4;
    if (long_rows) p.fours += nnz / 768, p.longest = PART; // R-MAT scales 12 to 14: a third more
    return best_launch(p, K, N).us;
}
// Worked out once for the plan's own width: 0.2 us of a call with 1,024 slices (65536 rows, N = 8 5.1 -> 4.9 of host time), nothing with 64 or fewer.
void resident_settle(ResidentPlan &p, size_t K, size_t N)
{
    p.n = N;
    p.own = best_launch(p, K, N);
}
ResidentLaunch resident_launch(const ResidentPlan &p, size_t K, size_t N)
{
    return N == p.n && !g_force_columns ? p.own : best_launch(p, K, N);
}
bool resident_forced() { return g_force_columns > 0; }
bool resident_holds(size_t K) { return lds_of(K, 2) <= MAX_LDS; }

hipError_t launch_resident(const SpmmArgs &a, const ResidentPlan &p, const ResidentLaunch &l, hipStream_t st)
{
    if (l.columns == 8) return a.c_f32 ? launch_as<8, true>(a, p, l, st) : launch_as<8, false>(a, p, l, st);
    if (l.columns == 4) return a.c_f32 ? launch_as<4, true>(a, p, l, st) : launch_as<4, false>(a, p, l, st);
    if (l.columns == 2) return a.c_f32 ? launch_as<2, true>(a, p, l, st) : launch_as<2, false>(a, p, l, st);
    return hipErrorInvalidValue;
}

void resident_destroy(ResidentPlan *p)
{
    if (!p) return;
    if (p->d_list) (void)dev_free(p->d_list);
    if (p->d_first) (void)dev_free(p->d_first - IN_FRONT);
    delete p;
}

hipError_t resident_build(const CompactPlan &c, size_t M, size_t K, int64_t nnz, ResidentPlan **out)
{
    *out = nullptr;
    if (c.n_items == 0 || nnz <= 0 || nnz > 0x3fffffff || M + (size_t)nnz / 32 >= PADDED || !resident_holds(K)) return hipSuccess;
    ResidentPlan *p = new (std::nothrow) ResidentPlan();
    if (!p) return hipErrorOutOfMemory;
    // A shared row takes a place for every 32 of its nonzeros or fewer.  Fours: those of the nonzeros, one more a slice for the first words, PART / 4 + 1 a
    // slice of shared rows, and what the longest rows leave the shorter ones of their slice.
    const size_t most_slices = (M + (size_t)nnz / 32) / 64 + 1;
    const size_t fours = ((size_t)nnz + 255) / 256 + most_slices + (PART / 4 + 1) * ((size_t)nnz / 2048 + 2) + 1;
    DevScratch tmp;
    uint32_t *places = nullptr;
    int32_t *lengths = nullptr, *parts = nullptr, *before = nullptr;
    ResidentTotals *totals = nullptr;
    hipError_t e = tmp.alloc((2 * M + 16 * (size_t)c.n_slots + 16 * BUILD_WAVES * (size_t)c.n_items) * sizeof(uint32_t));
    if (e == hipSuccess) {
        places = static_cast<uint32_t *>(tmp.p), lengths = reinterpret_cast<int32_t *>(places + M), parts = lengths + M, before = parts + 16 * (size_t)c.n_slots;
        e = dev_malloc(&p->d_list, fours * 1024);
    }
    if (e == hipSuccess) e = dev_malloc(&totals, (IN_FRONT + most_slices + 1) * sizeof(uint32_t));
    if (e == hipSuccess) {
        p->d_first = reinterpret_cast<uint32_t *>(totals) + IN_FRONT;
        e = hipMemsetAsync(totals, 0, IN_FRONT * sizeof(uint32_t), nullptr);
    }
    // the zeros of lanes that share rows are many: written beforehand
    const bool long_rows = c.n_split_rows > 0 || nnz > (int64_t)M * (PART / 2);
    if (e == hipSuccess && long_rows) e = hipMemsetD32Async((hipDeviceptr_t)p->d_list, (int)K, fours * 256, nullptr);
    if (e == hipSuccess) {
        const dim3 items((unsigned)c.n_items), rows((unsigned)((M + 1023) / 1024));
        hipLaunchKernelGGL(resident_lengths_kernel, items, dim3(64 * BUILD_WAVES), 0, nullptr, c.d_items, c.d_acol, c.d_entries, c.d_step_range, lengths, parts, before, totals);
        if (c.n_split_rows) hipLaunchKernelGGL(resident_parts_kernel, dim3((unsigned)c.n_split_rows), dim3(64), 0, nullptr, c.d_split, lengths, parts, totals);
        hipLaunchKernelGGL(resident_slices_kernel, dim3(1), dim3(1024), 0, nullptr, p->d_first, totals);
        hipLaunchKernelGGL(resident_places_kernel, rows, dim3(1024), 0, nullptr, lengths, (int)M, places, p->d_first, totals, (uint32_t)K, p->d_list);
        hipLaunchKernelGGL(resident_fill_kernel, items, dim3(64 * BUILD_WAVES), 0, nullptr, c.d_items, c.d_acol, c.d_entries, c.d_step_range, c.d_cols, lengths, parts, before,
                           places, p->d_first, (uint32_t)K, long_rows, p->d_list);
        e = hipGetLastError();
    }
    for (auto f : {prepare<2, false>, prepare<2, true>, prepare<4, false>, prepare<4, true>, prepare<8, false>, prepare<8, true>})
        if (e == hipSuccess) e = f();
    struct {
        uint32_t n_slices, fours, longest; // as ResidentTotals begins
    } n{};
    if (e == hipSuccess) e = hipMemcpy(&n, totals, sizeof n, hipMemcpyDeviceToHost);
    tmp.idle = e == hipSuccess;
    p->n_slices = (int)n.n_slices;
    p->fours = n.fours;
    p->longest = (int)std::min<uint32_t>(n.longest, PART);
    if (e != hipSuccess || n.longest > MAX_ROW) {
        (void)hipDeviceSynchronize();
        resident_destroy(p);
        return e;
    }
    *out = p;
    return hipSuccess;
}

} // namespace smat

// Test hook: the columns of B that a workgroup holds (2, 4 or 8; 0 = chosen, -1 = no plan takes the kernel) and the shares of the rows (0 = chosen).
extern "C" void smat_internal_resident_force(int columns, int shares) { smat::g_force_columns = columns; smat::g_force_shares = shares; }
// Test hook: launches that were worked out so far.
extern "C" int64_t smat_internal_resident_searches(void) { return smat::g_searches.load(); }
