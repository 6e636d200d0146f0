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
// end together and the wavefronts have equally much.  Lists are padded to fours of nonzeros by zeros that meet a row of zeros behind B.
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
constexpr int PADDED = 0x7fffffff;     // the row of a lane that has none
constexpr int AHEAD = 4;               // fours that a wavefront asks for ahead
constexpr int MAX_ROW = 2047;          // nonzeros of a row

size_t lds_of(size_t K, int T) { return ((K + 1) * 2 * T + 15) / 16 * 16; }

// ---- the lists, from the compact kernel's ----

// The steps of 32 listed columns of an item one after the other: of each the 8 values of row `lane % 16` in columns 8 * (lane / 16) .., asked
// for a step ahead (a wavefront that asked when it needed them waited for three loads in turn every step: 16384 rows of 16 25 -> 15 us).
constexpr int BUILD_WAVES = 4; // of a workgroup: as many as there are block rows would be too few workgroups
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
    __device__ __forceinline__ Steps(const WorkItem &it, const uint16_t *acol, const uint32_t *entries, const int2 *range, u32x4 *tile, int lane)
        : acol(acol), entries(entries), range(range), tile(reinterpret_cast<uint16_t *>(tile)), lane(lane), first(it.begin / 32), end(it.end / 32), next(first)
    {
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

// length[row] of every row, and how many rows are of every length.  A wavefront takes a block row.
__global__ __launch_bounds__(64 * BUILD_WAVES) void resident_lengths_kernel(const WorkItem *__restrict__ items, int n_items, const uint16_t *__restrict__ acol,
                                                                const uint32_t *__restrict__ entries, const int2 *__restrict__ range, int32_t *__restrict__ length,
                                                                uint32_t *__restrict__ rows_of)
{
    __shared__ u32x4 tiles[BUILD_WAVES][64];
    __shared__ uint32_t mine[MAX_ROW + 1];
    for (int i = threadIdx.x; i <= MAX_ROW; i += 64 * BUILD_WAVES) mine[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * BUILD_WAVES + w;
    if (i < n_items) {
        const WorkItem it = items[i];
        int n = 0;
        Steps steps(it, acol, entries, range, tiles[w], lane);
        for (long s = steps.first; s < steps.end; s++) n += nonzeros(steps.take());
        n += __shfl_xor(n, 16);
        n += __shfl_xor(n, 32);
        if (lane < 16) {
            length[it.block_row * 16 + lane] = n;
            atomicAdd(&mine[min(n, MAX_ROW)], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= MAX_ROW; i += 64 * BUILD_WAVES)
        if (mine[i]) atomicAdd(&rows_of[i], mine[i]);
}

// Longest rows first: rows_of[length] becomes the place of the first row of that length; first[s] the fours before slice s
// (64 rows), first[n_slices] those of all; *longest the longest row.  One workgroup.
__global__ __launch_bounds__(1024) void resident_slices_kernel(uint32_t *__restrict__ rows_of, int n_slices, uint32_t *__restrict__ first, uint32_t *__restrict__ longest)
{
    __shared__ uint32_t place[MAX_ROW + 2], part[1024], carry;
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
    const uint32_t a = rows_of[MAX_ROW - 2 * t], b = rows_of[MAX_ROW - 2 * t - 1];
    const uint32_t before = scan(a + b);
    place[2 * t] = before, place[2 * t + 1] = before + a; // of length MAX_ROW - index
    if (t == 0) place[MAX_ROW + 1] = 0xffffffffu, carry = 0;
    rows_of[MAX_ROW - 2 * t] = before, rows_of[MAX_ROW - 2 * t - 1] = before + a;
    __syncthreads();
    for (int s0 = 0; s0 < n_slices; s0 += 1024) {
        const int s = s0 + t;
        uint32_t fours = 0;
        if (s < n_slices) { // the last index whose place is not behind the slice's first row
            int lo = 0, hi = MAX_ROW + 1;
            while (hi - lo > 1) {
                const int mid = (lo + hi) / 2;
                if (place[mid] <= (uint32_t)s * 64u) lo = mid; else hi = mid;
            }
            const uint32_t len = (uint32_t)(MAX_ROW - lo);
            fours = (len + 4) / 4; // the row's number first
            if (s == 0) *longest = len;
        }
        const uint32_t at = scan(fours);
        if (s < n_slices) first[s] = carry + at;
        __syncthreads();
        if (t == 0) carry += part[1023];
        __syncthreads();
    }
    if (t == 0) first[n_slices] = carry;
}

// The place of every row among the sorted ones.
__global__ __launch_bounds__(1024) void resident_places_kernel(const int32_t *__restrict__ length, int M, uint32_t *__restrict__ next, uint32_t *__restrict__ place)
{
    __shared__ uint32_t mine[MAX_ROW + 1];
    for (int i = threadIdx.x; i <= MAX_ROW; i += 1024) mine[i] = 0;
    __syncthreads();
    const int row = (int)(blockIdx.x * 1024 + threadIdx.x);
    const int n = row < M ? min(length[row], MAX_ROW) : 0;
    uint32_t at = 0;
    if (row < M) at = atomicAdd(&mine[n], 1u);
    __syncthreads();
    for (int i = threadIdx.x; i <= MAX_ROW; i += 1024)
        if (mine[i]) mine[i] = atomicAdd(&next[i], mine[i]);
    __syncthreads();
    if (row < M) {
        at += mine[n];
        place[row] = at;
    }
}

// The number of every row and its nonzeros in the order of their columns.  list: of slice s from 256 * first[s] on, four words after the other for each lane.
__global__ __launch_bounds__(64 * BUILD_WAVES) void resident_fill_kernel(const WorkItem *__restrict__ items, int n_items, const uint16_t *__restrict__ acol,
                                                             const uint32_t *__restrict__ entries, const int2 *__restrict__ range, const int32_t *__restrict__ cols,
                                                             const uint32_t *__restrict__ place, const uint32_t *__restrict__ first, int M, uint32_t *__restrict__ list)
{
    __shared__ u32x4 tiles[BUILD_WAVES][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * BUILD_WAVES + w, g = lane >> 4;
    if (i == 0 && M + lane < (M + 63) / 64 * 64) list[(size_t)first[M / 64] * 256 + ((M + lane) & 63) * 4] = PADDED; // places without a row
    if (i >= n_items) return;
    const WorkItem it = items[i];
    const uint32_t at = place[it.block_row * 16 + (lane & 15)], slice = at / 64;
    uint32_t *const to = list + (size_t)first[slice] * 256 + (at & 63) * 4;
    const int room = (int)(first[slice + 1] - first[slice]) * 4;
    if (lane < 16) to[0] = (uint32_t)(it.block_row * 16 + lane);
    int done = 1;
    Steps steps(it, acol, entries, range, tiles[w], lane);
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
                if (o < room) to[(size_t)(o / 4) * 256 + (o & 3)] = h << 16 | here[j & 1][j >> 1];
                o++;
            }
        }
        done += all;
    }
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

    int j = 0, s = slice_of(0), row = -1;
    uint32_t left = 0;
    bool fresh;
    floats<T> acc;
    auto begin = [&] {
        left = first[s + 1] - first[s];
        acc = 0.0f;
        fresh = true;
    };
    auto store = [&] {
        if (row == PADDED) return;
        if constexpr (C_F32) {
            constexpr int V = T < 4 ? T : 4;
            float *const c = static_cast<float *>(C) + (size_t)row * N + n0;
#pragma unroll
            for (int t = 0; t < T; t += V) {
                floats<V> v;
#pragma unroll
                for (int i = 0; i < V; i++) v[i] = acc[t + i];
                *reinterpret_cast<floats<V> *>(c + t) = v;
            }
        } else {
            *reinterpret_cast<halves<T> *>(static_cast<uint16_t *>(C) + (size_t)row * N + n0) = __builtin_convertvector(acc, halves<T>);
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
            if (fresh) row = (int)e[0], e[0] = (uint32_t)K, fresh = false;
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

struct Launch {
    int groups, shares;
    double us;
};
// Workgroups of the same columns on one XCD, whose L2 then reads those columns of B alone, or workgroups of the same rows, whose
// parts of a row of C meet in one L2.  16384 rows, 16 a row, rows together -> columns together, us: N = 64, K = 8192 6.4 -> 8.0; N = 128, K = 1040
// 6.9 -> 8.2, K = 8192 10.1 -> 9.5; N = 256, K = 8192 13.7 -> 10.9, K = 16384 16.8 -> 14.0.
bool columns_together(size_t K, size_t N) { return N >= 128 && N * K >= (size_t)1 << 20; }

// The shares of the rows that take the least time with T columns a workgroup.  Of a round of 256 workgroups: B into LDS (70 KB/us), the
// fours one after the other (12, 14 or 23 ns on 2, 4 or 8 columns) and the ends of slices; of all: the pieces of C of a row and T columns, which
// the L2s take one by one, and bytes.  Fitted to 259 products of 40 uniform random matrices and 7 stencils, M and K 1,040 to 63,760, N = 8 to 816: 11 %
// standard deviation, and what it picks is 0.6 % from the best tried in the mean.  Estimate (measured), us: 18736 x 18704, 38 a row, N = 88, 4 columns,
// 11 shares 12.7 (13.4); 2000 x 6448, 40 a row, N = 816, 8 and 2 10.6 (10.6); 32400 x 2096, 17 a row, N = 680, fp32, 8 and 3 38 (51).
Launch launch_of(const ResidentPlan &p, size_t K, size_t N, int T)
{
    Launch best{(int)(N / T), 1, 1e30};
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

int best_columns(const ResidentPlan &p, size_t K, size_t N, Launch *l)
{
    int best = 0;
    l->us = 1e30;
    for (int T : {8, 4, 2}) {
        if (g_force_columns && T != g_force_columns) continue;
        const Launch x = launch_of(p, K, N, T);
        if (x.us < l->us) *l = x, best = T;
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
hipError_t launch_as(const SpmmArgs &a, const ResidentPlan &p, const Launch &l, hipStream_t st)
{
    const hipError_t e = prepare<T, C_F32>();
    if (e != hipSuccess) return e;
    const int units = l.groups * l.shares;
    hipLaunchKernelGGL((spmm_resident_kernel<T, C_F32>), dim3((unsigned)((units + 7) / 8 * 8)), dim3(1024), lds_of(a.K, T), st, (const u32x4 *)p.d_list, p.d_first, p.n_slices,
                       a.B, a.C, (int)a.N, (int)a.K, l.groups, l.shares, (int)columns_together(a.K, a.N));
    return hipGetLastError();
}

} // namespace

double resident_estimate_us(size_t M, size_t K, size_t N, int64_t nnz)
{
    ResidentPlan p;
    p.n_slices = (int)((M + 63) / 64);
    p.fours = nnz / 256 + (int64_t)p.n_slices * 3 / 4;
    Launch l;
    return best_columns(p, K, N, &l) ? l.us : 1e30;
}
double resident_launch_us(const ResidentPlan &p, size_t K, size_t N)
{
    Launch l;
    return best_columns(p, K, N, &l) ? l.us : 1e30;
}
bool resident_forced() { return g_force_columns > 0; }

hipError_t launch_resident(const SpmmArgs &a, const ResidentPlan &p, hipStream_t st)
{
    Launch l;
    const int T = best_columns(p, a.K, a.N, &l);
    if (T == 8) return a.c_f32 ? launch_as<8, true>(a, p, l, st) : launch_as<8, false>(a, p, l, st);
    if (T == 4) return a.c_f32 ? launch_as<4, true>(a, p, l, st) : launch_as<4, false>(a, p, l, st);
    if (T == 2) return a.c_f32 ? launch_as<2, true>(a, p, l, st) : launch_as<2, false>(a, p, l, st);
    return hipErrorInvalidValue;
}

void resident_destroy(ResidentPlan *p)
{
    if (!p) return;
    if (p->d_list) (void)dev_free(p->d_list);
    if (p->d_first) (void)dev_free(p->d_first);
    delete p;
}

hipError_t resident_build(const CompactPlan &c, size_t M, size_t K, int64_t nnz, ResidentPlan **out)
{
    *out = nullptr;
    if (c.n_split_rows || c.n_items == 0 || nnz <= 0 || nnz > 0x3fffffff || M > 0x3fffffff || lds_of(K, 2) > MAX_LDS) return hipSuccess;
    ResidentPlan *p = new (std::nothrow) ResidentPlan();
    if (!p) return hipErrorOutOfMemory;
    const int n_slices = p->n_slices = (int)((M + 63) / 64);
    // fours: those of the nonzeros and the rows' numbers, up to one more a slice, and what the longest rows leave the shorter ones of their slice
    const size_t fours = ((size_t)nnz + 255) / 256 + (size_t)n_slices + (MAX_ROW + 3) / 4 + 1;
    DevScratch tmp;
    uint32_t *lengths = nullptr, *places = nullptr, *rows_of = nullptr;
    hipError_t e = tmp.alloc((2 * M + MAX_ROW + 1) * sizeof(uint32_t));
    if (e == hipSuccess) {
        rows_of = static_cast<uint32_t *>(tmp.p), lengths = rows_of + MAX_ROW + 1, places = lengths + M;
        e = dev_malloc(&p->d_list, fours * 1024);
    }
    if (e == hipSuccess) e = dev_malloc(&p->d_first, ((size_t)n_slices + 2) * sizeof(uint32_t));
    if (e == hipSuccess) {
        e = hipMemsetAsync(rows_of, 0, (MAX_ROW + 1) * sizeof(uint32_t), nullptr);
    }
    if (e == hipSuccess) e = hipMemsetD32Async((hipDeviceptr_t)p->d_list, (int)K, fours * 256, nullptr);
    const unsigned wgs = (unsigned)((c.n_items + BUILD_WAVES - 1) / BUILD_WAVES);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(resident_lengths_kernel, dim3(wgs), dim3(64 * BUILD_WAVES), 0, nullptr, c.d_items, c.n_items, c.d_acol, c.d_entries, c.d_step_range, (int32_t *)lengths, rows_of);
        hipLaunchKernelGGL(resident_slices_kernel, dim3(1), dim3(1024), 0, nullptr, rows_of, n_slices, p->d_first, p->d_first + n_slices + 1);
        hipLaunchKernelGGL(resident_places_kernel, dim3((unsigned)((M + 1023) / 1024)), dim3(1024), 0, nullptr, (const int32_t *)lengths, (int)M, rows_of, places);
        hipLaunchKernelGGL(resident_fill_kernel, dim3(wgs), dim3(64 * BUILD_WAVES), 0, nullptr, c.d_items, c.n_items, c.d_acol, c.d_entries, c.d_step_range, c.d_cols, places, p->d_first,
                           (int)M, p->d_list);
        e = hipGetLastError();
    }
    for (auto f : {prepare<2, false>, prepare<2, true>, prepare<4, false>, prepare<4, true>, prepare<8, false>, prepare<8, true>})
        if (e == hipSuccess) e = f();
    uint32_t n[2] = {0, 0};
    if (e == hipSuccess) e = hipMemcpy(n, p->d_first + n_slices, sizeof n, hipMemcpyDeviceToHost);
    tmp.idle = e == hipSuccess;
    p->fours = n[0];
    p->longest = (int)n[1];
    if (e != hipSuccess || p->longest >= MAX_ROW) {
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
