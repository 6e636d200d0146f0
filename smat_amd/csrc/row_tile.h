// How a wavefront's accumulators map to C in the kernels that multiply whole 16x16 blocks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace smat {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f16x8 load_f16x8(const uint16_t *p)
{
    return *reinterpret_cast<const f16x8 *>(p);
}

// Column of C owned by MFMA output row i (0..15) of n-tile t inside a wave's
// panel.  Tiles are taken in groups of TG = min(TN, 4); inside a group the
// assignment interleaves tiles so that the 4*TG values a lane holds for one C
// row are consecutive columns.
template <int TN>
__device__ __forceinline__ int ncol_of(int t, int i)
{
    constexpr int TG = TN < 4 ? TN : 4;
    return 16 * TG * (t / TG) + 4 * TG * (i >> 2) + 4 * (t % TG) + (i & 3);
}

// acc[t][r] = C[br*16 + i16][n0 + ncol_of(t, 4*g + r)], to C or (dst >= 0) to workspace slot dst.
template <int TN, bool C_F32>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[TN], int br, int dst, int n0, int i16, int g, void *__restrict__ Cout,
                                           float *__restrict__ workspace, int N)
{
    constexpr int TG = TN < 4 ? TN : 4;
    const long m = (long)br * 16 + i16;
#pragma unroll
    for (int u = 0; u < TN / TG; u++) {
        const int nbase = n0 + 16 * TG * u + 4 * TG * g; // first of 4*TG consecutive columns
        if (dst >= 0) {
            // fp32 partial tile: slot-major, then the same row-major M x N addressing
            float *wrow = workspace + ((long)dst * 16 + i16) * (long)N;
#pragma unroll
            for (int tt = 0; tt < TG; tt++) {
                int n = nbase + 4 * tt;
                if (n < N) *reinterpret_cast<f32x4 *>(wrow + n) = acc[u * TG + tt];
            }
        } else if (C_F32) {
            float *crow = reinterpret_cast<float *>(Cout) + m * (long)N;
#pragma unroll
            for (int tt = 0; tt < TG; tt++) {
                int n = nbase + 4 * tt;
                if (n < N) *reinterpret_cast<f32x4 *>(crow + n) = acc[u * TG + tt];
            }
        } else {
            uint16_t *crow = reinterpret_cast<uint16_t *>(Cout) + m * (long)N;
            if constexpr (TG == 1) {
                f32x4 v = acc[u];
                f16x4 h = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                if (nbase < N) *reinterpret_cast<f16x4 *>(crow + nbase) = h;
            } else {
#pragma unroll
                for (int tt = 0; tt < TG; tt += 2) {
                    f32x4 v0 = acc[u * TG + tt], v1 = acc[u * TG + tt + 1];
                    f16x8 h = {(_Float16)v0[0], (_Float16)v0[1], (_Float16)v0[2], (_Float16)v0[3],
                               (_Float16)v1[0], (_Float16)v1[1], (_Float16)v1[2], (_Float16)v1[3]};
                    int n = nbase + 4 * tt;
                    if (n < N) *reinterpret_cast<f16x8 *>(crow + n) = h;
                }
            }
        }
    }
}

} // namespace smat
