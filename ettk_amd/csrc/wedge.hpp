// wedge.hpp -- device functions of the analytic missing wedge (shared by ccc.hip and avg.hip).
#pragma once
#include "common.hpp"

namespace ettk {

// ------------------------------------------------------------------ smoothed analytic wedge
// binary wedge (v1.d)(v2.d) <= 0, d = (i - N/2, j - N/2, k - N/2), on an N x N x nk grid: the half grid
// (nk = N/2 + 1, nbfWedge3D::getImageHalf, Wedge.h:313-360) or the full grid (nk = N, nbfWedge3D::getImage,
// Wedge.h:195-290, centre floor(N/2)); smoothed with the separable 3-tap Gaussian (sigma 2, radius factor 1/2:
// smoothWedgeImage, Wedge.h:432-445) clipped and renormalised at the borders of that grid
//
// Where the tilt axis runs along a direction of the lattice, a whole line of samples lies on both planes and its side is
// decided by the last bit of the two plane values; the CCC moves by 1e-4 with it.  The order in which a plane value is
// rounded is therefore written out, and is the same for every caller: v.x di, then v.y dj, then v.z dk, a product rounded by
// itself where that offset of the stencil is 0 and fused with the sum elsewhere, and at the centre v.y dj first.  So a
// sample on a plane may count as inside for one neighbour and as outside for another.  Of 36 rotations by multiples of
// 45 degrees, 32 distances agree with the FP64 oracle within 1.5e-5 at box 32; the other four are 1.7e-3 to 5.3e-3 off (5e-4
// to 1.3e-3 at 96), as they were when each kernel left the order to the compiler.  Rotations in general position have
// no such samples.
template <int A, int B, int C>
__device__ __forceinline__ float wedge_plane(const float* v, float di, float dj, float dk) {
#pragma clang fp contract(off)
    float s;
    if constexpr (A == 0 && B == 0) s = __builtin_fmaf(v[0], di, v[1] * dj);
    else if constexpr (B == 0) s = v[0] * di + v[1] * dj;
    else s = __builtin_fmaf(v[1], dj, v[0] * di);
    if constexpr (C == 0 && (A != 0 || B != 0)) return s + v[2] * dk;
    return __builtin_fmaf(v[2], dk, s);
}
template <int A, int B, int C>
__device__ __forceinline__ float wedge_bin(const float* v1, const float* v2, int i, int j, int k, int N) {
    const float di = (float)(i + A - N / 2), dj = (float)(j + B - N / 2), dk = (float)(k + C - N / 2);
    return wedge_plane<A, B, C>(v1, di, dj, dk) * wedge_plane<A, B, C>(v2, di, dj, dk) <= 0.f ? 1.f : 0.f;
}
// taps of a position: 3 inside, 2 at the borders, renormalised (constants: the same divisions at compile time)
__device__ __forceinline__ void tap3(int idx, int n, float* w) {
    constexpr float g = 0.88249690258459540286f;  // exp(-1/8)
    constexpr float in = 1.f / (g + 1.f + g), edge = 1.f / (1.f + g);
    const bool first = idx <= 0, last = idx >= n - 1;
    w[1] = first || last ? edge : in;
    w[0] = first ? 0.f : last ? g * edge : g * in;
    w[2] = last ? 0.f : first ? g * edge : g * in;
}
// Away from both planes the 27 binary samples all equal the centre's: true when they do, with that sample
__device__ __forceinline__ bool wedge_uniform(const float* v1, const float* v2, int i, int j, int k, int N, bool& in) {
    const float di = (float)(i - N / 2), dj = (float)(j - N / 2), dk = (float)(k - N / 2);
    const float a0 = v1[0] * di + v1[1] * dj + v1[2] * dk, b0 = v2[0] * di + v2[1] * dj + v2[2] * dk;
    const float r1 = fabsf(v1[0]) + fabsf(v1[1]) + fabsf(v1[2]), r2 = fabsf(v2[0]) + fabsf(v2[1]) + fabsf(v2[2]);
    in = !(a0 * b0 > 0.f);
    return fabsf(a0) > r1 * 1.001f + 1e-3f && fabsf(b0) > r2 * 1.001f + 1e-3f;
}
// the kernel's sum at (i, j, k), accumulated in the same order as the stencil of ones would be: the smoothed value where
// all samples are 1
__device__ __forceinline__ float wedge_ones(int i, int j, int k, int N, int nk) {
    float wi[3], wj[3], wk[3];
    tap3(i, N, wi);
    tap3(j, N, wj);
    tap3(k, nk, wk);
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (wi[a] == 0.f) continue;
        float sj = 0.f;
#pragma unroll
        for (int b = 0; b < 3; b++) {
            if (wj[b] == 0.f) continue;
            float sk = 0.f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (wk[c] == 0.f) continue;
                sk += wk[c] * 1.f;
            }
            sj += wj[b] * sk;
        }
        acc += wi[a] * sj;
    }
    return acc;
}
// the 27-sample stencil
template <int A, int B>
__device__ __forceinline__ float wedge_row(const float* v1, const float* v2, int i, int j, int k, int N, const float* wk) {
    float s = 0.f;
    if (wk[0] != 0.f) s += wk[0] * wedge_bin<A, B, -1>(v1, v2, i, j, k, N);
    s += wk[1] * wedge_bin<A, B, 0>(v1, v2, i, j, k, N);
    if (wk[2] != 0.f) s += wk[2] * wedge_bin<A, B, 1>(v1, v2, i, j, k, N);
    return s;
}
template <int A>
__device__ __forceinline__ float wedge_slab(const float* v1, const float* v2, int i, int j, int k, int N, const float* wj,
                                            const float* wk) {
    float s = 0.f;
    if (wj[0] != 0.f) s += wj[0] * wedge_row<A, -1>(v1, v2, i, j, k, N, wk);
    s += wj[1] * wedge_row<A, 0>(v1, v2, i, j, k, N, wk);
    if (wj[2] != 0.f) s += wj[2] * wedge_row<A, 1>(v1, v2, i, j, k, N, wk);
    return s;
}
__device__ inline float wedge_stencil(const float* v1, const float* v2, int i, int j, int k, int N, int nk) {
    float wi[3], wj[3], wk[3];
    tap3(i, N, wi);
    tap3(j, N, wj);
    tap3(k, nk, wk);
    float acc = 0.f;
    if (wi[0] != 0.f) acc += wi[0] * wedge_slab<-1>(v1, v2, i, j, k, N, wj, wk);
    acc += wi[1] * wedge_slab<0>(v1, v2, i, j, k, N, wj, wk);
    if (wi[2] != 0.f) acc += wi[2] * wedge_slab<1>(v1, v2, i, j, k, N, wj, wk);
    return acc;
}
__device__ inline float wedge_smooth(const float* v1, const float* v2, int i, int j, int k, int N, int nk) {
    bool in;
    if (wedge_uniform(v1, v2, i, j, k, N, in)) return in ? wedge_ones(i, j, k, N, nk) : 0.f;
    return wedge_stencil(v1, v2, i, j, k, N, nk);
}

}  // namespace ettk
