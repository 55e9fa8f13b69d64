// tricubic.hpp -- VTK's tricubic interpolation (Keys a = -1/2, taps clamped to the volume) of an 8x8x8 tile of output
// voxels from an LDS-staged box of the input; shared by the CCC reslice (ccc.hip) and the extraction (extract.hip).
//
// The input voxels the 64-tap stencils of a tile can touch lie in the bounding box of the tile's transformed corners:
// at most floor(7 sqrt 3) + 1 + 4 = 17 voxels per axis for a rigid map.  That box (its actual extent, about 14 voxels
// per axis for a random rotation), with the volume's border replicated where it reaches outside (the taps clamp to
// the border), is staged in LDS at fixed strides, so every tap is a plain LDS read and the 4 taps of a row are
// consecutive words.  A non-rigid map whose box does not fit reads the clamped taps from global memory instead.
// Each wavefront interpolates a 4x4x4 block of the tile: the taps of its voxels then cover a compact region of the
// box and, with the row and plane strides 17 and 300, fall on fewer common LDS banks than those of an 8x8 plane.  A
// 17^3 box at these strides (20 KB) lets 8 workgroups share a CU's 160 KB of LDS.
#pragma once
#include "common.hpp"

namespace ettk {

static constexpr int kTriThreads = 256;
static constexpr int kTile = 8, kBox = 17, kSY = 17, kSZ = 300;
static constexpr float kTriTol = 7.62939453125e-06f;  // VTK's floor tolerance (2^-17)

__device__ __forceinline__ void keys_w(float f, float* w) {  // vtkTricubicInterpWeights
    const float fm1 = f - 1.f, fd2 = f * 0.5f, ft3 = f * 3.f;
    w[0] = -fd2 * fm1 * fm1;
    w[1] = ((ft3 - 2.f) * fd2 - 1.f) * fm1;
    w[2] = -((ft3 - 4.f) * f - 1.f) * fd2;
    w[3] = f * fd2 * fm1;
}

// staged box [lo, hi] per input axis (x, y, z) of the tile at (i0, j0, k0) under the map m (columns of the output axes,
// then the offset); it may reach outside the volume.  False when the map's box does not fit.
__device__ __forceinline__ bool tile_box(const float* m, int i0, int j0, int k0, int lo[3], int hi[3]) {
    bool fits = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float c0 = m[a] * i0 + m[3 + a] * j0 + m[6 + a] * k0 + m[9 + a];
        float ext = (kTile - 1) * (fabsf(m[a]) + fabsf(m[3 + a]) + fabsf(m[6 + a]));
        float mn = c0 + (kTile - 1) * (fminf(m[a], 0.f) + fminf(m[3 + a], 0.f) + fminf(m[6 + a], 0.f));
        lo[a] = (int)floorf(mn + kTriTol) - 1;
        hi[a] = (int)floorf(mn + ext + kTriTol) + 2;
        if (!(hi[a] - lo[a] + 1 <= kBox) || !(fabsf(mn) < 1e6f)) fits = false;
    }
    return fits;
}

// the box into LDS (kBox * kSZ floats): a 2-D thread map over (y, x), a loop over z, coordinates clamped to the volume
__device__ __forceinline__ void stage_tile_box(const float* __restrict__ vol, int nx, int ny, int nz, const int lo[3],
                                               const int hi[3], float* box) {
    constexpr int kRows = kTriThreads / kBox;
    const int t = threadIdx.x;
    const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
    const int x = t % kBox, y0 = t / kBox;
    if (t < kBox * kRows && x < wx) {
        const int gx = min(max(lo[0] + x, 0), nx - 1);
        for (int y = y0; y < wy; y += kRows) {
            const int gy = min(max(lo[1] + y, 0), ny - 1);
            const float* src = vol + (size_t)gy * nx + gx;
#pragma unroll 6
            for (int z = 0; z < wz; z++) {
                const int gz = min(max(lo[2] + z, 0), nz - 1);
                box[z * kSZ + y * kSY + x] = src[(size_t)gz * ny * nx];
            }
        }
    }
}

// voxel (offset within the tile) of item t < 512: t >> 6 numbers the tile's eight 4x4x4 blocks, t & 63 the voxel
// within its block; axis c runs fastest
__device__ __forceinline__ void tile_voxel(int t, int& a, int& b, int& c) {
    const int sb = t >> 6, l = t & 63;
    a = 4 * (sb >> 2) + (l >> 4);
    b = 4 * ((sb >> 1) & 1) + ((l >> 2) & 3);
    c = 4 * (sb & 1) + (l & 3);
}

// the sample at (px, py, pz) from the staged box
__device__ __forceinline__ float sample_box(const float* box, const int lo[3], const int hi[3], float px, float py,
                                            float pz) {
    const float xx = px + kTriTol, yy = py + kTriTol, zz = pz + kTriTol;
    int ix = (int)floorf(xx), iy = (int)floorf(yy), iz = (int)floorf(zz);
    // the box was sized from the tile's corners; a sample within rounding of a voxel boundary can floor one voxel
    // outside it: take the neighbouring cubic piece at f just outside [0, 1) instead (the Keys kernel is C1, the
    // value agrees to O(f^2) of a few ulps)
    ix = min(max(ix, lo[0] + 1), hi[0] - 2);
    iy = min(max(iy, lo[1] + 1), hi[1] - 2);
    iz = min(max(iz, lo[2] + 1), hi[2] - 2);
    float wx[4], wy[4], wz[4];
    keys_w(xx - ix, wx);
    keys_w(yy - iy, wy);
    keys_w(zz - iz, wz);
    const float* b0 = box + (iz - 1 - lo[2]) * kSZ + (iy - 1 - lo[1]) * kSY + (ix - 1 - lo[0]);
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < 4; a++) {
        float ay = 0.f;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float* row = b0 + a * kSZ + b * kSY;
            ay += wy[b] * (wx[0] * row[0] + wx[1] * row[1] + wx[2] * row[2] + wx[3] * row[3]);
        }
        acc += wz[a] * ay;
    }
    return acc;
}

// the sample at (px, py, pz) from global memory, taps clamped to the volume
__device__ __forceinline__ float sample_global(const float* __restrict__ vol, int nx, int ny, int nz, float px, float py,
                                               float pz) {
    const float xx = px + kTriTol, yy = py + kTriTol, zz = pz + kTriTol;
    const int ix = (int)floorf(xx), iy = (int)floorf(yy), iz = (int)floorf(zz);
    float wx[4], wy[4], wz[4];
    keys_w(xx - ix, wx);
    keys_w(yy - iy, wy);
    keys_w(zz - iz, wz);
    int cx[4], cy[4], cz[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        cx[q] = min(max(ix - 1 + q, 0), nx - 1);
        cy[q] = min(max(iy - 1 + q, 0), ny - 1);
        cz[q] = min(max(iz - 1 + q, 0), nz - 1);
    }
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < 4; a++) {
        float ay = 0.f;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float* row = vol + ((size_t)cz[a] * ny + cy[b]) * nx;
            ay += wy[b] * (wx[0] * row[cx[0]] + wx[1] * row[cx[1]] + wx[2] * row[cx[2]] + wx[3] * row[cx[3]]);
        }
        acc += wz[a] * ay;
    }
    return acc;
}

}  // namespace ettk
