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
// 17^3 box at these strides (20 KB) lets 7 workgroups share a CU.
//
// Bound by LDS and VALU together (the LDS is busy for 87% of the kernel, 48% of that with bank conflicts, and the SIMDs
// issue for 89%, at four cycles an instruction), so the rest of a tile is kept cheap: the box's bounds and the staging's
// plane addresses are scalar, tiles away from the volume's border test no sample, the box has a margin instead of a clamp
// per sample, counts are ballots and sums DPP.
// 240 evaluations at 64^3: 605 us, 686 before; extraction of 60 boxes 157 against 176 us.  Layouts that trade bank
// conflicts for address arithmetic are slower: voxel (x, y, z) on bank (x & 3) + 4 (y & 3) + 16 (z & 1) with the taps
// visited in a lane's own conflict-free order 675 us (VALU-bound, 1.5 times the instructions), without the z digit 721;
// pairs or quads of words per voxel read 20% faster by themselves but leave 3 workgroups or fewer per CU.
#pragma once
#include "common.hpp"

namespace ettk {

static constexpr int kTriThreads = 256;
static constexpr int kTile = 8, kBox = 17;
static constexpr int kSY = 17, kSZ = 300, kBoxWords = kBox * kSZ;
static_assert(kBox % 6 == 5, "the staging writes planes in sixes, the last five");
static constexpr float kTriTol = 7.62939453125e-06f;  // VTK's floor tolerance (2^-17)

__device__ __forceinline__ void keys_w(float f, float* w) {  // vtkTricubicInterpWeights
    const float fm1 = f - 1.f, fd2 = f * 0.5f, ft3 = f * 3.f;
    w[0] = -fd2 * fm1 * fm1;
    w[1] = ((ft3 - 2.f) * fd2 - 1.f) * fm1;
    w[2] = -((ft3 - 4.f) * f - 1.f) * fd2;
    w[3] = f * fd2 * fm1;
}

// What the staged box reaches beyond the tile's transformed corners, so that every sample's stencil lies in it whatever
// FP32 rounding does to the positions.  A sample inside the volume has terms of m[0..2] x + ... + m[9..11] whose magnitudes
// add up to A <= n + 4 N for a volume of n and an output box of N voxels per axis (a map that fits has rows of absolute sum
// below 2).  In any order, fused or not, a position with its floor tolerance takes 7 roundings of at most 2^-24 A, a bound
// of the box 9: 2^-20 A together, and the small terms of 7 voxels below 1e-5, kTriTol below 1e-5.  Up to N = 128 the floor
// of 1e-3 covers it; with the floor alone a box of 1024^3 cut beyond coordinate 8192 read taps that were not staged.
// A rigid map (corners 12.13 voxels apart at most) fits kBox with margins up to 0.43, coordinates of 4e5.
static constexpr float kMarginMin = 1e-3f, kMarginUlp = 9.5367431640625e-07f, kMarginSmall = 2e-5f;
__device__ __forceinline__ float tile_margin(int n, int N) {
    return fmaxf(kMarginMin, kMarginUlp * ((float)n + 4.f * (float)N) + kMarginSmall);
}

// staged box [lo, hi] per input axis (x, y, z) of the tile at (i0, j0, k0) under the map m (columns of the output axes,
// then the offset); it may reach outside the volume.  False when the map's box does not fit.  `inside`: the box fits and
// every sample of the tile lies in an nx x ny x nz volume, more than 1e-3 away from its border, so that no sample's
// validity needs a test.
__device__ __forceinline__ bool tile_box(const float* m, int i0, int j0, int k0, int nx, int ny, int nz, float margin,
                                         int lo[3], int hi[3], bool& inside) {
    bool fits = true;
    inside = true;
    const int n[3] = {nx, ny, nz};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float c0 = m[a] * i0 + m[3 + a] * j0 + m[6 + a] * k0 + m[9 + a];
        float ext = (kTile - 1) * (fabsf(m[a]) + fabsf(m[3 + a]) + fabsf(m[6 + a]));
        float mn = c0 + (kTile - 1) * (fminf(m[a], 0.f) + fminf(m[3 + a], 0.f) + fminf(m[6 + a], 0.f));
        // the same for every thread: kept in scalar registers, and with them the staging's row and plane arithmetic
        lo[a] = __builtin_amdgcn_readfirstlane((int)floorf(mn - margin) - 1);
        hi[a] = __builtin_amdgcn_readfirstlane((int)floorf(mn + ext + margin) + 2);
        // a map too steep, or a tile too far away, for these whole numbers does not fit either
        if (!(ext < (float)kBox) || !(fabsf(mn) < 1e6f) || hi[a] - lo[a] + 1 > kBox) fits = false;
        if (!(mn > -0.499f + margin && mn + ext < (float)n[a] - 0.501f - margin)) inside = false;
    }
    if ((unsigned long long)nx * ny >= (1ull << 30)) fits = false;  // the staging's offsets within a plane are 32-bit bytes
    inside = inside && fits;
    return fits;
}

// the box into LDS (kBoxWords floats): a 2-D thread map over (y, x), a loop over z whose plane addresses are scalar,
// coordinates clamped to the volume
__device__ __forceinline__ void stage_tile_box(const float* __restrict__ vol, int nx, int ny, int nz, const int lo[3],
                                               const int hi[3], float* box) {
    constexpr int kRows = kTriThreads / kBox;
    const int x = threadIdx.x % kBox, y0 = threadIdx.x / kBox;
    const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
    const size_t plane = (size_t)nx * ny;
    const int gx = min(max(lo[0] + x, 0), nx - 1);
#pragma unroll
    for (int pass = 0; pass < (kBox + kRows - 1) / kRows; pass++) {
        const int y = y0 + pass * kRows;
        if (y0 < kRows && x < wx && y < wy) {
            const int gy = min(max(lo[1] + y, 0), ny - 1);
            const unsigned off = ((unsigned)gy * nx + gx) * 4u;
            float* dst = box + y * kSY + x;
            // the plane's address advances in scalar registers; it stays where the clamped coordinate does
            const float* src = vol + (size_t)min(max(lo[2], 0), nz - 1) * plane;
            for (int z = 0; z < wz; z += 6, dst += 6 * kSZ) {  // six loads in flight; planes past the box are written unused
                float r[6];
#pragma unroll
                for (int u = 0; u < 6; u++) {
                    r[u] = at_byte(src, off);
                    const unsigned g = (unsigned)(lo[2] + z + u);  // step from this plane to the next one inside the volume
                    src += g < (unsigned)(nz - 1) ? plane : 0;
                }
#pragma unroll
                for (int u = 0; u < 5; u++) dst[u * kSZ] = r[u];
                if (z + 5 < kBox) dst[5 * kSZ] = r[5];
            }
        }
    }
}

// Thread t of the workgroup takes voxel (a, b, c) of the tile and voxel (a + 4, b, c): a 4x4x4 block per wavefront, axis c
// fastest.
__device__ __forceinline__ void tile_voxel(int& a, int& b, int& c) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    a = l >> 4;
    b = 4 * ((w >> 1) & 1) + ((l >> 2) & 3);
    c = 4 * (w & 1) + (l & 3);
}

// sum over a wavefront, in its last lane: row shifts, then row broadcasts (a fixed order, no LDS)
__device__ __forceinline__ float wave_sum_last(float v) {
#define ETTK_DPP_ADD(ctrl, rows) \
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rows, 0xf, false))
    ETTK_DPP_ADD(0x111, 0xf);  // row_shr:1
    ETTK_DPP_ADD(0x112, 0xf);  // row_shr:2
    ETTK_DPP_ADD(0x114, 0xf);  // row_shr:4
    ETTK_DPP_ADD(0x118, 0xf);  // row_shr:8
    ETTK_DPP_ADD(0x142, 0xa);  // row_bcast:15
    ETTK_DPP_ADD(0x143, 0xc);  // row_bcast:31
#undef ETTK_DPP_ADD
    return v;
}

// the sample at (px, py, pz) from the staged box, whose voxel lo + 1 is lo1
__device__ __forceinline__ float sample_box(const float* box, const int lo1[3], float px, float py, float pz) {
    const float xx = px + kTriTol, yy = py + kTriTol, zz = pz + kTriTol;
    const float fx = floorf(xx), fy = floorf(yy), fz = floorf(zz);
    const int x0 = (int)fx - lo1[0], y0 = (int)fy - lo1[1], z0 = (int)fz - lo1[2];  // the stencil's start in the box
    float wx[4], wy[4], wz[4];
    keys_w(xx - fx, wx);
    keys_w(yy - fy, wy);
    keys_w(zz - fz, wz);
    const float* b0 = box + z0 * kSZ + y0 * kSY + x0;
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
