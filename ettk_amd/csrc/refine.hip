// refine.hip -- continuous constrained CCC and its adjoint for local pose refinement (gfx950).
//
// No reference counterpart: this replaces the Powell line searches of nbfFourierImageMetric::refine
// (inc/em/nbfFourierImageMetric.h:1702-1809), whose every function value is a full constrained CCC on a
// half-voxel shift grid, by gradient ascent on a differentiable score of the six pose parameters.
//
// The score lives in the particle's own frame, where the particle's missing wedge is fixed:
//   X2 = H r2c((I2 - mean I2) maskfft (-1)^(x+y+z))               particle, fixed: spectra computed once
//   X1 = H r2c(I1'(theta) maskfft (-1)^(x+y+z))                    reference resliced into the particle frame
//   I1'(p) = (I1 - mean I1)(q(p)),  q = G' (p - N/2, 1),  G' = fin(theta)^-1 plus (N/2, N/2, N/2 + cut)
//            (trilinear with clamped taps: the reference is extended by its border values, so that I1' and S
//            are continuous in theta)
//   S  = <X1, X2> / (|X1| |X2|),  <a, b> = sum_h c_h Re(a_h conj(b_h))  (c_h: exact Hermitian weights)
// with H = band-pass x binary particle wedge (lab frame) x binary reference wedge (rotated by the seed).
// Volumes stay in the particle's memory order [z][y][x]; the half axis of every spectrum is x.
// Adjoint: dS = <Z, dX1> with Z = X2/(n1 n2) - S X1/n1^2, so dS/dI1'(p) = maskfft (-1)^(x+y+z) c2r(H Z)(p),
// and through the interpolator dS/dtheta_r =
// sum_ab dG'_r[a][b] Q[a][b], Q[a][b] = sum_p gamma(p) dI1/dq_a(q(p)) w_b(p), w = (x-N/2, y-N/2, z-N/2, 1):
// twelve moments per evaluation, contracted with dG'_r = -G dfin_r G on the host in FP64.
#include <algorithm>
#include <cfloat>

#include "kernels.hpp"

namespace ettk {

static constexpr int kT = 256;

__device__ __forceinline__ float wsum64(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}
__device__ __forceinline__ double dsum64(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// trilinear sample of an x-fastest volume with clamped taps, and its gradient in (x, y, z)
__device__ __forceinline__ float trilin(const float* __restrict__ vol, int N, float px, float py, float pz, float* gr) {
    float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    float ax = px - fx, ay = py - fy, az = pz - fz;
    int x0 = min(max((int)fx, 0), N - 1), x1 = min(max((int)fx + 1, 0), N - 1);
    int y0 = min(max((int)fy, 0), N - 1), y1 = min(max((int)fy + 1, 0), N - 1);
    int z0 = min(max((int)fz, 0), N - 1), z1 = min(max((int)fz + 1, 0), N - 1);
    const int r00 = (z0 * N + y0) * N, r01 = (z0 * N + y1) * N, r10 = (z1 * N + y0) * N, r11 = (z1 * N + y1) * N;
    float v000 = vol[r00 + x0], v100 = vol[r00 + x1];
    float v010 = vol[r01 + x0], v110 = vol[r01 + x1];
    float v001 = vol[r10 + x0], v101 = vol[r10 + x1];
    float v011 = vol[r11 + x0], v111 = vol[r11 + x1];
    float c00 = v000 + ax * (v100 - v000), c10 = v010 + ax * (v110 - v010);
    float c01 = v001 + ax * (v101 - v001), c11 = v011 + ax * (v111 - v011);
    float c0 = c00 + ay * (c10 - c00), c1 = c01 + ay * (c11 - c01);
    if (gr) {
        float dx00 = v100 - v000, dx10 = v110 - v010, dx01 = v101 - v001, dx11 = v111 - v011;
        float dx0 = dx00 + ay * (dx10 - dx00), dx1 = dx01 + ay * (dx11 - dx01);
        gr[0] = dx0 + az * (dx1 - dx0);
        float dy0 = c10 - c00, dy1 = c11 - c01;
        gr[1] = dy0 + az * (dy1 - dy0);
        gr[2] = c1 - c0;
    }
    return c0 + az * (c1 - c0);
}

// sampling position in the reference of voxel (x, y, z) of the particle frame
__device__ __forceinline__ void ref_pos(const RefineGeom& g, int N, int x, int y, int z, float* q) {
    const float h = 0.5f * (float)N;
    const float wx = (float)x - h, wy = (float)y - h, wz = (float)z - h;
    q[0] = g.G[0] * wx + g.G[1] * wy + g.G[2] * wz + g.G[3];
    q[1] = g.G[4] * wx + g.G[5] * wy + g.G[6] * wz + g.G[7];
    q[2] = g.G[8] * wx + g.G[9] * wy + g.G[10] * wz + g.G[11];
}

// ---------------------------------------------------------------- LDS-staged trilinear sampling
// One workgroup handles an 8x8x8 tile of the particle frame.  The reference voxels its trilinear taps can
// touch lie in the bounding box [floor(min), floor(max) + 1] of the tile's mapped corners, at most
// floor(7 sqrt 3) + 1 + 2 = 15 voxels per axis for a rigid map (about 12 for a random rotation).  That box's
// actual extent, with the reference's border replicated where it reaches outside (the taps clamp to the
// border), is staged in LDS at fixed strides, so the divergent gathers become LDS reads and every sample equals
// the clamped-tap global one; a sample that rounds one voxel past the box keeps the box's edge cell with its
// fraction just outside [0, 1) (the same value to a few ulps).  A 15^3 box (13.5 KB) lets 10 workgroups share a
// CU, which hides the staging loads' latency (an 18^3 box staged whole took 1.2 times as long); the box's bounds and
// the staging's plane addresses are scalar.  40 evaluations at 64^3: reference reslice 48 us, adjoint moments 60, where
// addresses per lane took 51 and 65.  A map whose box does not fit samples from global memory instead.
static constexpr int kRT = 8, kRB = 15;

__device__ __forceinline__ bool stage_ref_box(const float* __restrict__ vol, int N, const RefineGeom& g, int x0,
                                              int y0, int z0, float* box, int lo[3], int hi[3]) {
    const float h = 0.5f * (float)N;
    bool fits = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float* r = g.G + a * 4;
        const float c0 = r[0] * ((float)x0 - h) + r[1] * ((float)y0 - h) + r[2] * ((float)z0 - h) + r[3];
        const float mn = c0 + (kRT - 1) * (fminf(r[0], 0.f) + fminf(r[1], 0.f) + fminf(r[2], 0.f));
        const float ext = (kRT - 1) * (fabsf(r[0]) + fabsf(r[1]) + fabsf(r[2]));
        // the same for every thread: in scalar registers, with the plane addresses of the staging below
        lo[a] = __builtin_amdgcn_readfirstlane((int)floorf(mn));
        hi[a] = __builtin_amdgcn_readfirstlane((int)floorf(mn + ext) + 1);
        if (!(hi[a] - lo[a] + 1 <= kRB) || !(fabsf(mn) < 1e6f)) fits = false;
    }
    if (fits) {
        // 2-D thread map over (y, x) of the box, loop over z; coordinates clamped to the volume
        static_assert(kT / kRB >= kRB && kRB % 5 == 0, "one pass over a plane, whole steps of z");
        const int x = threadIdx.x % kRB, y = threadIdx.x / kRB;
        const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
        if (x < wx && y < wy) {
            const int gx = min(max(lo[0] + x, 0), N - 1), gy = min(max(lo[1] + y, 0), N - 1);
            const unsigned off = ((unsigned)gy * N + gx) * 4u;
            float* dst = box + y * kRB + x;
            const size_t plane = (size_t)N * N;
            // the plane's address advances in scalar registers; it stays where the clamped coordinate does
            const float* src = vol + (size_t)min(max(lo[2], 0), N - 1) * plane;
            for (int z = 0; z < wz; z += 5, dst += 5 * kRB * kRB) {  // five loads in flight; planes past the box unused
                float r[5];
#pragma unroll
                for (int u = 0; u < 5; u++) {
                    r[u] = at_byte(src, off);
                    const unsigned g = (unsigned)(lo[2] + z + u);  // step from this plane to the next one inside the volume
                    src += g < (unsigned)(N - 1) ? plane : 0;
                }
#pragma unroll
                for (int u = 0; u < 5; u++) dst[u * kRB * kRB] = r[u];
            }
        }
    }
    __syncthreads();
    return fits;
}

// trilin() on the staged box: the same arithmetic, taps read from LDS
__device__ __forceinline__ float trilin_box(const float* box, const int lo[3], const int hi[3], float px, float py,
                                            float pz, float* gr) {
    float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    float ax = px - fx, ay = py - fy, az = pz - fz;
    int ix = (int)fx, iy = (int)fy, iz = (int)fz;
    if (ix < lo[0] || ix > hi[0] - 1) {
        ix = min(max(ix, lo[0]), hi[0] - 1);
        ax = px - (float)ix;
    }
    if (iy < lo[1] || iy > hi[1] - 1) {
        iy = min(max(iy, lo[1]), hi[1] - 1);
        ay = py - (float)iy;
    }
    if (iz < lo[2] || iz > hi[2] - 1) {
        iz = min(max(iz, lo[2]), hi[2] - 1);
        az = pz - (float)iz;
    }
    const float* p = box + ((iz - lo[2]) * kRB + (iy - lo[1])) * kRB + (ix - lo[0]);
    float v000 = p[0], v100 = p[1];
    float v010 = p[kRB], v110 = p[kRB + 1];
    float v001 = p[kRB * kRB], v101 = p[kRB * kRB + 1];
    float v011 = p[kRB * kRB + kRB], v111 = p[kRB * kRB + kRB + 1];
    float c00 = v000 + ax * (v100 - v000), c10 = v010 + ax * (v110 - v010);
    float c01 = v001 + ax * (v101 - v001), c11 = v011 + ax * (v111 - v011);
    float c0 = c00 + ay * (c10 - c00), c1 = c01 + ay * (c11 - c01);
    if (gr) {
        float dx00 = v100 - v000, dx10 = v110 - v010, dx01 = v101 - v001, dx11 = v111 - v011;
        float dx0 = dx00 + ay * (dx10 - dx00), dx1 = dx01 + ay * (dx11 - dx01);
        gr[0] = dx0 + az * (dx1 - dx0);
        float dy0 = c10 - c00, dy1 = c11 - c01;
        gr[1] = dy0 + az * (dy1 - dy0);
        gr[2] = c1 - c0;
    }
    return c0 + az * (c1 - c0);
}


// mean of each particle volume (FP64 accumulation): kMeanV voxels per workgroup, then one wave per particle over
// the workgroups' sums in a fixed order.  Bound by one read of the volumes; with one workgroup per particle, 96
// volumes of 64^3 took 413 us (0.24 TB/s: 96 of 256 CUs, each on one workgroup's load latency) and 40 of 96^3
// 1420 us; split like this the score and gradient of those particles went from 1092 to 690 us and from 2767 to
// 1334 us.  The 16-byte loads need 4-byte alignment only.
static constexpr int kMeanU = 8, kMeanV = kT * 4 * kMeanU;
// sum of the kMeanV voxels from `first` on over kT threads (t = 0 .. kT - 1), in thread 0; `sh` holds kT / 64 doubles
__device__ __forceinline__ double mean_part(const float* __restrict__ v, long first, long n3, int t, double* sh) {
    const long o0 = first + t * 4;
    float4 r[kMeanU];  // all loads in flight; n3 is a multiple of 4 (box sizes are multiples of 8)
#pragma unroll
    for (int u = 0; u < kMeanU; u++) {
        const long o = o0 + (long)u * kT * 4;
        r[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (o < n3) __builtin_memcpy(&r[u], v + o, sizeof(float4));
    }
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kMeanU; u++) s += ((double)r[u].x + r[u].y) + ((double)r[u].z + r[u].w);
    s = dsum64(s);
    if ((t & 63) == 0) sh[t >> 6] = s;
    __syncthreads();
    double sum = 0.0;
    if (t == 0)
        for (int w = 0; w < kT / 64; w++) sum += sh[w];
    return sum;
}
__global__ void __launch_bounds__(kT) k_vol_sum(const float* __restrict__ vols, long n3, double* __restrict__ part) {
    __shared__ double sh[kT / 64];
    const double t = mean_part(vols + (size_t)blockIdx.y * n3, (long)blockIdx.x * kMeanV, n3, threadIdx.x, sh);
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = t;
}
// Volumes of at most four parts (boxes of 16 and 32): one workgroup holds them all, and the sums, added in the order of
// k_vol_mean, need no second launch.  Score and gradient of one particle of 32^3: 101 us, 104 with two launches.
template <int NB>
__global__ void __launch_bounds__(kT * NB) k_vol_mean_small(const float* __restrict__ vols, long n3, float* __restrict__ mean) {
    __shared__ double sh[NB][kT / 64];
    __shared__ double part[NB];
    const int b = threadIdx.x / kT, t = threadIdx.x % kT;
    const double sum = mean_part(vols + (size_t)blockIdx.x * n3, (long)b * kMeanV, n3, t, sh[b]);
    if (t == 0) part[b] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = part[0];
        if constexpr (NB == 4) s = (part[0] + part[2]) + (part[1] + part[3]);
        mean[blockIdx.x] = (float)(s / (double)n3);
    }
}
__global__ void __launch_bounds__(64) k_vol_mean(const double* __restrict__ part, int nb, long n3,
                                                 float* __restrict__ mean) {
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) s += part[(size_t)blockIdx.x * nb + b];
    s = dsum64(s);
    if (threadIdx.x == 0) mean[blockIdx.x] = (float)(s / (double)n3);
}

// I1'(p) for every evaluation: out[e][z][y][x]; `ref` holds I1 - mean I1, x fastest
__global__ void __launch_bounds__(kT) k_reslice_ref(const float* __restrict__ ref, const RefineGeom* __restrict__ geom,
                                                     int N, float* __restrict__ out) {
    __shared__ float box[kRB * kRB * kRB];
    const int e = blockIdx.y;
    const RefineGeom g = geom[e];
    const size_t n3 = (size_t)N * N * N;
    const int nt = N / kRT;
    const int tb = xcd_tile(blockIdx.x, gridDim.x);
    const int z0 = (tb / (nt * nt)) * kRT, y0 = ((tb / nt) % nt) * kRT, x0 = (tb % nt) * kRT;
    int lo[3], hi[3];
    const bool fits = stage_ref_box(ref, N, g, x0, y0, z0, box, lo, hi);
    for (int t = threadIdx.x; t < kRT * kRT * kRT; t += kT) {
        const int x = x0 + (t & 7), y = y0 + ((t >> 3) & 7), z = z0 + (t >> 6);
        float q[3];
        ref_pos(g, N, x, y, z, q);
        const float v = fits ? trilin_box(box, lo, hi, q[0], q[1], q[2], nullptr) : trilin(ref, N, q[0], q[1], q[2], nullptr);
        out[(size_t)e * n3 + ((size_t)z * N + y) * N + x] = v;
    }
}

// sc[e] = {S, n1, n2} in FP64
__global__ void __launch_bounds__(64) k_refine_scalars(const double* __restrict__ part, int nb, int n_eval,
                                                       double* __restrict__ sc) {
    const int e = blockIdx.x, l = threadIdx.x;
    double d = 0, q1 = 0, q2 = 0;
    for (int b = l; b < nb; b += 64) {
        d += part[((size_t)e * nb + b) * 3];
        q1 += part[((size_t)e * nb + b) * 3 + 1];
        q2 += part[((size_t)e * nb + b) * 3 + 2];
    }
    for (int o = 32; o > 0; o >>= 1) {
        d += __shfl_xor(d, o, 64);
        q1 += __shfl_xor(q1, o, 64);
        q2 += __shfl_xor(q2, o, 64);
    }
    if (l != 0) return;
    const double n1 = sqrt(q1), n2 = sqrt(q2);
    sc[e * 4 + 0] = (n1 > 0 && n2 > 0) ? d / (n1 * n2) : 0.0;
    sc[e * 4 + 1] = n1;
    sc[e * 4 + 2] = n2;
}

// twelve moments per evaluation: per-workgroup partial sums of gamma(p) dI1/dq_a w_b(p) over kMT consecutive
// 8x8x8 tiles (one staged box per tile, one 12-value reduction per workgroup)
static constexpr int kMT = 4;
__global__ void __launch_bounds__(kT) k_refine_moments(const float* __restrict__ ref, const RefineGeom* __restrict__ geom,
                                                        const float* __restrict__ G, const float* __restrict__ maskfft,
                                                        int N, float* __restrict__ part) {
    __shared__ float box[kRB * kRB * kRB];
    __shared__ float sh[12][kT / 64];
    const int e = blockIdx.y;
    const RefineGeom g = geom[e];
    const size_t n3 = (size_t)N * N * N;
    const float* Ge = G + (size_t)e * n3;
    const float half = 0.5f * (float)N;
    const int nt = N / kRT, ntile = nt * nt * nt;
    const int wb = xcd_tile(blockIdx.x, gridDim.x);
    float q12[12];
#pragma unroll
    for (int r = 0; r < 12; r++) q12[r] = 0.f;
    for (int u = 0; u < kMT; u++) {
        const int tb = wb * kMT + u;
        if (tb >= ntile) break;
        const int z0 = (tb / (nt * nt)) * kRT, y0 = ((tb / nt) % nt) * kRT, x0 = (tb % nt) * kRT;
        if (u > 0) __syncthreads();  // the previous tile's box is no longer read
        int lo[3], hi[3];
        const bool fits = stage_ref_box(ref, N, g, x0, y0, z0, box, lo, hi);
        for (int t = threadIdx.x; t < kRT * kRT * kRT; t += kT) {
            const int x = x0 + (t & 7), y = y0 + ((t >> 3) & 7), z = z0 + (t >> 6);
            const size_t o = ((size_t)z * N + y) * N + x;
            float q[3];
            ref_pos(g, N, x, y, z, q);
            const float gam = maskfft[o] * (((x + y + z) & 1) ? -Ge[o] : Ge[o]);
            float gr[3];
            if (fits) trilin_box(box, lo, hi, q[0], q[1], q[2], gr);
            else trilin(ref, N, q[0], q[1], q[2], gr);
            const float w[4] = {(float)x - half, (float)y - half, (float)z - half, 1.f};
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const float ga = gam * gr[a];
#pragma unroll
                for (int b = 0; b < 4; b++) q12[a * 4 + b] += ga * w[b];
            }
        }
    }
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int r = 0; r < 12; r++) {
        const float t = wsum64(q12[r]);
        if ((threadIdx.x & 63) == 0) sh[r][wv] = t;
    }
    __syncthreads();
    if (threadIdx.x < 12) {
        float t = 0.f;
        for (int i = 0; i < kT / 64; i++) t += sh[threadIdx.x][i];
        part[((size_t)e * gridDim.x + wb) * 12 + threadIdx.x] = t;
    }
}

__global__ void __launch_bounds__(64) k_refine_reduce_moments(const float* __restrict__ part, int nb, int n_eval,
                                                              double* __restrict__ out) {
    const int e = blockIdx.x, l = threadIdx.x;
    double acc[12];
#pragma unroll
    for (int r = 0; r < 12; r++) acc[r] = 0.0;
    for (int b = l; b < nb; b += 64) {
        const float* p = part + ((size_t)e * nb + b) * 12;
#pragma unroll
        for (int r = 0; r < 12; r++) acc[r] += p[r];
    }
#pragma unroll
    for (int r = 0; r < 12; r++) {
        double v = acc[r];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (l == 0) out[e * 12 + r] = v;
    }
}

int refine_moment_blocks(int N) {
    const int nt = N / kRT;
    return (nt * nt * nt + kMT - 1) / kMT;
}
int vol_mean_blocks(int N) { return (int)(((long)N * N * N + kMeanV - 1) / kMeanV); }
void launch_vol_mean(const float* vols, int count, int N, double* part, float* mean, hipStream_t s) {
    ETTK_REQUIRE(N % 4 == 0, ETTK_ERR_ARG, "launch_vol_mean: box size must be a multiple of 4");
    const long n3 = (long)N * N * N;
    const int nb = vol_mean_blocks(N);
    if (nb <= 4) {
        if (nb == 1) k_vol_mean_small<1><<<count, kT, 0, s>>>(vols, n3, mean);
        else k_vol_mean_small<4><<<count, kT * 4, 0, s>>>(vols, n3, mean);
        ETTK_HIP(hipGetLastError());
        return;
    }
    // the particles run along the grid's second axis, at most 65535 per launch
    for (int c0 = 0; c0 < count; c0 += 65535) {
        const int c = std::min(65535, count - c0);
        k_vol_sum<<<dim3(nb, c), kT, 0, s>>>(vols + (size_t)c0 * n3, n3, part + (size_t)c0 * nb);
    }
    k_vol_mean<<<count, 64, 0, s>>>(part, nb, n3, mean);
    ETTK_HIP(hipGetLastError());
}
void launch_reslice_ref(const float* ref, const RefineGeom* geom, int E, int N, float* out, hipStream_t s) {
    ETTK_REQUIRE(N % kRT == 0, ETTK_ERR_ARG, "launch_reslice_ref: box size must be a multiple of 8");
    const int nt = N / kRT;
    k_reslice_ref<<<dim3(nt * nt * nt, E), kT, 0, s>>>(ref, geom, N, out);
    ETTK_HIP(hipGetLastError());
}
void launch_refine_scalars(const double* part, int nb, int E, double* sc, hipStream_t s) {
    k_refine_scalars<<<E, 64, 0, s>>>(part, nb, E, sc);
    ETTK_HIP(hipGetLastError());
}
void launch_refine_moments(const float* ref, const RefineGeom* geom, const float* G, const float* maskfft, int E, int N,
                           float* mpart, double* mom, hipStream_t s) {
    ETTK_REQUIRE(N % kRT == 0, ETTK_ERR_ARG, "launch_refine_moments: box size must be a multiple of 8");
    const int nb = refine_moment_blocks(N);
    k_refine_moments<<<dim3(nb, E), kT, 0, s>>>(ref, geom, G, maskfft, N, mpart);
    k_refine_reduce_moments<<<E, 64, 0, s>>>(mpart, nb, E, mom);
    ETTK_HIP(hipGetLastError());
}

}  // namespace ettk
