// ccc.hip -- the reslice, the wedges and the set-up kernels of the wedge-constrained FFT cross-correlation (gfx950).
//
// Device side of nbfFourierImageMetric::executeFourierNewHalf (inc/em/nbfFourierImageMetric.h:1078-1323)
// for a batch of (particle, transform) evaluations:
//   reslice -> nbfWedgedSubImage3D::getImage (inc/em/nbfWedgedSubImage3D.h:603-828), VTK tricubic
//   wedge overlap -> nbfCorrelationImageMetric::getWedgeOverlap (nbfCorrelationImageMetric.h:533-566)
// The transforms, the spectral weighting, the quadratic expression (FIM.h:1202-1203), the upsampled correlation on the
// search window (FIM.h:1209-1247) and its first maximum (nbfCorrelationImageMetric.h:304-323) are in fft.hip.
// Per-evaluation sums are written as per-block partials and reduced in a fixed order (deterministic).
#include "kernels.hpp"

#include <hip/hip_ext.h>
#include "tricubic.hpp"
#include "wedge.hpp"

#include <algorithm>
#include <cfloat>

namespace ettk {

static constexpr int kThreads = 256;

// ------------------------------------------------------------------ reslice
// Validity of a sample is decided in FP32 unless it lies within 1e-3 of the border, where the FP64 map decides
// (the reference places samples in FP64: a sample that FP32 rounding moves across the border would otherwise
// enter or leave the valid set and change the mean the volume is centred on).
__device__ __forceinline__ bool near_border(float p, float lo, float hi) {
    return fabsf(p - lo) < 1e-3f || fabsf(p - hi) < 1e-3f;
}
__device__ __forceinline__ bool inside_fp64(const double* md, int i, int j, int k, double lo, double hx, double hy,
                                            double hz) {
    const double x = md[0] * i + md[3] * j + md[6] * k + md[9];
    const double y = md[1] * i + md[4] * j + md[7] * k + md[10];
    const double z = md[2] * i + md[5] * j + md[8] * k + md[11];
    return x >= lo && x <= hx && y >= lo && y <= hy && z >= lo && z <= hz;
}

// One workgroup reslices an 8x8x8 tile of the output from the LDS-staged box of the particle (tricubic.hpp).
// kUse names the caller in kernel traces (0: CCC evaluations, 1: S^2 projection); the code is the same
template <int kUse>
__global__ void __launch_bounds__(kThreads, 7) k_reslice(const float* __restrict__ parts, const EvalGeom* __restrict__ geom,
                                                       int N, float* __restrict__ out, float* __restrict__ partials) {
    static_assert(kThreads == kTriThreads, "the staging's thread map");
    __shared__ float2 sh[kThreads / 64];
    __shared__ float box[kBoxWords];
    int e, tb;
    xcd_eval_tile(blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, e, tb);
    const EvalGeom& g = geom[e];
    const size_t n3 = (size_t)N * N * N;
    const float* vol = parts + g.particle * n3;
    const int nt = N / kTile;
    const int i0 = tb / (nt * nt) * kTile, j0 = (tb / nt) % nt * kTile, k0 = tb % nt * kTile;
    int lo[3], hi[3];
    bool inside;
    const bool fits = tile_box(g.m, i0, j0, k0, N, N, N, kMarginMin, lo, hi, inside);  // N <= 128
    if (fits) stage_tile_box(vol, N, N, N, lo, hi, box);
    const int lo1[3] = {lo[0] + 1, lo[1] + 1, lo[2] + 1};
    int i, j, k;
    tile_voxel(i, j, k);
    i += i0;
    j += j0;
    k += k0;
    const float fj = (float)j, fk = (float)k;
    float pjk[3];
#pragma unroll
    for (int a = 0; a < 3; a++) pjk[a] = g.m[3 + a] * fj + g.m[6 + a] * fk;
    float* __restrict__ oe = out + e * n3;
    const unsigned off = ((i * N + j) * N + k) * 4u;
    __syncthreads();
    float s = 0.f;
    int c = 0;
    const float lob = -0.5f, hib = (float)N - 0.5f;
#pragma unroll
    for (int h = 0; h < 2; h++, i += 4) {
        const float fi = (float)i;
        const float px = g.m[0] * fi + pjk[0] + g.m[9];
        const float py = g.m[1] * fi + pjk[1] + g.m[10];
        const float pz = g.m[2] * fi + pjk[2] + g.m[11];
        float v;
        if (inside) {
            v = sample_box(box, lo1, px, py, pz);
            s += v;
            c += 64;
        } else {
            bool in = px >= lob && px <= hib && py >= lob && py <= hib && pz >= lob && pz <= hib;
            if (near_border(px, lob, hib) || near_border(py, lob, hib) || near_border(pz, lob, hib))
                in = inside_fp64(g.md, i, j, k, -0.5, N - 0.5, N - 0.5, N - 0.5);
            v = -FLT_MAX;
            if (in) {
                v = fits ? sample_box(box, lo1, px, py, pz) : sample_global(vol, N, N, N, px, py, pz);
                s += v;
            }
            c += __popcll(__ballot(in));
        }
        at_byte(oe + (size_t)h * 4 * N * N, off) = v;
    }
    // the tile's (sum, count): per wavefront, then the wavefronts in order
    s = wave_sum_last(s);
    if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = make_float2(s, (float)c);
    __syncthreads();
    if (threadIdx.x == 0) {
        float ts = 0.f, tc = 0.f;
        for (int w = 0; w < kThreads / 64; w++) {
            ts += sh[w].x;
            tc += sh[w].y;
        }
        partials[((size_t)e * gridDim.x + tb) * 2 + 0] = ts;  // in tile order: the same sum order for any mapping
        partials[((size_t)e * gridDim.x + tb) * 2 + 1] = tc;
    }
}

// one wave per evaluation: lane l sums the partials b = l, l + 64, ... in FP64, then a fixed butterfly
__device__ __forceinline__ double wave_dsum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__global__ void __launch_bounds__(64) k_reslice_mean(const float* __restrict__ partials, int nb, int n_eval,
                                                     float* __restrict__ stats) {
    const int e = blockIdx.x, l = threadIdx.x;
    double s = 0, c = 0;
    for (int b = l; b < nb; b += 64) {
        s += partials[((size_t)e * nb + b) * 2];
        c += partials[((size_t)e * nb + b) * 2 + 1];
    }
    s = wave_dsum(s);
    c = wave_dsum(c);
    if (l == 0) stats[e] = (float)(s / (double)(float)c);  // meanInside is a float (WSub.h:794-797)
}

int reslice_blocks(int N) { return (N / kTile) * (N / kTile) * (N / kTile); }

void launch_reslice(const float* parts, const EvalGeom* geom, int n_eval, int N, float* out, float* partials,
                    int nb, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop) {
    ETTK_REQUIRE(N % kTile == 0 && nb == reslice_blocks(N), ETTK_ERR_ARG, "launch_reslice: block count mismatch");
    dim3 grid(nb, n_eval);
    if (ev_start || ev_stop)  // the events take the kernel's own start and end timestamps
        hipExtLaunchKernelGGL(k_reslice<0>, grid, dim3(kThreads), 0, s, ev_start, ev_stop, 0, parts, geom, N, out,
                              partials);
    else
        k_reslice<0><<<grid, kThreads, 0, s>>>(parts, geom, N, out, partials);
    ETTK_HIP(hipGetLastError());
}
void launch_reslice_projection(const float* parts, const EvalGeom* geom, int n, int N, float* out, float* partials,
                               int nb, hipStream_t s) {
    ETTK_REQUIRE(N % kTile == 0 && nb == reslice_blocks(N), ETTK_ERR_ARG, "launch_reslice: block count mismatch");
    k_reslice<1><<<dim3(nb, n), kThreads, 0, s>>>(parts, geom, N, out, partials);
    ETTK_HIP(hipGetLastError());
}
void launch_reslice_mean(const float* partials, int nb, int n_eval, float* stats, hipStream_t s) {
    k_reslice_mean<<<n_eval, 64, 0, s>>>(partials, nb, n_eval, stats);
    ETTK_HIP(hipGetLastError());
}

__global__ void k_wedge_ref(WedgeRef w, int N, float* __restrict__ W) {
    const int H = N / 2 + 1;
    long nh = (long)N * N * H;
    for (long h = blockIdx.x * (long)blockDim.x + threadIdx.x; h < nh; h += (long)gridDim.x * blockDim.x) {
        int i, j, k;
        split3((unsigned)h, (unsigned)N, (unsigned)H, i, j, k);
        W[h] = w.full ? 1.f : wedge_smooth(w.v1, w.v2, i, j, k, N, H);
    }
}
void launch_wedge_ref(const WedgeRef& w, int N, float* W, hipStream_t s) {
    k_wedge_ref<<<512, kThreads, 0, s>>>(w, N, W);
    ETTK_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ wedge overlap
// nbfCorrelationImageMetric::getWedgeOverlap (CorrMetric.h:533-566): sum(W1 W2(t) filter) over the half grid,
// W2 the particle's smoothed wedge at the evaluation's transform (all ones when geom.full).  Per-block FP64
// partials, then one sum per evaluation.
__global__ void __launch_bounds__(kThreads) k_wedge_overlap(const float* __restrict__ W1, const float* __restrict__ filter,
                                                             const EvalGeom* __restrict__ geom, int N,
                                                             double* __restrict__ part) {
    __shared__ double sh[kThreads / 64];
    const int e = blockIdx.y, H = N / 2 + 1;
    const unsigned nh = (unsigned)N * N * H;
    const EvalGeom& g = geom[e];
    double acc = 0.0;
    for (unsigned h = blockIdx.x * kThreads + threadIdx.x; h < nh; h += gridDim.x * kThreads) {
        int i, j, k;
        split3(h, (unsigned)N, (unsigned)H, i, j, k);
        float w = W1[h] * (g.full ? 1.f : wedge_smooth(g.v1, g.v2, i, j, k, N, H));
        acc += (double)(w * filter[h]);
    }
    for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int q = 0; q < kThreads / 64; q++) t += sh[q];
        part[(size_t)e * gridDim.x + blockIdx.x] = t;
    }
}
__global__ void k_sum_partials(const double* __restrict__ part, int nb, int n_eval, double* __restrict__ out) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_eval) return;
    double t = 0.0;
    for (int b = 0; b < nb; b++) t += part[(size_t)e * nb + b];
    out[e] = t;
}
void launch_wedge_overlap(const float* W1, const float* filter, const EvalGeom* geom, int E, int N, double* part,
                          double* out, hipStream_t s) {
    const int nb = 64;
    k_wedge_overlap<<<dim3(nb, E), kThreads, 0, s>>>(W1, filter, geom, N, part);
    k_sum_partials<<<(E + 127) / 128, 128, 0, s>>>(part, nb, E, out);
    ETTK_HIP(hipGetLastError());
}

template <class T>
__global__ void k_fill_zero(T* __restrict__ p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = T(0);
}
template <class T>
static void fill_zero(T* p, size_t n, hipStream_t s) {
    if (n == 0) return;
    const unsigned blocks = (unsigned)std::min<size_t>((n + kThreads - 1) / kThreads, 4096);
    k_fill_zero<T><<<blocks, kThreads, 0, s>>>(p, n);
    ETTK_HIP(hipGetLastError());
}
void launch_fill_zero(int* p, size_t n, hipStream_t s) { fill_zero(p, n, s); }
void launch_fill_zero(double* p, size_t n, hipStream_t s) { fill_zero(p, n, s); }

// ------------------------------------------------------------------ helpers used by the plan set-up
__global__ void k_xfast_to_internal(const float* __restrict__ in, float* __restrict__ out, int N) {
    long n3 = (long)N * N * N;
    for (long o = blockIdx.x * (long)blockDim.x + threadIdx.x; o < n3; o += (long)gridDim.x * blockDim.x) {
        int i, j, k;
        split3((unsigned)o, (unsigned)N, (unsigned)N, i, j, k);
        out[o] = in[((size_t)k * N + j) * N + i];
    }
}
void launch_xfast_to_internal(const float* in, float* out, int N, hipStream_t s) {
    k_xfast_to_internal<<<1024, kThreads, 0, s>>>(in, out, N);
    ETTK_HIP(hipGetLastError());
}
__global__ void k_internal_to_xfast(const float* __restrict__ in, float* __restrict__ out, int N) {
    long n3 = (long)N * N * N;
    for (long o = blockIdx.x * (long)blockDim.x + threadIdx.x; o < n3; o += (long)gridDim.x * blockDim.x) {
        int zz, y, x;
        split3((unsigned)o, (unsigned)N, (unsigned)N, zz, y, x);
        out[o] = in[((size_t)x * N + y) * N + zz];
    }
}
void launch_internal_to_xfast(const float* in, float* out, int N, hipStream_t s) {
    k_internal_to_xfast<<<1024, kThreads, 0, s>>>(in, out, N);
    ETTK_HIP(hipGetLastError());
}
__global__ void k_mcf_inplace(float2* __restrict__ F, long n) {
    for (long h = blockIdx.x * (long)blockDim.x + threadIdx.x; h < n; h += (long)gridDim.x * blockDim.x) {
        float2 z = F[h];
        float C = sqrtf(sqrtf(z.x * z.x + z.y * z.y));
        if (C > 0.f) F[h] = make_float2(z.x / C, z.y / C);
    }
}
void launch_mcf_inplace(float2* F, long n, hipStream_t s) {
    k_mcf_inplace<<<1024, kThreads, 0, s>>>(F, n);
    ETTK_HIP(hipGetLastError());
}

}  // namespace ettk
