// extract.hip -- sub-volumes cut from a tomogram: nbfWedgedSubImage3D::getImage with the tomogram loaded
// (inc/em/nbfWedgedSubImage3D.h:603-802, normalize off), the step before the alignment path
// (src/CutVolumes3DFromPositions.cpp).
//
// Output voxel q of particle p reads the tomogram at  position_p + fin_p (q - N/2 - cut_p z),
// fin = Euler(normal) matrix, with VTK's tricubic (Keys a = -1/2, taps clamped to the tomogram); samples outside
// [-0.5, n - 0.5] on any axis are invalid.  The mean of the valid samples is subtracted and invalid voxels are 0,
// as getImage does before handing the sub-volume to the metric.  Outputs are N^3 floats, x fastest.
#include "kernels.hpp"
#include "plan.hpp"
#include "tricubic.hpp"

#include <cfloat>

namespace ettk {

namespace {

constexpr int kExT = kTriThreads;

// Magnification of a map (the root mean square of its rows' lengths: 1 for a rotation, whichever it is, so that the boxes of
// a call take one form) from which a box is cut without tiles.  Tiles / runs of voxels in us: 200 boxes of 32^3 at 2.0
// 461 / 431, at 2.5 560 / 472, at 4 555 / 469; 10 of 100^3 548 / 642, 472 / 540, 248 / 213; 4 of 128^3 377 / 396, 394 / 299,
// 285 / 171; one of 64^3 50 / 47, 55 / 62, 65 / 49.
constexpr double kSteep = 2.25;

// Validity of the sample at (px, py, pz) of output voxel (x, y, z): FP32 unless it lies within 1e-3 of the border
__device__ __forceinline__ bool sample_inside(const ExtractGeom& g, int x, int y, int z, float px, float py, float pz, int nx,
                                              int ny, int nz) {
    const float hx = nx - 0.5f, hy = ny - 0.5f, hz = nz - 0.5f;
    auto near = [](float p, float hi) { return fabsf(p + 0.5f) < 1e-3f || fabsf(p - hi) < 1e-3f; };
    if (near(px, hx) || near(py, hy) || near(pz, hz)) {
        const double* md = g.md;
        const double qx = md[0] * x + md[3] * y + md[6] * z + md[9];
        const double qy = md[1] * x + md[4] * y + md[7] * z + md[10];
        const double qz = md[2] * x + md[5] * y + md[8] * z + md[11];
        return qx >= -0.5 && qx <= nx - 0.5 && qy >= -0.5 && qy <= ny - 0.5 && qz >= -0.5 && qz <= nz - 0.5;
    }
    return px >= -0.5f && px <= hx && py >= -0.5f && py <= hy && pz >= -0.5f && pz <= hz;
}

// STAGED: one workgroup per 8x8x8 tile of an output box (tiles at the far sides of a box whose size is not a multiple of 8
// are partial), interpolated from the LDS-staged box of the tomogram that its stencils touch (tricubic.hpp).  Bound by the
// LDS reads of the taps, as the CCC reslice.  The call on 60 boxes of 64^3 takes 201 us; with every tap read from global
// memory it took 1558 us.  The other form serves steep maps, whose input boxes don't fit: 256 consecutive voxels, taps from
// global memory, bound by the latency of its gathers.  The tiles sample from global memory too where their box does not fit,
// and a compact tile's lines are still shared: the line between the forms (kSteep) lies where that stops to pay, see there.
// A launch skips the boxes of the other form.  Per workgroup the (sum, count) of the valid samples (the sum in FP32: up to
// two samples per thread, then a tree; the workgroups in FP64); workgroups past a form's share leave zeros.
template <bool STAGED>
__global__ void __launch_bounds__(kExT, STAGED ? 7 : 4) k_extract(const float* __restrict__ tomo, int nx, int ny, int nz,
                                                  const ExtractGeom* __restrict__ geom, int N, float* __restrict__ out,
                                                  float* __restrict__ partials) {
    __shared__ float box[STAGED ? kBoxWords : 1];
    __shared__ float sh[2][kExT / 64];
    int p = blockIdx.y, tb = blockIdx.x;
    if constexpr (STAGED)  // neighbouring tiles share their lines in one L2
        xcd_eval_tile(blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, p, tb);
    const ExtractGeom& g = geom[p];
    if ((g.steep == 0) != STAGED) return;
    const size_t n3 = (size_t)N * N * N;
    const int nt = (N + kTile - 1) / kTile;
    float* __restrict__ part = partials + ((size_t)p * gridDim.x + tb) * 2;
    if (tb >= (STAGED ? nt * nt * nt : (int)((n3 + kExT - 1) / kExT))) {
        if (threadIdx.x < 2) part[threadIdx.x] = 0.f;
        return;
    }
    int x, y, z;
    int lo[3], hi[3], lo1[3];
    bool inside, fits;
    if constexpr (STAGED) {
        const int z0 = (tb / (nt * nt)) * kTile, y0 = ((tb / nt) % nt) * kTile, x0 = (tb % nt) * kTile;
        fits = tile_box(g.m, x0, y0, z0, nx, ny, nz, tile_margin(max(nx, max(ny, nz)), N), lo, hi, inside);
        if (fits) stage_tile_box(tomo, nx, ny, nz, lo, hi, box);
        for (int a = 0; a < 3; a++) lo1[a] = lo[a] + 1;
        tile_voxel(z, y, x);
        x += x0;
        y += y0;
        z += z0;
        __syncthreads();
    } else {
        split3((unsigned)min((size_t)tb * kExT + threadIdx.x, n3 - 1), (unsigned)N, (unsigned)N, z, y, x);
    }
    float s = 0.f;
    int c = 0;
#pragma unroll 1
    for (int h = 0; h < (STAGED ? 2 : 1); h++, z += 4) {
        const bool live = STAGED ? x < N && y < N && z < N : (size_t)tb * kExT + threadIdx.x < n3;
        const float px = g.m[0] * x + g.m[3] * y + g.m[6] * z + g.m[9];
        const float py = g.m[1] * x + g.m[4] * y + g.m[7] * z + g.m[10];
        const float pz = g.m[2] * x + g.m[5] * y + g.m[8] * z + g.m[11];
        float v = -FLT_MAX;
        const bool in = live && ((STAGED && inside) || sample_inside(g, x, y, z, px, py, pz, nx, ny, nz));
        if (in) {
            v = STAGED && fits ? sample_box(box, lo1, px, py, pz) : sample_global(tomo, nx, ny, nz, px, py, pz);
            s += v;
        }
        c += __popcll(__ballot(in));
        if (live) out[(size_t)p * n3 + ((size_t)z * N + y) * N + x] = v;
    }
    s = wave_sum_last(s);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 63) {
        sh[0][w] = s;
        sh[1][w] = (float)c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float ts = 0.f, tc = 0.f;
        for (int q = 0; q < kExT / 64; q++) {
            ts += sh[0][q];
            tc += sh[1][q];
        }
        part[0] = ts;
        part[1] = tc;
    }
}

// valid samples minus their mean, invalid (-FLT_MAX) to 0
__global__ void __launch_bounds__(kExT) k_extract_finish(float* __restrict__ out, const float* __restrict__ mean, long n3) {
    const int p = blockIdx.y;
    const long o = (long)blockIdx.x * kExT + threadIdx.x;
    if (o >= n3) return;
    float* v = out + (size_t)p * n3 + o;
    const float a = *v;
    *v = a > -FLT_MAX ? a - mean[p] : 0.f;
}

}  // namespace

void extract_batch(ettk_ctx* ctx, const float* d_tomo, int nx, int ny, int nz, int n, const double* positions,
                   const ettk_particle* descs, int N, float* d_out) {
    hipStream_t s = ctx->stream;
    std::vector<ExtractGeom> g(n);
    const double half = N / 2.0;
    bool any_tiles = false, any_steep = false;
    for (int i = 0; i < n; i++) {
        Mat4 fin = euler_of(descs[i]) * Mat4::from(descs[i].matrix);
        if (mat_det(fin) == 0.0) fin = Mat4::ident();
        double square = 0;
        const double w0[3] = {-half, -half, -half - descs[i].cut_offset};
        for (int r = 0; r < 3; r++) {
            g[i].md[0 + r] = fin(r, 0);
            g[i].md[3 + r] = fin(r, 1);
            g[i].md[6 + r] = fin(r, 2);
            g[i].md[9 + r] = fin(r, 0) * w0[0] + fin(r, 1) * w0[1] + fin(r, 2) * w0[2] + fin(r, 3) + positions[3 * i + r];
            for (int c = 0; c < 4; c++) g[i].m[3 * c + r] = (float)g[i].md[3 * c + r];
            square += fin(r, 0) * fin(r, 0) + fin(r, 1) * fin(r, 1) + fin(r, 2) * fin(r, 2);
        }
        g[i].steep = square >= 3 * kSteep * kSteep;
        (g[i].steep ? any_steep : any_tiles) = true;
    }
    const long n3 = (long)N * N * N;
    const int nt = (N + kTile - 1) / kTile, nbt = nt * nt * nt, nbs = (int)((n3 + kExT - 1) / kExT);
    const int nb = std::max(any_tiles ? nbt : 0, any_steep ? nbs : 0);
    // the context's buffers, held until the call's work is done: calls of several host threads on one context take turns
    std::lock_guard<std::mutex> hold(ctx->extract_mu);
    ctx->extract_geom.upload(g.data(), n, s);
    ctx->extract_part.ensure((size_t)2 * nb * n);
    ctx->extract_mean.ensure(n);
    const dim3 grid(nb, n);
    const ExtractGeom* geom = ctx->extract_geom.p;
    if (any_tiles) k_extract<true><<<grid, kExT, 0, s>>>(d_tomo, nx, ny, nz, geom, N, d_out, ctx->extract_part.p);
    if (any_steep) k_extract<false><<<grid, kExT, 0, s>>>(d_tomo, nx, ny, nz, geom, N, d_out, ctx->extract_part.p);
    ETTK_HIP(hipGetLastError());
    launch_reslice_mean(ctx->extract_part.p, nb, n, ctx->extract_mean.p, s);
    k_extract_finish<<<dim3((unsigned)((n3 + kExT - 1) / kExT), n), kExT, 0, s>>>(d_out, ctx->extract_mean.p, n3);
    ETTK_HIP(hipGetLastError());
    ETTK_HIP(hipStreamSynchronize(s));
}

}  // namespace ettk

using namespace ettk;

extern "C" int ettk_extract_batch(ettk_ctx* ctx, const float* d_tomogram, int nx, int ny, int nz, int n,
                                  const double* positions, const ettk_particle* descs, int N, float* d_out) {
    try {
        ETTK_REQUIRE(ctx && d_tomogram && positions && descs && d_out, ETTK_ERR_ARG, "ettk_extract_batch: null argument");
        ETTK_REQUIRE(nx > 0 && ny > 0 && nz > 0 && n >= 0 && N > 0 && N <= 1024, ETTK_ERR_ARG,
                     "ettk_extract_batch: bad sizes");
        ETTK_REQUIRE((long long)nx * ny * nz < (1LL << 40), ETTK_ERR_ARG, "ettk_extract_batch: tomogram too large");
        if (n > 0) {
            ETTK_HIP(hipSetDevice(ctx->device));
            extract_batch(ctx, d_tomogram, nx, ny, nz, n, positions, descs, N, d_out);
        }
    } catch (const Error& e) {
        set_error(e.msg);
        return e.code;
    } catch (const std::exception& e) {
        set_error(e.what());
        return ETTK_ERR_ALLOC;
    }
    set_error("");
    return ETTK_OK;
}
