// project.hip -- magnitude of the padded particle spectrum that the S^2 projection samples
// (cartesianToSpherical, ProjRot.h:265-338).
//
// The masked image v = (image - mean) * mask + mean sits in the corner [0, N)^3 of a box of M = 2N whose rest holds the
// constant c (voxel (0,0,0) of v), times (-1)^(i+j+k).  The transform of the constant alone is c M^3 at (N, N, N) and
// 0 elsewhere, so v - c is transformed, of whose M^2 rows only N^2 and of whose M planes only N are not zero, and the
// constant is added to one element.  Two kernels: rows and columns of a plane (N planes per image), then the pencils
// along i with the magnitude as their epilogue.  Elements farther than `rad` from the centre are never sampled and are
// neither written nor read.
//
// HBM passes per image: 4 N^3 bytes in, 8 N M (N + 2) out and in again, 4 M^2 (N + 2) out; the general transform of the
// M^3 box followed by a magnitude pass moved 8 M^2 (N + 1) five times.
#include "kernels.hpp"
#include "regfft.hpp"

#include <cfloat>

namespace ettk {

namespace {

constexpr int kPmT = 256;

template <int M> struct PadShape {
    static constexpr int N = M / 2, T = ColShape<M>::T, E = ColShape<M>::E, HS = N + 2;
    static constexpr int RP = kPmT / T;               // row pairs per step
    static constexpr int CP = M == 256 ? 8 : kPmT / T;  // columns per step (M = 256: the exchange has to fit the LDS)
    static constexpr int LDZ = kRowLd<M>;
    static_assert(T % 2 == 0 && E % 2 == 0 && LDZ >= M, "row pairs and halves");
};

// Plane i of image b: N rows of N values, packed in pairs as one complex row of length M, transformed by T lanes each;
// the columns read their element of the two rows straight from the packed spectrum (Z(k) and Z(M - k)), so no split
// pass is stored.  Columns 0 and N are real before the column transform and share one.  Column N + 1 repeats column
// N - 1 conjugated and mirrored: with it every 4-tap stencil of the sampler reads one row.
// Bound by the stores of the spectrum: 32 images of 64^3 (2048 planes, 110 MB inside the radius) take 47 us; the row,
// column and plane passes over the whole box took 260 us.
template <int M>
__global__ void __launch_bounds__(kPmT) k_pad_planes(PadMagArgs a, const float2* __restrict__ twg) {
    using S = PadShape<M>;
    constexpr int N = S::N, T = S::T, E = S::E, HS = S::HS, LDZ = S::LDZ, CP = S::CP;
    __shared__ float2 Z[(N / 2) * LDZ];
    __shared__ float2 ex[M * CP];
    __shared__ float2 z0[M];
    __shared__ float2 tw[M];
    const int i = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
    for (int q = tid; q < M; q += kPmT) tw[q] = twg[q];
    const float* st = a.stats + b * 4;
    const float vmean = st[0], mean = st[1], padc = st[2];
    const bool mask_on = st[3] != 0.f;
    const float* __restrict__ in = a.in + ((size_t)b * N + i) * N * N;
    const float* __restrict__ msk = a.mask + (size_t)i * N * N;
    __syncthreads();
    {
        const int t = tid % T;
#pragma unroll 1
        for (int pp = tid / T; pp < N / 2; pp += S::RP) {
            float2 x[E];
            float r0[E / 2], r1[E / 2], m0[E / 2], m1[E / 2];
#pragma unroll
            for (int u = 0; u < E / 2; u++) {
                const int o = 2 * pp * N + t + T * u;
                r0[u] = in[o];
                r1[u] = in[o + N];
                m0[u] = mask_on ? msk[o] : 1.f;
                m1[u] = mask_on ? msk[o + N] : 1.f;
            }
#pragma unroll
            for (int u = 0; u < E / 2; u++) {
                const float i0 = r0[u] == -FLT_MAX ? 0.f : r0[u] - vmean, i1 = r1[u] == -FLT_MAX ? 0.f : r1[u] - vmean;
                const float v0 = (mask_on ? (i0 - mean) * m0[u] + mean : i0) - padc;
                const float v1 = (mask_on ? (i1 - mean) * m1[u] + mean : i1) - padc;
                const float sg = (i + t + T * u) & 1 ? -1.f : 1.f;  // rows 2 pp (even) and 2 pp + 1
                x[u] = make_float2(v0 * sg, -(v1 * sg));
            }
#pragma unroll
            for (int u = E / 2; u < E; u++) x[u] = make_float2(0.f, 0.f);
            float2* pen = Z + pp * LDZ;
            row_fft<M, false>(x, t, pen, tw);
#pragma unroll
            for (int u = 0; u < E; u++) pen[t + T * u] = x[u];
        }
    }
    __syncthreads();
    const int t = tid / CP, p = tid % CP;
    const bool on = t < T;
    float2* out = a.F + ((size_t)b * N + i) * M * HS;
    const int r2 = a.rad * a.rad;
#pragma unroll 1
    for (int k0 = 0; k0 < N; k0 += CP) {
        const int k = k0 + p;
        const bool live = on && k < N;
        float2 x[E];
        if (live)
#pragma unroll
            for (int u = 0; u < E; u++) {
                x[u] = make_float2(0.f, 0.f);
                if (u >= E / 2) continue;
                const int j = t + T * u;
                const float2 z = Z[(j >> 1) * LDZ + k], zm = Z[(j >> 1) * LDZ + (k ? M - k : N)];
                if (k == 0) x[u] = j & 1 ? make_float2(z.y, zm.y) : make_float2(z.x, zm.x);
                else x[u] = j & 1 ? make_float2(0.5f * (z.y + zm.y), 0.5f * (zm.x - z.x))
                                  : make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
            }
        col_fft<M, false, CP>(x, t, ex + p, tw, live);
        if (!live) continue;
        const int lim = r2 - (N - k) * (N - k);
#pragma unroll
        for (int u = 0; u < E; u++) {
            const int j = t + T * u;
            if (k == 0) {
                z0[j] = x[u];
                continue;
            }
            if ((j - N) * (j - N) > lim) continue;
            out[j * HS + k] = x[u];
            if (k == N - 1) out[((M - j) % M) * HS + N + 1] = cconj(x[u]);
        }
    }
    __syncthreads();
    for (int j = tid; j < M; j += kPmT) {
        const float2 z = z0[j], zc = cconj(z0[(M - j) % M]);
        const int dj = (j - N) * (j - N);
        if (dj + N * N <= r2) out[j * HS] = make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y + zc.y));
        if (dj <= r2) out[j * HS + N] = make_float2(0.5f * (z.y - zc.y), -0.5f * (z.x - zc.x));
    }
}

// pencils along i: N values in, M magnitudes out (their square roots with MCF)
// Bound by the traffic and the one exchange per pencil: 32 images of 64^3 take 61 us (180 MB); the strided pass over the
// whole box and the magnitude pass took 200 us.
template <int M>
__global__ void __launch_bounds__(kPmT) k_pad_mag(PadMagArgs a, const float2* __restrict__ twg) {
    using S = PadShape<M>;
    constexpr int N = S::N, T = S::T, E = S::E, HS = S::HS, P = kPmT / T, PL = M * HS;
    __shared__ float2 ex[M * P];
    __shared__ float2 tw[M];
    const int t = threadIdx.x / P, q = blockIdx.x * P + threadIdx.x % P, b = blockIdx.y;
    for (int w = threadIdx.x; w < M; w += kPmT) tw[w] = twg[w];
    const int j = q / HS, k = q % HS, dj = j - N, dk = N - k;
    const int lim = a.rad * a.rad - dj * dj - dk * dk;
    const bool live = q < PL && lim >= 0;
    const float2* in = a.F + (size_t)b * N * PL;
    float2 x[E];
    if (live)
#pragma unroll
        for (int u = 0; u < E; u++) x[u] = u < E / 2 ? at_byte(in + (size_t)u * T * PL, (unsigned)(t * PL + q) * 8) : make_float2(0.f, 0.f);
    __syncthreads();
    col_fft<M, false>(x, t, ex + threadIdx.x % P, tw, live);
    if (!live) return;
    float* out = a.mag + (size_t)b * M * PL;
    const float dc = dj == 0 && dk == 0 ? a.stats[b * 4 + 2] * ((float)M * M * M) : 0.f;
#pragma unroll
    for (int u = 0; u < E; u++) {
        const int di = t + T * u - N;
        if (di * di > lim) continue;
        const float re = x[u].x + (di == 0 ? dc : 0.f);
        const float m2 = re * re + x[u].y * x[u].y;
        at_byte(out + (size_t)u * T * PL, (unsigned)(t * PL + q) * 4) = a.mcf ? sqrtf(sqrtf(m2)) : sqrtf(m2);
    }
}

template <int M>
void launch_pad_mag(const FftTables& T, const PadMagArgs& a, hipStream_t s) {
    using S = PadShape<M>;
    constexpr int P = kPmT / S::T, PL = M * S::HS;
    const float2* tw = T.tw.p + T.offset[fft_len_index(M)];
    const double spec = (double)a.batch * S::N * PL * sizeof(float2), vol = (double)a.batch * PL * M * sizeof(float);
    {
        ProfScope ps(T.prof, "k_pad_planes", (double)a.batch * S::N * S::N * S::N * sizeof(float) + spec, s);
        k_pad_planes<M><<<dim3(S::N, a.batch), kPmT, 0, s>>>(a, tw);
    }
    ETTK_HIP(hipGetLastError());
    ProfScope ps(T.prof, "k_pad_mag", spec + vol, s);
    k_pad_mag<M><<<dim3((PL + P - 1) / P, a.batch), kPmT, 0, s>>>(a, tw);
    ETTK_HIP(hipGetLastError());
}

}  // namespace

void fft3_pad_magnitude(const FftTables& T, const PadMagArgs& a, int n, hipStream_t s) {
    switch (n) {
        case 16: launch_pad_mag<32>(T, a, s); break;
        case 32: launch_pad_mag<64>(T, a, s); break;
        case 48: launch_pad_mag<96>(T, a, s); break;
        case 64: launch_pad_mag<128>(T, a, s); break;
        case 96: launch_pad_mag<192>(T, a, s); break;
        case 128: launch_pad_mag<256>(T, a, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_pad_magnitude: unsupported size " + std::to_string(n)};
    }
}

}  // namespace ettk
