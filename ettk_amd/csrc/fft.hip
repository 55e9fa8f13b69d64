// fft.hip -- batched 3-D FFTs for gfx950, and the steps of the CCC and of the refinement that run inside their passes.
//
// Replaces the FFTW double-precision plans of nbfFourierFilter::initializeFFTWhalf
// (inc/em/nbfFourierFilter.h:270-358): fftw_plan_dft_r2c_3d / fftw_plan_dft_c2r_3d on [i][j][k] arrays
// with the half spectrum along k.  Every pass reads and writes each element of HBM once.
//   r2c: pass k (pairs of real rows packed as one complex row, split after the transform), pass j, pass i
//   c2r: pass i, pass j (complex, backward), then pass k (pairs of half rows -> two real rows)
// Up to 128 the k and j passes of a (b, i) plane run in one workgroup.  Two forms of a pass stand side by side: pencils
// staged in LDS (Stockham stages of radix 4/3/2, or of 8 in registers), which the plain and the refinement's transforms
// use, and pencils held in registers with one LDS exchange (regfft.hpp), which the CCC's kernels and the strided passes
// above 64 use.
#include "kernels.hpp"
#include "regfft.hpp"
#include "wedge.hpp"

#include <cfloat>
#include <cmath>

namespace ettk {

static const int kLens[9] = {16, 32, 48, 64, 96, 128, 192, 256, 0};

int fft_len_index(int L) {
    for (int i = 0; kLens[i]; i++)
        if (kLens[i] == L) return i;
    return -1;
}

void fft_tables_init(FftTables& T, hipStream_t s) {
    std::vector<float2> h;
    for (int i = 0; kLens[i]; i++) {
        T.offset[i] = (int)h.size();
        int L = kLens[i];
        for (int t = 0; t < L; t++) {
            double a = -2.0 * M_PI * (double)t / (double)L;
            h.push_back(make_float2((float)std::cos(a), (float)std::sin(a)));
        }
    }
    T.tw.upload(h.data(), h.size(), s);
    ETTK_HIP(hipStreamSynchronize(s));
}

template <int L> struct Shape {
    static constexpr int TPP = L / 4;                       // threads per pencil
    static constexpr int P = (1024 / L) > 0 ? 1024 / L : 1; // pencils per workgroup
    static constexpr int THREADS = P * TPP;
    static constexpr int LD = L + 1;                        // padded LDS row
    static_assert(THREADS >= L, "one twiddle per thread");
};

template <int L, int R>
__device__ __forceinline__ void stockham_stage(float2* pen, int lane, int Ns, const float2* tw, bool inv) {
    constexpr int NB = L / R;
    constexpr int TPP = Shape<L>::TPP;
    constexpr int MAXB = (NB + TPP - 1) / TPP;
    float2 v[MAXB][R];
    int base[MAXB];
    const int step = L / (Ns * R);
#pragma unroll
    for (int c = 0; c < MAXB; c++) {
        int bf = lane + c * TPP;
        base[c] = -1;
        if (bf < NB) {
            int k = bf % Ns;
#pragma unroll
            for (int m = 0; m < R; m++) {
                float2 x = pen[bf + m * NB];
                if (m > 0) {
                    float2 w = tw[m * k * step];
                    if (inv) w.y = -w.y;
                    x = cmul(x, w);
                }
                v[c][m] = x;
            }
            butterfly<R>(v[c], inv);
            base[c] = (bf / Ns) * Ns * R + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < MAXB; c++)
        if (base[c] >= 0)
#pragma unroll
            for (int m = 0; m < R; m++) pen[base[c] + m * Ns] = v[c][m];
    __syncthreads();
}

template <int L, int S>
__device__ __forceinline__ void run_stage(float2* pen, int lane, int& Ns, const float2* tw, bool inv) {
    using RD = Radices<L>;
    if constexpr (S < RD::n) {
        constexpr int R = RD::r[S];
        stockham_stage<L, R>(pen, lane, Ns, tw, inv);
        Ns *= R;
    }
}

// in-LDS transform of one pencil (every thread of the block must call it: it synchronises)
template <int L>
__device__ __forceinline__ void lds_fft(float2* pen, int lane, const float2* tw, bool inv) {
    int Ns = 1;
    run_stage<L, 0>(pen, lane, Ns, tw, inv);
    run_stage<L, 1>(pen, lane, Ns, tw, inv);
    run_stage<L, 2>(pen, lane, Ns, tw, inv);
    run_stage<L, 3>(pen, lane, Ns, tw, inv);
}

// ------------------------------------------------------------------ length 64 in registers (8 x 8)
// 64 = 8 x 8 Cooley-Tukey: each of 8 threads holds x[t + 8m] (m = 0..7), runs an 8-point DFT in registers,
// applies W64^(t k1), and the 8 x 8 block is transposed through the pencil's own LDS row; an 8-point DFT per
// thread finishes X[k1 + 8 k2].  One LDS exchange instead of three radix-4 stages.
// the twiddles a thread of a length-64 pencil applies, w[k] = exp(-2 pi i lane k / 64), held in registers
// for all the pencil transforms of a kernel (length 64 only; other lengths read the LDS table)
template <int L> struct TwCache {
    float2 w[L == 64 ? 8 : 1];
};
template <int L>
__device__ __forceinline__ TwCache<L> tw_cache(const float2* tw, int lane) {
    TwCache<L> c;
    if constexpr (L == 64) {
#pragma unroll
        for (int k = 0; k < 8; k++) c.w[k] = tw[(lane * k) & 63];
    } else {
        c.w[0] = make_float2(1.f, 0.f);
    }
    return c;
}

// every thread of the workgroup must call it (it ends with a workgroup barrier, after which the whole pencil is
// visible to every thread).  The 8 threads of a pencil (lanes 8q .. 8q+7 of the workgroup) share a wavefront,
// so the exchange inside needs only wavefront ordering.  The 8 x 8 exchange goes through rows of 9
// (pen[k * 9 + t] = element k of thread t), so neither its writes nor its reads collide in LDS banks; the
// pencil's storage therefore spans 72 entries.
__device__ __forceinline__ void fft64_reg(float2* pen, int lane, const TwCache<64>& tc, bool inv) {
    float2 x[8];
#pragma unroll
    for (int m = 0; m < 8; m++) x[m] = pen[lane + 8 * m];
    dft8(x, inv);
#pragma unroll
    for (int k = 1; k < 8; k++) {
        float2 w = tc.w[k];
        if (inv) w.y = -w.y;
        x[k] = cmul(x[k], w);
    }
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < 8; k++) pen[k * 9 + lane] = x[k];
    wave_lds_order();
#pragma unroll
    for (int t = 0; t < 8; t++) x[t] = pen[lane * 9 + t];
    dft8(x, inv);
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < 8; k++) pen[lane + 8 * k] = x[k];
    __syncthreads();
}

// The same for 96 = 12 x 8 and 128 = 16 x 8: an (L/8)-point DFT per thread, the exchange, then L/8 8-point DFTs over the
// 8 threads (two per thread; at 96 half of the threads' second one is idle).  The pencil's storage spans 9 L/8 entries.
template <int L, bool INV>
__device__ __forceinline__ void fft_reg8(float2* pen, int lane, const float2* tw) {
    constexpr int N1 = L / 8, NR = (N1 + 7) / 8;
    float2 x[N1];
#pragma unroll
    for (int m = 0; m < N1; m++) x[m] = pen[lane + 8 * m];
    Dft<N1, INV>::run(x);
#pragma unroll
    for (int k = 1; k < N1; k++) {
        float2 w = tw[lane * k];
        if (INV) w.y = -w.y;
        x[k] = cmul(x[k], w);
    }
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < N1; k++) pen[k * 9 + lane] = x[k];
    wave_lds_order();
    float2 y[NR][8];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k1 = lane + 8 * r;
        if (k1 < N1) {
#pragma unroll
            for (int b = 0; b < 8; b++) y[r][b] = pen[k1 * 9 + b];
            Dft<8, INV>::run(y[r]);
        }
    }
    wave_lds_order();
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k1 = lane + 8 * r;
        if (k1 < N1)
#pragma unroll
            for (int k = 0; k < 8; k++) pen[k1 + N1 * k] = y[r][k];
    }
    __syncthreads();
}

// threads per pencil of the pencil FFT used by the fused and strided passes, and the LDS stride of a pencil
template <int L> struct PenT {
    static constexpr bool kReg = L == 64 || L == 96 || L == 128;
    static constexpr int TPP = kReg ? 8 : Shape<L>::TPP;
    static constexpr int LD = kReg ? 9 * (L / 8) + 1 : L + 1;
};
template <int L>
__device__ __forceinline__ void pencil_fft(float2* pen, int lane, const float2* tw, const TwCache<L>& tc, bool inv) {
    if constexpr (L == 64) fft64_reg(pen, lane, tc, inv);
    else if constexpr (PenT<L>::kReg) {
        if (inv) fft_reg8<L, true>(pen, lane, tw);
        else fft_reg8<L, false>(pen, lane, tw);
    } else lds_fft<L>(pen, lane, tw, inv);
}

// ------------------------------------------------------------------ r2c, pass along k (real rows)
template <int L>
__global__ void __launch_bounds__(Shape<L>::THREADS) k_r2c_rows(R2CArgs a, const float2* __restrict__ twg) {
    using S = Shape<L>;
    constexpr int H = L / 2 + 1;
    __shared__ float2 lds[S::P * S::LD];
    __shared__ float2 tw[L];
    const long npairs = (long)a.batch * L * L / 2;
    const long p0 = (long)blockIdx.x * S::P;
    const float2 twv = twg[threadIdx.x % L];  // stored after the staging loads are in flight
    // load P pairs of rows (2L contiguous floats each) and pack row 2q + i*row 2q+1
    for (int t = threadIdx.x; t < S::P * 2 * L; t += blockDim.x) {
        int q = t / (2 * L), r = t % (2 * L);
        long pair = p0 + q;
        float x = 0.0f;
        if (pair < npairs) {
            long row = pair * 2 + r / L;
            x = a.in[row * L + r % L];
        }
        float* f = reinterpret_cast<float*>(&lds[q * S::LD + (r % L)]);
        f[r / L] = x;
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / S::TPP, lane = threadIdx.x % S::TPP;
    lds_fft<L>(&lds[q * S::LD], lane, tw, false);
    // split Z = A + iB into the half spectra of the two rows
    for (int t = threadIdx.x; t < S::P * 2 * H; t += blockDim.x) {
        int qq = t / (2 * H), r = t % (2 * H);
        long pair = p0 + qq;
        if (pair >= npairs) continue;
        int which = r / H, k = r % H;
        float2 z = lds[qq * S::LD + k], zc = cconj(lds[qq * S::LD + ((L - k) % L)]);
        float2 o = which == 0 ? cscale(cadd(z, zc), 0.5f) : make_float2(0.5f * (z.y - zc.y), -0.5f * (z.x - zc.x));
        a.out[(pair * 2 + which) * H + k] = o;
    }
}

// ------------------------------------------------------------------ complex pass along a strided axis
struct StridedArgs {
    const float2* in;
    float2* out;
    long npencils;
    long inner;         // pencils with consecutive addresses
    long outer_stride;  // address step between groups of `inner` pencils
    long es;            // element stride along the transformed axis
    int inv;
};

template <int L> struct StridedShape {
    static constexpr int TPP = PenT<L>::TPP;
    static constexpr int P = Shape<L>::THREADS / TPP;  // pencils per workgroup
    static constexpr int THREADS = Shape<L>::THREADS;
    static constexpr int LD = PenT<L>::LD;
};

template <int L>
__global__ void __launch_bounds__(StridedShape<L>::THREADS) k_fft_strided(StridedArgs a, const float2* __restrict__ twg) {
    using S = StridedShape<L>;
    __shared__ float2 lds[S::P * S::LD];
    __shared__ float2 tw[L];
    // consecutive pencil groups on one XCD: at L = 128 a group's rows are half cache lines, whose other halves
    // belong to the neighbouring groups (fetched into one L2 instead of two)
    const long q0 = (long)xcd_tile(blockIdx.x, gridDim.x) * S::P;
    const float2 twv = twg[threadIdx.x % L];  // stored after the staging loads are in flight
    // THREADS is a multiple of P: a thread moves the elements l = t / P, t / P + THREADS / P, ... of the one
    // pencil t % P, so the pencil's base address is computed once
    const int qm = threadIdx.x % S::P;
    const long pen = q0 + qm;
    const bool valid = pen < a.npencils;
    const long base = valid ? (pen / a.inner) * a.outer_stride + (pen % a.inner) : 0;
    constexpr int STEP = S::THREADS / S::P, NL = L / STEP;
    static_assert(L % STEP == 0, "pencil elements per thread");
    const int l0 = threadIdx.x / S::P;
    {
        float2 v[NL];  // all loads in flight before the first LDS store (an invalid pencil re-reads pencil 0)
#pragma unroll
        for (int u = 0; u < NL; u++) v[u] = a.in[base + (long)(l0 + u * STEP) * a.es];
#pragma unroll
        for (int u = 0; u < NL; u++) lds[qm * S::LD + l0 + u * STEP] = valid ? v[u] : make_float2(0.f, 0.f);
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / S::TPP, lane = threadIdx.x % S::TPP;
    pencil_fft<L>(&lds[q * S::LD], lane, tw, tw_cache<L>(tw, lane), a.inv != 0);
    if (valid)
#pragma unroll
        for (int u = 0; u < NL; u++) a.out[base + (long)(l0 + u * STEP) * a.es] = lds[qm * S::LD + l0 + u * STEP];
}

// Pencils in registers (regfft.hpp): loads and stores in rows of P consecutive pencils, one LDS exchange.  Bound by HBM.
template <int L, bool INV>
__global__ void __launch_bounds__(ColShape<L>::THREADS) k_fft_col(StridedArgs a, const float2* __restrict__ twg) {
    using S = ColShape<L>;
    __shared__ float2 ex[L * S::P];
    __shared__ float2 tw[L];
    // consecutive pencil groups on one XCD: a group's rows share cache lines with the neighbouring groups' where the
    // rows are not aligned to them
    const long pen = (long)xcd_tile(blockIdx.x, gridDim.x) * S::P + threadIdx.x % S::P;
    const int t = threadIdx.x / S::P;
    const bool valid = pen < a.npencils;  // an invalid pencil transforms pencil 0 and stores nothing
    const long base = valid ? (pen / a.inner) * a.outer_stride + (pen % a.inner) : 0;
    float2 x[S::E];
#pragma unroll
    for (int j = 0; j < S::E; j++) x[j] = a.in[base + (long)(t + j * S::T) * a.es];
    for (int q = threadIdx.x; q < L; q += S::THREADS) tw[q] = twg[q];
    __syncthreads();
    col_fft<L, INV>(x, t, ex + threadIdx.x % S::P, tw);
    if (valid)
#pragma unroll
        for (int j = 0; j < S::E; j++) a.out[base + (long)(t + j * S::T) * a.es] = x[j];
}

// ------------------------------------------------------------------ CCC spectra: one pass along i (L <= 128)
// deterministic sum over the NT threads of a workgroup (NT need not be a multiple of 64), valid in thread 0
template <int NT>
__device__ __forceinline__ float block_sum_nt(float v, float* sred) {
    constexpr int NFW = NT / 64, REM = NT % 64;
    const int w = threadIdx.x >> 6;
    if (w < NFW) {
        for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
        if ((threadIdx.x & 63) == 0) sred[w] = v;
    } else {
        sred[NFW + (threadIdx.x & 63)] = v;
    }
    __syncthreads();
    float tot = 0.f;
    if (threadIdx.x == 0)
        for (int i = 0; i < NFW + REM; i++) tot += sred[i];
    __syncthreads();
    return tot;
}

// Between the k/j plane passes of the particle's r2c and the fused plane kernels, every step of the CCC runs on
// pencils along i, so one kernel does them all per pencil (j, k) of an evaluation:
//   F2 = forward i-transform of the plane-pass output (completes the particle's r2c)
//   fw = filter * W1 * W2(e) (the smoothed particle wedge at the evaluation's transform, computed once)
//   X2 = mcf(F2) * fw, DC term zeroed -> S2 (the combine's F2), and its inverse i-transform -> S3
//   X1 = F1mcf * fw, DC term zeroed -> inverse i-transform -> S1
//   per-block partials of sum hw |X1|^2, sum fw, sum hw |X2|^2 (hw = 2 off the last half plane), FP32 over the
//   workgroup's L P elements (E per thread, then a tree), the workgroups in FP64
// Distances of 128 to 480 evaluations differ from FP64 by an rms of 2.0e-7, 1.6e-7, 1.7e-7, 2.0e-7 and 6.3e-7 relative at
// 32, 48, 64, 96 and 128; with partials of 1024 elements everywhere above 64 and the transforms staged in LDS they differed
// by 2.3e-7, 2.4e-7, 1.6e-7, 2.8e-7 and 7.3e-7.
// The element-wise arithmetic is that of nbfFourierFilter::executeHalf (FFilt.h:587-606) and normalizeFourierHalf
// (CorrMetric.h:498-530).
// Each thread keeps its E elements of a pencil in registers through the three transforms (regfft.hpp).
template <int L>
__global__ void __launch_bounds__(ColShape<L>::THREADS) k_ccc_ipass(CccIpassArgs a, const float2* __restrict__ twg) {
    using S = ColShape<L>;
    constexpr int H = L / 2 + 1, LH = L * H, NE = S::E;
    __shared__ float2 ex[L * S::P];
    __shared__ float2 tw[L];
    __shared__ float sred[S::THREADS / 64 + 1];
    __shared__ int n_near;
    if (threadIdx.x == 0) n_near = 0;
    const int e = blockIdx.y;
    const int t = threadIdx.x / S::P;
    const int p = blockIdx.x * S::P + threadIdx.x % S::P;  // pencil (j, k) = (p / H, p % H) of evaluation e
    const bool valid = p < LH;
    const int pc = valid ? p : 0, pj = pc / H, pk = pc % H;
    const size_t vol = (size_t)e * L * LH;
    const unsigned lo = (t * LH + pc) * 8;  // byte offset of this thread's first element of a spectrum
    float2* __restrict__ xp = ex + threadIdx.x % S::P;
    float2 x[NE];
#pragma unroll
    for (int u = 0; u < NE; u++) x[u] = ld_stream(&at_byte(a.S2 + vol + u * S::T * LH, lo));
    for (int q = threadIdx.x; q < L; q += S::THREADS) tw[q] = twg[q];
    __syncthreads();
    col_fft<L, false>(x, t, xp, tw);
    // filter weights of this thread's elements (i = t + u T of pencil p), the particle side in place
    const EvalGeom& g = a.geom[e];
    const int dc_i = L / 2, dc_j = L / 2, dc_k = H - 1;
    const float hw = pk < H - 1 ? 2.f : 1.f;
    float fw[NE], w1[NE];
    float s2 = 0.f, swf = 0.f;
#pragma unroll
    for (int u = 0; u < NE; u++) {
        fw[u] = at_byte(a.filter + u * S::T * LH, lo / 2);
        w1[u] = a.W1 ? at_byte(a.W1 + u * S::T * LH, lo / 2) : 1.f;
    }
    if (!g.full) {
        // Smoothed wedge W2.  About one element in ten lies near a plane and needs the 27-sample stencil, but nearly
        // every wavefront holds one: the near ones are listed in LDS (the exchange buffer, free here) and evaluated by
        // all threads evenly.  240 evaluations at 64^3: 234 us, 302 with the stencil where its element lies and 215
        // without a wedge (the HBM rate); 36 at 128^3: 361 against 455 us.
        float* __restrict__ near_w = reinterpret_cast<float*>(ex);                   // [u][thread]
        int* __restrict__ list = reinterpret_cast<int*>(ex) + NE * S::THREADS;
        unsigned far = 0, inside = 0;  // bits of this thread's elements
#pragma unroll
        for (int u = 0; u < NE; u++) {
            bool in;
            const bool uni = wedge_uniform(g.v1, g.v2, t + u * S::T, pj, pk, L, in);
            if (uni) far |= 1u << u;
            if (in) inside |= 1u << u;
            if (!uni && valid) list[atomicAdd(&n_near, 1)] = u * S::THREADS + threadIdx.x;
        }
        __syncthreads();
        for (int q = threadIdx.x; q < n_near; q += S::THREADS) {
            const int m = list[q], th = m % S::THREADS, pp = blockIdx.x * S::P + th % S::P;
            near_w[m] = wedge_stencil(g.v1, g.v2, th / S::P + m / S::THREADS * S::T, pp / H, pp % H, L, H);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NE; u++) {
            if (far >> u & 1) w1[u] *= inside >> u & 1 ? wedge_ones(t + u * S::T, pj, pk, L, H) : 0.f;
            else if (valid) w1[u] *= near_w[u * S::THREADS + threadIdx.x];
        }
        __syncthreads();  // the exchange buffer is reused by the transforms below
    }
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const int i = t + u * S::T;
        fw[u] *= w1[u];
        float2 z = x[u];
        if (a.mcf) {
            const float m2 = z.x * z.x + z.y * z.y;
            const float C = sqrtf(sqrtf(m2));
            if (C > 0.f) z = make_float2(z.x / C, z.y / C);
        }
        if (a.apply) z = cscale(z, fw[u]);
        if (i == dc_i && pj == dc_j && pk == dc_k) z = make_float2(0.f, 0.f);
        if (valid) {
            st_stream(&at_byte(a.S2 + vol + u * S::T * LH, lo), z);
            s2 += hw * (z.x * z.x + z.y * z.y);
            swf += fw[u];
        }
        x[u] = z;
    }
    col_fft<L, true>(x, t, xp, tw);
    // reference side: its spectrum loads are issued before the particle side's inverse transform is stored
    float2 f1[NE];
#pragma unroll
    for (int u = 0; u < NE; u++) f1[u] = at_byte(a.F1mcf + u * S::T * LH, lo);
    if (valid)
#pragma unroll
        for (int u = 0; u < NE; u++) st_stream(&at_byte(a.S3 + vol + u * S::T * LH, lo), x[u]);
    float s1 = 0.f;
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const int i = t + u * S::T;
        float2 z = f1[u];
        if (a.apply) z = cscale(z, fw[u]);
        if (i == dc_i && pj == dc_j && pk == dc_k) z = make_float2(0.f, 0.f);
        if (valid) s1 += hw * (z.x * z.x + z.y * z.y);
        x[u] = z;
    }
    col_fft<L, true>(x, t, xp, tw);
    if (valid)
#pragma unroll
        for (int u = 0; u < NE; u++) st_stream(&at_byte(a.S1 + vol + u * S::T * LH, lo), x[u]);
    const float t1 = block_sum_nt<S::THREADS>(s1, sred);
    const float tf = block_sum_nt<S::THREADS>(swf, sred);
    const float t2 = block_sum_nt<S::THREADS>(s2, sred);
    if (threadIdx.x == 0) {
        const size_t o = (size_t)e * gridDim.x + blockIdx.x;
        a.p_n1[o] = t1;
        a.p_wf[o] = tf;
        a.p_n2[o] = t2;
    }
}

// ------------------------------------------------------------------ c2r, pass along k (half rows)
template <int L>
__global__ void __launch_bounds__(Shape<L>::THREADS) k_c2r_rows(const float2* __restrict__ in, float* __restrict__ out,
                                                                  long npairs, const float2* __restrict__ twg) {
    using S = Shape<L>;
    constexpr int H = L / 2 + 1;
    __shared__ float2 lds[S::P * S::LD];
    __shared__ float2 tw[L];
    const long p0 = (long)blockIdx.x * S::P;
    const float2 twv = twg[threadIdx.x % L];  // stored after the staging loads are in flight
    // Z(k) = A(k) + i B(k) over the full length, with A(L-k) = conj(A(k)) and real A(0), A(L/2)
    for (int t = threadIdx.x; t < S::P * L; t += blockDim.x) {
        int q = t / L, k = t % L;
        long pair = p0 + q;
        float2 z = make_float2(0.f, 0.f);
        if (pair < npairs) {
            const float2* ra = in + (pair * 2) * H;
            const float2* rb = ra + H;
            float2 A, Bv;
            if (k <= L / 2) {
                A = ra[k];
                Bv = rb[k];
                if (k == 0 || k == L / 2) { A.y = 0.f; Bv.y = 0.f; }
            } else {
                A = cconj(ra[L - k]);
                Bv = cconj(rb[L - k]);
            }
            z = make_float2(A.x - Bv.y, A.y + Bv.x);
        }
        lds[q * S::LD + k] = z;
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / S::TPP, lane = threadIdx.x % S::TPP;
    lds_fft<L>(&lds[q * S::LD], lane, tw, true);
    for (int t = threadIdx.x; t < S::P * 2 * L; t += blockDim.x) {
        int qq = t / (2 * L), r = t % (2 * L);
        long pair = p0 + qq;
        if (pair >= npairs) continue;
        float2 z = lds[qq * S::LD + (r % L)];
        out[pair * 2 * L + r] = (r < L) ? z.x : z.y;
    }
}

// ------------------------------------------------------------------ fused plane passes (L <= 128)
// One workgroup per (batch, i) plane of L x L reals: the k pass (pairs of real rows packed as complex rows) and
// the j pass run back to back in LDS, so an r2c moves each element through HBM twice (plane pass + i pass)
// instead of three times.  H pencil groups of TPP threads; the spare group of the k pass works on a dummy row.
// The k pass works on the L/2 row pairs.  The j pass works on L/2 pencils as well: the DC (k = 0) and Nyquist
// (k = L/2) columns of a real plane's row transforms are real, so they travel as one complex pencil
// DC + i Nyquist (pencil 0) and are separated after the transform by Hermitian symmetry; the other pencils
// are the columns k = 1 .. L/2 - 1.  Slot L/2 of the buffer holds the Nyquist column while a c2r packs it.
template <int L> struct Plane {
    static constexpr int H = L / 2 + 1;
    static constexpr int TPP = PenT<L>::TPP;
    static constexpr int THREADS = (L / 2) * TPP;
    static constexpr int LD = PenT<L>::LD;
    static_assert(THREADS >= L, "one twiddle per thread");
};

// c2r: pencil 0 <- h(column 0) + i h(column L/2), h(c)(j) = (c(j) + conj c(-j)) / 2.  The c2r keeps only the real
// part of the inverse i/j transforms on these two planes (FFTW's c2r; a spectrum that is not exactly Hermitian
// there, such as one weighted by a border-clipped smoothed wedge, has an imaginary part that is dropped).  The
// inverse transform of h(c) is exactly that real part, so the two columns share one transform: its real and
// imaginary parts.  Every thread of the workgroup must call it (it synchronises).
template <int L>
__device__ __forceinline__ void pack_dc_nyquist(float2* buf) {
    constexpr int LD = Plane<L>::LD;
    const int t = threadIdx.x, tm = (L - t) % L;
    float2 z = make_float2(0.f, 0.f);
    if (t < L) {
        const float2 c0 = buf[t], c0m = cconj(buf[tm]), cn = buf[(L / 2) * LD + t], cnm = cconj(buf[(L / 2) * LD + tm]);
        const float2 h0 = make_float2(0.5f * (c0.x + c0m.x), 0.5f * (c0.y + c0m.y));
        const float2 hn = make_float2(0.5f * (cn.x + cnm.x), 0.5f * (cn.y + cnm.y));
        z = make_float2(h0.x - hn.y, h0.y + hn.x);
    }
    __syncthreads();
    if (t < L) buf[t] = z;
}
// c2r along k: Z(k) = A(k) + i B(k) of rows 2pp, 2pp+1 over the full length from the inverse-j-transformed
// pencils, A(L-k) = conj(A(k)), A(0) and A(L/2) real (the real and imaginary parts of pencil 0)
template <int L>
__device__ __forceinline__ float2 c2r_row_pair(const float2* buf, int pp, int k) {
    constexpr int LD = Plane<L>::LD;
    float2 A, Bv;
    if (k == 0 || k == L / 2) {
        const float2 a = buf[2 * pp], b = buf[2 * pp + 1];
        A = make_float2(k == 0 ? a.x : a.y, 0.f);
        Bv = make_float2(k == 0 ? b.x : b.y, 0.f);
    } else if (k < L / 2) {
        A = buf[k * LD + 2 * pp];
        Bv = buf[k * LD + 2 * pp + 1];
    } else {
        A = cconj(buf[(L - k) * LD + 2 * pp]);
        Bv = cconj(buf[(L - k) * LD + 2 * pp + 1]);
    }
    return make_float2(A.x - Bv.y, A.y + Bv.x);
}
// r2c: value o of column k of row 2pp + which into the j-pass pencils; at k = 0 and k = L/2 the row transform of
// a real row is real (o.y is exactly 0) and goes to the real or imaginary part of pencil 0
template <int L>
__device__ __forceinline__ void r2c_split_store(float2* buf, int pp, int which, int k, float2 o) {
    constexpr int LD = Plane<L>::LD;
    if (k > 0 && k < L / 2) buf[k * LD + 2 * pp + which] = o;
    else reinterpret_cast<float*>(&buf[2 * pp + which])[k == 0 ? 0 : 1] = o.x;
}
// r2c: element (j, k) of the half plane after the forward j pass; DC and Nyquist from pencil 0 Z:
// X0(j) = (Z(j) + conj Z(-j)) / 2, XN(j) = (Z(j) - conj Z(-j)) / 2i
template <int L>
__device__ __forceinline__ float2 r2c_half_at(const float2* buf, int j, int k) {
    constexpr int LD = Plane<L>::LD;
    if (k > 0 && k < L / 2) return buf[k * LD + j];
    const float2 z = buf[j], zc = cconj(buf[(L - j) % L]);
    if (k == 0) return make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y + zc.y));
    return make_float2(0.5f * (z.y - zc.y), -0.5f * (z.x - zc.x));
}

// the k-pass input of plane i for one preprocessing mode, staged as packed row pairs buf[(j/2) LD + x]
// (.x row j even, .y row j odd); MSK: aux0 holds the N^3 mask
template <int L, int PRO, bool MSK>
__device__ __forceinline__ void r2c_stage_plane(const R2CArgs& a, int pi, const float* __restrict__ src, float mean,
                                                float2* buf) {
    constexpr int LD = Plane<L>::LD;
    const float* __restrict__ msk = MSK ? a.aux0 + (size_t)pi * L * L : nullptr;
    block_copy<Plane<L>::THREADS, L * L>(
        [&](int t) { return make_float2(src[t], MSK ? msk[t] : 1.0f); },
        [&](int t, float2 v) {
            const int j = t / L, x = t % L;
            const float sg = ((pi + j + x) & 1) ? -1.0f : 1.0f;
            float r;
            if constexpr (PRO == PRO_NONE) r = v.x;
            else if constexpr (PRO == PRO_SHIFT) r = v.x * sg;
            else if constexpr (PRO == PRO_MASK_SHIFT) r = v.x * v.y * sg;
            else r = (v.x == -3.402823466e+38f) ? 0.0f : (v.x - mean) * v.y * sg;  // PRO_RESLICED
            reinterpret_cast<float*>(&buf[(j >> 1) * LD + x])[j & 1] = r;
        });
}

template <int L>
__global__ void __launch_bounds__(Plane<L>::THREADS) k_r2c_plane(R2CArgs a, const float2* __restrict__ twg) {
    using PL = Plane<L>;
    constexpr int H = PL::H, LD = PL::LD;
    constexpr int NS = ((L / 2) * 2 * H + PL::THREADS - 1) / PL::THREADS;  // split outputs per thread
    __shared__ float2 buf[H * LD];  // k pass: L/2 packed row pairs; then j pass: L/2 column pencils
    __shared__ float2 tw[L];
    const long plane = blockIdx.x;  // b * L + i
    const int pb = (int)(plane / L), pi = (int)(plane % L);
    const float* src = a.in + plane * L * L;
    const float mean = a.pro == PRO_RESLICED ? a.stats[pb] : 0.0f;
    const float2 twv = twg[threadIdx.x % L];  // stored after the staging loads are in flight
    switch (a.pro) {
        case PRO_NONE: r2c_stage_plane<L, PRO_NONE, false>(a, pi, src, mean, buf); break;
        case PRO_SHIFT: r2c_stage_plane<L, PRO_SHIFT, false>(a, pi, src, mean, buf); break;
        case PRO_MASK_SHIFT: r2c_stage_plane<L, PRO_MASK_SHIFT, true>(a, pi, src, mean, buf); break;
        case PRO_RESLICED:
            if (a.aux0) r2c_stage_plane<L, PRO_RESLICED, true>(a, pi, src, mean, buf);
            else r2c_stage_plane<L, PRO_RESLICED, false>(a, pi, src, mean, buf);
            break;
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / PL::TPP, lane = threadIdx.x % PL::TPP;
    const TwCache<L> twc = tw_cache<L>(tw, lane);
    pencil_fft<L>(&buf[q * LD], lane, tw, twc, false);
    // split Z = A + iB of each pair into the half spectra of its two rows, through registers
    float2 o[NS];
#pragma unroll
    for (int u = 0; u < NS; u++) {
        const int t = threadIdx.x + u * PL::THREADS;
        if (t < (L / 2) * 2 * H) {
            const int pp = t / (2 * H), r = t % (2 * H), which = r / H, k = r % H;
            const float2 z = buf[pp * LD + k], zc = cconj(buf[pp * LD + ((L - k) % L)]);
            o[u] = which == 0 ? cscale(cadd(z, zc), 0.5f) : make_float2(0.5f * (z.y - zc.y), -0.5f * (z.x - zc.x));
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NS; u++) {
        const int t = threadIdx.x + u * PL::THREADS;
        if (t < (L / 2) * 2 * H) {
            const int pp = t / (2 * H), r = t % (2 * H), which = r / H, k = r % H;
            r2c_split_store<L>(buf, pp, which, k, o[u]);
        }
    }
    __syncthreads();
    pencil_fft<L>(&buf[q * LD], lane, tw, twc, false);
    float2* op = a.out + plane * L * H;
    for (int t = threadIdx.x; t < L * H; t += blockDim.x) op[t] = r2c_half_at<L>(buf, t / H, t % H);
}

template <int L>
__global__ void __launch_bounds__(Plane<L>::THREADS) k_c2r_plane(const float2* __restrict__ in, float* __restrict__ out,
                                                                   const float2* __restrict__ twg) {
    using PL = Plane<L>;
    constexpr int H = PL::H, LD = PL::LD;
    constexpr int NZ = ((L / 2) * L + PL::THREADS - 1) / PL::THREADS;
    __shared__ float2 buf[H * LD];
    __shared__ float2 tw[L];
    const long plane = blockIdx.x;
    const float2 twv = twg[threadIdx.x % L];  // stored after the staging loads are in flight
    const float2* ip = in + plane * L * H;
    block_copy<PL::THREADS, L * H>([&](int t) { return ip[t]; }, [&](int t, float2 v) { buf[(t % H) * LD + t / H] = v; });
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    pack_dc_nyquist<L>(buf);
    __syncthreads();
    const int q = threadIdx.x / PL::TPP, lane = threadIdx.x % PL::TPP;
    const TwCache<L> twc = tw_cache<L>(tw, lane);
    pencil_fft<L>(&buf[q * LD], lane, tw, twc, true);
    float2 zr[NZ];
#pragma unroll
    for (int u = 0; u < NZ; u++) {
        const int t = threadIdx.x + u * PL::THREADS;
        if (t < (L / 2) * L) zr[u] = c2r_row_pair<L>(buf, t / L, t % L);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NZ; u++) {
        const int t = threadIdx.x + u * PL::THREADS;
        if (t < (L / 2) * L) buf[(t / L) * LD + (t % L)] = zr[u];
    }
    __syncthreads();
    pencil_fft<L>(&buf[q * LD], lane, tw, twc, true);
    float* op = out + plane * L * L;
    for (int t = threadIdx.x; t < L * L; t += blockDim.x) {
        const int j = t / L, x = t % L;
        const float2 z = buf[(j >> 1) * LD + x];
        op[t] = (j & 1) ? z.y : z.x;
    }
}

// ------------------------------------------------------------------ fused c2r -> pointwise op -> r2c (L <= 128)
// Between the inverse and the forward transform of one volume, a (b, i) plane is complete in a workgroup after the c2r
// plane passes: the pointwise operation and the r2c plane passes run there, so the real volume never goes
// through HBM.  `io` holds the half spectrum after the inverse i pass and receives the forward j/k passes.
//   PLANE_OP_MASK:          r <- r m (m = aux, N^3), partials[plane] = sum r^2 m over the plane (FP32: 2E terms per
//                           thread, then the threads as a tree; the planes are added in FP64)
//   PLANE_OP_SQUARE_SHIFT:  r <- r^2 (-1)^(i+j+k)
// One launch runs one or two batches of `planes` planes, each with its operation: the CCC's two sides together fill the
// chip where one evaluation's N planes would not.
struct PlaneOps {
    float2 *io0, *io1;
    int op0, op1;
    unsigned planes;
    const float* mask;  // PLANE_OP_MASK
    float* partials;    // PLANE_OP_MASK
};
// The columns (transforms along j, one per k) and the row pairs (transforms along k) of the plane take turns in
// registers: inverse j on the columns straight from global memory, one pass through LDS to the row pairs, both k
// transforms and the operation in registers, one pass back, forward j, store.  The L/2 columns below Nyquist and the
// L/2 row pairs occupy the workgroup's threads exactly; the Nyquist column goes through one wavefront beside them.  The
// inverse keeps the real part of the DC and Nyquist columns, as FFTW's c2r does.  Bound by LDS (14 accesses per element
// of the half plane, against 26 with every transform's pencils staged in LDS and the DC and Nyquist columns packed into
// one pencil): both sides of 240 evaluations at 64^3 take 228 us against 402, of 36 at 128^3 375 against 596.
template <int L> struct OpPlane {
    using S = ColShape<L>;
    static constexpr int H = L / 2 + 1, T = S::T, E = S::E, LR = kRowLd<L>;
    static constexpr int HS = T == 8 ? (H + 7) / 8 * 8 - 4 : H + 1;  // row stride of the plane: row pairs spread as LR does
    static constexpr int THREADS = L / 2 * T;
    static constexpr int LDS = L * HS > L / 2 * LR ? L * HS : L / 2 * LR;  // columns' exchange, the plane, or row pencils
    static_assert(HS >= H && (T == 8 ? HS % 8 == 4 : HS % 4 == 2), "row stride");
    // wavefronts per SIMD with which as many workgroups share a CU as its LDS holds
    static constexpr int WAVES = L == 96 ? 3 : 4;
};
template <int L>
__global__ void __launch_bounds__(OpPlane<L>::THREADS, OpPlane<L>::WAVES) k_c2r_r2c_plane(PlaneOps a,
                                                                                          const float2* __restrict__ twg) {
    using O = OpPlane<L>;
    constexpr int H = O::H, HS = O::HS, T = O::T, E = O::E, LR = O::LR, NT = O::THREADS, C = L / 2;
    __shared__ float2 buf[O::LDS];
    __shared__ float2 nyq_pen[LR];
    __shared__ float nyq[L];
    __shared__ float2 tw[L];
    __shared__ float sred[NT / 64 + NT % 64 + 1];
    const bool second = blockIdx.x >= a.planes;
    const long plane = second ? blockIdx.x - a.planes : blockIdx.x;
    const int op = second ? a.op1 : a.op0;
    const int pi = (int)(plane % L);
    float2* __restrict__ ip = (second ? a.io1 : a.io0) + plane * L * H;
    // columns: c = k, elements j = ct + T u; row pairs: rows 2 q and 2 q + 1, elements k = rt + T u
    const int c = threadIdx.x % C, ct = threadIdx.x / C, q = threadIdx.x / T, rt = threadIdx.x % T;
    float2 x[E];
#pragma unroll
    for (int u = 0; u < E; u++) x[u] = at_byte(ip + T * u * H, (ct * H + c) * 8);
    for (int i = threadIdx.x; i < L; i += NT) tw[i] = twg[i];
    __syncthreads();
    col_fft<L, true, C>(x, ct, buf + c, tw);
#pragma unroll
    for (int u = 0; u < E; u++) {
        if (c == 0) x[u].y = 0.f;
        buf[(ct + T * u) * HS + c] = x[u];
    }
    if (threadIdx.x < T) {
#pragma unroll
        for (int u = 0; u < E; u++) x[u] = at_byte(ip + T * u * H, (rt * H + C) * 8);
        row_fft<L, true>(x, rt, nyq_pen, tw);
#pragma unroll
        for (int u = 0; u < E; u++) nyq[rt + T * u] = x[u].x;
    }
    __syncthreads();
    // Z(k) = A(k) + i B(k) of rows 2q and 2q + 1 over the full length, A(L - k) = conj A(k)
#pragma unroll
    for (int u = 0; u < E; u++) {
        if (E > 8 && u % 4 == 0) __builtin_amdgcn_sched_barrier(0);  // at most 8 LDS reads ahead of their use
        const int k = rt + T * u;
        if (k == C) {
            x[u] = make_float2(nyq[2 * q], nyq[2 * q + 1]);
            continue;
        }
        const int kk = k < C ? k : L - k;
        const float2 A = buf[2 * q * HS + kk], B = buf[(2 * q + 1) * HS + kk];
        x[u] = k < C ? make_float2(A.x - B.y, A.y + B.x) : make_float2(A.x + B.y, B.x - A.y);
    }
    __syncthreads();  // the plane is read: its storage becomes the row pencils'
    float sacc = 0.f;
    float2* __restrict__ pen = buf + q * LR;
    const float* __restrict__ mp = a.mask + (size_t)pi * L * L;
    const unsigned mo = (2 * q * L + rt) * 4;
    row_fft<L, true>(x, rt, pen, tw);
    // x[u] = (r(row 2q), r(row 2q + 1)) at rt + T u
    if (op == PLANE_OP_MASK) {
#pragma unroll
        for (int u0 = 0; u0 < E; u0 += 4) {  // eight mask values in flight at a time: the registers hold the pencils
            __builtin_amdgcn_sched_barrier(0);
            float2 m[4];
#pragma unroll
            for (int u = 0; u < 4; u++) m[u] = make_float2(at_byte(mp + T * (u0 + u), mo), at_byte(mp + T * (u0 + u) + L, mo));
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float2& z = x[u0 + u];
                sacc += z.x * z.x * m[u].x;
                sacc += z.y * z.y * m[u].y;
                z.x *= m[u].x;
                z.y *= m[u].y;
            }
        }
    } else {
        const float sg = ((pi + rt) & 1) ? -1.0f : 1.0f;  // T and 2 q are even
#pragma unroll
        for (int u = 0; u < E; u++) x[u] = make_float2(x[u].x * x[u].x * sg, x[u].y * x[u].y * -sg);
    }
    row_fft<L, false>(x, rt, pen, tw);
#pragma unroll
    for (int u = 0; u < E; u++) pen[rt + T * u] = x[u];
    if (op == PLANE_OP_MASK) {
        const float tot = block_sum_nt<NT>(sacc, sred);
        if (threadIdx.x == 0) a.partials[plane] = tot;
    }
    __syncthreads();
    const int cm = (L - c) % L;
    // column c of row j from the packed pair: (Z(c) + conj Z(-c)) / 2 for even rows, (Z(c) - conj Z(-c)) / 2i for odd
    // ones; j = ct + T u has ct's parity
    if (threadIdx.x < T) {
#pragma unroll
        for (int u = 0; u < E; u++) {
            const float2 z = buf[((rt >> 1) + T / 2 * u) * LR + C];  // real rows: Z(C) = X(C) of the one + i X(C) of the other
            x[u] = make_float2(rt & 1 ? z.y : z.x, 0.f);
        }
        row_fft<L, false>(x, rt, nyq_pen, tw);
#pragma unroll
        for (int u = 0; u < E; u++) at_byte(ip + T * u * H, (rt * H + C) * 8) = x[u];
    }
#pragma unroll
    for (int u = 0; u < E; u++) {
        if (E > 8 && u % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        const float2* pp = buf + ((ct >> 1) + T / 2 * u) * LR;
        const float2 z = pp[c], zc = cconj(pp[cm]);
        x[u] = ct & 1 ? make_float2(0.5f * (z.y - zc.y), -0.5f * (z.x - zc.x)) : cscale(cadd(z, zc), 0.5f);
    }
    __syncthreads();
    col_fft<L, false, C>(x, ct, buf + c, tw);
#pragma unroll
    for (int u = 0; u < E; u++) at_byte(ip + T * u * H, (ct * H + c) * 8) = x[u];
}

// ------------------------------------------------------------------ combine + first DFT axis by FFT
// norms of both sides of evaluation e from the i pass's partials, in the lanes of one wavefront (FP64, a fixed order)
__device__ __forceinline__ double wave_xsum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float ccc_norm(const float* __restrict__ part, int nb, int e, double n3) {
    double s = 0;
    for (int b = threadIdx.x & 63; b < nb; b += 64) s += part[(size_t)e * nb + b];
    return (float)sqrt(wave_xsum(s) / n3);
}

// e^{+2 pi i (i - L/2) / 2L} for i = 0 .. L-1 from the forward twiddles of length 2L
template <int L>
__device__ __forceinline__ float2 half_step(const float2* __restrict__ tw2, int i) {
    return cconj(tw2[(i - L / 2 + 2 * L) % (2 * L)]);
}
// Window index (from u = I0 - L) of element n of the parity-par transform: n stands for m = n or n - L, u = 2m + par
template <int L>
__device__ __forceinline__ int window_at(int n, int par, int I0) {
    return 2 * (n < L / 2 ? n : n - L) + par - (I0 - L);
}

// The first axis of the zero-padded 2L-point inverse transform on the search window, A[x][i] = (-1)^f e^{+i pi f u / L},
// f = i - L/2, u = I0 + x - L, as two length-L FFTs per pencil: with u = 2m + b,
// G(u) = sum_f [(-1)^f C(f) e^{+2 pi i f b / 2L}] e^{+2 pi i f m / L}, a backward L-point transform of the twiddled
// pencil (f periodic mod L) for each parity b, read at m mod L.  F1m and Q arrive before their forward i transform
// (the fused plane kernels' outputs), which runs here first.  A workgroup holds P pencils (j, k) of one evaluation in
// registers through all four transforms (regfft.hpp); rows of P neighbouring pencils of every array are whole cache
// lines.  Bound by HBM (3H read, the window's rows written): 240 evaluations at 64^3 take 148 us (6.1 TB/s), where a
// workgroup per (j, evaluation) with its 66 pencils staged in LDS took 305; 36 at 128^3 take 219 us, where the table
// product (an LDS-resident plane and table: one workgroup of 4 waves per CU) took 861.
template <int L>
__global__ void __launch_bounds__(ColShape<L>::THREADS) k_ccc_combine(const float2* __restrict__ F1m, const float2* __restrict__ F2,
                                                                  const float2* __restrict__ Q, const float2* __restrict__ Mfft,
                                                                  const float* __restrict__ p_n1, const float* __restrict__ p_n2,
                                                                  int nb, CccSizes z, float2* __restrict__ G1,
                                                                  const float2* __restrict__ twg, const float2* __restrict__ tw2) {
    using S = ColShape<L>;
    constexpr int H = L / 2 + 1, LH = L * H, NE = S::E, T = S::T, HS = L / 2 / T;  // HS: half the pencil in slots
    __shared__ float2 ex[L * S::P];
    __shared__ float2 tw[L];
    __shared__ float2 wb[L];
    __shared__ float sn[2];
    const int e = blockIdx.y, t = threadIdx.x / S::P;
    const int p = blockIdx.x * S::P + threadIdx.x % S::P;  // pencil (j, k) = (p / H, p % H)
    const bool valid = p < LH;
    const int pc = valid ? p : 0;
    const size_t vol = (size_t)e * L * LH;
    const unsigned lo = (t * LH + pc) * 8;  // byte offset of this thread's first element of a spectrum
    float2* __restrict__ xp = ex + threadIdx.x % S::P;
    float2 f1[NE], q[NE];
#pragma unroll
    for (int u = 0; u < NE; u++) {
        f1[u] = ld_stream(&at_byte(F1m + vol + u * T * LH, lo));
        q[u] = ld_stream(&at_byte(Q + vol + u * T * LH, lo));
    }
    for (int i = threadIdx.x; i < L; i += S::THREADS) {
        tw[i] = twg[i];
        wb[i] = half_step<L>(tw2, i);
    }
    if (threadIdx.x < 128) {
        const float n = ccc_norm(threadIdx.x < 64 ? p_n1 : p_n2, nb, e, (double)L * L * L);
        if ((threadIdx.x & 63) == 0) sn[threadIdx.x >> 6] = n;
    }
    __syncthreads();
    col_fft<L, false>(f1, t, xp, tw);
    col_fft<L, false>(q, t, xp, tw);
    // C = (-M conj(Q)/n2^2 + 2 F1m/n1 conj(F2 N^3/n2)) (-1)^(i+j+k), times (-1)^f: i cancels
    const float n1 = sn[0], n2 = sn[1];
    const float sg = ((pc / H + pc % H + L / 2) & 1) ? -1.f : 1.f;
    const float a = sg * (2.f * (float)(L * L * L) / (n1 * n2)), b = sg / (n2 * n2);
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const float2 f2 = ld_stream(&at_byte(F2 + vol + u * T * LH, lo)), m = at_byte(Mfft + u * T * LH, lo);
        f1[u] = csub(cscale(cmulc(f1[u], f2), a), cscale(cmulc(m, q[u]), b));
        q[u] = cmul(f1[u], wb[t + u * T]);
    }
    // element f mod L = i + L/2 mod L: a rotation of the slots by HS
#pragma unroll
    for (int par = 0; par < 2; par++) {
        float2 x[NE];
#pragma unroll
        for (int u = 0; u < NE; u++) x[(u + HS) % NE] = par ? q[u] : f1[u];
        col_fft<L, true>(x, t, xp, tw);
        if (valid)
#pragma unroll
            for (int u = 0; u < NE; u++) {
                const int xi = window_at<L>(t + u * T, par, z.I0);
                if (xi >= 0 && xi < z.E) G1[((size_t)e * z.E + xi) * LH + p] = x[u];
            }
    }
}

// The second axis the same way on the pencils along j of one (x, evaluation), in rounds of P columns k; then the third
// axis on the crop, T = sum_k Re(G2(y, k) K(z, k)) as 3 x 3 register tiles of (y, z), the spherical mask and the first
// maximum (value descending, then index ascending).  The tiles read 6 values for 9 outputs from LDS instead of 18: 93 us
// for 240 evaluations at 64^3 against 171, 71 us for 36 at 128^3 against 219 with the second axis as a table product.
template <int L> struct BcShape {
    static constexpr int H = L / 2 + 1;
    static constexpr int ROUNDS = L == 128 ? 2 : 1;  // at 128 all columns' exchange (67 KB) would leave one workgroup per CU
    static constexpr int P = (H + ROUNDS - 1) / ROUNDS;
    static constexpr int T = ColShape<L>::T;
    static constexpr int THREADS = (P * T + 63) / 64 * 64;
};
template <int L>
__global__ void __launch_bounds__(BcShape<L>::THREADS) k_ccc_dftBC(const float2* __restrict__ G1, const float2* __restrict__ tabK,
                                                               CccSizes z, float* __restrict__ best_val, int* __restrict__ best_idx,
                                                               const float2* __restrict__ twg, const float2* __restrict__ tw2) {
    using B = BcShape<L>;
    constexpr int H = B::H, P = B::P, T = B::T, NE = L / T, HS = L / 2 / T, NT = B::THREADS;
    extern __shared__ float2 dyn[];  // G2 [y][k], then K [zz][k], each E x H
    __shared__ float2 ex[L * P];
    __shared__ float2 tw[L];
    __shared__ float2 wb[L];
    __shared__ float sv[NT / 64];
    __shared__ int si[NT / 64];
    const int xi = blockIdx.x, e = blockIdx.y, E = z.E;
    float2 *g2 = dyn, *K = dyn + (size_t)E * H;
    const int t = threadIdx.x / P, c = threadIdx.x % P;
    const float2* __restrict__ src = G1 + ((size_t)e * E + xi) * L * H;  // [j][k]
#pragma unroll
    for (int r = 0; r < B::ROUNDS; r++) {
        const int k = r * P + c;
        const bool live = t < T && k < H;
        float2 v[NE];
#pragma unroll
        for (int u = 0; u < NE; u++) v[u] = live ? at_byte(src + u * T * H, (t * H + k) * 8) : make_float2(0.f, 0.f);
        if (r == 0) {
            for (int i = threadIdx.x; i < L; i += NT) {
                tw[i] = twg[i];
                wb[i] = half_step<L>(tw2, i);
            }
            block_copy_rt<4>(E * H, [&](int q) { return tabK[q]; }, [&](int q, float2 w) { K[q] = w; });
            __syncthreads();
        }
        const float sg = ((t + L / 2) & 1) ? -1.f : 1.f;  // (-1)^f of the table: T is even, so it is the thread's
#pragma unroll
        for (int par = 0; par < 2; par++) {
            float2 x[NE];
#pragma unroll
            for (int u = 0; u < NE; u++) {
                const float2 w = cscale(v[u], sg);
                x[(u + HS) % NE] = par && live ? cmul(w, wb[t + u * T]) : w;
            }
            col_fft<L, true, P>(x, t, ex + c, tw, live);
            if (live)
#pragma unroll
                for (int u = 0; u < NE; u++) {
                    const int y = window_at<L>(t + u * T, par, z.I0);
                    if (y >= 0 && y < E) g2[y * H + k] = x[u];
                }
        }
    }
    __syncthreads();
    const float scale = 8.f / ((float)(2 * L) * (float)(2 * L) * (float)(2 * L));
    float bv = -FLT_MAX;
    int bi = 0x7fffffff;
    const int dx = z.ub2 - xi, nt = (E + 2) / 3;
    for (int q = threadIdx.x; q < nt * nt; q += NT) {
        const int y0 = 3 * (q / nt), z0 = 3 * (q % nt);
        const float2 *gp[3], *kp[3];
        bool any = false;
#pragma unroll
        for (int r = 0; r < 3; r++) {
            gp[r] = g2 + min(y0 + r, E - 1) * H;
            kp[r] = K + min(z0 + r, E - 1) * H;
#pragma unroll
            for (int w = 0; w < 3; w++) {
                const int dy = z.ub2 - (y0 + r), dz = z.ub2 - (z0 + w);
                any = any || (float)(dx * dx + dy * dy + dz * dz) < z.restr2;
            }
        }
        if (!any) continue;
        float acc[3][3] = {};
#pragma unroll 2
        for (int k = 0; k < H; k++) {
            float2 g[3], w[3];
#pragma unroll
            for (int r = 0; r < 3; r++) {
                g[r] = gp[r][k];
                w[r] = kp[r][k];
            }
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int s = 0; s < 3; s++) {
                    acc[r][s] = fmaf(g[r].x, w[s].x, acc[r][s]);
                    acc[r][s] = fmaf(-g[r].y, w[s].y, acc[r][s]);
                }
        }
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int s = 0; s < 3; s++) {
                const int y = y0 + r, zz = z0 + s, dy = z.ub2 - y, dz = z.ub2 - zz, id = y * E + zz;
                if (y >= E || zz >= E || !((float)(dx * dx + dy * dy + dz * dz) < z.restr2)) continue;
                const float val = acc[r][s] * scale;
                if (val > bv || (val == bv && id < bi)) {
                    bv = val;
                    bi = id;
                }
            }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float v2 = __shfl_xor(bv, o, 64);
        const int i2 = __shfl_xor(bi, o, 64);
        if (v2 > bv || (v2 == bv && i2 < bi)) {
            bv = v2;
            bi = i2;
        }
    }
    if ((threadIdx.x & 63) == 0) {
        sv[threadIdx.x >> 6] = bv;
        si[threadIdx.x >> 6] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < NT / 64; w++)
            if (sv[w] > bv || (sv[w] == bv && si[w] < bi)) {
                bv = sv[w];
                bi = si[w];
            }
        best_val[(size_t)e * E + xi] = bv;
        best_idx[(size_t)e * E + xi] = bi;
    }
}

// One wavefront per evaluation: the first maximum over x, then k1_m and sum(W filter) from their partials, the
// distance and the shift (FIM.h:1249-1322)
__global__ void __launch_bounds__(64) k_peak_final(const float* __restrict__ best_val, const int* __restrict__ best_idx,
                                                   const float* __restrict__ p_n1, const float* __restrict__ p_wf, int nb,
                                                   const float* __restrict__ p_k1, float sum_filter, int overlap, CccSizes z,
                                                   float* __restrict__ out) {
    const int e = blockIdx.x, l = threadIdx.x, E = z.E;
    const double n3 = (double)z.N * z.N * z.N;
    const float n1 = ccc_norm(p_n1, nb, e, n3);
    double wf = 0, k1 = 0;
    for (int b = l; b < nb; b += 64) wf += p_wf[(size_t)e * nb + b];
    for (int b = l; b < z.N; b += 64) k1 += p_k1[(size_t)e * z.N + b];
    wf = wave_xsum(wf);
    k1 = wave_xsum(k1);
    float bv = -FLT_MAX;
    int bx = 0x7fffffff, byz = 0x7fffffff;  // byz 0x7fffffff: nothing inside the mask
    for (int x = l; x < E; x += 64) {
        const float v = best_val[(size_t)e * E + x];
        const int id = best_idx[(size_t)e * E + x];
        if (id != 0x7fffffff && (byz == 0x7fffffff || v > bv)) {
            bv = v;
            bx = x;
            byz = id;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float v2 = __shfl_xor(bv, o, 64);
        const int x2 = __shfl_xor(bx, o, 64), id2 = __shfl_xor(byz, o, 64);
        if (id2 != 0x7fffffff && (byz == 0x7fffffff || v2 > bv || (v2 == bv && x2 < bx))) {
            bv = v2;
            bx = x2;
            byz = id2;
        }
    }
    if (l != 0) return;
    float px = 0.f, py = 0.f, pz = 0.f;
    double maxT = -(double)FLT_MAX;
    if (byz != 0x7fffffff) {
        px = (float)bx;
        py = (float)(byz / E);
        pz = (float)(byz % E);
        maxT = bv;
    }
    const float k1m = (float)(k1 / ((double)n1 * (double)n1));  // k1_m of the normalised reference
    double peak = fmax(0.0, (double)k1m - maxT);
    if (overlap) peak = peak / (double)(float)wf * (double)sum_filter;
    float cp = (float)peak;
    const double big = (double)(2 * z.N) * (2 * z.N) * (2 * z.N);
    cp = (float)((double)cp / big / big);
    const float c = (E - 1) / 2.0f;
    out[e * 4 + 0] = cp;
    out[e * 4 + 1] = (px - c) / 2.0f;
    out[e * 4 + 2] = (py - c) / 2.0f;
    out[e * 4 + 3] = (pz - c) / 2.0f;
}

// ------------------------------------------------------------------ host launchers
// Which form a strided pass takes.  In registers it is faster at every length: over 0.5 GB at 16, 32, 48, 64, 96 and 128,
// 6.1, 6.7, 6.2, 6.5, 6.2 and 6.6 TB/s against 5.7, 6.0, 3.8, 6.3, 3.9 and 6.3 staged in LDS.  Up to 64 it stays staged for
// its rounding, not its accuracy: the 20 steps of the refinement amplify a last bit of these spectra to 1e-2 of a pose,
// and poses at 48 and 64 are kept as earlier versions gave them.
template <int L>
static constexpr bool staged_pencils() {
    return L <= 64;
}

// profile record names: k_r2c_rows<L>, the strided pass that runs (k_fft_strided<L> or k_fft_col<L>), k_c2r_rows<L>
template <int L>
static const char* plane_name(int which) {
    static const std::string n[2] = {"k_r2c_plane<" + std::to_string(L) + ">", "k_c2r_plane<" + std::to_string(L) + ">"};
    return n[which].c_str();
}
template <int L>
static const char* prof_name(int which) {
    static const std::string n[3] = {"k_r2c_rows<" + std::to_string(L) + ">",
                                     (staged_pencils<L>() ? "k_fft_strided<" : "k_fft_col<") + std::to_string(L) + ">",
                                     "k_c2r_rows<" + std::to_string(L) + ">"};
    return n[which].c_str();
}

template <int L>
static void launch_strided(const StridedArgs& a, const float2* tw, hipStream_t s) {
    if constexpr (staged_pencils<L>()) {
        using S = StridedShape<L>;
        k_fft_strided<L><<<(unsigned)((a.npencils + S::P - 1) / S::P), S::THREADS, 0, s>>>(a, tw);
    } else {
        using S = ColShape<L>;
        const unsigned nb = (unsigned)((a.npencils + S::P - 1) / S::P);
        if (a.inv) k_fft_col<L, true><<<nb, S::THREADS, 0, s>>>(a, tw);
        else k_fft_col<L, false><<<nb, S::THREADS, 0, s>>>(a, tw);
    }
}

template <int L>
static void launch_r2c(const FftTables& T, const R2CArgs& a, float2* scratch, hipStream_t s) {
    using S = Shape<L>;
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    long npairs = (long)a.batch * L * L / 2;
    const double vol_c = (double)a.batch * L * L * H * sizeof(float2);  // one pass over the half spectrum
    const double vol_r = (double)a.batch * L * L * L * sizeof(float);
    if constexpr (L <= 128) {
        // passes k and j fused per (b, i) plane
        ProfScope ps(T.prof, plane_name<L>(0), vol_r + vol_c, s);
        k_r2c_plane<L><<<(unsigned)((long)a.batch * L), Plane<L>::THREADS, 0, s>>>(a, tw);
    } else {
        // pass k: real rows -> a.out (half rows); only ettk_fft3 transforms such boxes, without a prologue
        ETTK_REQUIRE(a.pro == PRO_NONE, ETTK_ERR_UNSUPPORTED, "fft3_r2c: prologues are for n <= 128");
        {
            ProfScope ps(T.prof, prof_name<L>(0), vol_r + vol_c, s);
            k_r2c_rows<L><<<(unsigned)((npairs + S::P - 1) / S::P), S::THREADS, 0, s>>>(a, tw);
        }
        // pass j: pencils over (b, i, k), element stride H
        StridedArgs sj{a.out, a.out, (long)a.batch * L * H, (long)H, (long)L * H, (long)H, 0};
        {
            ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
            launch_strided<L>(sj, tw, s);
        }
    }
    // pass i: pencils over (b, j, k), element stride L*H
    StridedArgs si{a.out, a.out, (long)a.batch * L * H, (long)L * H, (long)L * L * H, (long)L * H, 0};
    {
        ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
        launch_strided<L>(si, tw, s);
    }
    (void)scratch;
}

template <int L>
static void launch_c2r(const FftTables& T, const float2* in, float2* tmp, float* out, int batch, hipStream_t s) {
    using S = Shape<L>;
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    const double vol_c = (double)batch * L * L * H * sizeof(float2), vol_r = (double)batch * L * L * L * sizeof(float);
    StridedArgs si{in, tmp, (long)batch * L * H, (long)L * H, (long)L * L * H, (long)L * H, 1};
    {
        ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
        launch_strided<L>(si, tw, s);
    }
    if constexpr (L <= 128) {
        ProfScope ps(T.prof, plane_name<L>(1), vol_c + vol_r, s);
        k_c2r_plane<L><<<(unsigned)((long)batch * L), Plane<L>::THREADS, 0, s>>>(tmp, out, tw);
    } else {
        StridedArgs sj{tmp, tmp, (long)batch * L * H, (long)H, (long)L * H, (long)H, 1};
        {
            ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
            launch_strided<L>(sj, tw, s);
        }
        long npairs = (long)batch * L * L / 2;
        {
            ProfScope ps(T.prof, prof_name<L>(2), vol_c + vol_r, s);
            k_c2r_rows<L><<<(unsigned)((npairs + S::P - 1) / S::P), S::THREADS, 0, s>>>(tmp, out, npairs, tw);
        }
    }
}

template <int L>
static void launch_planes(const FftTables& T, const PlaneOps& a, hipStream_t s) {
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    const unsigned nb = a.planes * (a.io1 ? 2 : 1);
    static const std::string name = "k_c2r_r2c_plane<" + std::to_string(L) + ">";
    ProfScope ps(T.prof, name.c_str(), 2.0 * nb * L * (L / 2 + 1) * sizeof(float2), s);
    k_c2r_r2c_plane<L><<<nb, OpPlane<L>::THREADS, 0, s>>>(a, tw);
}
template <int L>
static void launch_c2r_op_r2c(const FftTables& T, const float2* in, float2* io, int batch, int op, const float* aux,
                              float* partials, hipStream_t s) {
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    const double vol_c = (double)batch * L * L * H * sizeof(float2);
    const StridedArgs si{in, io, (long)batch * L * H, (long)L * H, (long)L * L * H, (long)L * H, 1};
    {
        ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
        launch_strided<L>(si, tw, s);
    }
    launch_planes<L>(T, PlaneOps{io, nullptr, op, op, (unsigned)(batch * L), aux, partials}, s);
    const StridedArgs sf{io, io, (long)batch * L * H, (long)L * H, (long)L * L * H, (long)L * H, 0};
    ProfScope ps(T.prof, prof_name<L>(1), 2 * vol_c, s);
    launch_strided<L>(sf, tw, s);
}

template <int L>
static size_t window_lds(int E) {  // k_ccc_dftBC's dynamic LDS: two E x (L / 2 + 1) tables
    return (size_t)2 * E * (L / 2 + 1) * sizeof(float2);
}
template <int L>
static size_t window_lds_all(int E) {
    hipFuncAttributes at{};
    ETTK_HIP(hipFuncGetAttributes(&at, (const void*)k_ccc_dftBC<L>));
    return at.sharedSizeBytes + window_lds<L>(E);
}
size_t fft3_ccc_window_lds(int n, int E) {
    switch (n) {
        case 16: return window_lds_all<16>(E);
        case 32: return window_lds_all<32>(E);
        case 48: return window_lds_all<48>(E);
        case 64: return window_lds_all<64>(E);
        case 96: return window_lds_all<96>(E);
        case 128: return window_lds_all<128>(E);
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_ccc_window_lds: unsupported size " + std::to_string(n)};
    }
}

template <int L>
static void launch_ccc_tail(const FftTables& T, const CccTailArgs& a, hipStream_t s) {
    constexpr int H = L / 2 + 1;
    const float2 *tw = T.tw.p + T.offset[fft_len_index(L)], *tw2 = T.tw.p + T.offset[fft_len_index(2 * L)];
    const int nb = fft3_ccc_ipass_blocks(L), E = a.z.E;
    const double Hb = (double)a.batch * L * L * H * sizeof(float2), Gb = (double)a.batch * E * L * H * sizeof(float2);
    launch_planes<L>(T, PlaneOps{a.S1, a.S3, PLANE_OP_MASK, PLANE_OP_SQUARE_SHIFT, (unsigned)(a.batch * L), a.m1, a.p_k1}, s);
    {
        ProfScope ps(T.prof, "k_ccc_combine", 3 * Hb + Gb, s);
        k_ccc_combine<L><<<dim3((L * H + ColShape<L>::P - 1) / ColShape<L>::P, a.batch), ColShape<L>::THREADS, 0, s>>>(
            a.S1, a.S2, a.S3, a.Mfft, a.p_n1, a.p_n2, nb, a.z, a.G1, tw, tw2);
    }
    {
        ProfScope ps(T.prof, "k_ccc_dftBC", Gb, s);
        const size_t shm = window_lds<L>(E);
        ensure_dynamic_lds((const void*)k_ccc_dftBC<L>, shm);
        k_ccc_dftBC<L><<<dim3(E, a.batch), BcShape<L>::THREADS, shm, s>>>(a.G1, a.tabK, a.z, a.bval, a.bidx, tw, tw2);
    }
    k_peak_final<<<a.batch, 64, 0, s>>>(a.bval, a.bidx, a.p_n1, a.p_wf, nb, a.p_k1, a.sum_filter, a.overlap, a.z, a.out4);
}
void fft3_ccc_tail(const FftTables& T, const CccTailArgs& a, hipStream_t s) {
    switch (a.z.N) {
        case 16: launch_ccc_tail<16>(T, a, s); break;
        case 32: launch_ccc_tail<32>(T, a, s); break;
        case 48: launch_ccc_tail<48>(T, a, s); break;
        case 64: launch_ccc_tail<64>(T, a, s); break;
        case 96: launch_ccc_tail<96>(T, a, s); break;
        case 128: launch_ccc_tail<128>(T, a, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_ccc_tail: unsupported size " + std::to_string(a.z.N)};
    }
    ETTK_HIP(hipGetLastError());
}

template <int L>
static int ccc_ipass_blocks_t() {
    return (L * (L / 2 + 1) + ColShape<L>::P - 1) / ColShape<L>::P;
}
int fft3_ccc_ipass_blocks(int n) {
    switch (n) {
        case 16: return ccc_ipass_blocks_t<16>();
        case 32: return ccc_ipass_blocks_t<32>();
        case 48: return ccc_ipass_blocks_t<48>();
        case 64: return ccc_ipass_blocks_t<64>();
        case 96: return ccc_ipass_blocks_t<96>();
        case 128: return ccc_ipass_blocks_t<128>();
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_ccc_ipass: unsupported size " + std::to_string(n)};
    }
}

template <int L>
static void launch_ccc_ipass(const FftTables& T, const CccIpassArgs& a, int batch, hipStream_t s) {
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    const double vol_c = (double)batch * L * L * H * sizeof(float2);
    static const std::string name = "k_ccc_ipass<" + std::to_string(L) + ">";
    ProfScope ps(T.prof, name.c_str(), 4 * vol_c, s);  // S2 read and written, S3 and S1 written
    k_ccc_ipass<L><<<dim3((unsigned)ccc_ipass_blocks_t<L>(), (unsigned)batch), ColShape<L>::THREADS, 0, s>>>(a, tw);
}
void fft3_ccc_ipass(const FftTables& T, const CccIpassArgs& a, int n, int batch, hipStream_t s) {
    switch (n) {
        case 16: launch_ccc_ipass<16>(T, a, batch, s); break;
        case 32: launch_ccc_ipass<32>(T, a, batch, s); break;
        case 48: launch_ccc_ipass<48>(T, a, batch, s); break;
        case 64: launch_ccc_ipass<64>(T, a, batch, s); break;
        case 96: launch_ccc_ipass<96>(T, a, batch, s); break;
        case 128: launch_ccc_ipass<128>(T, a, batch, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_ccc_ipass: unsupported size " + std::to_string(n)};
    }
    ETTK_HIP(hipGetLastError());
}

template <int L>
static void launch_r2c_planes(const FftTables& T, const R2CArgs& a, hipStream_t s) {
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    const double vol_c = (double)a.batch * L * L * H * sizeof(float2), vol_r = (double)a.batch * L * L * L * sizeof(float);
    ProfScope ps(T.prof, plane_name<L>(0), vol_r + vol_c, s);
    k_r2c_plane<L><<<(unsigned)((long)a.batch * L), Plane<L>::THREADS, 0, s>>>(a, tw);
}
// ------------------------------------------------------------------ refinement: score and adjoint in the i passes
// FP64 sums of the three score terms over a workgroup (halving tree, any thread count), valid in thread 0
template <int NT>
__device__ __forceinline__ void block_sum3_f64(double v0, double v1, double v2, double* sred) {
    sred[threadIdx.x] = v0;
    sred[NT + threadIdx.x] = v1;
    sred[2 * NT + threadIdx.x] = v2;
    __syncthreads();
    for (int cnt = NT; cnt > 1;) {
        const int st = (cnt + 1) / 2;
        if ((int)threadIdx.x < cnt - st)
#pragma unroll
            for (int r = 0; r < 3; r++) sred[r * NT + threadIdx.x] += sred[r * NT + threadIdx.x + st];
        __syncthreads();
        cnt = st;
    }
}

// The forward i pass of X1 (in place, after the plane passes of its r2c) and the score's terms on the transformed
// elements: per workgroup (P pencils (j, k) of one evaluation, 32 at 64 and 128, 30 at 96) the FP64 partials of
// <H X1, H X2>, |H X1|^2 and |H X2|^2 with the Hermitian weights (2 off the k = 0 and k = N/2 planes).
template <int L>
__global__ void __launch_bounds__(StridedShape<L>::THREADS) k_refine_ipass_dot(
    float2* __restrict__ X1, const float2* __restrict__ FP, const float* __restrict__ filter,
    const float* __restrict__ wbin, const RefineGeom* __restrict__ geom, double* __restrict__ part,
    const float2* __restrict__ twg) {
    using S = StridedShape<L>;
    constexpr int H = L / 2 + 1, LH = L * H, STEP = S::THREADS / S::P, NL = L / STEP;
    static_assert(L % STEP == 0, "pencil elements per thread");
    __shared__ float2 lds[S::P * S::LD];
    __shared__ float2 tw[L];
    __shared__ double sred[3 * S::THREADS];
    const int e = blockIdx.y;
    const float2 twv = twg[threadIdx.x % L];
    const int qm = threadIdx.x % S::P, l0 = threadIdx.x / S::P;
    const int p = blockIdx.x * S::P + qm;  // pencil (j, k) = (p / H, p % H) of evaluation e
    const bool valid = p < LH;
    const int pc = valid ? p : 0, pj = pc / H, pk = pc % H;
    const RefineGeom g = geom[e];
    float2* x1p = X1 + (size_t)e * L * LH;
    const float2* x2p = FP + (size_t)g.spec * L * LH;
    float2* __restrict__ pen = &lds[qm * S::LD];
    float2 v2[NL];
    {
        float2 v[NL];
#pragma unroll
        for (int u = 0; u < NL; u++) {
            v[u] = x1p[(size_t)(l0 + u * STEP) * LH + pc];
            v2[u] = x2p[(size_t)(l0 + u * STEP) * LH + pc];
        }
#pragma unroll
        for (int u = 0; u < NL; u++) pen[l0 + u * STEP] = valid ? v[u] : make_float2(0.f, 0.f);
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / S::TPP, lane = threadIdx.x % S::TPP;
    pencil_fft<L>(&lds[q * S::LD], lane, tw, tw_cache<L>(tw, lane), false);
    __syncthreads();
    double sd = 0.0, s1 = 0.0, s2 = 0.0;
    if (valid) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = l0 + u * STEP;
            const size_t h = (size_t)i * LH + pc;
            const float2 z = pen[i];
            x1p[h] = z;
            const float w = refine_hweight(filter, wbin, g, (long)h, i, pj, pk, L, H);
            const double ww = (pk == 0 || pk == H - 1) ? (double)w * w : 2.0 * (double)w * w;
            const float2 v = v2[u];
            sd += ww * ((double)z.x * v.x + (double)z.y * v.y);
            s1 += ww * ((double)z.x * z.x + (double)z.y * z.y);
            s2 += ww * ((double)v.x * v.x + (double)v.y * v.y);
        }
    }
    block_sum3_f64<S::THREADS>(sd, s1, s2, sred);
    if (threadIdx.x < 3) part[((size_t)e * gridDim.x + blockIdx.x) * 3 + threadIdx.x] = sred[threadIdx.x * S::THREADS];
}

// The adjoint spectrum H (H X2 / (n1 n2) - S H X1 / n1^2), formed as the pencils are loaded, then the inverse i pass
// into `out` (X1 is left unchanged)
template <int L>
__global__ void __launch_bounds__(StridedShape<L>::THREADS) k_refine_ipass_adj(
    const float2* __restrict__ X1, const float2* __restrict__ FP, const float* __restrict__ filter,
    const float* __restrict__ wbin, const RefineGeom* __restrict__ geom, const double* __restrict__ sc,
    float2* __restrict__ out, const float2* __restrict__ twg) {
    using S = StridedShape<L>;
    constexpr int H = L / 2 + 1, LH = L * H, STEP = S::THREADS / S::P, NL = L / STEP;
    static_assert(L % STEP == 0, "pencil elements per thread");
    __shared__ float2 lds[S::P * S::LD];
    __shared__ float2 tw[L];
    const int e = blockIdx.y;
    const float2 twv = twg[threadIdx.x % L];
    const int qm = threadIdx.x % S::P, l0 = threadIdx.x / S::P;
    const int p = blockIdx.x * S::P + qm;
    const bool valid = p < LH;
    const int pc = valid ? p : 0, pj = pc / H, pk = pc % H;
    const RefineGeom g = geom[e];
    const double Sv = sc[e * 4], n1 = sc[e * 4 + 1], n2 = sc[e * 4 + 2];
    const float ca = (n1 > 0 && n2 > 0) ? (float)(1.0 / (n1 * n2)) : 0.f;
    const float cb = n1 > 0 ? (float)(Sv / (n1 * n1)) : 0.f;
    const float2* x1p = X1 + (size_t)e * L * LH;
    const float2* x2p = FP + (size_t)g.spec * L * LH;
    float2* __restrict__ pen = &lds[qm * S::LD];
    {
        float2 x[NL], v[NL];
#pragma unroll
        for (int u = 0; u < NL; u++) {
            x[u] = x1p[(size_t)(l0 + u * STEP) * LH + pc];
            v[u] = x2p[(size_t)(l0 + u * STEP) * LH + pc];
        }
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = l0 + u * STEP;
            const float w = refine_hweight(filter, wbin, g, (long)((size_t)i * LH + pc), i, pj, pk, L, H);
            const float w2 = w * w;
            pen[i] = valid ? make_float2(w2 * (ca * v[u].x - cb * x[u].x), w2 * (ca * v[u].y - cb * x[u].y))
                           : make_float2(0.f, 0.f);
        }
    }
    if (threadIdx.x < L) tw[threadIdx.x] = twv;
    __syncthreads();
    const int q = threadIdx.x / S::TPP, lane = threadIdx.x % S::TPP;
    pencil_fft<L>(&lds[q * S::LD], lane, tw, tw_cache<L>(tw, lane), true);
    __syncthreads();
    if (valid) {
        float2* op = out + (size_t)e * L * LH;
#pragma unroll
        for (int u = 0; u < NL; u++) op[(size_t)(l0 + u * STEP) * LH + pc] = pen[l0 + u * STEP];
    }
}

template <int L>
static int refine_ipass_blocks_t() {
    return (L * (L / 2 + 1) + StridedShape<L>::P - 1) / StridedShape<L>::P;
}
template <int L>
static void launch_refine_dot_t(const FftTables& T, float2* X1, const float2* FP, const float* filter,
                                const float* wbin, const RefineGeom* geom, int batch, double* part, hipStream_t s) {
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    ProfScope ps(T.prof, "k_refine_ipass_dot", 3.0 * batch * L * L * (L / 2 + 1) * sizeof(float2), s);
    k_refine_ipass_dot<L><<<dim3((unsigned)refine_ipass_blocks_t<L>(), (unsigned)batch), StridedShape<L>::THREADS, 0, s>>>(
        X1, FP, filter, wbin, geom, part, tw);
}
template <int L>
static void launch_refine_adj_c2r_t(const FftTables& T, const float2* X1, const float2* FP, const float* filter,
                                    const float* wbin, const RefineGeom* geom, const double* sc, int batch,
                                    float2* tmp, float* out, hipStream_t s) {
    constexpr int H = L / 2 + 1;
    const float2* tw = T.tw.p + T.offset[fft_len_index(L)];
    {
        ProfScope ps(T.prof, "k_refine_ipass_adj", 3.0 * batch * L * L * H * sizeof(float2), s);
        k_refine_ipass_adj<L><<<dim3((unsigned)refine_ipass_blocks_t<L>(), (unsigned)batch), StridedShape<L>::THREADS, 0,
                                s>>>(X1, FP, filter, wbin, geom, sc, tmp, tw);
    }
    ETTK_HIP(hipGetLastError());
    const double vol_c = (double)batch * L * L * H * sizeof(float2), vol_r = (double)batch * L * L * L * sizeof(float);
    ProfScope ps(T.prof, plane_name<L>(1), vol_c + vol_r, s);
    k_c2r_plane<L><<<(unsigned)((long)batch * L), Plane<L>::THREADS, 0, s>>>(tmp, out, tw);
}
int fft3_refine_ipass_blocks(int n) {
    switch (n) {
        case 16: return refine_ipass_blocks_t<16>();
        case 32: return refine_ipass_blocks_t<32>();
        case 48: return refine_ipass_blocks_t<48>();
        case 64: return refine_ipass_blocks_t<64>();
        case 96: return refine_ipass_blocks_t<96>();
        case 128: return refine_ipass_blocks_t<128>();
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_refine_ipass: unsupported size " + std::to_string(n)};
    }
}
void fft3_refine_dot(const FftTables& T, float2* X1, const float2* FP, const float* filter, const float* wbin,
                     const RefineGeom* geom, int n, int batch, double* part, hipStream_t s) {
    switch (n) {
        case 16: launch_refine_dot_t<16>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        case 32: launch_refine_dot_t<32>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        case 48: launch_refine_dot_t<48>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        case 64: launch_refine_dot_t<64>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        case 96: launch_refine_dot_t<96>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        case 128: launch_refine_dot_t<128>(T, X1, FP, filter, wbin, geom, batch, part, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_refine_dot: unsupported size " + std::to_string(n)};
    }
    ETTK_HIP(hipGetLastError());
}
void fft3_refine_adj_c2r(const FftTables& T, const float2* X1, const float2* FP, const float* filter,
                         const float* wbin, const RefineGeom* geom, const double* sc, int n, int batch, float2* tmp,
                         float* out, hipStream_t s) {
    switch (n) {
        case 16: launch_refine_adj_c2r_t<16>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        case 32: launch_refine_adj_c2r_t<32>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        case 48: launch_refine_adj_c2r_t<48>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        case 64: launch_refine_adj_c2r_t<64>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        case 96: launch_refine_adj_c2r_t<96>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        case 128: launch_refine_adj_c2r_t<128>(T, X1, FP, filter, wbin, geom, sc, batch, tmp, out, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_refine_adj_c2r: unsupported size " + std::to_string(n)};
    }
    ETTK_HIP(hipGetLastError());
}

void fft3_r2c_planes(const FftTables& T, const R2CArgs& a, hipStream_t s) {
    switch (a.n) {
        case 16: launch_r2c_planes<16>(T, a, s); break;
        case 32: launch_r2c_planes<32>(T, a, s); break;
        case 48: launch_r2c_planes<48>(T, a, s); break;
        case 64: launch_r2c_planes<64>(T, a, s); break;
        case 96: launch_r2c_planes<96>(T, a, s); break;
        case 128: launch_r2c_planes<128>(T, a, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_r2c_planes: unsupported size " + std::to_string(a.n)};
    }
    ETTK_HIP(hipGetLastError());
}

void fft3_c2r_op_r2c(const FftTables& T, const float2* in, float2* io, int n, int batch, int op, const float* aux,
                     float* partials, hipStream_t s) {
    ETTK_REQUIRE(in != nullptr, ETTK_ERR_ARG, "fft3_c2r_op_r2c: null input");
    switch (n) {
        case 16: launch_c2r_op_r2c<16>(T, in, io, batch, op, aux, partials, s); break;
        case 32: launch_c2r_op_r2c<32>(T, in, io, batch, op, aux, partials, s); break;
        case 48: launch_c2r_op_r2c<48>(T, in, io, batch, op, aux, partials, s); break;
        case 64: launch_c2r_op_r2c<64>(T, in, io, batch, op, aux, partials, s); break;
        case 96: launch_c2r_op_r2c<96>(T, in, io, batch, op, aux, partials, s); break;
        case 128: launch_c2r_op_r2c<128>(T, in, io, batch, op, aux, partials, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_c2r_op_r2c: unsupported size " + std::to_string(n)};
    }
    ETTK_HIP(hipGetLastError());
}

void fft3_r2c(const FftTables& T, const R2CArgs& a, float2* scratch, hipStream_t s) {
    switch (a.n) {
        case 16: launch_r2c<16>(T, a, scratch, s); break;
        case 32: launch_r2c<32>(T, a, scratch, s); break;
        case 48: launch_r2c<48>(T, a, scratch, s); break;
        case 64: launch_r2c<64>(T, a, scratch, s); break;
        case 96: launch_r2c<96>(T, a, scratch, s); break;
        case 128: launch_r2c<128>(T, a, scratch, s); break;
        case 192: launch_r2c<192>(T, a, scratch, s); break;
        case 256: launch_r2c<256>(T, a, scratch, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_r2c: unsupported size " + std::to_string(a.n)};
    }
    ETTK_HIP(hipGetLastError());
}

void fft3_c2r(const FftTables& T, const float2* in, float2* tmp, float* out, int n, int batch, hipStream_t s) {
    switch (n) {
        case 16: launch_c2r<16>(T, in, tmp, out, batch, s); break;
        case 32: launch_c2r<32>(T, in, tmp, out, batch, s); break;
        case 48: launch_c2r<48>(T, in, tmp, out, batch, s); break;
        case 64: launch_c2r<64>(T, in, tmp, out, batch, s); break;
        case 96: launch_c2r<96>(T, in, tmp, out, batch, s); break;
        case 128: launch_c2r<128>(T, in, tmp, out, batch, s); break;
        case 192: launch_c2r<192>(T, in, tmp, out, batch, s); break;
        case 256: launch_c2r<256>(T, in, tmp, out, batch, s); break;
        default: throw Error{ETTK_ERR_UNSUPPORTED, "fft3_c2r: unsupported size " + std::to_string(n)};
    }
    ETTK_HIP(hipGetLastError());
}

}  // namespace ettk
