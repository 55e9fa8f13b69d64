// regfft.hpp -- DFTs of a few points in registers, and pencils along a strided axis held in registers (gfx950).
//
// L = N1 N2 (Cooley-Tukey): T threads share a pencil, thread t holding the elements t + T j (j = 0 .. L/T - 1) in
// natural order before and after.  Each thread runs N2/T DFTs of N1 points in registers, applies the twiddles, and
// the pencil is exchanged once through LDS before N1/T DFTs of N2 points.  T divides N1 and N2, so no thread idles and
// the elements a thread ends with are those it started with: pointwise work between two transforms stays in registers.
//
// The pencils of a workgroup run along a strided axis (P consecutive pencils are neighbours in memory, threadIdx =
// t P + p), so global loads and stores go straight between registers and memory in rows of P elements, and the LDS
// exchange, laid out [element][p], has no bank conflicts.  Against pencils staged in LDS (load, three radix-4 stages
// with two barriers each, store) this leaves one LDS round trip and two barriers per transform.
#pragma once
#include "common.hpp"

namespace ettk {

// ------------------------------------------------------------------ compile-time radix plans
template <int L> struct Radices;
template <> struct Radices<16>  { static constexpr int n = 2; static constexpr int r[4] = {4, 4, 1, 1}; };
template <> struct Radices<32>  { static constexpr int n = 3; static constexpr int r[4] = {4, 4, 2, 1}; };
template <> struct Radices<48>  { static constexpr int n = 3; static constexpr int r[4] = {4, 4, 3, 1}; };
template <> struct Radices<64>  { static constexpr int n = 3; static constexpr int r[4] = {4, 4, 4, 1}; };
template <> struct Radices<96>  { static constexpr int n = 4; static constexpr int r[4] = {4, 4, 3, 2}; };
template <> struct Radices<128> { static constexpr int n = 4; static constexpr int r[4] = {4, 4, 4, 2}; };
template <> struct Radices<192> { static constexpr int n = 4; static constexpr int r[4] = {4, 4, 4, 3}; };
template <> struct Radices<256> { static constexpr int n = 4; static constexpr int r[4] = {4, 4, 4, 4}; };

// ------------------------------------------------------------------ DFTs in registers
__device__ __forceinline__ float2 mul_i(float2 z, bool inv) {  // forward: -i z, inverse: +i z
    return inv ? make_float2(-z.y, z.x) : make_float2(z.y, -z.x);
}

template <int R>
__device__ __forceinline__ void butterfly(float2* x, bool inv) {
    if constexpr (R == 2) {
        float2 a = x[0], b = x[1];
        x[0] = cadd(a, b);
        x[1] = csub(a, b);
    } else if constexpr (R == 3) {
        const float s = inv ? 0.86602540378443864676f : -0.86602540378443864676f;
        float2 t1 = cadd(x[1], x[2]);
        float2 t2 = make_float2(x[0].x - 0.5f * t1.x, x[0].y - 0.5f * t1.y);
        float2 d = csub(x[1], x[2]);
        float2 id = make_float2(-s * d.y, s * d.x);  // i*s*d
        x[0] = cadd(x[0], t1);
        x[1] = cadd(t2, id);
        x[2] = csub(t2, id);
    } else if constexpr (R == 4) {
        float2 a = cadd(x[0], x[2]), b = csub(x[0], x[2]);
        float2 c = cadd(x[1], x[3]), d = csub(x[1], x[3]);
        float2 md = mul_i(d, inv);  // forward: -i d
        x[0] = cadd(a, c);
        x[2] = csub(a, c);
        x[1] = cadd(b, md);
        x[3] = csub(b, md);
    }
}
__device__ __forceinline__ float2 mul_w8(float2 z, int n, bool inv) {  // z * exp(-+2 pi i n / 8), n = 1..3
    const float r = 0.70710678118654752440f;
    switch (n) {
        case 1: return inv ? make_float2(r * (z.x - z.y), r * (z.x + z.y)) : make_float2(r * (z.x + z.y), r * (z.y - z.x));
        case 2: return mul_i(z, inv);
        default: return inv ? make_float2(-r * (z.x + z.y), r * (z.x - z.y)) : make_float2(r * (z.y - z.x), -r * (z.x + z.y));
    }
}
// in place, natural order in and out: a[k] = sum_n a[n] exp(-+2 pi i n k / 8)
__device__ __forceinline__ void dft8(float2* a, bool inv) {
    float2 b0 = cadd(a[0], a[4]), b4 = csub(a[0], a[4]);
    float2 b1 = cadd(a[1], a[5]), b5 = mul_w8(csub(a[1], a[5]), 1, inv);
    float2 b2 = cadd(a[2], a[6]), b6 = mul_i(csub(a[2], a[6]), inv);
    float2 b3 = cadd(a[3], a[7]), b7 = mul_w8(csub(a[3], a[7]), 3, inv);
    float2 c0 = cadd(b0, b2), c2 = csub(b0, b2), c1 = cadd(b1, b3), c3 = mul_i(csub(b1, b3), inv);
    float2 c4 = cadd(b4, b6), c6 = csub(b4, b6), c5 = cadd(b5, b7), c7 = mul_i(csub(b5, b7), inv);
    a[0] = cadd(c0, c1);
    a[4] = csub(c0, c1);
    a[2] = cadd(c2, c3);
    a[6] = csub(c2, c3);
    a[1] = cadd(c4, c5);
    a[5] = csub(c4, c5);
    a[3] = cadd(c6, c7);
    a[7] = csub(c6, c7);
}

// exp(-2 pi i m / 48)
struct W48 {
    double c, s;
};
static constexpr W48 kW48[48] = {
    {1.0, 0.0}, {0.9914448613738104, -0.13052619222005157}, {0.9659258262890683, -0.25881904510252074},
    {0.9238795325112867, -0.3826834323650898}, {0.8660254037844387, -0.49999999999999994}, {0.7933533402912352, -0.6087614290087207},
    {0.7071067811865476, -0.7071067811865475}, {0.6087614290087207, -0.7933533402912352}, {0.5000000000000001, -0.8660254037844386},
    {0.38268343236508984, -0.9238795325112867}, {0.25881904510252074, -0.9659258262890683}, {0.1305261922200517, -0.9914448613738104},
    {0.0, -1.0}, {-0.1305261922200516, -0.9914448613738104}, {-0.25881904510252063, -0.9659258262890683},
    {-0.3826834323650895, -0.9238795325112868}, {-0.4999999999999998, -0.8660254037844387}, {-0.6087614290087207, -0.7933533402912352},
    {-0.7071067811865475, -0.7071067811865476}, {-0.793353340291235, -0.6087614290087209}, {-0.8660254037844387, -0.49999999999999994},
    {-0.9238795325112867, -0.3826834323650899}, {-0.9659258262890682, -0.258819045102521}, {-0.9914448613738104, -0.130526192220052},
    {-1.0, 0.0}, {-0.9914448613738104, 0.13052619222005177}, {-0.9659258262890683, 0.2588190451025208},
    {-0.9238795325112868, 0.38268343236508967}, {-0.8660254037844388, 0.4999999999999997}, {-0.7933533402912352, 0.6087614290087207},
    {-0.7071067811865479, 0.7071067811865471}, {-0.6087614290087209, 0.7933533402912349}, {-0.5000000000000004, 0.8660254037844384},
    {-0.3826834323650895, 0.9238795325112868}, {-0.25881904510252063, 0.9659258262890683}, {-0.13052619222005163, 0.9914448613738104},
    {0.0, 1.0}, {0.13052619222005127, 0.9914448613738105}, {0.2588190451025203, 0.9659258262890684},
    {0.38268343236508917, 0.923879532511287}, {0.5000000000000001, 0.8660254037844386}, {0.6087614290087199, 0.7933533402912357},
    {0.7071067811865474, 0.7071067811865477}, {0.7933533402912349, 0.6087614290087209}, {0.8660254037844384, 0.5000000000000004},
    {0.9238795325112868, 0.38268343236508956}, {0.9659258262890681, 0.25881904510252157}, {0.9914448613738104, 0.13052619222005168}};

template <int R, bool INV> __device__ __forceinline__ float2 mul_root(float2 z, int m) {  // z exp(-+2 pi i m / R), R | 48
    static_assert(48 % R == 0, "tabulated roots");
    const W48 w = kW48[(m % R) * (48 / R)];
    if (m % R == 0) return z;
    const float c = (float)w.c, s = (float)(INV ? -w.s : w.s);
    return make_float2(z.x * c - z.y * s, z.x * s + z.y * c);
}

// DFTs of R points in registers, natural order in and out
template <int R, bool INV> struct Dft {
    // R = A B: B DFTs of A points over the elements b, b + B, ..., then A DFTs of B points
    static constexpr int A = R == 24 ? 8 : 4, B = R / A;
    static __device__ __forceinline__ void run(float2* x) {
        float2 y[R];
#pragma unroll
        for (int b = 0; b < B; b++) {
            float2 v[A];
#pragma unroll
            for (int a = 0; a < A; a++) v[a] = x[B * a + b];
            Dft<A, INV>::run(v);
#pragma unroll
            for (int k = 0; k < A; k++) y[k * B + b] = mul_root<R, INV>(v[k], b * k);
        }
#pragma unroll
        for (int k = 0; k < A; k++) {
            Dft<B, INV>::run(y + k * B);
#pragma unroll
            for (int q = 0; q < B; q++) x[k + A * q] = y[k * B + q];
        }
    }
};
template <bool INV> struct Dft<3, INV> {
    static __device__ __forceinline__ void run(float2* x) { butterfly<3>(x, INV); }
};
template <bool INV> struct Dft<4, INV> {
    static __device__ __forceinline__ void run(float2* x) { butterfly<4>(x, INV); }
};
template <bool INV> struct Dft<8, INV> {
    static __device__ __forceinline__ void run(float2* x) { dft8(x, INV); }
};

// ------------------------------------------------------------------ pencils along a strided axis
template <int L> struct Col;
template <> struct Col<16> { static constexpr int N1 = 4, T = 4; };
template <> struct Col<32> { static constexpr int N1 = 8, T = 4; };
template <> struct Col<48> { static constexpr int N1 = 12, T = 4; };
template <> struct Col<64> { static constexpr int N1 = 8, T = 8; };
template <> struct Col<96> { static constexpr int N1 = 12, T = 4; };
template <> struct Col<128> { static constexpr int N1 = 16, T = 8; };
template <> struct Col<192> { static constexpr int N1 = 24, T = 8; };
template <> struct Col<256> { static constexpr int N1 = 16, T = 16; };
template <int L> struct ColShape {
    static constexpr int N1 = Col<L>::N1, N2 = L / N1;
    static constexpr int T = Col<L>::T;         // threads per pencil
    static constexpr int THREADS = 256;
    static constexpr int P = THREADS / T;       // pencils per workgroup
    static constexpr int E = L / T;             // elements per thread
    static_assert(N1 % T == 0 && N2 % T == 0, "balanced steps");
};

// Transforms the pencil whose elements t + T j are in x[j]; `ex` is the workgroup's exchange buffer (L P complex
// values, [element][p]) plus p, `tw` the forward twiddles of length L in LDS (written before a barrier that every
// thread has passed).  Every thread of the workgroup must call it: it synchronises after the exchange's writes and
// after its reads.  P: pencils of the workgroup; threads without a pencil pass live = false.
template <int L, bool INV, int P = ColShape<L>::P>
__device__ __forceinline__ void col_fft(float2* x, int t, float2* ex, const float2* tw, bool live = true) {
    using S = ColShape<L>;
    constexpr int T = S::T, N1 = S::N1, N2 = S::N2, S2 = N2 / T, S1 = N1 / T;
    if (live)
#pragma unroll
        for (int i = 0; i < S2; i++) {
            float2 v[N1];
#pragma unroll
            for (int m = 0; m < N1; m++) v[m] = x[i + S2 * m];
            Dft<N1, INV>::run(v);
            const int b = t + T * i;
#pragma unroll
            for (int k = 0; k < N1; k++) {
                if (k > 0) {
                    float2 w = tw[b * k];  // b k <= (N2 - 1)(N1 - 1) < L
                    if (INV) w.y = -w.y;
                    v[k] = cmul(v[k], w);
                }
                ex[(k * N2 + b) * P] = v[k];
            }
        }
    __syncthreads();
    if (live)
#pragma unroll
        for (int i = 0; i < S1; i++) {
            float2 v[N2];
            const int k1 = t + T * i;
#pragma unroll
            for (int b = 0; b < N2; b++) v[b] = ex[(k1 * N2 + b) * P];
            Dft<N2, INV>::run(v);
#pragma unroll
            for (int k = 0; k < N2; k++) x[i + S1 * k] = v[k];
        }
    __syncthreads();
}

// The same transform for a pencil whose T threads are consecutive lanes of one wavefront: `pen` is the pencil's own
// exchange storage, kRowLd<L> complex values, and the exchange needs only the wavefront's LDS order.  Rows of N2 + 1 and a
// pencil stride of 16 banks (T = 8) or 8 or 24 banks (T = 4) modulo 32 let neither the writes nor the reads of half a
// wavefront collide in LDS banks.
template <int L>
static constexpr int kRowLd = ColShape<L>::N1 * (ColShape<L>::N2 + 1) + (L == 128 ? 8 : L == 32 ? 4 : 0);
// Orders the LDS accesses of one wavefront: the LDS instructions of a wavefront execute in order, so threads of
// one wavefront exchanging data through LDS only need the compiler kept from reordering those accesses.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int L, bool INV>
__device__ __forceinline__ void row_fft(float2* x, int t, float2* pen, const float2* tw) {
    using S = ColShape<L>;
    constexpr int T = S::T, N1 = S::N1, N2 = S::N2, S2 = N2 / T, S1 = N1 / T;
#pragma unroll
    for (int i = 0; i < S2; i++) {
        float2 v[N1];
#pragma unroll
        for (int m = 0; m < N1; m++) v[m] = x[i + S2 * m];
        Dft<N1, INV>::run(v);
        const int b = t + T * i;
#pragma unroll
        for (int k = 0; k < N1; k++) {
            if (k > 0) {
                float2 w = tw[b * k];
                if (INV) w.y = -w.y;
                v[k] = cmul(v[k], w);
            }
            pen[k * (N2 + 1) + b] = v[k];
        }
    }
    wave_lds_order();
#pragma unroll
    for (int i = 0; i < S1; i++) {
        float2 v[N2];
        const int k1 = t + T * i;
#pragma unroll
        for (int b = 0; b < N2; b++) v[b] = pen[k1 * (N2 + 1) + b];
        Dft<N2, INV>::run(v);
#pragma unroll
        for (int k = 0; k < N2; k++) x[i + S1 * k] = v[k];
    }
    wave_lds_order();
}

}  // namespace ettk
