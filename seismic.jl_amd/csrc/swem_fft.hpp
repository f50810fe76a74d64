// swem_fft.hpp -- register/LDS Stockham FFT for gfx950 and complex helpers.
//
// A subgroup of T = N/P threads transforms N points.  Thread t holds its points in the
// "strided mapping" v[q] = x[t + q*T], q = 0..P-1.  Each pass of radix R (R | P) does P/R
// butterflies per thread; butterfly j = t + b*T reads x[j + r*N/R] -- exactly register slot
// b + r*P/R of the strided mapping -- twiddles them, runs an R-point DFT in registers and
// writes the self-sorting Stockham position (j/Ns)*Ns*R + j%Ns + r*Ns to LDS.  The last pass
// (Ns*R == N) writes back to the same register slots, so both the input and the output of a
// transform are in the strided mapping and the output is in natural order: the forward FFT
// leaves X[k = t + q*T] in v[q].  A transform costs (passes - 1) LDS round trips.
//
// LDS: each subgroup owns two buffers of LdsLen<N> complex and alternates between them
// (parity `pp`, carried across calls), so one barrier per round trip suffices: a buffer written
// in round trip k is rewritten in round trip k+2, after every thread has passed barrier k+1 and
// hence finished reading it.  Indices are padded per pass (PassPad) to spread the stores and
// loads over the banks.
// Sign convention as FFTW: SIGN = -1 forward exp(-i...), SIGN = +1 backward, unnormalised.
#pragma once
#include <hip/hip_runtime.h>

namespace swem {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b)
{
    return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
// multiply by SIGN*i
template <int SIGN>
__device__ __forceinline__ float2 mul_si(float2 a)
{
    return SIGN < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

// exp(SIGN i pi M / 8) for a compile-time M in 0..3 (and i times it for 4..7, by mul_si)
constexpr float kCos8[4] = {1.f, 0.92387953251128675613f, 0.70710678118654752440f, 0.38268343236508977173f};
constexpr float kSin8[4] = {0.f, 0.38268343236508977173f, 0.70710678118654752440f, 0.92387953251128675613f};

// a, b <- a + w b, a - w b in six fused multiply-adds: y = a + w b by four, a - w b = 2 a - y by
// two (a complex product and two sums are ten operations, eight after contraction; the radix-2
// butterfly of Linzer and Feig, "Implementation of efficient FFT algorithms on fused multiply-add
// architectures", IEEE Trans. Signal Processing 41 (1993), in its unscaled form).
__device__ __forceinline__ void bfly(float2& a, float2& b, float2 w)
{
    const float yr = fmaf(-w.y, b.y, fmaf(w.x, b.x, a.x));
    const float yi = fmaf(w.y, b.x, fmaf(w.x, b.y, a.y));
    b = make_float2(fmaf(2.f, a.x, -yr), fmaf(2.f, a.y, -yi));
    a = make_float2(yr, yi);
}
// The same with the product formed once (eight operations, the two results rounded alike): radix-2
// passes are a chain of dependent exchanges with little arithmetic between, where two operations
// less buy nothing and the unequal rounding of 2 a - y shows over the many passes.
__device__ __forceinline__ void bfly_prod(float2& a, float2& b, float2 w)
{
    const float2 t = make_float2(fmaf(w.x, b.x, -(w.y * b.y)), fmaf(w.x, b.y, w.y * b.x));
    b = csub(a, t);
    a = cadd(a, t);
}
__device__ __forceinline__ void bfly1(float2& a, float2& b)
{
    const float2 t = csub(a, b);
    a = cadd(a, b);
    b = t;
}

constexpr int bitrev(int i, int n) { return n <= 1 ? 0 : (i & 1) * (n / 2) + bitrev(i >> 1, n / 2); }

// Twiddles of a radix-R butterfly, R = 2, 4, 8 or 16, whose input r is multiplied by w^r, in two forms.
// Staged: log2 R radix-2 stages on inputs in bit-reversed order; the stage of block size S takes
// w^(R/S) W_S^m, m < S / 4 (m < 1 for S = 2); the upper quarter is SIGN i times these, a swap.
// So R / 2 seeds in all: [S = 2: w^(R/2)] [S = 4: w^(R/4)] [S = 8: w^(R/8), w^(R/8) W_8]
// [S = 16: w, w W_16, w W_8, w W_16^3], each one entry of the twiddle table.  An input passes up to
// log2 R of them, whose roundings add up.
// Direct: an input passes one table entry per radix-4 level (radix 4: w, w^2, w^3; radix 16 as 4 x 4:
// w^4, w^8, w^12, then w^c W_16^(c m), c = 1, 3 with m < 4 and c = 2 with m < 2, the rest by a swap; radix 8:
// w .. w^7 before a plain butterfly), in as many operations at radix 4 and 16 but with up to half as many
// seeds again.  The entries' rounding is the same at every depth of a march and adds up: error against 64 bits
// of 200 steps FFT, phase, IFFT in float arithmetic, powers by one product of two entries | staged | direct:
//   256 points  9.3e-6 (four radix-4 passes, no products) | 12.6e-6 | 9.3e-6, in radix-4 or in radix-16 passes
//   128 points  12.0e-6 (seven radix-2 passes) | 11.9e-6 as 16 x 8
//   512, 1024, 2048 points  14.6e-6, 16.2e-6, 18.3e-6 | 12.7e-6, 13.2e-6, 13.5e-6
// So lines of 256 points take the direct form (128 x 128 3-D modelling 35.4 -> 37.3 ms, PSPI migration 49.4 ->
// 50.5 ms, one 2-D shot of 128 traces 0.381 -> 0.374 ms); the longer lines' kernels hold their seeds in registers
// and have none left for more.
constexpr bool direct_twiddles(int N) { return N == 256; }
template <int R, bool DIRECT>
constexpr int seed_count()
{
    return !DIRECT ? R / 2 : R == 16 ? 13 : R - 1;
}
constexpr int seed_off(int S) { return S <= 2 ? 0 : S / 4; }

// Radix-4 butterfly in place, natural order: inputs 1, 2, 3 times w1, w2, w3 (ONE2: w2 = 1).
template <int SIGN, bool ONE2 = false>
__device__ __forceinline__ void radix4(float2& x0, float2& x1, float2& x2, float2& x3, float2 w1, float2 w2, float2 w3)
{
    if constexpr (ONE2) bfly1(x0, x2);
    else bfly(x0, x2, w2);
    float2 t = make_float2(fmaf(w1.x, x1.x, -(w1.y * x1.y)), fmaf(w1.x, x1.y, w1.y * x1.x));
    bfly(t, x3, w3);
    const float2 d = mul_si<SIGN>(x3), a = x0, b = x2;
    x0 = cadd(a, t);
    x2 = csub(a, t);
    x1 = cadd(b, d);
    x3 = csub(b, d);
}
// The same with unit twiddles; HIN: x2 = x3 = 0, not read.
template <int SIGN, bool HIN = false>
__device__ __forceinline__ void radix4_plain(float2& x0, float2& x1, float2& x2, float2& x3)
{
    if constexpr (HIN) {
        const float2 a = x0, t = x1, d = mul_si<SIGN>(x1);
        x0 = cadd(a, t);
        x2 = csub(a, t);
        x1 = cadd(a, d);
        x3 = csub(a, d);
    } else {
        bfly1(x0, x2);
        bfly1(x1, x3);
        const float2 t = x1, d = mul_si<SIGN>(x3), a = x0, b = x2;
        x0 = cadd(a, t);
        x2 = csub(a, t);
        x1 = cadd(b, d);
        x3 = csub(b, d);
    }
}

// The radix-R butterfly in place on x[0..R), natural order in and out.  TW: with the seeds s
// (those of exp(-...), conjugated here for SIGN > 0); otherwise w = 1 and the constants are
// immediate.  HIN: inputs r >= R / 2 are zero and are not read.
template <int R, int SIGN, bool TW, bool HIN = false>
__device__ __forceinline__ void dft_pow2(float2 (&x)[R], const float2* s)
{
    float2 y[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int r = bitrev(i, R);
        if (!HIN || r < R / 2) y[i] = x[r];
    }
#pragma unroll
    for (int S = 2; S <= R; S *= 2) {
#pragma unroll
        for (int base = 0; base < R; base += S)
#pragma unroll
            for (int m = 0; m < S / 2; ++m) {
                float2 &a = y[base + m], &b = y[base + m + S / 2];
                if (HIN && S == 2) {
                    b = a;
                    continue;
                }
                const int q = S >= 4 ? S / 4 : 1, mm = m % q;
                if (m >= q) b = mul_si<SIGN>(b);
                if constexpr (TW) {
                    const float2 w = s[seed_off(S) + mm];
                    if constexpr (R == 2) bfly_prod(a, b, SIGN > 0 ? cconj(w) : w);
                    else bfly(a, b, SIGN > 0 ? cconj(w) : w);
                } else if (mm == 0) {
                    bfly1(a, b);
                } else {
                    const int k = mm * (16 / S);  // W_S^mm = W_16^k
                    bfly(a, b, make_float2(kCos8[k], SIGN * kSin8[k]));
                }
            }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) x[i] = y[i];
}

// The direct form.  Seeds s (of exp(-...), conjugated here for SIGN > 0) in the order named above.
template <int R, int SIGN, bool TW, bool HIN = false>
__device__ __forceinline__ void dft_direct(float2 (&x)[R], const float2* s)
{
    auto seed = [&](int i) { return SIGN > 0 ? cconj(s[i]) : s[i]; };
    if constexpr (R <= 2 || (R == 4 && !TW)) {
        dft_pow2<R, SIGN, TW, HIN>(x, s);
    } else if constexpr (R == 4) {
        radix4<SIGN>(x[0], x[1], x[2], x[3], seed(0), seed(1), seed(2));
    } else if constexpr (R == 8) {
        if constexpr (TW) {
#pragma unroll
            for (int r = 1; r < 8; ++r) {
                const float2 w = seed(r - 1), v = x[r];
                x[r] = make_float2(fmaf(w.x, v.x, -(w.y * v.y)), fmaf(w.x, v.y, w.y * v.x));
            }
        }
        dft_pow2<8, SIGN, false, HIN>(x, nullptr);
    } else {
        // x[4 a + c]: over a, then over c with the twiddles w^c W_16^(c m)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (TW) radix4<SIGN>(x[c], x[4 + c], x[8 + c], x[12 + c], seed(0), seed(1), seed(2));
            else radix4_plain<SIGN, HIN>(x[c], x[4 + c], x[8 + c], x[12 + c]);
        }
        // slot 4 m + c now holds the m-th output of column c
        float2 y[16];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float2 c0 = x[4 * m], c1 = x[4 * m + 1], c2 = m < 2 ? x[4 * m + 2] : mul_si<SIGN>(x[4 * m + 2]), c3 = x[4 * m + 3];
            if constexpr (TW) {
                radix4<SIGN>(c0, c1, c2, c3, seed(3 + m), seed(7 + (m & 1)), seed(9 + m));
            } else if (m == 0) {
                radix4_plain<SIGN>(c0, c1, c2, c3);
            } else {
                // W_16^m, W_16^(2 m) (m odd: W_8, for m = 3 after the swap), W_16^(3 m)
                const float2 w1 = make_float2(kCos8[m], SIGN * kSin8[m]);
                const float2 w3 = m == 1 ? make_float2(kCos8[3], SIGN * kSin8[3])
                                : m == 2 ? make_float2(-kCos8[2], SIGN * kSin8[2])
                                         : make_float2(-kCos8[1], -SIGN * kSin8[1]);
                if (m == 2) radix4<SIGN, true>(c0, c1, c2, c3, w1, w1, w3);
                else radix4<SIGN>(c0, c1, c2, c3, w1, make_float2(kCos8[2], SIGN * kSin8[2]), w3);
            }
            y[m] = c0;
            y[m + 4] = c1;
            y[m + 8] = c2;
            y[m + 12] = c3;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = y[i];
    }
}

// A pass's butterfly of a line of N points.
template <int N, int R, int SIGN, bool TW, bool HIN = false>
__device__ __forceinline__ void dft_pass(float2 (&x)[R], const float2* s)
{
    if constexpr (direct_twiddles(N)) dft_direct<R, SIGN, TW, HIN>(x, s);
    else dft_pow2<R, SIGN, TW, HIN>(x, s);
}

template <int R, int SIGN>
struct Dft {  // R = 2, 4, 8, 16
    static __device__ __forceinline__ void run(float2 (&v)[R]) { dft_pow2<R, SIGN, false>(v, nullptr); }
};

template <int SIGN>
struct Dft<3, SIGN> {
    // X1,2 = x0 - (x1 + x2) / 2 +- SIGN i (sqrt(3) / 2) (x1 - x2)
    static __device__ __forceinline__ void run(float2 (&v)[3])
    {
        const float h = 0.86602540378443864676f;
        const float2 a = cadd(v[1], v[2]), b = cscale(mul_si<SIGN>(csub(v[1], v[2])), h);
        const float2 c = csub(v[0], cscale(a, 0.5f));
        v[0] = cadd(v[0], a);
        v[1] = cadd(c, b);
        v[2] = csub(c, b);
    }
};

template <int SIGN>
struct Dft<5, SIGN> {
    // with a1 = x1 + x4, a2 = x2 + x3, b1 = x1 - x4, b2 = x2 - x3 and w = exp(SIGN 2 pi i / 5):
    // X1,4 = x0 + c1 a1 + c2 a2 +- SIGN i (s1 b1 + s2 b2), X2,3 = x0 + c2 a1 + c1 a2 +- SIGN i (s2 b1 - s1 b2)
    static __device__ __forceinline__ void run(float2 (&v)[5])
    {
        const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
        const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
        const float2 a1 = cadd(v[1], v[4]), a2 = cadd(v[2], v[3]);
        const float2 b1 = csub(v[1], v[4]), b2 = csub(v[2], v[3]);
        const float2 x0 = v[0];
        const float2 p1 = make_float2(x0.x + c1 * a1.x + c2 * a2.x, x0.y + c1 * a1.y + c2 * a2.y);
        const float2 p2 = make_float2(x0.x + c2 * a1.x + c1 * a2.x, x0.y + c2 * a1.y + c1 * a2.y);
        const float2 q1 = mul_si<SIGN>(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y));
        const float2 q2 = mul_si<SIGN>(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y));
        v[0] = cadd(x0, cadd(a1, a2));
        v[1] = cadd(p1, q1);
        v[4] = csub(p1, q1);
        v[2] = cadd(p2, q2);
        v[3] = csub(p2, q2);
    }
};

// cos and sin of 2 pi m / R, m = 1 .. (R - 1) / 2
template <int R>
struct OddTable;
template <>
struct OddTable<7> {
    static constexpr float c[3] = {0.62348980185873359439f, -0.22252093395631433737f, -0.90096886790241903498f};
    static constexpr float s[3] = {0.78183148246802980363f, 0.97492791218182361934f, 0.43388373911755823142f};
};
template <>
struct OddTable<11> {
    static constexpr float c[5] = {0.84125353283118120551f, 0.41541501300188643508f, -0.1423148382732850048f, -0.65486073394528498959f, -0.95949297361449736865f};
    static constexpr float s[5] = {0.54064081745559755543f, 0.90963199535451833011f, 0.98982144188093279524f, 0.7557495743542582689f, 0.28173255684142967104f};
};
template <>
struct OddTable<13> {
    static constexpr float c[6] = {0.88545602565320991051f, 0.56806474673115592289f, 0.12053668025532300601f, -0.35460488704253545489f, -0.74851074817110119231f, -0.9709418174260520118f};
    static constexpr float s[6] = {0.46472317204376850652f, 0.82298386589365635224f, 0.99270887409805397272f, 0.93501624268541483342f, 0.66312265824079519305f, 0.23931566428755768339f};
};

// Prime radices 7, 11, 13: with a_j = x_j + x_(R-j), b_j = x_j - x_(R-j), j = 1 .. H = (R - 1) / 2,
// X_k and X_(R-k) = x_0 + sum_j cos(2 pi j k / R) a_j +- SIGN i sum_j sin(2 pi j k / R) b_j.
template <int R, int SIGN>
struct DftOdd {
    static __device__ __forceinline__ void run(float2 (&v)[R])
    {
        constexpr int H = (R - 1) / 2;
        float2 a[H], b[H];
        const float2 x0 = v[0];
        float2 sum = x0;
#pragma unroll
        for (int j = 0; j < H; ++j) {
            a[j] = cadd(v[j + 1], v[R - 1 - j]);
            b[j] = csub(v[j + 1], v[R - 1 - j]);
            sum = cadd(sum, a[j]);
        }
        v[0] = sum;
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            float2 p = x0, q = make_float2(0.f, 0.f);
#pragma unroll
            for (int j = 0; j < H; ++j) {
                const int m = ((j + 1) * k) % R;  // angle 2 pi m / R: m <= H, or the mirrored R - m
                const float c = OddTable<R>::c[(m <= H ? m : R - m) - 1];
                const float s = m <= H ? OddTable<R>::s[m - 1] : -OddTable<R>::s[R - m - 1];
                p = make_float2(fmaf(c, a[j].x, p.x), fmaf(c, a[j].y, p.y));
                q = make_float2(fmaf(s, b[j].x, q.x), fmaf(s, b[j].y, q.y));
            }
            q = mul_si<SIGN>(q);
            v[k] = cadd(p, q);
            v[R - k] = csub(p, q);
        }
    }
};
template <int SIGN>
struct Dft<7, SIGN> : DftOdd<7, SIGN> {};
template <int SIGN>
struct Dft<11, SIGN> : DftOdd<11, SIGN> {};
template <int SIGN>
struct Dft<13, SIGN> : DftOdd<13, SIGN> {};

// Bank-conflict padding: one complex inserted every 2^SH.  The LDS has 64 banks of 4 bytes (32
// complex per row).  A Stockham pass writes at lane stride R (first pass) or in groups of NS
// lanes, then reads back at unit lane stride; SH is chosen per pass so both the writes and the
// reads of a 64-lane instruction touch every bank exactly twice (the minimum for 8-byte
// accesses), except the radix-8 NS = 8 and radix-4 NS > 1 passes, which keep one 3-way access.
template <int SH>
__device__ __forceinline__ int padsh(int i)
{
    return i + (i >> SH);
}
// Padding of the strided-mapping accesses x[t + q T] outside a transform (hand-offs).
__device__ __forceinline__ int lds_pad(int i) { return padsh<5>(i); }
template <int NS, int R>
struct PassPad {
    static constexpr int value = (R == 8)   ? (NS == 8 ? 3 : 5)
                                 : (R == 4) ? (NS == 1 ? 5 : 3)
                                 : (R == 2) ? ((NS == 8 || NS == 16) ? 3 : 5)
                                            : 5;
};
// Complex elements per LDS buffer: the largest padded index (shift 3), rounded to a multiple of
// 32 plus 4, so consecutive buffers start 8 banks apart (tiles staged across buffers spread
// over all banks).
template <int N>
struct LdsLen {
    static constexpr int value = ((N + N / 8 + 31) & ~31) + 4;
};

// Number of radix passes of fft<N,P> (for flop accounting and tests).
template <int N, int P>
constexpr int fft_passes()
{
    int n = 1, p = 0;
    while (n < N) {
        int rem = N / n;
        n *= rem >= P ? P : rem;
        ++p;
    }
    return p;
}

// One pass of fft<N,P>.  Twiddle seeds of a pass after the first (NS > 1, radix R): for each
// butterfly b of a thread the seeds of dft_pass with w = exp(-2 pi i k / (NS R)),
// k = (t + b T) mod NS: w^(R/S) W_S^m is the table entry N / (S NS) (k + m NS), below N / 2;
// w^e W_R^(e m) the entry e N / (R NS) (k + m NS), below N.
template <int N, int P, int NS>
struct FPass {
    static constexpr int T = N / P;
    static constexpr int REM = N / NS;
    static constexpr int R = REM >= P ? P : REM;
    static constexpr int B = P / R;
    static constexpr bool LAST = (NS * R == N);
    static constexpr int S = seed_count<R, direct_twiddles(N)>();
    static constexpr int NTW = NS > 1 ? B * S : 1;  // twiddle seeds per thread (1: unused slot)
};

// The seeds of one radix-R butterfly of pass NS, k = its index mod NS.
template <int N, int NS, int R>
__device__ __forceinline__ void pass_seeds(const float2* __restrict__ tw, uint32_t k, float2* s)
{
    const char* table = reinterpret_cast<const char*>(tw);
    if constexpr (direct_twiddles(N)) {
        auto entry = [&](int e, int m) {  // w^e W_R^(e m)
            return *reinterpret_cast<const float2*>(table + k * (uint32_t)(8 * e * (N / (R * NS))) + 8 * e * m * (N / R));
        };
        if constexpr (R == 16) {
#pragma unroll
            for (int a = 1; a < 4; ++a) s[a - 1] = entry(4 * a, 0);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                s[3 + m] = entry(1, m);
                if (m < 2) s[7 + m] = entry(2, m);
                s[9 + m] = entry(3, m);
            }
        } else {
#pragma unroll
            for (int r = 1; r < R; ++r) s[r - 1] = entry(r, 0);
        }
        return;
    }
#pragma unroll
    for (int S = 2; S <= R; S *= 2)
#pragma unroll
        for (int m = 0; m < (S >= 4 ? S / 4 : 1); ++m)
            s[seed_off(S) + m] =
                *reinterpret_cast<const float2*>(table + k * (uint32_t)(8 * (N / (S * NS))) + 8 * m * (N / S));
}

// The seeds of pass NS.  Byte offsets from the wave-uniform table: one 32-bit offset register and an
// immediate per load instead of a 64-bit address.
template <int N, int P, int NS>
__device__ __forceinline__ void fft_seeds(const float2* __restrict__ tw, int t,
                                          float2 (&w)[FPass<N, P, NS>::NTW])
{
    using S = FPass<N, P, NS>;
    if constexpr (NS > 1) {
#pragma unroll
        for (int b = 0; b < S::B; ++b) {
            // opaque: the loads stay in the transform instead of pinning registers across the
            // caller's loops
            uint32_t k = (uint32_t)(t + b * S::T) & (NS - 1);
            asm volatile("" : "+v"(k));
            pass_seeds<N, NS, S::R>(tw, k, &w[b * S::S]);
        }
    }
}

// Seeds of every pass of fft<N,P>, in pass order.
template <int N, int P, int NS = 1>
constexpr int fft_seed_total()
{
    using S = FPass<N, P, NS>;
    const int own = NS > 1 ? S::NTW : 0;
    if constexpr (S::LAST) return own;
    else return own + fft_seed_total<N, P, NS * S::R>();
}
template <int N, int P>
struct FftSeeds {
    static constexpr int count = fft_seed_total<N, P>();
    float2 w[count > 0 ? count : 1];
    template <int NS = 1>
    __device__ __forceinline__ void load(const float2* __restrict__ tw, int t)
    {
        using S = FPass<N, P, NS>;
        if constexpr (NS > 1) {
            constexpr int off = count - fft_seed_total<N, P, NS>();
            float2 q[S::NTW];
            fft_seeds<N, P, NS>(tw, t, q);
#pragma unroll
            for (int i = 0; i < S::NTW; ++i) w[off + i] = q[i];
        }
        if constexpr (!S::LAST) load<NS * S::R>(tw, t);
    }
};

// Where a transform's seeds come from.
//   kSeedPass   each pass loads its own (every load in flight before the first use: under register
//               pressure the scheduler would otherwise pair each load with its use and serialise
//               the latencies)
//   kSeedAhead  a pass loads the next one's at its start, so that their latency overlaps its
//               butterflies
//   kSeedHeld   the caller holds all of them in registers (FftSeeds): they depend on the thread
//               only, so a march reads them once
enum { kSeedPass = 0, kSeedAhead = 1, kSeedHeld = 2 };

// One Stockham pass and the passes after it on one wavefield v in the strided mapping.
// lds: the subgroup's two buffers (2 * LdsLen<N> complex); pp: buffer parity, toggled per
// round trip; w: this pass's twiddle seeds (kSeedHeld: those of this and the later passes).
template <int N, int P, int SIGN, int NS, int SEED, bool HIN>
__device__ __forceinline__ void fft_pass(float2 (&v)[P], float2* lds, const float2* __restrict__ tw,
                                         const float2* w, int t, int& pp)
{
    using S = FPass<N, P, NS>;
    constexpr int T = S::T, R = S::R, B = S::B;
    constexpr int L = LdsLen<N>::value;
    constexpr int SH = PassPad<NS, R>::value;
    constexpr int NSN = S::LAST ? NS : NS * R;
    float2* buf = lds + pp * L;
    float2 wn[SEED == kSeedHeld ? 1 : FPass<N, P, NSN>::NTW];
    if constexpr (!S::LAST && SEED == kSeedAhead) {
        fft_seeds<N, P, NSN>(tw, t, wn);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = t + b * T;
        const int k = j & (NS - 1);
        float2 x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = v[b + r * B];
        if constexpr (NS > 1) dft_pass<N, R, SIGN, true>(x, &w[b * S::S]);
        else dft_pass<N, R, SIGN, false, HIN>(x, nullptr);
        if constexpr (S::LAST) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[b + r * B] = x[r];
        } else {
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[padsh<SH>(base + r * NS)] = x[r];
        }
    }
    if constexpr (!S::LAST) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = buf[padsh<SH>(t + q * T)];
        pp ^= 1;
        if constexpr (SEED == kSeedPass) {
            fft_seeds<N, P, NSN>(tw, t, wn);
            __builtin_amdgcn_sched_barrier(0);
        }
        fft_pass<N, P, SIGN, NSN, SEED, false>(v, lds, tw, SEED == kSeedHeld ? w + (NS > 1 ? S::NTW : 0) : wn, t, pp);
    }
}

// The transform of one wavefield v in the strided mapping.  tw[m] = exp(-2 pi i m/N).  SEED: see
// above (held: the seeds).  HIN: the points N/2 .. N-1 (slots q >= P/2) are zero on input and are
// not read (the first pass runs half-input DFTs).
template <int N, int P, int SIGN, int SEED = kSeedPass, bool HIN = false>
__device__ __forceinline__ void fft(float2 (&v)[P], float2* lds, const float2* __restrict__ tw, int t, int& pp,
                                    const float2* held = nullptr)
{
    fft_pass<N, P, SIGN, 1, SEED, HIN>(v, lds, tw, held, t, pp);
}

// Wave-level variant: G lanes of a wave (G a power of two, 64 / G lines side by side) transform
// N = G P points held as v[q] = x[t + G q].  All exchanges stay inside the wave, whose LDS instructions execute in program order, so a
// read issued after a write observes it and one buffer (LdsLen<N> complex, private to the line)
// suffices with no s_barrier; wave_barrier only stops the compiler from reordering the LDS
// accesses across the exchange.
template <int N, int NS, int G = 64>
struct WPass {
    static constexpr int P = N / G;
    static constexpr int REM = N / NS;
    static constexpr int RMAX = P < 16 ? P : 16;
    static constexpr int R = REM >= RMAX ? RMAX : REM;
    static constexpr int B = P / R;
    static constexpr bool LAST = (NS * R == N);
    static constexpr int S = seed_count<R, direct_twiddles(N)>();
    static constexpr int NTW = NS > 1 ? B * S : 1;  // twiddle seeds per lane (1: unused slot)
};

// The twiddle seeds of pass NS of wfft<N> (as in fft).
template <int N, int NS, int G = 64>
__device__ __forceinline__ void wfft_seeds(const float2* __restrict__ tw, int t, float2 (&w)[WPass<N, NS, G>::NTW])
{
    using S = WPass<N, NS, G>;
    if constexpr (NS > 1) {
#pragma unroll
        for (int b = 0; b < S::B; ++b) {
            uint32_t k = (uint32_t)(t + b * G) & (NS - 1);
            asm volatile("" : "+v"(k));  // keep the loads in the transform (see fft)
            pass_seeds<N, NS, S::R>(tw, k, &w[b * S::S]);
        }
    }
}

template <int N, int NS = 1>
constexpr int wfft_seed_total()
{
    using S = WPass<N, NS>;
    const int own = NS > 1 ? S::NTW : 0;
    if constexpr (S::LAST) return own;
    else return own + wfft_seed_total<N, NS * S::R>();
}
template <int N>
struct WfftSeeds {
    static constexpr int count = wfft_seed_total<N>();
    float2 w[count > 0 ? count : 1];
    template <int NS = 1>
    __device__ __forceinline__ void load(const float2* __restrict__ tw, int t)
    {
        using S = WPass<N, NS>;
        if constexpr (NS > 1) {
            constexpr int off = count - wfft_seed_total<N, NS>();
            float2 q[S::NTW];
            wfft_seeds<N, NS>(tw, t, q);
#pragma unroll
            for (int i = 0; i < S::NTW; ++i) w[off + i] = q[i];
        }
        if constexpr (!S::LAST) load<NS * S::R>(tw, t);
    }
};

// One pass and the passes after it; w: this pass's seeds (kSeedHeld: and those of the later ones).
// Otherwise the next pass's seeds are loaded at the start of this one where that costs at most 8
// complex registers; larger transforms load their seeds in the pass that uses them.
template <int N, int SIGN, int NS, int SEED, bool HIN, int G>
__device__ __forceinline__ void wfft_pass(float2 (&v)[N / G], float2* buf, const float2* __restrict__ tw, int t,
                                          const float2* w)
{
    using S = WPass<N, NS, G>;
    constexpr int P = S::P, R = S::R, B = S::B;
    constexpr int T = G;
    constexpr int SH = PassPad<NS, R>::value;
    static_assert(P % R == 0, "radix must divide the points per lane");
    constexpr int NSN = S::LAST ? NS : NS * R;
    constexpr bool PRE = WPass<N, NSN, G>::NTW <= 8;
    float2 wn[SEED == kSeedHeld ? 1 : WPass<N, NSN, G>::NTW];
    if constexpr (!S::LAST && PRE && SEED != kSeedHeld) wfft_seeds<N, NSN, G>(tw, t, wn);
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = t + b * T;
        const int k = j & (NS - 1);
        float2 x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = v[b + r * B];
        if constexpr (NS > 1) dft_pass<N, R, SIGN, true>(x, &w[b * S::S]);
        else dft_pass<N, R, SIGN, false, HIN>(x, nullptr);
        if constexpr (S::LAST) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[b + r * B] = x[r];
        } else {
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[padsh<SH>(base + r * NS)] = x[r];
        }
    }
    if constexpr (!S::LAST) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = buf[padsh<SH>(t + q * T)];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (!PRE && SEED != kSeedHeld) wfft_seeds<N, NSN, G>(tw, t, wn);
        wfft_pass<N, SIGN, NSN, SEED, false, G>(v, buf, tw, t, SEED == kSeedHeld ? w + (NS > 1 ? S::NTW : 0) : wn);
    }
}

// SEED: kSeedHeld with the lane's WfftSeeds in `held`, else read in the transform.  HIN: the points
// N/2 .. N-1 (slots q >= P/2) are zero on input and are not read.
template <int N, int SIGN, int SEED = kSeedAhead, bool HIN = false, int G = 64>
__device__ __forceinline__ void wfft(float2 (&v)[N / G], float2* buf, const float2* __restrict__ tw, int t,
                                     const float2* held = nullptr)
{
    wfft_pass<N, SIGN, 1, SEED, HIN, G>(v, buf, tw, t, held);
}

// Two wavefields transformed in lockstep, one LDS buffer each: every barrier serves both, and one's
// butterflies overlap the other's exchange.  T = N / P threads; `sync` orders the LDS accesses of
// those threads (a wave fence for T = 64).  A buffer is read before the next pass writes it, so a
// pass takes two syncs.  held: the FftSeeds of the thread.
template <int N, int P, int SIGN, int NS, bool HIN, class Sync>
__device__ __forceinline__ void fft2_pass(float2 (&u)[P], float2 (&v)[P], float2* bu, float2* bv, const float2* w, int t,
                                          Sync sync)
{
    using S = FPass<N, P, NS>;
    constexpr int T = S::T, R = S::R, B = S::B;
    constexpr int SH = PassPad<NS, R>::value;
    auto butterflies = [&](float2(&f)[P], float2* buf) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int j = t + b * T;
            const int k = j & (NS - 1);
            float2 x[R];
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = f[b + r * B];
            if constexpr (NS > 1) dft_pass<N, R, SIGN, true>(x, &w[b * S::S]);
            else dft_pass<N, R, SIGN, false, HIN>(x, nullptr);
            if constexpr (S::LAST) {
#pragma unroll
                for (int r = 0; r < R; ++r) f[b + r * B] = x[r];
            } else {
                const int base = (j - k) * R + k;
#pragma unroll
                for (int r = 0; r < R; ++r) buf[padsh<SH>(base + r * NS)] = x[r];
            }
        }
    };
    butterflies(u, bu);
    butterflies(v, bv);
    if constexpr (!S::LAST) {
        sync();
#pragma unroll
        for (int q = 0; q < P; ++q) u[q] = bu[padsh<SH>(t + q * T)];
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = bv[padsh<SH>(t + q * T)];
        sync();
        fft2_pass<N, P, SIGN, NS * R, false>(u, v, bu, bv, w + (NS > 1 ? S::NTW : 0), t, sync);
    }
}
template <int N, int P, int SIGN, bool HIN, class Sync>
__device__ __forceinline__ void fft2(float2 (&u)[P], float2 (&v)[P], float2* bu, float2* bv, const float2* held, int t,
                                     Sync sync)
{
    fft2_pass<N, P, SIGN, 1, HIN>(u, v, bu, bv, held, t, sync);
}

// ------------------------------------------------------------------ mixed-radix transforms
// A length n = 2^a 3^b 5^c 7^d 11^e 13^f held in an array of M >= n points (M a power of two; T = M / P
// threads, point j = t + q T in v[q]; entries j >= n are zero on input and on output).  The
// transform runs in LDS: the points are stored in natural order; every pass of radix R (in the
// plan's order) reads butterfly b < n / R at b + r n / R, multiplies input r by
// exp(SIGN 2 pi i r k / (NS R)) with k = b mod NS, runs the R-point DFT and writes the
// self-sorting Stockham position (b - k) R + k + r NS, NS being the product of the radices before
// the pass; the points are then loaded back.  Each thread holds at most IT = ceil(P / R)
// butterflies of a pass.  PP: two buffers alternated per pass (one barrier per pass), parity `pp`
// carried as in fft; otherwise one buffer with a barrier between a pass's loads and its stores.
// Twiddles from the table tw[j] = exp(-2 pi i j / n).  Lengths of 2, 3 and 5: w = tw[k n / (NS R)], its powers by
// products, w^r = w^h w^(r-h) with h the largest power of two below r (one load per butterfly:
// seeds as in fft, four loads per radix-8 butterfly, measured slower here, 818 -> 943 ms for a
// 250 x 250 3-D shot).  With a radix 7, 11 or 13 (TABLE): every power is its own entry.  The products' rounding is
// the same at every depth and adds up; those lengths ran Bluestein's identity before, which has no products of
// entries, and the packed PSPI march at 700 points came out at 2.1e-5 of its image by products, 1.7e-6 by
// entries and 1.4e-6 by Bluestein (split step: 1.07e-6, 8.1e-7, 2.7e-6).  It costs 3 to 40 % of the march (one
// shot of 350 traces 377 -> 398 us, eight linear ones of 550 traces 2.85 -> 4.05 ms); Bluestein took 522 us and 12.1 ms.
// LDS indices are unpadded: the loads and the later passes' stores run at unit lane
// stride, the first pass's stores at stride R.
template <int R, int SIGN, int IT, bool PP, bool TABLE, class Sync>
__device__ __forceinline__ void mixed_pass(const float2* src, float2* dst, const float2* __restrict__ tw, int n,
                                           int ns, int tws, uint32_t magic, int t, int T, Sync sync)
{
    const int nb = n / R;
    float2 x[IT][R];
    int base[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int b = t + i * T;
        if (i == 0 || b < nb) {
            const int k = ns > 1 ? b - (int)__umulhi((uint32_t)b, magic) * ns : 0;
            base[i] = (b - k) * R + k;
            float2 pw[R];
            if (TABLE && ns > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    const float2 w = b < nb ? tw[r * k * tws] : make_float2(1.f, 0.f);
                    pw[r] = SIGN > 0 ? cconj(w) : w;
                }
            }
            float2 w1 = make_float2(1.f, 0.f);
            if (!TABLE && ns > 1 && b < nb) w1 = tw[k * tws];
#pragma unroll
            for (int r = 0; r < R; ++r) x[i][r] = b < nb ? src[b + r * nb] : make_float2(0.f, 0.f);
            if (ns > 1) {
                if constexpr (!TABLE) {
                    pw[1] = SIGN > 0 ? cconj(w1) : w1;
#pragma unroll
                    for (int r = 2; r < R; ++r) {
                        int h = 1;
                        while (2 * h < r) h *= 2;
                        pw[r] = cmul(pw[h], pw[r - h]);
                    }
                }
#pragma unroll
                for (int r = 1; r < R; ++r) x[i][r] = cmul(x[i][r], pw[r]);
            }
            Dft<R, SIGN>::run(x[i]);
        }
    }
    if constexpr (!PP) sync();
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int b = t + i * T;
        if (b < nb) {
#pragma unroll
            for (int r = 0; r < R; ++r) dst[base[i] + r * ns] = x[i][r];
        }
    }
    sync();
}

// PRIME: the plan may hold the radices 7, 11 and 13.
template <int M, int P, int SIGN, bool PP, bool PRIME, class Plan, class Sync>
__device__ __forceinline__ void mixed_fft(float2 (&v)[P], float2* buf0, float2* buf1, const float2* __restrict__ tw,
                                          const Plan& mr, int t, int& pp, Sync sync)
{
    constexpr int T = M / P;
    const int n = mr.n;
    float2* cur = (PP && pp) ? buf1 : buf0;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int j = t + q * T;
        if (j < n) cur[j] = v[q];
    }
    sync();
    for (int p = 0; p < mr.np; ++p) {
        float2* nxt = PP ? (cur == buf0 ? buf1 : buf0) : cur;
        const int ns = mr.ns[p], tws = mr.tws[p];
        const uint32_t mg = mr.magic[p];
        const int r = mr.r[p];
        if constexpr (PRIME) {
            if (r == 7 || r > 8) {
                if (r == 7) mixed_pass<7, SIGN, (P + 6) / 7, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync);
                else if (r == 11) mixed_pass<11, SIGN, (P + 10) / 11, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync);
                else mixed_pass<13, SIGN, (P + 12) / 13, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync);
                cur = nxt;
                continue;
            }
        }
        switch (r) {
        case 8: mixed_pass<8, SIGN, (P + 7) / 8, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync); break;
        case 4: mixed_pass<4, SIGN, (P + 3) / 4, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync); break;
        case 2: mixed_pass<2, SIGN, (P + 1) / 2, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync); break;
        case 3: mixed_pass<3, SIGN, (P + 2) / 3, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync); break;
        default: mixed_pass<5, SIGN, (P + 4) / 5, PP, PRIME>(cur, nxt, tw, n, ns, tws, mg, t, T, sync); break;
        }
        cur = nxt;
    }
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int j = t + q * T;
        v[q] = j < n ? cur[j] : make_float2(0.f, 0.f);
    }
    if constexpr (PP) pp = cur == buf0 ? 1 : 0;  // the next transform writes the other buffer
    else sync();
}

}  // namespace swem
