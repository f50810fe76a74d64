// The butterflies and twiddle seeds of swem_fft.hpp on the host: whole lines, pass by pass, for the error
// of the transforms against 64 bits (test_fft_lines.py).  Threads become loops: a pass gathers butterfly j
// from the line, runs the header's own dft_pass with the header's own pass_seeds, and scatters it.
#include <cmath>
#include <complex>
#include <vector>

// device builtins of the kernels around them, unused here
inline void __syncthreads() {}
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }
#define __builtin_amdgcn_sched_barrier(x) (void)0
#define __builtin_amdgcn_wave_barrier() (void)0
#define __builtin_amdgcn_fence(...) (void)0
#include "swem_fft.hpp"

using swem::cmul;

// entry j: exp(-2 pi i j / N)
template <int N>
static const float2* table()
{
    static std::vector<float2> t;
    if (t.empty())
        for (int j = 0; j < N; j++) {
            const double a = -2.0 * M_PI * j / N;
            t.push_back(make_float2((float)std::cos(a), (float)std::sin(a)));
        }
    return t.data();
}

// the radices of fft / wfft on P points per thread
template <int N, int P, int SIGN, bool HIN = false, int NS = 1>
static void line(std::vector<float2>& v)
{
    constexpr int RMAX = P < 16 ? P : 16, REM = N / NS, R = REM >= RMAX ? RMAX : REM;
    std::vector<float2> out(N);
    for (int j = 0; j < N / R; j++) {
        const int k = j % NS;
        float2 x[R], s[16];
        for (int r = 0; r < R; r++) x[r] = v[j + r * (N / R)];
        if constexpr (NS > 1) {
            swem::pass_seeds<N, NS, R>(table<N>(), (uint32_t)k, s);
            swem::dft_pass<N, R, SIGN, true>(x, s);
        } else {
            swem::dft_pass<N, R, SIGN, false, HIN>(x, s);
        }
        for (int r = 0; r < R; r++) out[(j - k) * R + k + r * NS] = x[r];
    }
    v.swap(out);
    if constexpr (NS * R < N) line<N, P, SIGN, false, NS * R>(v);
}

// radix-4 passes of plain complex products and sums, each input times one table entry
template <int N, int SIGN>
static void plain4(std::vector<float2>& v)
{
    const float2* tw = table<N>();
    std::vector<float2> out(N);
    for (int ns = 1; ns < N; ns *= 4) {
        for (int j = 0; j < N / 4; j++) {
            const int k = j % ns;
            float2 x[4];
            for (int r = 0; r < 4; r++) {
                float2 w = tw[r * k * (N / (4 * ns))];
                if (SIGN > 0) w.y = -w.y;
                x[r] = r && ns > 1 ? cmul(v[j + r * (N / 4)], w) : v[j + r * (N / 4)];
            }
            const float2 a = swem::cadd(x[0], x[2]), b = swem::csub(x[0], x[2]), c = swem::cadd(x[1], x[3]);
            const float2 d = swem::mul_si<SIGN>(swem::csub(x[1], x[3]));
            const float2 y[4] = {swem::cadd(a, c), swem::cadd(b, d), swem::csub(a, c), swem::csub(b, d)};
            for (int r = 0; r < 4; r++) out[(j - k) * 4 + k + r * ns] = y[r];
        }
        v.swap(out);
    }
}

// steps of FFT, phase, inverse FFT on [steps] depths; the upper half of the line is cleared after each.
// P = 0: plain4.  x, phase: [2 N] interleaved, x in place.
template <int N, int P>
static void march(float* x, const float* phase, int steps)
{
    std::vector<float2> v(N);
    for (int i = 0; i < N; i++) v[i] = make_float2(x[2 * i], x[2 * i + 1]);
    for (int s = 0; s < steps; s++) {
        if constexpr (P) line<N, P, -1>(v);
        else plain4<N, -1>(v);
        for (int i = 0; i < N; i++) v[i] = cmul(v[i], make_float2(phase[2 * i], phase[2 * i + 1]));
        if constexpr (P) line<N, P, +1>(v);
        else plain4<N, +1>(v);
        for (int i = N / 2; i < N; i++) v[i] = make_float2(0.f, 0.f);
    }
    for (int i = 0; i < N; i++) x[2 * i] = v[i].x, x[2 * i + 1] = v[i].y;
}

// half: the upper half of the line is not to be read (half-input first pass)
extern "C" int fft_lines(int n, int p, int sign, int half, float* x)
{
#define CASE(N, P)                                                                    \
    if (n == N && p == P) {                                                           \
        std::vector<float2> v(N);                                                     \
        for (int i = 0; i < N; i++) v[i] = make_float2(x[2 * i], x[2 * i + 1]);       \
        if (half && sign < 0) line<N, P, -1, true>(v);                                \
        else if (half) line<N, P, +1, true>(v);                                       \
        else if (sign < 0) line<N, P, -1>(v);                                         \
        else line<N, P, +1>(v);                                                       \
        for (int i = 0; i < N; i++) x[2 * i] = v[i].x, x[2 * i + 1] = v[i].y;         \
        return 0;                                                                     \
    }
    CASE(128, 2) CASE(128, 8) CASE(128, 16) CASE(256, 4) CASE(256, 8) CASE(256, 16) CASE(512, 8) CASE(1024, 8) CASE(1024, 16)
    CASE(2048, 8) CASE(2048, 16) CASE(4096, 16)
    return 1;
}

extern "C" int fft_march_256(int p, float* x, const float* phase, int steps)
{
    if (p == 0) march<256, 0>(x, phase, steps);
    else if (p == 4) march<256, 4>(x, phase, steps);
    else if (p == 8) march<256, 8>(x, phase, steps);
    else if (p == 16) march<256, 16>(x, phase, steps);
    else return 1;
    return 0;
}
