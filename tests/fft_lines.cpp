// The butterflies and twiddle seeds of swem_fft.hpp on the host: whole lines, pass by pass, for the error
// of the transforms against 64 bits (test_fft_lines.py).  Threads become loops: a pass gathers butterfly j
// from the line, runs the header's own dft_pass with the header's own pass_seeds, and scatters it.
// Mixed-radix lines run the header's mixed_fft itself, one context per thread that yields at each barrier.
#include <ucontext.h>

#include <cmath>
#include <functional>
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

// ---------------------------------------------------------------- mixed radix
struct Plan {
    int n, np = 0, ns[12], tws[12];
    uint32_t magic[12];
    uint8_t r[12];
    explicit Plan(int len) : n(len)
    {
        int rest = len, done = 1;
        for (int q : {13, 11, 7, 5, 3, 8, 4, 2})
            while (rest % q == 0) {
                r[np] = (uint8_t)q;
                ns[np] = done;
                tws[np] = len / (done * q);
                magic[np] = done > 1 ? (uint32_t)(((1ull << 32) + done - 1) / done) : 0;
                done *= q;
                rest /= q;
                np++;
            }
    }
};

// body(t, sync) for t = 0 .. T - 1 side by side, sync a barrier of all of them
static void side_by_side(int T, const std::function<void(int, const std::function<void()>&)>& body)
{
    static std::vector<std::vector<char>> stacks;
    static std::vector<ucontext_t> at;
    static ucontext_t home;
    static const std::function<void(int, const std::function<void()>&)>* run;
    static int now;
    static std::vector<char> done;
    run = &body;
    at.resize(T);
    done.assign(T, 0);
    while ((int)stacks.size() < T) stacks.emplace_back(64 << 10);
    void (*enter)() = [] {
        const int t = now;
        (*run)(t, [] { swapcontext(&at[now], &home); });
        done[t] = 1;
        swapcontext(&at[t], &home);
    };
    for (int t = 0; t < T; t++) {
        getcontext(&at[t]);
        at[t].uc_stack.ss_sp = stacks[t].data();
        at[t].uc_stack.ss_size = stacks[t].size();
        at[t].uc_link = &home;
        makecontext(&at[t], enter, 0);
    }
    for (bool more = true; more;) {
        more = false;
        for (now = 0; now < T; now++)
            if (!done[now]) {
                swapcontext(&home, &at[now]);
                more = true;
            }
    }
}

// the same radices with each input times one table entry
template <int R, int SIGN>
static void plain_pass(std::vector<float2>& v, const float2* tw, int n, int ns)
{
    std::vector<float2> out(n);
    for (int b = 0; b < n / R; b++) {
        const int k = b % ns;
        float2 x[R];
        for (int r = 0; r < R; r++) {
            float2 w = tw[r * k * (n / (ns * R))];
            if (SIGN > 0) w.y = -w.y;
            x[r] = r && ns > 1 ? cmul(v[b + r * (n / R)], w) : v[b + r * (n / R)];
        }
        swem::Dft<R, SIGN>::run(x);
        for (int r = 0; r < R; r++) out[(b - k) * R + k + r * ns] = x[r];
    }
    v.swap(out);
}

template <int M, bool PRIME, int SIGN>
static void mixed_line(std::vector<float2>& v, const Plan& pl, const float2* tw, bool plain)
{
    if (plain) {
        for (int p = 0; p < pl.np; p++) switch (pl.r[p]) {
#define PASS(R) case R: plain_pass<R, SIGN>(v, tw, pl.n, pl.ns[p]); break;
            PASS(13) PASS(11) PASS(7) PASS(5) PASS(3) PASS(8) PASS(4) PASS(2)
        }
        return;
    }
    constexpr int P = M >= 1024 ? 8 : M / 64;
    std::vector<float2> b0(M), b1(M);
    side_by_side(M / P, [&](int t, const std::function<void()>& sync) {
        float2 u[P];
        int pp = 0;
        for (int q = 0; q < P; q++) u[q] = t + q * (M / P) < pl.n ? v[t + q * (M / P)] : make_float2(0.f, 0.f);
        swem::mixed_fft<M, P, SIGN, true, PRIME>(u, b0.data(), b1.data(), tw, pl, t, pp, sync);
        for (int q = 0; q < P; q++)
            if (t + q * (M / P) < pl.n) v[t + q * (M / P)] = u[q];
    });
}

// as fft_march_256 on a line of n points; steps = 0: one transform of the sign
extern "C" int mixed_march(int n, int plain, float* x, const float* phase, int steps, int sign)
{
    const Plan pl(n);
    std::vector<float2> tw(n), v(n);
    for (int j = 0; j < n; j++) {
        const double a = -2.0 * M_PI * j / n;
        tw[j] = make_float2((float)std::cos(a), (float)std::sin(a));
        v[j] = make_float2(x[2 * j], x[2 * j + 1]);
    }
    const bool prime = pl.r[0] > 5 && pl.r[0] % 2;
    auto run = [&](int s) {
#define LEN(M)                                                                             \
    if (n <= M) {                                                                          \
        if (prime && s < 0) return mixed_line<M, true, -1>(v, pl, tw.data(), plain);       \
        if (prime) return mixed_line<M, true, +1>(v, pl, tw.data(), plain);                \
        if (s < 0) return mixed_line<M, false, -1>(v, pl, tw.data(), plain);               \
        return mixed_line<M, false, +1>(v, pl, tw.data(), plain);                          \
    }
        LEN(128) LEN(256) LEN(1024) LEN(2048)
    };
    if (steps == 0) run(sign);
    for (int s = 0; s < steps; s++) {
        run(-1);
        for (int i = 0; i < n; i++) v[i] = cmul(v[i], make_float2(phase[2 * i], phase[2 * i + 1]));
        run(+1);
        for (int i = n / 2; i < n; i++) v[i] = make_float2(0.f, 0.f);
    }
    for (int i = 0; i < n; i++) x[2 * i] = v[i].x, x[2 * i + 1] = v[i].y;
    return 0;
}
