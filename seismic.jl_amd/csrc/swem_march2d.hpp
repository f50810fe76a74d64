// swem_march2d.hpp -- fused 2-D depth-march kernels (split-step Fourier and PSPI).
//
// Migration (adjoint): a workgroup holds F frequencies of one shot; each frequency has a source
// and a receiver wavefield, each owned by its own subgroup (a 64-lane wave holding N/64 points
// per lane, or N/P threads holding P points), kept in registers for the whole depth march.  Each
// depth step runs the x-FFTs through LDS, multiplies by the kz phase and the split-step phase
// read from the FP64-built phase tables (swem_phase.hip), applies the taper (SSF) or the per-vref
// propagation and selection (PSPI).  The source subgroup then hands its wavefield to the receiver
// subgroup through LDS for the cross-correlation image; the image of the F frequencies is summed
// in a fixed order and written once per depth step to a partial image, which reduce_image sums
// over frequency groups and shots with compensated sums -- so a shot's image does not depend on
// what else was launched with it.
//
// The default migration kernels keep both wavefields of a frequency in one subgroup instead:
// PAIR steps them in turn (image register-local), and for PSPI compat PACKED steps both with one
// transform per vref (their real parts packed in one complex array, see adj_body_packed).
//
// Modelling (forward): each subgroup owns one frequency, marches the source down storing it per
// depth in HBM, then marches the receiver up injecting m * source before each step.
//
// Reference semantics (src/Imaging/c/wem.c):
//   extrap1f adjoint   wem.c:229-250  source marched with -dz, receiver with +dz, image
//                                     m[x][iz] += factor Re(ur conj(us)), factor 2 (1 at iw=0)
//   extrap1f forward   wem.c:252-281  source stored per depth, receiver marched upward from
//                                     nz-1 with injection ur += m us before each step
//   ssop               wem.c:289-378  adj: FFT, kz phase, IFFT, split-step phase, taper;
//                                     forward branch: taper, split-step phase, FFT, kz, IFFT
//   pspiop             wem.c:380-471  FFT, per vref (phase, IFFT), per-x selection with the
//                                     real-part cut of linear_interp (wem.c:473-478)
// A step of -dz uses the complex conjugate of the +dz phases (the evanescent factor is real).
#pragma once
#include <type_traits>

#include "swem_esep.hpp"
#include "swem_fft.hpp"
#include "swem_internal.hpp"

namespace swem {

template <int N>
struct Pts {
    static constexpr int value = N >= 512 ? 8 : (N >= 256 ? 4 : 2);
};

constexpr int kModeSSF = 0, kModePspiCompat = 1, kModePspiLinear = 2;

// Block index -> (frequency group, shot).  Workgroups are dispatched to the 8 XCDs round
// robin, so block b runs on XCD b % 8; consecutive blocks of one XCD take the shots of one
// frequency group, which then read the same phase-table rows from that XCD's L2.
__device__ __forceinline__ void decode_block(int ngroups, int nshot, int& g, int& shot)
{
    const int b = blockIdx.x, x = b & 7, m = b >> 3;
    shot = m % nshot;
    g = (m / nshot) * 8 + x;
    if (g >= ngroups) g = -1;
}

// Raw buffer access: a resource of `bytes` bytes at `base` (wave-uniform); loads beyond it
// return zero and stores beyond it are dropped by the hardware, so edge lanes need no branch.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float2 buf_load2(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
__device__ __forceinline__ float buf_load1(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
__device__ __forceinline__ void buf_store1(__amdgpu_buffer_rsrc_t r, uint32_t off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, 0);
}
// Partial-image rows are written once and read once by the reduction: stored non-temporal (cache
// policy NT), so they stream through L2 instead of evicting the phase-table rows that the shots
// of one frequency share there.
constexpr int kCachePolicyNT = 2;
__device__ __forceinline__ void buf_store1_nt(__amdgpu_buffer_rsrc_t r, uint32_t off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, kCachePolicyNT);
}
__device__ __forceinline__ void buf_store2(__amdgpu_buffer_rsrc_t r, uint32_t off, float2 v)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, v), r,
                                          (int)off, 0, 0);
}

// kz phase of the point k = t + q T of the strided mapping from a table row (L is even in kx,
// the row holds kk = 0..N/2): kk = k for q < P/2, N - k = (P - q) T - t above.  Byte offsets of 32
// bits from the wave-uniform row: two offset registers and immediates for all P loads.
template <int N, int P>
__device__ __forceinline__ float2 kload(const float2* __restrict__ row, int t, int q)
{
    constexpr int T = N / P;
    const char* r = reinterpret_cast<const char*>(row);
    const uint32_t lo = 8u * (uint32_t)t, hi = 8u * (uint32_t)(T - t);
    return *reinterpret_cast<const float2*>(q < P / 2 ? r + lo + q * T * 8 : r + hi + (P - 1 - q) * T * 8);
}

__device__ __forceinline__ float2 cmul_c(float2 x, float2 L, bool conj) { return conj ? cmulc(x, L) : cmul(x, L); }

// A table row of the strided mapping into registers with every load issued before the first
// use (under register pressure the scheduler otherwise pairs each load with its use and
// serialises the latencies).
template <int N, int P>
__device__ __forceinline__ void kload_row(float2 (&L)[P], const float2* __restrict__ row, int t)
{
#pragma unroll
    for (int q = 0; q < P; ++q) L[q] = kload<N, P>(row, t, q);
    __builtin_amdgcn_sched_barrier(0);
}

// Transform policies of the step functions, one object per thread.  XPow2: the transform length is
// the register array length N (a power of two), a wave-level transform (WAVE, P = N/64, no
// barriers) or a subgroup transform through ping-pong buffers; SEED: where its twiddle seeds come
// from (swem_fft.hpp).  XBlue: a transform of runtime length n = nkx (any length) through
// two power-of-two transforms of the array length M >= 2 n - 1 (Bluestein): with
// w_j = exp(SIGN i pi j^2 / n),  X_k = w_k sum_j (x_j w_j) conj(w_(k-j)),  the sum a cyclic
// convolution of length M taken as IFFT_M(FFT_M(x w) B) with B = FFT_M(conj w, wrapped) / M
// built in FP64.  Entries j, k >= n of the array are zero on input and on output.  The PSPI
// selection tables keep the array length as their row stride (0x7f padding beyond nmx) in both.
template <int N, int P, bool WAVE_, int SEED>
struct HeldSeeds {
    __device__ __forceinline__ HeldSeeds(const float2*, int) {}
    __device__ __forceinline__ const float2* ptr() const { return nullptr; }
};
template <int N, int P>
struct HeldSeeds<N, P, false, kSeedHeld> {
    FftSeeds<N, P> s;
    __device__ __forceinline__ HeldSeeds(const float2* tw, int t) { s.load(tw, t); }
    __device__ __forceinline__ const float2* ptr() const { return s.w; }
};
template <int N, int P>
struct HeldSeeds<N, P, true, kSeedHeld> {
    WfftSeeds<N> s;
    __device__ __forceinline__ HeldSeeds(const float2* tw, int t) { s.load(tw, t); }
    __device__ __forceinline__ const float2* ptr() const { return s.w; }
};

template <int N, int P, bool WAVE_ = false, int SEED = kSeedAhead, bool AHEAD = true>
struct XPow2 {
    static constexpr bool kAhead = AHEAD, kPow2 = true;
    HeldSeeds<N, P, WAVE_, SEED> held;
    __device__ __forceinline__ XPow2(const March2DArgs& a, int t) : held(a.tw, t) {}
    // HIN: slots q >= P/2 are zero on input (see fft)
    template <int SIGN, bool WAVE, bool HIN = false>
    __device__ __forceinline__ void fft(float2 (&v)[P], float2* lds, const March2DArgs& a, int t, int& pp) const
    {
        static_assert(WAVE == WAVE_, "transform of another shape");
        if constexpr (WAVE) {
            static_assert(P * 64 == N, "wave transforms hold N/64 points per lane");
            wfft<N, SIGN, SEED, HIN>(v, lds, a.tw, t, held.ptr());
        } else
            swem::fft<N, P, SIGN, SEED, HIN>(v, lds, a.tw, t, pp, held.ptr());
    }
    __device__ __forceinline__ void kload_row(float2 (&L)[P], const float2* __restrict__ row, const March2DArgs&, int t) const
    {
        swem::kload_row<N, P>(L, row, t);
    }
};

template <int M, int P>
struct XBlue {
    static constexpr bool kAhead = true, kPow2 = false;
    static constexpr int T = M / P;
    uint32_t koff[P];  // byte offsets of the thread's points in a kz row (0 beyond n)
    __device__ __forceinline__ XBlue(const March2DArgs& a, int t)
    {
        const int n = a.nkx;
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const int k = t + q * T;
            koff[q] = 8u * (uint32_t)(k < n ? (k <= n / 2 ? k : n - k) : 0);
        }
    }
    template <int SIGN, bool WAVE, bool HIN = false>
    __device__ __forceinline__ void fft(float2 (&v)[P], float2* lds, const March2DArgs& a, int t, int& pp) const
    {
        static_assert(!WAVE, "Bluestein transforms use the subgroup FFT");
        chirp_mul<SIGN>(v, a, t);
        swem::fft<M, P, -1>(v, lds, a.tw, t, pp);
        const float2* B = a.bchirp + (SIGN < 0 ? 0 : M);
        {
            float2 bq[P];
#pragma unroll
            for (int q = 0; q < P; ++q) bq[q] = B[t + q * T];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < P; ++q) v[q] = cmul(v[q], bq[q]);
        }
        swem::fft<M, P, +1>(v, lds, a.tw, t, pp);
        chirp_mul<SIGN>(v, a, t);
    }
    // v_j <- v_j w_j for j < n, 0 beyond (the chirp is reloaded rather than kept in registers)
    template <int SIGN>
    __device__ __forceinline__ void chirp_mul(float2 (&v)[P], const March2DArgs& a, int t) const
    {
        const int n = a.nkx;
        float2 w[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const int j = t + q * T;
            const float2 c = j < n ? a.chirp[j] : make_float2(0.f, 0.f);  // exp(-i pi j^2 / n)
            w[q] = SIGN < 0 ? c : make_float2(c.x, -c.y);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = cmul(v[q], w[q]);
    }
    __device__ __forceinline__ void kload_row(float2 (&L)[P], const float2* __restrict__ row, const March2DArgs&, int) const
    {
#pragma unroll
        for (int q = 0; q < P; ++q) L[q] = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(row) + koff[q]);
        __builtin_amdgcn_sched_barrier(0);
    }
};

// XMixed: a mixed-radix length n = nkx (PRIME: with factors 7, 11, 13) in the power-of-two array of M >= n points,
// transformed in the subgroup's two LDS buffers (mixed_fft); entries j >= n stay zero.
template <int M, int P, bool PRIME = false, bool AHEAD = true>
struct XMixed {
    static constexpr bool kAhead = AHEAD, kPow2 = false;
    XBlue<M, P> b;  // the kz row offsets
    __device__ __forceinline__ XMixed(const March2DArgs& a, int t) : b(a, t) {}
    template <int SIGN, bool WAVE, bool HIN = false>
    __device__ __forceinline__ void fft(float2 (&v)[P], float2* lds, const March2DArgs& a, int t, int& pp) const
    {
        static_assert(!WAVE, "mixed-radix transforms use the subgroup buffers");
        mixed_fft<M, P, SIGN, true, PRIME>(v, lds, lds + LdsLen<M>::value, a.tw, a.mr, t, pp, []() { __syncthreads(); });
    }
    __device__ __forceinline__ void kload_row(float2 (&L)[P], const float2* __restrict__ row, const March2DArgs& a, int t) const
    {
        b.kload_row(L, row, a, t);
    }
};

template <int T>
__device__ __forceinline__ void subgroup_sync()
{
    if constexpr (T == 64) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

struct StepCtx {
    int t, iz, fc;  // thread within the subgroup, depth index, frequency index within the chunk
                    // (fc and iz are wave-uniform: table rows are addressed from scalar registers)
};

__device__ __forceinline__ const float2* krow(const March2DArgs& a, const StepCtx& c, int ir)
{
    return a.ktab + (((size_t)c.fc * a.nz + c.iz) * a.nref + ir) * a.nkh;
}

// Split-step phase row of (fc, iz) as a buffer of nmx entries: lanes x >= nmx read zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ss_row(const March2DArgs& a, const StepCtx& c)
{
    return buf_rsrc(a.stab + ((size_t)c.fc * a.nz + c.iz) * a.nmx, (uint32_t)a.nmx * 8u);
}

// The split-step phases (taper included) of the live slots q < Q; lanes x >= nmx read zero, so the
// product zeroes them.
template <int T, int Q>
__device__ __forceinline__ void ss_load(float2 (&sp)[Q], const March2DArgs& a, const StepCtx& c)
{
    StepCtx u = c;
    u.iz = __builtin_amdgcn_readfirstlane(c.iz);
    const auto sr = ss_row(a, u);
#pragma unroll
    for (int q = 0; q < Q; ++q) sp[q] = buf_load2(sr, (uint32_t)(c.t + q * T) * 8u);
    __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first use
}

template <int P, int Q>
__device__ __forceinline__ void zero_tail(float2 (&u)[P])
{
#pragma unroll
    for (int q = Q; q < P; ++q) u[q] = make_float2(0.f, 0.f);
}

// Step functions.  HALF (2 nmx <= N): the slots q >= P / 2 of a wavefield are zero before and after a
// step, so the first pass of its transform runs half-input butterflies, the last pass of the inverse
// drops the upper outputs and the pointwise work covers Q = P / 2 slots.

// ssop adjoint branch (wem.c:313-320, 334-359) on one wavefield: FFT, kz phase, IFFT, split-step
// phase and taper.  ACT = false turns the step into FFT / IFFT with unit phases (a numerical
// identity) so every subgroup of a workgroup runs the same barriers when only one of the two
// wavefields is stepped at a depth.
template <int N, int P, bool WAVE, bool ACT, bool HALF, class X>
__device__ __forceinline__ void ssf_adj_step(float2 (&u)[P], float2* lds, int& pp, const March2DArgs& a,
                                             const X& xf, const StepCtx& c, bool conj)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    float2 L[P], sp[Q];
    if constexpr (ACT && X::kAhead) xf.kload_row(L, krow(a, c, 0), a, c.t);
    xf.template fft<-1, WAVE, HALF>(u, lds, a, c.t, pp);
    if constexpr (ACT) {
        if constexpr (!X::kAhead) xf.kload_row(L, krow(a, c, 0), a, c.t);
#pragma unroll
        for (int q = 0; q < P; ++q) u[q] = cmul_c(u[q], L[q], conj);
        if constexpr (X::kAhead) ss_load<T, Q>(sp, a, c);
    } else {
#pragma unroll
        for (int q = 0; q < P; ++q) u[q] = cscale(u[q], a.inv_nk);
    }
    xf.template fft<+1, WAVE>(u, lds, a, c.t, pp);
    if constexpr (ACT) {
        if constexpr (!X::kAhead) ss_load<T, Q>(sp, a, c);
#pragma unroll
        for (int q = 0; q < Q; ++q) u[q] = cmul_c(u[q], sp[q], conj);
    } else {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (c.t + q * T >= a.nmx) u[q] = make_float2(0.f, 0.f);
    }
    zero_tail<P, Q>(u);
}

// ssop forward branch with dz < 0 (wem.c:321-332, 334-348, 362-369): taper and split-step phase,
// FFT, kz phase, IFFT.
template <int N, int P, bool WAVE, bool HALF, class X>
__device__ __forceinline__ void ssf_fwd_step(float2 (&u)[P], float2* lds, int& pp, const March2DArgs& a,
                                             const X& xf, const StepCtx& c, const float2 (&sp)[HALF ? P / 2 : P])
{
    constexpr int Q = HALF ? P / 2 : P;
    float2 L[P];
    xf.kload_row(L, krow(a, c, 0), a, c.t);
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] = cmulc(u[q], sp[q]);
    xf.template fft<-1, WAVE, HALF>(u, lds, a, c.t, pp);
#pragma unroll
    for (int q = 0; q < P; ++q) u[q] = cmulc(u[q], L[q]);
    xf.template fft<+1, WAVE>(u, lds, a, c.t, pp);
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (c.t + q * (N / P) >= a.nmx) u[q] = make_float2(0.f, 0.f);
    zero_tail<P, Q>(u);
}

// Weight of reference velocity ir at a point with selection byte s1 (iref1 | cut<<7), iref2
// s2 and interpolation weight w2 (linear mode: the formula at wem.c:476).
__device__ __forceinline__ float pspi_linear_weight(int ir, uint8_t s1, uint8_t s2, float w2)
{
    const int i1 = s1 & 0x7f;
    if (!(s1 >> 7)) return i1 == ir ? 1.f : 0.f;
    float wt = 0.f;
    if (i1 == ir) wt += 1.f - w2;
    if ((int)s2 == ir) wt += w2;
    return wt;
}

// pspiop with the reference structure (wem.c:409-460): FFT, for each vref phase + IFFT, then
// per-x selection.  Compat: u = Re(dref[iref1]) when cut else dref[iref1]; linear: weights.
// The selection rows are padded to N columns (0x7f beyond nmx: no vref selected).
template <int N, int P, int MODE, bool WAVE, bool ACT, bool HALF, class X>
__device__ __forceinline__ void pspi_select_step(float2 (&u)[P], float2* lds, int& pp, const March2DArgs& a, const X& xf,
                                                 const StepCtx& c, bool conj)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    uint32_t todo = a.used[c.iz] & ((1u << a.nref) - 1u);
    const int first = __builtin_ctz(todo | 0x80000000u);
    // each vref's row is read while the transform before its use runs (kAhead)
    float2 L[P];
    auto next_row = [&]() {
        if (ACT && todo) xf.kload_row(L, krow(a, c, __builtin_ctz(todo)), a, c.t);
    };
    if constexpr (X::kAhead) next_row();
    float2 U[Q];
    uint8_t s1[Q], s2[Q];
    float w2[Q];
    auto selection = [&]() {
        const size_t rowx = (size_t)c.iz * N;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int x = c.t + q * T;
            s1[q] = a.sel[rowx + x];
            if constexpr (MODE == kModePspiLinear) {
                s2[q] = a.sel2[rowx + x];
                w2[q] = a.w2[rowx + x];
            }
            U[q] = make_float2(0.f, 0.f);
        }
    };
    if constexpr (X::kAhead) selection();
    xf.template fft<-1, WAVE, HALF>(u, lds, a, c.t, pp);
    if constexpr (!X::kAhead) selection();
    while (todo) {
        const int ir = __builtin_ctz(todo);
        if constexpr (!X::kAhead) next_row();
        todo &= todo - 1u;
        float2 B[P];
#pragma unroll
        for (int q = 0; q < P; ++q) B[q] = ACT ? cmul_c(u[q], L[q], conj) : cscale(u[q], a.inv_nk);
        if constexpr (X::kAhead) next_row();
        xf.template fft<+1, WAVE>(B, lds, a, c.t, pp);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if constexpr (!ACT) {
                if (ir == first) U[q] = B[q];
            } else if constexpr (MODE == kModePspiCompat) {
                if ((s1[q] & 0x7f) == ir) U[q] = (s1[q] >> 7) ? make_float2(B[q].x, 0.f) : B[q];
            } else {
                const float wt = pspi_linear_weight(ir, s1[q], s2[q], w2[q]);
                U[q] = make_float2(fmaf(B[q].x, wt, U[q].x), fmaf(B[q].y, wt, U[q].y));
            }
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] = (c.t + q * T < a.nmx) ? U[q] : make_float2(0.f, 0.f);
    zero_tail<P, Q>(u);
}

// Exact adjoint of the linear select-after step, for the forward receiver (dz < 0):
// u <- IFFT( sum_ir conj(L_ir) FFT(W_ir u) ).
template <int N, int P, bool WAVE, bool HALF, class X>
__device__ __forceinline__ void pspi_weight_step(float2 (&u)[P], float2* lds, int& pp, const March2DArgs& a, const X& xf,
                                                 const StepCtx& c)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    float2 acc[P];
    uint8_t s1[Q], s2[Q];
    float w2[Q];
    const size_t rowx = (size_t)c.iz * N;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int x = c.t + q * T;
        s1[q] = a.sel[rowx + x];
        s2[q] = a.sel2[rowx + x];
        w2[q] = a.w2[rowx + x];
    }
#pragma unroll
    for (int q = 0; q < P; ++q) acc[q] = make_float2(0.f, 0.f);
    for (uint32_t todo = a.used[c.iz] & ((1u << a.nref) - 1u); todo; todo &= todo - 1u) {
        const int ir = __builtin_ctz(todo);
        float2 L[P], B[P];
        if constexpr (X::kAhead) xf.kload_row(L, krow(a, c, ir), a, c.t);
#pragma unroll
        for (int q = 0; q < Q; ++q) B[q] = cscale(u[q], pspi_linear_weight(ir, s1[q], s2[q], w2[q]));
        zero_tail<P, Q>(B);
        xf.template fft<-1, WAVE, HALF>(B, lds, a, c.t, pp);
        if constexpr (!X::kAhead) xf.kload_row(L, krow(a, c, ir), a, c.t);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            acc[q].x = fmaf(B[q].x, L[q].x, fmaf(B[q].y, L[q].y, acc[q].x));
            acc[q].y = fmaf(B[q].y, L[q].x, fmaf(-B[q].x, L[q].y, acc[q].y));
        }
    }
    xf.template fft<+1, WAVE>(acc, lds, a, c.t, pp);
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] = (c.t + q * T < a.nmx) ? acc[q] : make_float2(0.f, 0.f);
    zero_tail<P, Q>(u);
}

// Source / adjoint-receiver step of either method (select-after for PSPI).  act is uniform
// over the subgroup: the branch is taken once per step, not per element.
template <int N, int P, int MODE, bool WAVE, bool HALF, class X>
__device__ __forceinline__ void adj_step(float2 (&u)[P], float2* lds, int& pp, const March2DArgs& a, const X& xf,
                                         const StepCtx& c, bool act, bool conj)
{
    if constexpr (MODE == kModeSSF) {
        if (act)
            ssf_adj_step<N, P, WAVE, true, HALF, X>(u, lds, pp, a, xf, c, conj);
        else
            ssf_adj_step<N, P, WAVE, false, HALF, X>(u, lds, pp, a, xf, c, conj);
    } else {
        if (act)
            pspi_select_step<N, P, MODE, WAVE, true, HALF, X>(u, lds, pp, a, xf, c, conj);
        else
            pspi_select_step<N, P, MODE, WAVE, false, HALF, X>(u, lds, pp, a, xf, c, conj);
    }
}

// Migration march shared by both kernel families.  The workgroup has 2F subgroups of T
// threads; subgroup s = 2f is the source and 2f + 1 the receiver of frequency f.  BUFS LDS
// buffers of LdsLen<N> complex per subgroup (1 for wave transforms, 2 for ping-pong).
template <int N, int P, int MODE, bool WAVE, class X = XPow2<N, P, WAVE>>
__device__ __forceinline__ void adj_body(const March2DArgs& a)
{
    constexpr int T = N / P;
    constexpr int L = LdsLen<N>::value;
    constexpr int BUFS = WAVE ? 1 : 2;
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(a.ngroups, a.nshot, g, shot);
    if (g < 0) return;  // padding block of the XCD-aware grid: exits before any barrier
    const int F = blockDim.x / (2 * T);
    const int tid = threadIdx.x, s = tid / T, t = tid - s * T;
    const int f = s >> 1;
    const bool src = (s & 1) == 0;
    const int fc = g * F + f;  // frequency within the chunk
    const bool active = fc < a.nfc;
    const int fl = a.f0 + fc;  // frequency within the band
    const int iw = a.ifmin + fl;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    const float factor = iw == 0 ? 1.f : 2.f;
    float2* lds = smem + (size_t)s * BUFS * L;
    const float2* xsrc = smem + (size_t)(2 * f) * BUFS * L;
    int pp = 0;
    const X xf(a, t);

    float2 u[P];
    const int igx = a.igx[shot];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        if (src)
            u[q] = (active && x == igx) ? a.spec_s[fl] : make_float2(0.f, 0.f);
        else
            u[q] = (active && x < a.nmx) ? a.spec_r[((size_t)shot * a.nmx + x) * a.nf + fl] : make_float2(0.f, 0.f);
    }
    float* part = a.partial + ((size_t)shot * a.ngroups + g) * (size_t)a.nz * a.nmx;

    for (int iz = 0; iz < a.nz; ++iz) {
        c.iz = iz;
        const float z = a.oz + a.dz * (float)iz;
        const bool ds = z >= a.sz, dr = z >= a.gz;
        if (ds || dr) adj_step<N, P, MODE, WAVE, false, X>(u, lds, pp, a, xf, c, src ? ds : dr, src);
        // imaging condition (wem.c:243-247): the source subgroup hands its wavefield over in LDS
        const int xb = pp * L;
        if (src) {
#pragma unroll
            for (int q = 0; q < P; ++q) lds[xb + lds_pad(t + q * T)] = u[q];
        }
        __syncthreads();
        float cc[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const float2 us = xsrc[xb + lds_pad(t + q * T)];
            cc[q] = dr ? factor * (u[q].x * us.x + u[q].y * us.y) : 0.f;
        }
        if constexpr (!WAVE) pp ^= 1;
        if (F == 1) {
            if (!src) {
                const auto pr = buf_rsrc(part + (size_t)iz * a.nmx, (uint32_t)a.nmx * 4u);
#pragma unroll
                for (int q = 0; q < P; ++q) buf_store1_nt(pr, (uint32_t)(t + q * T) * 4u, cc[q]);
            }
        } else {
            if constexpr (WAVE) __syncthreads();  // single buffer: the source copy is read
            // the receiver subgroup parks its image row in its own buffer; all threads then sum
            // over the F frequencies in a fixed order
            const int rb = pp * L;
            if (!src) {
                float* red = reinterpret_cast<float*>(lds + rb);
#pragma unroll
                for (int q = 0; q < P; ++q) red[t + q * T] = cc[q];
            }
            __syncthreads();
            for (int x = tid; x < a.nmx; x += blockDim.x) {
                float sum = 0.f;
                for (int ff = 0; ff < F; ++ff)
                    sum += reinterpret_cast<const float*>(smem + (size_t)(2 * ff + 1) * BUFS * L + rb)[x];
                part[(size_t)iz * a.nmx + x] = sum;
            }
            if constexpr (!WAVE) pp ^= 1;
        }
        if constexpr (WAVE) __syncthreads();  // readers of the single buffers are done
    }
}

// Modelling march: NSUB subgroups, one frequency each, no interaction between subgroups.
//
// The receiver's depth reads (stored source, image, split-step phases) are issued one depth ahead (kAhead):
// they come from HBM and would otherwise be waited for at the start of every step.
template <int N, int P, int MODE, bool WAVE, bool HALF, class X = XPow2<N, P, WAVE>>
__device__ __forceinline__ void fwd_body(const March2DArgs& a)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    constexpr int L = LdsLen<N>::value;
    constexpr int BUFS = WAVE ? 1 : 2;
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(a.ngroups, a.nshot, g, shot);
    if (g < 0) return;
    const int NSUB = blockDim.x / T;
    const int tid = threadIdx.x, s = tid / T, t = tid - s * T;
    const int fc = __builtin_amdgcn_readfirstlane(g * NSUB + s);  // uniform: T >= 64
    const bool active = fc < a.nfc;
    const int fl = a.f0 + fc;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    float2* lds = smem + (size_t)s * BUFS * L;
    int pp = 0;
    const X xf(a, t);
    const int igx = a.igx[shot];
    // from the wave-uniform fc: a buffer resource of a base the compiler cannot prove uniform costs a
    // loop over the lanes at every access
    float2* sm = a.smig + ((size_t)shot * a.nfc + c.fc) * (size_t)a.nz * a.nmx;

    float2 u[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        u[q] = (active && x == igx) ? a.spec_s[fl] : make_float2(0.f, 0.f);
    }
    // source march, stored per depth (wem.c:254-265)
    for (int iz = 0; iz < a.nz; ++iz) {
        c.iz = iz;
        const float z = a.oz + a.dz * (float)iz;
        const bool ds = z >= a.sz;
        if (ds) adj_step<N, P, MODE, WAVE, HALF, X>(u, lds, pp, a, xf, c, true, true);
        if (active) {
            const auto sr = buf_rsrc(sm + (size_t)iz * a.nmx, (uint32_t)a.nmx * 8u);
#pragma unroll
            for (int q = 0; q < Q; ++q)
                buf_store2(sr, (uint32_t)(t + q * T) * 8u, ds ? u[q] : make_float2(0.f, 0.f));
        }
    }
    // receiver march upward with injection (wem.c:266-276)
#pragma unroll
    for (int q = 0; q < P; ++q) u[q] = make_float2(0.f, 0.f);
    float2 sv[Q], sp[Q];
    float mv[Q];
    auto fetch = [&](int iz) {
        c.iz = iz;
        if (active) {
            const auto sr = buf_rsrc(sm + (size_t)iz * a.nmx, (uint32_t)a.nmx * 8u);
            const auto mr = buf_rsrc(a.mT + (size_t)iz * a.nmx, (uint32_t)a.nmx * 4u);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const uint32_t x = (uint32_t)(t + q * T);
                sv[q] = buf_load2(sr, x * 8u);
                mv[q] = buf_load1(mr, x * 4u);
            }
        } else {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                sv[q] = make_float2(0.f, 0.f);
                mv[q] = 0.f;
            }
        }
        if constexpr (MODE == kModeSSF) ss_load<T, Q>(sp, a, c);
        __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first use
    };
    auto stepped = [&](int iz) { return a.oz + a.dz * (float)iz >= a.gz; };
    int iz = a.nz - 1;
    while (iz >= 0 && !stepped(iz)) --iz;
    if (X::kAhead && iz >= 0) fetch(iz);
    while (iz >= 0) {
        int next = iz - 1;
        while (next >= 0 && !stepped(next)) --next;
        if constexpr (!X::kAhead) fetch(iz);
#pragma unroll
        for (int q = 0; q < Q; ++q) u[q] = make_float2(fmaf(sv[q].x, mv[q], u[q].x), fmaf(sv[q].y, mv[q], u[q].y));
        if constexpr (MODE == kModeSSF) {
            float2 L1[P];
            c.iz = iz;
            if constexpr (X::kAhead) xf.kload_row(L1, krow(a, c, 0), a, t);
#pragma unroll
            for (int q = 0; q < Q; ++q) u[q] = cmulc(u[q], sp[q]);
            if (X::kAhead && next >= 0) fetch(next);
            xf.template fft<-1, WAVE, HALF>(u, lds, a, t, pp);
            if constexpr (!X::kAhead) xf.kload_row(L1, krow(a, c, 0), a, t);
#pragma unroll
            for (int q = 0; q < P; ++q) u[q] = cmulc(u[q], L1[q]);
            xf.template fft<+1, WAVE>(u, lds, a, t, pp);
            zero_tail<P, Q>(u);  // within the live slots the next split-step row cuts at nmx
        } else {
            if (X::kAhead && next >= 0) fetch(next);
            c.iz = iz;
            if constexpr (MODE == kModePspiCompat)
                pspi_select_step<N, P, MODE, WAVE, true, HALF, X>(u, lds, pp, a, xf, c, true);
            else
                pspi_weight_step<N, P, WAVE, HALF, X>(u, lds, pp, a, xf, c);
        }
        iz = next;
    }
    if (active) {
        const auto dr = buf_rsrc(a.dgw + (size_t)shot * a.nmx * a.nf, (uint32_t)a.nmx * a.nf * 8u);
#pragma unroll
        for (int q = 0; q < Q; ++q) buf_store2(dr, ((uint32_t)(t + q * T) * (uint32_t)a.nf + (uint32_t)fl) * 8u, u[q]);
    }
}

// Migration march with one subgroup per frequency that steps the source, then the receiver,
// through the same LDS buffers (variant PAIR).  One frequency per workgroup; the imaging
// condition is register-local.
template <int N, int P, int MODE, bool WAVE, bool HALF, class X = XPow2<N, P, WAVE>>
__device__ __forceinline__ void adj_body_pair(const March2DArgs& a)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    // split-step steps on a power-of-two length: both wavefields in lockstep (fft2)
    constexpr bool LOCK = MODE == kModeSSF && std::is_same<X, XPow2<N, P, WAVE, kSeedHeld>>::value;
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(a.ngroups, a.nshot, g, shot);
    if (g < 0) return;  // padding block of the XCD-aware grid
    const int t = threadIdx.x;
    const int fc = g;  // one frequency per workgroup
    const bool active = fc < a.nfc;
    const int fl = a.f0 + fc;
    const int iw = a.ifmin + fl;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    const float factor = iw == 0 ? 1.f : 2.f;
    int pp = 0;
    const X xf(a, t);
    const int igx = a.igx[shot];
    float2 us[P], ur[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        us[q] = (active && x == igx) ? a.spec_s[fl] : make_float2(0.f, 0.f);
        ur[q] = (active && x < a.nmx) ? a.spec_r[((size_t)shot * a.nmx + x) * a.nf + fl] : make_float2(0.f, 0.f);
    }
    float* part = a.partial + ((size_t)shot * a.ngroups + g) * (size_t)a.nz * a.nmx;
    auto image = [&](int iz, bool dr) {  // imaging condition (wem.c:243-247)
        const auto pr = buf_rsrc(part + (size_t)iz * a.nmx, (uint32_t)a.nmx * 4u);
#pragma unroll
        for (int q = 0; q < Q; ++q)
            buf_store1_nt(pr, (uint32_t)(t + q * T) * 4u, dr ? factor * (ur[q].x * us[q].x + ur[q].y * us[q].y) : 0.f);
    };
    // the depths above the deeper of source and receivers, where one of the two steps alone
    int iz = 0;
    for (; iz < a.nz; ++iz) {
        c.iz = iz;
        const float z = a.oz + a.dz * (float)iz;
        const bool ds = z >= a.sz, dr = z >= a.gz;
        if (LOCK && ds && dr) break;
        if (ds) adj_step<N, P, MODE, WAVE, HALF, X>(us, smem, pp, a, xf, c, true, true);
        if (dr) adj_step<N, P, MODE, WAVE, HALF, X>(ur, smem, pp, a, xf, c, true, false);
        image(iz, dr);
    }
    if constexpr (LOCK) {
        // Both step: one read of each phase row for the two, a depth ahead (the rows stream from
        // HBM; a 256-point step lasts less than their latency), and the transforms in lockstep.  One shot of
        // 128 traces x 200 depths: 533 us in turn, 316 so (FMA butterflies and held seeds included); the
        // latency of the depths in series bounds it.
        auto sync = [] { subgroup_sync<T>(); };
        const float2* held = xf.held.ptr();
        float2 *bu = smem, *bv = smem + LdsLen<N>::value;
        float2 L[P], sp[Q];
        sync();  // the single steps above leave their last exchange unread by slower waves
        if (iz < a.nz) {
            c.iz = iz;
            xf.kload_row(L, krow(a, c, 0), a, t);
            ss_load<T, Q>(sp, a, c);
        }
        for (; iz < a.nz; ++iz) {
            const float z = a.oz + a.dz * (float)iz;
            if (!(z >= a.sz && z >= a.gz)) {  // a depth axis that turns back (dz < 0)
                c.iz = iz;
                if (z >= a.sz) adj_step<N, P, MODE, WAVE, HALF, X>(us, smem, pp, a, xf, c, true, true);
                if (z >= a.gz) adj_step<N, P, MODE, WAVE, HALF, X>(ur, smem, pp, a, xf, c, true, false);
                image(iz, z >= a.gz);
                sync();
                c.iz = min(iz + 1, a.nz - 1);
                xf.kload_row(L, krow(a, c, 0), a, t);
                ss_load<T, Q>(sp, a, c);
                continue;
            }
            c.iz = min(iz + 1, a.nz - 1);
            fft2<N, P, -1, HALF>(us, ur, bu, bv, held, t, sync);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                us[q] = cmulc(us[q], L[q]);
                ur[q] = cmul(ur[q], L[q]);
            }
            xf.kload_row(L, krow(a, c, 0), a, t);
            fft2<N, P, +1, false>(us, ur, bu, bv, held, t, sync);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                us[q] = cmulc(us[q], sp[q]);
                ur[q] = cmul(ur[q], sp[q]);
            }
            zero_tail<P, Q>(us);
            zero_tail<P, Q>(ur);
            ss_load<T, Q>(sp, a, c);
            image(iz, true);
        }
    }
}

// ---------------------------------------------------------------- packed PSPI compat migration
// In compat mode pspiop keeps only the real part of its result wherever vref2 - vref1 > 10
// (wem.c:450-458 with linear_interp, wem.c:473-478), so after a step both wavefields are real
// except at the few points of each depth with iref1 == iref2 (v at the depth's maximum, or every
// point of a depth with vmax <= vmin + 10).  With s = s_R + i s_I, r = r_R + i r_I the state is
//   z = s_R + i a r_R        e = s_I - i a r_I          (a: balances the two magnitudes)
// and, because L_ir(k) is even in kx and FFTs of real sequences are Hermitian,
//   Re P_src(s) + i a Re P_rec(r) = IFFT( Re L Z + Im L E )                        (all x)
//   Im P_src(s) - i a Im P_rec(r) = IFFT( Re L E - Im L Z )                        (all x)
// with Z = FFT(z), E = FFT(e), P_src using conj(L) (-dz) and P_rec using L.  One inverse
// transform per vref thus steps both wavefields; one more, with the vref of the uncut points,
// gives their new e: 2 + nref + 1 transforms per depth instead of 2 (1 + nref).  The image is
// factor Re(r conj s) = factor (Re z Im z - Re e Im e) / a.

// Sum over the 64 lanes of a wave, in every lane: four steps inside the rows of 16 lanes by DPP and
// two across them by the row swaps (vector-ALU instructions: a butterfly of LDS permutes waits for
// the LDS six times in turn).
__device__ __forceinline__ float wave_sum(float v)
{
    auto dpp = [](float x, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value,
                                                                     0xf, 0xf, true));
    };
    v += dpp(v, std::integral_constant<int, 0xb1>{});   // quad_perm 1 0 3 2
    v += dpp(v, std::integral_constant<int, 0x4e>{});   // quad_perm 2 3 0 1
    v += dpp(v, std::integral_constant<int, 0x141>{});  // half-row mirror
    v += dpp(v, std::integral_constant<int, 0x140>{});  // row mirror
    auto add = [](unsigned a, unsigned b) { return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b); };
    const unsigned a = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane16_swap(a, a, false, false);
    v = add(r[0], r[1]);
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const auto h = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return add(h[0], h[1]);
}

// Sum over the T threads of a subgroup in a fixed order (red: T/64 floats of LDS scratch).
template <int T>
__device__ __forceinline__ float subgroup_sum(float v, float* red)
{
    v = wave_sum(v);
    if constexpr (T == 64) {
        return v;
    } else {
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < T / 64; ++i) s += red[i];
        __syncthreads();
        return s;
    }
}

// HALF: nmx <= N / 2, so the points q >= P / 2 (x >= N / 2) are zero in the state and never selected:
// those constants let the first forward pass and the last inverse pass drop their work.
// X: the transform policy (XPow2: nkx = N; XMixed: a mixed-radix nkx <= N, whose twiddle table
// holds nkx entries and whose spectra are zero at k >= nkx).
//
// What bounds it (nkx 2048, two waves per workgroup, two waves per SIMD): vector-ALU issue and the
// latencies that two waves cannot hide, so nothing that can be known early is waited for: the seeds
// of the transforms stay in registers for the whole march, a kz row is read while the transform
// before it runs, the selection bytes and the direct sums' twiddles at the start of the depth, and
// the wave sums take no LDS.  64 shots of 1024 traces x 500 depths x 641 frequencies: 282 -> 217 ms, VALUs
// 90 % busy at 2906 instructions per wave and depth.
template <int N, int P, bool WAVE, bool HALF, class X = XPow2<N, P, WAVE, kSeedHeld>>
__device__ __forceinline__ void adj_body_packed(const March2DArgs& a)
{
    constexpr int T = N / P;
    constexpr int Q = HALF ? P / 2 : P;  // live slots
    constexpr int K = kUncutSparse;
    constexpr int NW = T / 64;  // waves of the subgroup
    constexpr bool POW2 = X::kPow2;
    // Bluestein lengths: the table tw is of the array length, not of nkx, so no direct sums (the
    // uncut points' e and output always come from transforms)
    constexpr bool BLUE = std::is_same<X, XBlue<N, P>>::value;
    // exp(-2 pi i m / nkx) for the direct sums (m >= 0)
    auto twid = [&](int m) { return POW2 ? a.tw[m & (N - 1)] : a.tw[m % a.nkx]; };
    static_assert(4 + K + 2 * NW * K <= kPackedScratch, "packed scratch");
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(a.ngroups, a.nshot, g, shot);
    if (g < 0) return;  // padding block of the XCD-aware grid
    const int t = threadIdx.x;
    const int fc = g;  // one frequency per workgroup
    const bool active = fc < a.nfc;
    const int fl = a.f0 + fc;
    const int iw = a.ifmin + fl;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    const float factor = iw == 0 ? 1.f : 2.f;
    int pp = 0;
    const X xf(a, t);
    const int igx = a.igx[shot];
    const float2 ss = active ? a.spec_s[fl] : make_float2(0.f, 0.f);
    // scratch after the transform buffers: reduction slots, e at the previous depth's second and
    // later uncut points, per-wave partial sums of the direct sums
    float2* scr = smem + (WAVE ? 1 : 2) * LdsLen<N>::value;
    float* red = reinterpret_cast<float*>(scr);
    float2* scr_e = scr + 4;
    float2* scr_v = scr + 4 + K;
    float2 z[P], e[P];
    float nr = 0.f;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        e[q] = (active && x < a.nmx) ? a.spec_r[((size_t)shot * a.nmx + x) * a.nf + fl] : make_float2(0.f, 0.f);
        nr += e[q].x * e[q].x + e[q].y * e[q].y;
    }
    nr = subgroup_sum<T>(nr, red);
    const float ns = sqrtf(ss.x * ss.x + ss.y * ss.y);
    float* part = a.partial + ((size_t)shot * a.ngroups + g) * (size_t)a.nz * a.nmx;
    if (nr == 0.f || ns == 0.f) {
        // a zero receiver or source spectrum images to zero at every depth (the march is linear
        // in each): the packed pair would leave rounding noise of the other wavefield instead
        // (a NaN in either takes the march and reaches the image)
        for (int iz = 0; iz < a.nz; ++iz) {
            const auto pr = buf_rsrc(part + (size_t)iz * a.nmx, (uint32_t)a.nmx * 4u);
#pragma unroll
            for (int q = 0; q < P; ++q) buf_store1_nt(pr, (uint32_t)(t + q * T) * 4u, 0.f);
        }
        return;
    }
    float alpha = ns / sqrtf(nr);
    float inv_alpha = 1.f / alpha;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        const float2 us = x == igx ? ss : make_float2(0.f, 0.f);
        z[q] = make_float2(us.x, alpha * e[q].x);
        e[q] = make_float2(us.y, -alpha * e[q].y);
        if (HALF && q >= P / 2) z[q] = e[q] = make_float2(0.f, 0.f);
    }
    // e before the step: dense in e (the initial imaginary parts; more than K uncut points), or
    // nonzero only at the prev_cnt <= K uncut points of the previous depth: its value at the first
    // of them (ev, known to every thread) with the twiddles of that point (w0 = w^(t x), st =
    // w^(T x), w = exp(-2 pi i / nkx)), the others in scr_e
    int prev_cnt = -1;  // -1: dense
    const int* prev_row = a.cref;
    float2 ev = make_float2(0.f, 0.f), w0 = ev, st = ev;
    for (int iz = 0; iz < a.nz; ++iz) {
        c.iz = iz;
        const int* crow = a.cref + (size_t)iz * kCrefStride;
        const int cr = crow[0], cnt = crow[1];
        const bool sparse = !BLUE && cnt > 0 && cnt <= K;
        // Few uncut points, and no cut point selecting their vref cr: their output under cr, like
        // their new e, comes from direct sums instead of an inverse transform of cr (HALF kernels:
        // the others have no registers left for the second set of sums).
        const bool direct_cr = HALF && sparse && crow[2] != 0;
        uint32_t todo = a.used[iz] & ((1u << a.nref) - 1u);
        if (direct_cr) todo &= ~(1u << cr);
        // the rows of the depth in turn: those of todo, then cr's for the uncut points; each is
        // read while the transform before its use runs (kAhead)
        float2 Lr[P];
        auto next_row = [&](uint32_t left) {
            if (left || cnt > 0) xf.kload_row(Lr, krow(a, c, left ? __builtin_ctz(left) : cr), a, t);
        };
        if constexpr (X::kAhead) next_row(todo);
        uint32_t s1[Q];
        auto selection = [&]() {
#pragma unroll
            for (int q = 0; q < Q; ++q) s1[q] = a.sel[(size_t)iz * N + t + q * T];
        };
        if constexpr (X::kAhead) selection();
        // HALF: slots q >= P/2 of z and e are zero (x >= N/2 >= nmx is never selected)
        xf.template fft<-1, WAVE, HALF>(z, smem, a, t, pp);
        if (prev_cnt < 0 || prev_cnt > (BLUE ? 0 : K)) {
            xf.template fft<-1, WAVE, HALF>(e, smem, a, t, pp);
        } else if (prev_cnt > 0) {
            // E(k) = sum_j e(x_j) w^(k x_j), by recurrence over the thread's points k = t + q T
            float2 p = cmul(ev, w0);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                e[q] = p;
                p = cmul(p, st);
            }
#pragma unroll 1
            for (int j = 1; j < prev_cnt; ++j) {
                const int xj = prev_row[3 + j];
                const float2 sj = twid(T * xj);
                p = cmul(scr_e[j], twid(t * xj));
#pragma unroll
                for (int q = 0; q < P; ++q) {
                    e[q] = cadd(e[q], p);
                    p = cmul(p, sj);
                }
            }
            if constexpr (!POW2) {  // the spectrum of a length nkx < N ends at nkx
#pragma unroll
                for (int q = 0; q < P; ++q)
                    if (t + q * T >= a.nkx) e[q] = make_float2(0.f, 0.f);
            }
        } else {
#pragma unroll
            for (int q = 0; q < P; ++q) e[q] = make_float2(0.f, 0.f);
        }
        if (sparse) {  // for this depth's sums and the next depth's E
            w0 = twid(t * crow[3]);
            st = twid(T * crow[3]);
        }
        if constexpr (!X::kAhead) selection();
        float2 out[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) out[q] = make_float2(0.f, 0.f);
        while (todo) {
            const uint32_t ir = (uint32_t)__builtin_ctz(todo);
            if constexpr (!X::kAhead) next_row(todo);
            todo &= todo - 1u;
            float2 w[P];
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const float2 L = Lr[q];
                w[q] = make_float2(z[q].x * L.x + e[q].x * L.y, z[q].y * L.x + e[q].y * L.y);
            }
            if constexpr (X::kAhead) next_row(todo);
            xf.template fft<+1, WAVE>(w, smem, a, t, pp);
#pragma unroll
            for (int q = 0; q < Q; ++q)
                if ((s1[q] & 0x7fu) == ir) out[q] = w[q];
        }
        if constexpr (!X::kAhead) next_row(0);
        float2 en[Q];  // the new e
#pragma unroll
        for (int q = 0; q < Q; ++q) en[q] = make_float2(0.f, 0.f);
        if (cnt > 0 && !sparse) {
            // imaginary parts at the uncut points of this depth (all select vref cr):
            // e_new = IFFT(Re L E - Im L Z), the conjugate of IFFT(V) by L(-k) = L(k)
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const float2 L = Lr[q];
                e[q] = make_float2(L.x * e[q].x - L.y * z[q].x, L.x * e[q].y - L.y * z[q].y);
            }
            xf.template fft<+1, WAVE>(e, smem, a, t, pp);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int x = t + q * T;
                if (x < a.nmx && !(s1[q] >> 7)) en[q] = e[q];
            }
        } else if (sparse) {
            // e_new(x_j) = sum_k U(k) conj(w^(k x_j)) with U = Re L E - Im L Z at the few uncut points
            // and, when direct_cr, out(x_j) = sum_k W(k) conj(w^(k x_j)) with W = Re L Z + Im L E:
            // per thread by Horner's rule over its points k = t + q T, then over the subgroup in
            // a fixed order.  U into e and W into z, in place (the spectra end here).
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const float2 L = Lr[q];
                const float2 u = make_float2(L.x * e[q].x - L.y * z[q].x, L.x * e[q].y - L.y * z[q].y);
                if (HALF) z[q] = make_float2(z[q].x * L.x + e[q].x * L.y, z[q].y * L.x + e[q].y * L.y);
                e[q] = u;
            }
            auto sums = [&](float2 w, float2 s, int j, float2& su, float2& sw) {
                su = e[P - 1];
                sw = HALF ? z[P - 1] : su;
#pragma unroll
                for (int q = P - 2; q >= 0; --q) {
                    su = make_float2(fmaf(su.x, s.x, fmaf(su.y, s.y, e[q].x)), fmaf(su.y, s.x, fmaf(-su.x, s.y, e[q].y)));
                    if (HALF)
                        sw = make_float2(fmaf(sw.x, s.x, fmaf(sw.y, s.y, z[q].x)), fmaf(sw.y, s.x, fmaf(-sw.x, s.y, z[q].y)));
                }
                su = cmulc(su, w);
                su = make_float2(wave_sum(su.x), wave_sum(su.y));
                if (HALF) {
                    sw = cmulc(sw, w);
                    sw = make_float2(wave_sum(sw.x), wave_sum(sw.y));
                }
                if constexpr (NW > 1)
                    if ((t & 63) == 0) {
                        scr_v[(t >> 6) * K + j] = su;
                        scr_v[(NW + (t >> 6)) * K + j] = sw;
                    }
            };
            float2 wn, wc;
            sums(w0, st, 0, wn, wc);
            // the second and later points: rare (equal maxima of the depth's velocity)
#pragma unroll 1
            for (int j = 1; j < cnt; ++j) {
                const int xj = crow[3 + j];
                float2 su, sw;
                sums(twid(t * xj), twid(T * xj), j, su, sw);
                if (NW == 1 && t == 0) scr_v[j] = su, scr_v[K + j] = sw;
            }
            subgroup_sync<T>();
            auto total = [&](int j, float2& su, float2& sw) {
                su = scr_v[j];
                sw = scr_v[NW * K + j];
#pragma unroll
                for (int wv = 1; wv < NW; ++wv) {
                    su = cadd(su, scr_v[wv * K + j]);
                    sw = cadd(sw, scr_v[(NW + wv) * K + j]);
                }
            };
            auto place = [&](int xj, float2 su, float2 sw) {
                const int tj = xj & (T - 1), qj = xj / T;  // the owner's thread and slot
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    if (q == qj && t == tj) {
                        en[q] = su;
                        if (direct_cr) out[q] = sw;
                    }
            };
            if constexpr (NW > 1) total(0, wn, wc);
            ev = wn;
            place(crow[3], wn, wc);
#pragma unroll 1
            for (int j = 1; j < cnt; ++j) {
                float2 su, sw;
                total(j, su, sw);
                place(crow[3 + j], su, sw);
                if (t == 0) scr_e[j] = su;
            }
        }
        prev_cnt = cnt;
        prev_row = crow;
        // imaging condition (wem.c:243-247): factor Re(ur conj(us))
        const auto pr = buf_rsrc(part + (size_t)iz * a.nmx, (uint32_t)a.nmx * 4u);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            if (q >= Q) {  // x >= nmx: nothing to image
                z[q] = e[q] = make_float2(0.f, 0.f);
                continue;
            }
            z[q] = out[q];
            e[q] = en[q];
            buf_store1_nt(pr, (uint32_t)(t + q * T) * 4u, factor * (z[q].x * z[q].y - e[q].x * e[q].y) * inv_alpha);
        }
        // keep the two packed wavefields of comparable size (the rounding of each transform is
        // relative to their sum): every 8 depths, rescale the receiver part when the ratio of
        // their energies leaves [1/4, 4]
        if ((iz & 7) != 7) continue;
        float n2s = 0.f, n2r = 0.f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            n2s += z[q].x * z[q].x + e[q].x * e[q].x;
            n2r += z[q].y * z[q].y + e[q].y * e[q].y;
        }
        n2s = subgroup_sum<T>(n2s, red);
        n2r = subgroup_sum<T>(n2r, red);
        if (n2s > 0.f && n2r > 0.f && (n2s > 4.f * n2r || n2r > 4.f * n2s)) {
            const float beta = sqrtf(n2s / n2r);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                z[q].y *= beta;
                e[q].y *= beta;
            }
            ev.y *= beta;
            if (t == 0)
                for (int j = 1; j < cnt && j < K; ++j) scr_e[j].y *= beta;
            alpha *= beta;
            inv_alpha = 1.f / alpha;
        }
    }
}

#define SWEM_SUBGROUP_BOUNDS(P) __launch_bounds__((P) == 16 ? 512 : kMaxBlock)

// Where the marches keep their twiddle seeds, and whether they read rows, selections and the stored source
// ahead of their use.  Seeds held in registers drop the table loads and address arithmetic of every transform;
// the half-line kernels have the registers for it, the general form at 16 points per thread spills
// and so does the 128-register budget of the large workgroups with 8.  Read ahead -> held, 8 shots x 100 depths,
// 1024 / 512 traces, and 16 shots of 256: split-step modelling 4.9 -> 3.8, 2.3 -> 1.8, 2.5 -> 1.6 ms; PSPI modelling
// 10.9 -> 9.2, 5.1 -> 4.2, 5.4 -> 4.0; linear modelling 11.5 -> 10.1, 5.3 -> 4.6, 5.5 -> 4.3; linear migration 11.3 ->
// 9.9, 5.3 -> 4.7, 5.9 -> 4.7.  Two vrefs of a PSPI step in lockstep on top spill (188 bytes): 76 -> 81 ms
// where held alone gives 63.
// The read-ahead needs 16 to 80 registers more.  The general lines at 16 points per thread (and 8 in the large
// workgroups) read at the use and step the two wavefields in turn: 16 shots x 20 depths of 4096 points (pad
// factor 1), ahead -> at the use: split-step migration 4.1 -> 3.0 ms, modelling 5.0 -> 3.2, linear migration 12.3 -> 7.6,
// linear modelling 11.1 -> 6.8.  So do the mixed-radix marches but the half-line migration and split-step
// modelling, whose workgroups would lose a wave per SIMD: 8 shots x 20 depths, nkx 3000, PSPI modelling 8.4 -> 5.1 ms.
constexpr int held_if(bool fits) { return fits ? kSeedHeld : kSeedAhead; }

template <int N, int P, bool HALF>
__global__ __launch_bounds__(N / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_packed(March2DArgs a)
{
    adj_body_packed<N, P, false, HALF, XPow2<N, P, false, held_if(HALF), HALF>>(a);
}

template <int N, bool HALF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_packed_w(March2DArgs a)
{
    adj_body_packed<N, N / 64, true, HALF>(a);
}

// Packed compat migration of a mixed-radix or Bluestein nkx on the array length M (the subgroup
// shape of the other non-power-of-two kernels: M / 8 threads from M = 1024, one wave below).
template <int M, int P, bool HALF, bool PRIME>
__global__ __launch_bounds__(M / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_packed_mixed(March2DArgs a)
{
    adj_body_packed<M, P, false, HALF, XMixed<M, P, PRIME>>(a);
}
template <int M, int P, bool HALF>
__global__ __launch_bounds__(M / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_packed_blue(March2DArgs a)
{
    adj_body_packed<M, P, false, HALF, XBlue<M, P>>(a);
}

template <int N, int MODE, int P>
__global__ SWEM_SUBGROUP_BOUNDS(P) void march2d_adj(March2DArgs a)
{
    adj_body<N, P, MODE, false, XPow2<N, P, false, P < 16 ? kSeedAhead : kSeedPass, P < 8>>(a);
}

template <int N, int MODE, int P, bool HALF>
__global__ SWEM_SUBGROUP_BOUNDS(P) void march2d_fwd(March2DArgs a)
{
    fwd_body<N, P, MODE, false, HALF, XPow2<N, P, false, held_if(HALF && P == 16), HALF || P < 8>>(a);
}

template <int N, int MODE>
__global__ __launch_bounds__(kWaveBlock) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_w(March2DArgs a)
{
    adj_body<N, N / 64, MODE, true, XPow2<N, N / 64, true, kSeedAhead, N < 1024>>(a);
}

template <int N, int MODE, bool HALF>
__global__ __launch_bounds__(kWaveBlock) __attribute__((amdgpu_waves_per_eu(2))) void march2d_fwd_w(March2DArgs a)
{
    fwd_body<N, N / 64, MODE, true, HALF, XPow2<N, N / 64, true, held_if(HALF && N <= 1024), HALF || N < 1024>>(a);
}

// PAIR: 16 points per thread from nkx = 1024 (nkx/16 threads, radix-16 passes), one wave with
// nkx/64 points per lane below it.
template <int N, int MODE, int P, bool HALF>
__global__ __launch_bounds__(N / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_pair(March2DArgs a)
{
    adj_body_pair<N, P, MODE, false, HALF,
                  XPow2<N, P, false, held_if(HALF || (MODE == kModeSSF && P < 16)), HALF || P < 16>>(a);
}

template <int N, int MODE, bool HALF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_pair_w(March2DArgs a)
{
    adj_body_pair<N, N / 64, MODE, true, HALF, XPow2<N, N / 64, true, held_if(HALF || MODE == kModeSSF)>>(a);
}

// Transform lengths that are not powers of two: Bluestein through the array length M (one
// subgroup of M/P threads marches both wavefields of a frequency in migration, as PAIR does;
// modelling takes F frequencies per workgroup of at most 512 threads).  P = 8 from M = 1024:
// the chirp products add live registers, and 16 points per thread would spill.
template <int M, int MODE, int P>
__global__ __launch_bounds__(M / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_blue(March2DArgs a)
{
    adj_body_pair<M, P, MODE, false, true, XBlue<M, P>>(a);
}

template <int M, int MODE, int P>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void march2d_fwd_blue(March2DArgs a)
{
    fwd_body<M, P, MODE, false, true, XBlue<M, P>>(a);
}

template <int M, int MODE, int P, bool HALF, bool PRIME>
__global__ __launch_bounds__(M / P) __attribute__((amdgpu_waves_per_eu(2))) void march2d_adj_mixed(March2DArgs a)
{
    adj_body_pair<M, P, MODE, false, HALF, XMixed<M, P, PRIME, HALF>>(a);
}

template <int M, int MODE, int P, bool HALF, bool PRIME>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void march2d_fwd_mixed(March2DArgs a)
{
    fwd_body<M, P, MODE, false, HALF, XMixed<M, P, PRIME, HALF && MODE == kModeSSF>>(a);
}

// ------------------------------------------------------------------ launches of one array length
template <typename K>
static int launch_kernel(K kernel, const March2DArgs& a, dim3 block, size_t lds, hipStream_t st)
{
    SWEM_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    dim3 grid(march2d_grid_blocks(a.ngroups, a.nshot));
    hipLaunchKernelGGL(kernel, grid, block, lds, st, a);
    SWEM_HIP(hipGetLastError());
    return SWEM_OK;
}

template <int N, int MODE>
static int launch_one(const March2DArgs& a, const March2DShape& sh, int F, int adj, hipStream_t st)
{
    const size_t lds = march2d_lds_bytes(N, sh, F);
    dim3 block(sh.T * sh.per_freq * F);
    if (sh.variant == SWEM_VARIANT_PACKED && MODE == kModePspiCompat && adj) {
        const size_t lds_p = lds + kPackedScratch * sizeof(float2);
        const bool half = 2 * a.nmx <= N;
        if constexpr (N < 1024)
            return half ? launch_kernel(march2d_adj_packed_w<N, true>, a, block, lds_p, st)
                        : launch_kernel(march2d_adj_packed_w<N, false>, a, block, lds_p, st);
        else
            return half ? launch_kernel(march2d_adj_packed<N, 16, true>, a, block, lds_p, st)
                        : launch_kernel(march2d_adj_packed<N, 16, false>, a, block, lds_p, st);
    }
    const bool half = 2 * a.nmx <= N;
    auto go = [&](auto with_half, auto without) { return launch_kernel(half ? with_half : without, a, block, lds, st); };
    if (sh.variant == SWEM_VARIANT_PAIR || sh.variant == SWEM_VARIANT_PACKED) {
        if constexpr (N < 1024)
            return go(march2d_adj_pair_w<N, MODE, true>, march2d_adj_pair_w<N, MODE, false>);
        else
            return go(march2d_adj_pair<N, MODE, 16, true>, march2d_adj_pair<N, MODE, 16, false>);
    }
    if (sh.variant == SWEM_VARIANT_PAIR8) {
        if constexpr (N >= 512) return go(march2d_adj_pair<N, MODE, 8, true>, march2d_adj_pair<N, MODE, 8, false>);
    }
    if constexpr (N <= 2048) {
        if (sh.variant == SWEM_VARIANT_WAVE)
            return adj ? launch_kernel(march2d_adj_w<N, MODE>, a, block, lds, st)
                       : go(march2d_fwd_w<N, MODE, true>, march2d_fwd_w<N, MODE, false>);
    }
    if constexpr (N >= 1024) {
        if (sh.variant == SWEM_VARIANT_SUBGROUP16)
            return adj ? launch_kernel(march2d_adj<N, MODE, 16>, a, block, lds, st)
                       : go(march2d_fwd<N, MODE, 16, true>, march2d_fwd<N, MODE, 16, false>);
    }
    constexpr int P = Pts<N>::value;
    return adj ? launch_kernel(march2d_adj<N, MODE, P>, a, block, lds, st)
               : go(march2d_fwd<N, MODE, P, true>, march2d_fwd<N, MODE, P, false>);
}

template <int M, int MODE>
static int launch_blue_mode(const March2DArgs& a, const March2DShape& sh, int F, int adj, hipStream_t st)
{
    constexpr int P = M >= 1024 ? 8 : M / 64;
    const size_t lds = march2d_lds_bytes(a.nkx, sh, F);
    dim3 block(sh.T * sh.per_freq * F);
    const bool half = 2 * a.nmx <= M;
    // one launch of the mixed-radix kernels with or without the radices 7, 11, 13 (lengths up to 2048)
    auto mixed = [&](auto prime) {
        constexpr bool PR = decltype(prime)::value;
        if constexpr (MODE == kModePspiCompat) {
            if (adj && sh.variant == SWEM_VARIANT_PACKED) {
                const size_t lds_p = lds + kPackedScratch * sizeof(float2);
                return launch_kernel(half ? march2d_adj_packed_mixed<M, P, true, PR> : march2d_adj_packed_mixed<M, P, false, PR>, a,
                                     block, lds_p, st);
            }
        }
        if (adj)
            return launch_kernel(half ? march2d_adj_mixed<M, MODE, P, true, PR> : march2d_adj_mixed<M, MODE, P, false, PR>, a, block,
                                 lds, st);
        return launch_kernel(half ? march2d_fwd_mixed<M, MODE, P, true, PR> : march2d_fwd_mixed<M, MODE, P, false, PR>, a, block, lds,
                             st);
    };
    if (sh.mixed == 1) return mixed(std::false_type{});
    if constexpr (M <= 2048)
        if (sh.mixed == 2) return mixed(std::true_type{});
    if constexpr (MODE == kModePspiCompat)
        if (adj && sh.variant == SWEM_VARIANT_PACKED)
            // Bluestein: M >= 2 nkx - 1 >= 2 nmx - 1, and M even, so the upper half is always zero
            return launch_kernel(march2d_adj_packed_blue<M, P, true>, a, block, lds + kPackedScratch * sizeof(float2), st);
    return adj ? launch_kernel(march2d_adj_blue<M, MODE, P>, a, block, lds, st)
               : launch_kernel(march2d_fwd_blue<M, MODE, P>, a, block, lds, st);
}

template <int M>
int launch_blue(const March2DArgs& a, const March2DShape& sh, int F, int mode, int adj, hipStream_t st)
{
    if (mode == kModeSSF) return launch_blue_mode<M, kModeSSF>(a, sh, F, adj, st);
    if (mode == kModePspiCompat) return launch_blue_mode<M, kModePspiCompat>(a, sh, F, adj, st);
    return launch_blue_mode<M, kModePspiLinear>(a, sh, F, adj, st);
}

template <int N>
int launch_n(const March2DArgs& a, const March2DShape& sh, int F, int mode, int adj, hipStream_t st)
{
    if (mode == kModeSSF) return launch_one<N, kModeSSF>(a, sh, F, adj, st);
    if (mode == kModePspiCompat) return launch_one<N, kModePspiCompat>(a, sh, F, adj, st);
    return launch_one<N, kModePspiLinear>(a, sh, F, adj, st);
}


// ------------------------------------------------------------------ source incidence angles
// compute_angles (wem.c:566-776) for 2-D.  The source march is the modelling receiver's step
// (ssop with adj = false and -dz, which is ssop_source, wem.c:778-826) stored at every depth.
// The derivatives of calculate_derivatives (wem.c:828-981) are separable: the inverse 3-D
// transform of i kx FFT3(u), divided by nkx nky nkz, equals IFFT_x(i kx FFT_x(u)) / nkx, so the
// x parts run along rows and the z part along columns of the stored volume.
template <int N, int P, class X>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void angle_march(March2DArgs a)
{
    constexpr int T = N / P;
    constexpr int L = LdsLen<N>::value;
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(a.ngroups, a.nshot, g, shot);
    if (g < 0) return;
    const int NSUB = blockDim.x / T;
    const int tid = threadIdx.x, s = tid / T, t = tid - s * T;
    const int fc = g * NSUB + s;
    const bool active = fc < a.nfc;
    const int fl = a.f0 + fc;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    float2* lds = smem + (size_t)s * 2 * L;
    int pp = 0;
    const X xf(a, t);
    const int igx = a.igx[shot];
    float2* vol = a.smig + (size_t)c.fc * a.nz * a.nmx;
    float2 u[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        u[q] = (active && x == igx) ? a.spec_s[fl] : make_float2(0.f, 0.f);
    }
    for (int iz = 0; iz < a.nz; ++iz) {  // extrapolate_source, wem.c:712-719
        c.iz = iz;
        const float z = a.oz + a.dz * (float)iz;
        const bool ds = z >= a.sz;
        if (ds) {
            float2 sp[P];
            ss_load<T, P>(sp, a, c);
            ssf_fwd_step<N, P, false, false, X>(u, lds, pp, a, xf, c, sp);
        }
        if (active) {
            const auto sr = buf_rsrc(vol + (size_t)iz * a.nmx, (uint32_t)a.nmx * 8u);
#pragma unroll
            for (int q = 0; q < P; ++q) buf_store2(sr, (uint32_t)(t + q * T) * 8u, ds ? u[q] : make_float2(0.f, 0.f));
        }
    }
}

__device__ __forceinline__ float kbin(int k, int n, float dk)
{
    return k <= n / 2 ? dk * (float)k : -(dk * (float)n - dk * (float)k);
}

__device__ __forceinline__ float2 times_i(float2 v, float k) { return make_float2(-v.y * k, v.x * k); }

// z pass (wem.c:888-899): |IFFT_z(i kz FFT_z(u))| / nz along the z line of one (frequency, point).
template <int N, int P, class X>
__global__ __launch_bounds__(N / P) void angle_cols(March2DArgs az, AngleArgs b)
{
    constexpr int T = N / P;
    extern __shared__ float2 smem[];
    const int l = blockIdx.x;
    const size_t base = (size_t)(l / b.inner) * b.outer + (size_t)(l % b.inner) * b.inner_stride;
    const int t = threadIdx.x;
    int pp = 0;
    const X xf(az, t);
    const float2* col = b.vol + base;
    float2 v[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int iz = t + q * T;
        v[q] = iz < b.nz ? col[(size_t)iz * b.elem] : make_float2(0.f, 0.f);
    }
    __builtin_amdgcn_sched_barrier(0);
    xf.template fft<-1, false>(v, smem, az, t, pp);
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int k = t + q * T;
        v[q] = times_i(v[q], k < b.nz ? kbin(k, b.nz, b.dkz) : 0.f);
    }
    xf.template fft<+1, false>(v, smem, az, t, pp);
    float* out = b.dzmag + base;
    const float inv = 1.f / (float)b.nz;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int iz = t + q * T;
        if (iz < b.nz) out[(size_t)iz * b.elem] = sqrtf(v[q].x * v[q].x + v[q].y * v[q].y) * inv;
    }
}

// Lateral pass along one x (or y) line of one depth: per frequency in order, the derivative along
// the line (wem.c:858-887) against the z pass's |u_z| (wem.c:747-748) and the left / right split
// (wem.c:901-970, wem.c:739-740), added to the sums of earlier chunks.
template <int N, int P, class X>
__global__ __launch_bounds__(N / P) void angle_rows(March2DArgs ax, AngleArgs b)
{
    constexpr int T = N / P;
    extern __shared__ float2 smem[];
    const int l = blockIdx.x;
    const size_t base = (size_t)(l / b.inner) * b.outer + (size_t)(l % b.inner) * b.inner_stride;
    const int t = threadIdx.x;
    int pp = 0;
    const X xf(ax, t);
    const int n = ax.nkx;
    const float deg = (float)(180.0 / 3.141592653589793);
    const float inv = 1.f / (float)n;
    const float inv_nw = 1.f / (float)b.nw;
    float acc[P], sgn[P], kx[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        const size_t i = base + (size_t)x * b.elem;
        acc[q] = x < b.len ? b.acc[i] : 0.f;
        sgn[q] = x < b.len ? b.sgn[i] : 0.f;
        kx[q] = x < n ? kbin(x, n, b.dk) : 0.f;
    }
    for (int f = 0; f < b.nfc; ++f) {
        const float2* ur = b.vol + (size_t)f * b.item + base;
        const float* zr = b.dzmag + (size_t)f * b.item + base;
        float2 A[P];
        float mu[P], mz[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const int x = t + q * T;
            A[q] = x < b.len ? ur[(size_t)x * b.elem] : make_float2(0.f, 0.f);
            mz[q] = x < b.len ? zr[(size_t)x * b.elem] : 0.f;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < P; ++q) mu[q] = sqrtf(A[q].x * A[q].x + A[q].y * A[q].y);
        xf.template fft<-1, false>(A, smem, ax, t, pp);
        float mx[P], ml[P];
        float2 B[P];
#pragma unroll
        for (int q = 0; q < P; ++q) B[q] = times_i(A[q], kx[q]);
        xf.template fft<+1, false>(B, smem, ax, t, pp);
#pragma unroll
        for (int q = 0; q < P; ++q) mx[q] = sqrtf(B[q].x * B[q].x + B[q].y * B[q].y) * inv;
        // negative wavenumbers only (k > n/2), then positive only (k <= n/2)
#pragma unroll
        for (int q = 0; q < P; ++q) B[q] = times_i(A[q], (t + q * T) <= n / 2 ? 0.f : kx[q]);
        xf.template fft<+1, false>(B, smem, ax, t, pp);
#pragma unroll
        for (int q = 0; q < P; ++q) ml[q] = sqrtf(B[q].x * B[q].x + B[q].y * B[q].y);
#pragma unroll
        for (int q = 0; q < P; ++q) B[q] = times_i(A[q], (t + q * T) <= n / 2 ? kx[q] : 0.f);
        xf.template fft<+1, false>(B, smem, ax, t, pp);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const float mr = sqrtf(B[q].x * B[q].x + B[q].y * B[q].y);
            sgn[q] += (ml[q] >= mr ? mu[q] : -mu[q]) * inv_nw;
            acc[q] += deg * atanf(mx[q] / (mz[q] + 1e-10f));
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int x = t + q * T;
        if (x < b.len) {
            const size_t i = base + (size_t)x * b.elem;
            b.acc[i] = acc[q];
            b.sgn[i] = sgn[q];
        }
    }
}

template <int N, class X>
static int launch_angles_n(int which, const March2DArgs& ax, const March2DArgs& az, const AngleArgs& b, int F,
                           hipStream_t st)
{
    constexpr int P = N >= 1024 ? 8 : N / 64, T = N / P;
    const size_t len = (size_t)LdsLen<N>::value * sizeof(float2);
    if (which == 0) {
        if (F < 1 || F * T > 512 || F * 2 * len > 160 * 1024) return set_error(SWEM_EINVAL, "angles: %d frequencies per block", F);
        return launch_kernel(angle_march<N, P, X>, ax, dim3(T * F), F * 2 * len, st);
    }
    auto k = which == 1 ? angle_cols<N, P, X> : angle_rows<N, P, X>;
    const March2DArgs& a = which == 1 ? az : ax;
    const unsigned grid = (unsigned)b.lines;
    SWEM_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * len)));
    hipLaunchKernelGGL(k, dim3(grid), dim3(T), 2 * len, st, a, b);
    SWEM_HIP(hipGetLastError());
    return SWEM_OK;
}

template <int N>
int launch_angles_len(int which, int kind, const March2DArgs& ax, const March2DArgs& az, const AngleArgs& b,
                             int F, hipStream_t st)
{
    constexpr int P = N >= 1024 ? 8 : N / 64;
    if (kind == kLenMixed) return launch_angles_n<N, XMixed<N, P>>(which, ax, az, b, F, st);
    if constexpr (N <= 2048)
        if (kind == kLenMixedPrime) return launch_angles_n<N, XMixed<N, P, true>>(which, ax, az, b, F, st);
    return kind == kLenBluestein ? launch_angles_n<N, XBlue<N, P>>(which, ax, az, b, F, st)
                                 : launch_angles_n<N, XPow2<N, P>>(which, ax, az, b, F, st);
}


// ------------------------------------------------------------------------ elastic WEM (2-D)
// ewem (ewem.c:3-366).  Per frequency: the P source (vp, -dz, adjoint order) normalised by the
// largest source sample, and the receiver components (ux, uz).  Per depth the components are
// separated into the P and second S potentials (elastic_separate_3d, ewem.c:553-741; the first
// S potential is never formed), each propagated with its own velocity's split-step step, and
// recombined; the P and S images correlate the potentials with the source.  The separation
// matrix of wavenumber kx (kx = dkx ikx for ikx < nkx/2, else -(dkx nkx - dkx ikx)) uses the
// depth's layer velocities vp0 = 1/po_p, vs0 = 1/po_s and is computed in place.
// Two wavefields through the transform: in lockstep on a power-of-two length (fft2), else in turn.
// A depth takes seven dependent pairs of transforms at two waves per SIMD (200 VGPRs), so barriers and
// exchanges, not the vector ALUs, bound the march; the potentials and the components always go in pairs.
// 4 shots of 512 traces x 300 depths x 576 frequencies, adjoint: 22.0 ms in turn over whole lines, 20.8
// with the zero half dropped, 17.5 in lockstep as well.  Three waves per SIMD spill (216 bytes): no faster.
template <int N, int P, int SIGN, bool HIN, class X>
__device__ __forceinline__ void ewem_fft(float2 (&u)[P], float2 (&v)[P], float2* lds, int& pp, const March2DArgs& a,
                                         const X& xf, int t)
{
    if constexpr (std::is_same<X, XPow2<N, P, false, kSeedHeld>>::value) {
        fft2<N, P, SIGN, HIN>(u, v, lds, lds + LdsLen<N>::value, xf.held.ptr(), t, [] { subgroup_sync<N / P>(); });
    } else {
        xf.template fft<SIGN, false, HIN>(u, lds, a, t, pp);
        xf.template fft<SIGN, false, HIN>(v, lds, a, t, pp);
    }
}

// The split-step steps of the two potentials, each with its own phase tables: BACK the forward
// operator (split step first, then the phases of -dz), else the adjoint one.
template <int N, int P, bool HALF, bool BACK, class X>
__device__ __forceinline__ void ewem_step(float2 (&u)[P], float2 (&v)[P], float2* lds, int& pp, const March2DArgs& ap,
                                          const March2DArgs& as, const X& xf, const StepCtx& c)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    float2 L[P], sp[Q], ss[Q];
    if constexpr (BACK) {
        ss_load<T, Q>(sp, ap, c);
        ss_load<T, Q>(ss, as, c);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            u[q] = cmulc(u[q], sp[q]);
            v[q] = cmulc(v[q], ss[q]);
        }
    }
    xf.kload_row(L, krow(ap, c, 0), ap, c.t);
    ewem_fft<N, P, -1, HALF>(u, v, lds, pp, ap, xf, c.t);
#pragma unroll
    for (int q = 0; q < P; ++q) u[q] = cmul_c(u[q], L[q], BACK);
    xf.kload_row(L, krow(as, c, 0), as, c.t);
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cmul_c(v[q], L[q], BACK);
    if constexpr (!BACK) {
        ss_load<T, Q>(sp, ap, c);
        ss_load<T, Q>(ss, as, c);
    }
    ewem_fft<N, P, +1, false>(u, v, lds, pp, ap, xf, c.t);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if constexpr (BACK) {
            if (c.t + q * T >= ap.nmx) u[q] = v[q] = make_float2(0.f, 0.f);
        } else {
            u[q] = cmul(u[q], sp[q]);
            v[q] = cmul(v[q], ss[q]);
        }
    }
    zero_tail<P, Q>(u);
    zero_tail<P, Q>(v);
}

// (i1, i2) -> (o1, o2) through the wavenumber domain; o1, o2 are zero at x >= nmx.
template <int N, int P, bool HALF, class X>
__device__ __forceinline__ void esep(const float2 (&i1)[P], const float2 (&i2)[P], float2 (&o1)[P], float2 (&o2)[P],
                                     float2* lds, int& pp, const March2DArgs& a, const X& xf, const EwemArgs& e, int t, float w,
                                     float vp, float vs, bool sep, bool adj)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    const int n = a.nkx;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        o1[q] = i1[q];
        o2[q] = i2[q];
    }
    ewem_fft<N, P, -1, HALF>(o1, o2, lds, pp, a, xf, t);
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int k = t + q * T;
        const float kx = k < n ? ((float)k < (float)n / 2.f ? e.dkx * (float)k : -(e.dkx * (float)n - e.dkx * (float)k))
                               : 0.f;
        float2 r1, r2;
        esep_k(kx, w, vp, vs, sep, adj, o1[q], o2[q], r1, r2);
        o1[q] = k < n ? cscale(r1, a.inv_nk) : make_float2(0.f, 0.f);
        o2[q] = k < n ? cscale(r2, a.inv_nk) : make_float2(0.f, 0.f);
    }
    ewem_fft<N, P, +1, false>(o1, o2, lds, pp, a, xf, t);
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (t + q * T >= a.nmx) o1[q] = o2[q] = make_float2(0.f, 0.f);
    zero_tail<P, Q>(o1);
    zero_tail<P, Q>(o2);
}

template <int N, int P, bool HALF, class X, bool ADJ>
__global__ __launch_bounds__(N / P) __attribute__((amdgpu_waves_per_eu(2))) void ewem_march(March2DArgs ap,
                                                                                             March2DArgs as, EwemArgs e)
{
    constexpr int T = N / P, Q = HALF ? P / 2 : P;
    extern __shared__ float2 smem[];
    int g, shot;
    decode_block(ap.ngroups, ap.nshot, g, shot);
    if (g < 0) return;
    const int t = threadIdx.x;
    const int fc = g;
    const bool active = fc < ap.nfc;
    const int fl = ap.f0 + fc;
    const int iw = ap.ifmin + fl;
    const float w = (float)iw * e.dwf;
    StepCtx c;
    c.t = t;
    c.fc = __builtin_amdgcn_readfirstlane(active ? fc : 0);
    int pp = 0;
    const X xf(ap, t);
    const int igx = ap.igx[shot];
    const float factor = iw == 0 ? 1.f : 2.f;
    const size_t sp = (size_t)shot * ap.nmx * e.nf;  // this shot's spectra
    float2 us[P], rx[P], rz[P];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int x = t + q * T;
        us[q] = (active && x == igx) ? ap.spec_s[fl] : make_float2(0.f, 0.f);
        rx[q] = (ADJ && active && x < ap.nmx) ? e.spx[sp + (size_t)x * e.nf + fl] : make_float2(0.f, 0.f);
        rz[q] = (ADJ && active && x < ap.nmx) ? e.spz[sp + (size_t)x * e.nf + fl] : make_float2(0.f, 0.f);
    }
    zero_tail<P, Q>(us);
    zero_tail<P, Q>(rx);
    zero_tail<P, Q>(rz);
    // partial images / stored source of (shot, frequency)
    const size_t vol = ((size_t)shot * ap.ngroups + (active ? fc : 0)) * ap.nz * ap.nmx;
    if constexpr (ADJ) {
        for (int iz = 0; iz < ap.nz; ++iz) {  // elastic_extrap1f, ewem.c:302-327
            c.iz = iz;
            const float z = ap.oz + ap.dz * (float)iz;
            const bool ds = z >= ap.sz, dr = z >= ap.gz;
            if (ds) ssf_adj_step<N, P, false, true, HALF, X>(us, smem, pp, ap, xf, c, true);
            subgroup_sync<T>();  // the lockstep transforms write both buffers, the single one's last exchange with them
            float2 up[P], u2[P];
            if (dr) {
                const float vp = e.vp0[iz], vs = e.vs0[iz];
                esep<N, P, HALF, X>(rx, rz, up, u2, smem, pp, ap, xf, e, t, w, vp, vs, true, true);
                ewem_step<N, P, HALF, false, X>(up, u2, smem, pp, ap, as, xf, c);
                esep<N, P, HALF, X>(up, u2, rx, rz, smem, pp, ap, xf, e, t, w, vp, vs, false, true);
            }
            if (active) {
                const auto rp = buf_rsrc(e.ppart + vol + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 4u);
                const auto rs = buf_rsrc(e.spart + vol + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 4u);
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const float2 sm = ds ? cscale(us[q], e.inv_maxs) : make_float2(0.f, 0.f);
                    const uint32_t off = (uint32_t)(t + q * T) * 4u;
                    buf_store1(rp, off, dr ? factor * (sm.x * up[q].x + sm.y * up[q].y) : 0.f);
                    buf_store1(rs, off, dr ? factor * (sm.x * u2[q].x + sm.y * u2[q].y) : 0.f);
                }
            }
        }
    } else {
        for (int iz = 0; iz < ap.nz; ++iz) {  // source, stored per depth (ewem.c:302-310)
            c.iz = iz;
            const float z = ap.oz + ap.dz * (float)iz;
            const bool ds = z >= ap.sz;
            if (ds) ssf_adj_step<N, P, false, true, HALF, X>(us, smem, pp, ap, xf, c, true);
            if (active) {
                const auto sr = buf_rsrc(e.smig + vol + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 8u);
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    buf_store2(sr, (uint32_t)(t + q * T) * 8u, ds ? cscale(us[q], e.inv_maxs) : make_float2(0.f, 0.f));
            }
        }
        subgroup_sync<T>();  // as in the migration
        for (int iz = ap.nz - 1; iz >= 0; --iz) {  // receiver upward (ewem.c:328-346)
            c.iz = iz;
            const float z = ap.oz + ap.dz * (float)iz;
            if (!(z >= ap.gz)) continue;
            const float vp = e.vp0[iz], vs = e.vs0[iz];
            float2 up[P], u2[P];
            esep<N, P, HALF, X>(rx, rz, up, u2, smem, pp, ap, xf, e, t, w, vp, vs, true, false);
            if (active) {
                const auto sr = buf_rsrc(e.smig + vol + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 8u);
                const auto mp = buf_rsrc(e.mppT + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 4u);
                const auto ms = buf_rsrc(e.mpsT + (size_t)iz * ap.nmx, (uint32_t)ap.nmx * 4u);
                float2 sv[Q];
                float mpv[Q], msv[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const uint32_t x = (uint32_t)(t + q * T);
                    sv[q] = buf_load2(sr, x * 8u);
                    mpv[q] = buf_load1(mp, x * 4u);
                    msv[q] = buf_load1(ms, x * 4u);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    up[q] = cadd(up[q], cscale(sv[q], mpv[q]));
                    u2[q] = cadd(u2[q], cscale(sv[q], msv[q]));
                }
            }
            ewem_step<N, P, HALF, true, X>(up, u2, smem, pp, ap, as, xf, c);
            esep<N, P, HALF, X>(up, u2, rx, rz, smem, pp, ap, xf, e, t, w, vp, vs, false, false);
        }
        if (active) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int x = t + q * T;
                if (x < ap.nmx) {
                    e.dgx[sp + (size_t)x * e.nf + fl] = rx[q];
                    e.dgz[sp + (size_t)x * e.nf + fl] = rz[q];
                }
            }
        }
    }
}

template <int N, class X, bool HALF = false>
static int launch_ewem_n(const March2DArgs& ap, const March2DArgs& as, const EwemArgs& e, int adj, hipStream_t st)
{
    constexpr int P = N >= 1024 ? 8 : N / 64, T = N / P;
    const size_t lds = (size_t)LdsLen<N>::value * 2 * sizeof(float2);
    auto k = adj ? ewem_march<N, P, HALF, X, true> : ewem_march<N, P, HALF, X, false>;
    SWEM_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3(march2d_grid_blocks(ap.ngroups, ap.nshot)), dim3(T), lds, st, ap, as, e);
    SWEM_HIP(hipGetLastError());
    return SWEM_OK;
}

template <int N>
int launch_ewem_len(int kind, const March2DArgs& ap, const March2DArgs& as, const EwemArgs& e, int adj,
                           hipStream_t st)
{
    constexpr int P = N >= 1024 ? 8 : N / 64;
    if (kind == kLenMixed) return launch_ewem_n<N, XMixed<N, P>>(ap, as, e, adj, st);
    if constexpr (N <= 2048)
        if (kind == kLenMixedPrime) return launch_ewem_n<N, XMixed<N, P, true>>(ap, as, e, adj, st);
    return kind == kLenBluestein ? launch_ewem_n<N, XBlue<N, P>>(ap, as, e, adj, st)
           : 2 * ap.nmx <= N         ? launch_ewem_n<N, XPow2<N, P, false, kSeedHeld>, true>(ap, as, e, adj, st)
                                     : launch_ewem_n<N, XPow2<N, P, false, kSeedHeld>>(ap, as, e, adj, st);
}

}  // namespace swem
