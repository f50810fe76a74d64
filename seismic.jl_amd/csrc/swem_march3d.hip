// swem_march3d.hip -- dispatch of the 3-D marches (swem_march3d.hpp).  The kernels of each transform
// array length are compiled in an object of their own (swem_march3d_len.hip).
#include "swem_internal.hpp"

namespace swem {

// Launches of one array length and length kind, instantiated in swem_march3d_len.hip.
template <int N, int BL>
int launch_ewem3d_n(int which, const March3DArgs& ap, const March3DArgs& as, const Ewem3DArgs& e, int F, int phase,
                    hipStream_t st);
template <int N, int BL>
int launch3_n(int which, const March3DArgs& a, int F, int phase, hipStream_t st);

// Array length of a 3-D line transform of n points: n for powers of two 128..1024, the next power of two
// for mixed-radix lengths (2, 3, 5 up to 1024; with factors 7, 11, 13 up to 512), else the Bluestein length (the power of two >= max(128, 2n - 1), up to 1024: n <= 512; n = 1 is the
// nkx of a single inline, nmx = 1); 0 if neither.
int march3d_kind(int n)
{
    if (n >= 128 && !(n & (n - 1))) return kLenPow2;
    return mixed_kind(n);
}

int march3d_len(int n)
{
    if (n < 1) return 0;
    const int kind = march3d_kind(n);
    if (kind == kLenPow2) return n <= 1024 ? n : 0;
    int m = 128;
    if (is_mixed(kind)) {
        if (kind == kLenMixedPrime && n > 512) return 0;
        while (m < n) m <<= 1;
        return m <= 1024 ? m : 0;
    }
    if (n > 512) return 0;
    while (m < 2 * n - 1) m <<= 1;
    return m;
}

bool march3d_supported(int nkx, int nky) { return march3d_len(nkx) > 0 && march3d_len(nky) > 0; }

// which: 0 init (y-FFT of the initial wavefields), 1 x-pass, 2 adjoint y-pass, 3 forward y-pass
// (phase 0 source, 1 receiver, 2 output).  F: frequencies per y-pass workgroup.
int launch_ewem3d(int which, const March3DArgs& ap, const March3DArgs& as, const Ewem3DArgs& e, int F, int phase,
                  hipStream_t st)
{
    const bool xpass = which == 1;
    const int n = xpass ? ap.nkx : ap.nky, m = march3d_len(n);
    if (!march3d_supported(ap.nkx, ap.nky) || ap.nmx > ap.nkx || ap.nmy > ap.nky || ap.nitem < 1 || !e.W)
        return set_error(SWEM_EINVAL, "3-D ewem: inconsistent launch (nkx=%d nky=%d)", ap.nkx, ap.nky);
    if (which == 2 && (F < 1 || F > 8))  // the y-pass holds three rows per line of lanes: 512 threads
        return set_error(SWEM_EINVAL, "3-D ewem: %d frequencies per workgroup (1..8)", F);
    const int kind = march3d_kind(n);
    if ((kind == kLenBluestein && (xpass ? !(ap.chx && ap.bchx) : !(ap.chy && ap.bchy))) ||
        (is_mixed(kind) && (xpass ? ap.mrx.n : ap.mry.n) != n))
        return set_error(SWEM_EINVAL, "3-D ewem: transform tables missing (n=%d)", n);
    switch (kind * 16 + m / 128) {
#define SWEM_E3(M, K) \
    case K * 16 + M / 128: return launch_ewem3d_n<M, K>(which, ap, as, e, F, phase, st);
        SWEM_E3(128, 0) SWEM_E3(256, 0) SWEM_E3(512, 0) SWEM_E3(1024, 0)
        SWEM_E3(128, 1) SWEM_E3(256, 1) SWEM_E3(512, 1) SWEM_E3(1024, 1)
        SWEM_E3(128, 2) SWEM_E3(256, 2) SWEM_E3(512, 2) SWEM_E3(1024, 2)
        SWEM_E3(128, 3) SWEM_E3(256, 3) SWEM_E3(512, 3)
#undef SWEM_E3
    }
    return set_error(SWEM_EUNSUPPORTED, "3-D ewem: n=%d", n);
}

int launch_march3d(int which, const March3DArgs& a, int F, int phase, hipStream_t st)
{
    const bool xpass = which == 1 || which == 4 || which == 6;
    const int n = xpass ? a.nkx : a.nky, m = march3d_len(n);
    if (!march3d_supported(a.nkx, a.nky) || a.nmx > a.nkx || a.nmy > a.nky || a.nitem < 1)
        return set_error(SWEM_EINVAL, "3-D march: inconsistent launch (nkx=%d nky=%d)", a.nkx, a.nky);
    const int kind = march3d_kind(n);
    if (kind == kLenBluestein && (xpass ? !(a.chx && a.bchx) : !(a.chy && a.bchy)))
        return set_error(SWEM_EINVAL, "3-D march: Bluestein tables missing (n=%d)", n);
    if (is_mixed(kind) && (xpass ? a.mrx.n : a.mry.n) != n)
        return set_error(SWEM_EINVAL, "3-D march: mixed-radix plan missing (n=%d)", n);
    // y-passes: up to 16 frequencies per workgroup (8 on a Bluestein y axis, whose kernels are
    // compiled for 512 threads to keep their longer transforms in registers; 8 for PSPI)
    const int fmax = which == 5 ? 8 : (!xpass && kind != kLenPow2 ? 8 : 16);
    if (((which == 2 || which == 3 || which == 5) && F > fmax) || F < 1)
        return set_error(SWEM_EINVAL, "3-D march: %d frequencies per workgroup (at most %d here)", F, fmax);
    if ((which == 4 || which == 5 || which == 6) && (!a.R || !a.sel || !a.used || a.nref < 1 || a.nref > 31))
        return set_error(SWEM_EINVAL, "3-D PSPI march: tables missing");
    if ((a.linear || which == 6) && (!a.sel2 || !a.w2))
        return set_error(SWEM_EINVAL, "3-D PSPI march: linear-mode tables missing");
    switch (kind * 16 + m / 128) {
#define SWEM_M3(M, K) \
    case K * 16 + M / 128: return launch3_n<M, K>(which, a, F, phase, st);
        SWEM_M3(128, 0) SWEM_M3(256, 0) SWEM_M3(512, 0) SWEM_M3(1024, 0)
        SWEM_M3(128, 1) SWEM_M3(256, 1) SWEM_M3(512, 1) SWEM_M3(1024, 1)
        SWEM_M3(128, 2) SWEM_M3(256, 2) SWEM_M3(512, 2) SWEM_M3(1024, 2)
        SWEM_M3(128, 3) SWEM_M3(256, 3) SWEM_M3(512, 3)
#undef SWEM_M3
    }
    return set_error(SWEM_EUNSUPPORTED, "3-D march: n=%d", n);
}

}  // namespace swem
