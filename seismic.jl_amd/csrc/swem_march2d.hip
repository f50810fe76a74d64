// swem_march2d.hip -- kernel shapes and dispatch of the 2-D marches (swem_march2d.hpp).  The kernels
// of each transform array length are compiled in an object of their own (swem_march2d_len.hip).
#include "swem_internal.hpp"

namespace swem {

// Launches of one array length, instantiated in swem_march2d_len.hip.
template <int N>
int launch_n(const March2DArgs& a, const March2DShape& sh, int F, int mode, int adj, hipStream_t st);
template <int M>
int launch_blue(const March2DArgs& a, const March2DShape& sh, int F, int mode, int adj, hipStream_t st);
template <int N>
int launch_angles_len(int which, int kind, const March2DArgs& ax, const March2DArgs& az, const AngleArgs& b, int F,
                      hipStream_t st);
template <int N>
int launch_ewem_len(int kind, const March2DArgs& ap, const March2DArgs& as, const EwemArgs& e, int adj, hipStream_t st);

// Kernel shape of a variant: threads per wavefield subgroup T, subgroups per frequency
// (2 = source and receiver in separate subgroups, 1 = one subgroup marches both), the largest
// workgroup, LDS buffers per subgroup.
//   WAVE         one 64-lane wave per wavefield, no barrier inside a transform (nkx <= 2048)
//   SUBGROUP     nkx/8 threads per wavefield (nkx/4, nkx/2 below 512), ping-pong LDS
//   SUBGROUP16   nkx/16 threads per wavefield, radix-16 passes (nkx >= 1024)
//   PAIR         (migration) one subgroup per frequency marches source and receiver in turn:
//                the imaging needs no hand-off and a barrier holds only that subgroup's waves;
//                a wave (nkx <= 1024) or nkx/16 threads.  Modelling uses the AUTO shape.
//   PACKED       PAIR's shape; PSPI compat migration with both wavefields in one transform
//                (the host selects it only where every depth steps both wavefields and the
//                uncut points of a depth share one vref; other modes run PAIR).
//   Bluestein    any other transform length up to 2048 (nkx = 1 too: one trace, nmx = 1, whose
//                transform is the identity): the PAIR body (migration) or the
//                subgroup body (modelling) over the array length M = blue (P = 8 from M = 1024,
//                one wave below); the variant option does not apply.
int march2d_kind(int nkx)
{
    if (nkx >= 128 && !(nkx & (nkx - 1))) return kLenPow2;
    return mixed_kind(nkx);
}

int march2d_blue_len(int nkx)
{
    if (nkx < 1 || (nkx >= 128 && !(nkx & (nkx - 1)))) return 0;
    int m = 128;
    if (is_mixed(march2d_kind(nkx))) {
        while (m < nkx) m <<= 1;
        return m <= 4096 ? m : 0;
    }
    if (nkx > 2048) return 0;
    while (m < 2 * nkx - 1) m <<= 1;
    return m;
}

March2DShape march2d_shape(int nkx, int variant, int adj)
{
    March2DShape sh{};
    if (const int m = march2d_blue_len(nkx)) {
        sh.blue = m;
        sh.mixed = march2d_kind(nkx) == kLenMixed ? 1 : march2d_kind(nkx) == kLenMixedPrime ? 2 : 0;
        sh.variant = adj ? SWEM_VARIANT_PAIR : SWEM_VARIANT_SUBGROUP;
        if (adj && variant == SWEM_VARIANT_PACKED) sh.variant = SWEM_VARIANT_PACKED;
        sh.T = m >= 1024 ? m / 8 : 64;
        sh.per_freq = 1;
        sh.max_block = adj ? sh.T : 512;
        sh.bufs = 2;
        return sh;
    }
    if (nkx < 128 || nkx > 4096 || (nkx & (nkx - 1))) return sh;
    int v = variant;
    if ((v == SWEM_VARIANT_PAIR || v == SWEM_VARIANT_PAIR8 || v == SWEM_VARIANT_PACKED) && !adj) v = SWEM_VARIANT_AUTO;
    if (v == SWEM_VARIANT_PAIR8 && nkx < 512) v = SWEM_VARIANT_PAIR;
    if (v == SWEM_VARIANT_AUTO) v = adj ? SWEM_VARIANT_PAIR : (nkx <= 512 ? SWEM_VARIANT_WAVE : SWEM_VARIANT_SUBGROUP16);
    if (v == SWEM_VARIANT_WAVE && nkx > 2048) v = SWEM_VARIANT_SUBGROUP16;
    if (v == SWEM_VARIANT_SUBGROUP16 && nkx < 1024) v = SWEM_VARIANT_SUBGROUP;
    sh.variant = v;
    sh.per_freq = adj ? 2 : 1;
    switch (v) {
    case SWEM_VARIANT_WAVE:
        sh.T = 64, sh.max_block = kWaveBlock, sh.bufs = 1;
        break;
    case SWEM_VARIANT_SUBGROUP16:
        sh.T = nkx / 16, sh.max_block = 512, sh.bufs = 2;
        break;
    case SWEM_VARIANT_PAIR:
    case SWEM_VARIANT_PACKED:
        sh.T = nkx >= 1024 ? nkx / 16 : 64, sh.per_freq = 1, sh.max_block = sh.T, sh.bufs = 2;
        break;
    case SWEM_VARIANT_PAIR8:
        sh.T = nkx / 8, sh.per_freq = 1, sh.max_block = sh.T, sh.bufs = 2;
        break;
    default:
        sh.variant = SWEM_VARIANT_SUBGROUP;
        sh.T = nkx / (nkx >= 512 ? 8 : (nkx >= 256 ? 4 : 2)), sh.max_block = kMaxBlock, sh.bufs = 2;
    }
    return sh;
}

bool march2d_supported(int nkx) { return march2d_shape(nkx, SWEM_VARIANT_AUTO, 1).T > 0; }

size_t march2d_lds_bytes(int nkx, const March2DShape& sh, int F)
{
    if (sh.blue) nkx = sh.blue;
    const size_t len = (size_t)(((nkx + nkx / 8 + 31) & ~31) + 4);  // LdsLen<nkx>
    return (size_t)F * sh.per_freq * sh.bufs * len * sizeof(float2);
}

int march2d_grid_blocks(int ngroups, int nshot) { return ((ngroups + 7) / 8) * 8 * nshot; }

// F = frequencies per workgroup (migration: 2F subgroups, or F for PAIR; modelling: F subgroups).
int launch_march2d(const March2DArgs& a, int nkx, int F, int mode, int adj, int variant, hipStream_t st)
{
    const March2DShape sh = march2d_shape(nkx, variant, adj);
    if (sh.T <= 0)
        return set_error(SWEM_EUNSUPPORTED,
                         "2-D march: nkx=%d is neither a power of two 128..4096, 2^a 3^b 5^c up to 4096 nor 1..2048", nkx);
    if (F < 1 || sh.T * sh.per_freq * F > sh.max_block)
        return set_error(SWEM_EINVAL, "2-D march: %d frequencies of %d subgroups of %d threads exceed %d", F,
                         sh.per_freq, sh.T, sh.max_block);
    if (a.nmx > nkx || a.nref < 1 || a.nref > 31 || a.ngroups < 1 || a.nshot < 1 || a.nkh != nkx / 2 + 1 ||
        a.f0 < 0 || a.nfc < 1 || a.f0 + a.nfc > a.nf)
        return set_error(SWEM_EINVAL, "2-D march: inconsistent launch (nmx=%d nkx=%d nref=%d)", a.nmx, nkx, a.nref);
    if (march2d_lds_bytes(nkx, sh, F) > 160 * 1024)
        return set_error(SWEM_EINVAL, "2-D march: LDS for %d frequencies at nkx=%d exceeds 160 KiB", F, nkx);
    if (sh.blue) {
        if (a.nkx != nkx || (sh.mixed ? a.mr.n != nkx : (!a.chirp || !a.bchirp)))
            return set_error(SWEM_EINVAL, "2-D march: %s tables missing", sh.mixed ? "mixed-radix" : "Bluestein");
        switch (sh.blue) {
        case 128: return launch_blue<128>(a, sh, F, mode, adj, st);
        case 256: return launch_blue<256>(a, sh, F, mode, adj, st);
        case 512: return launch_blue<512>(a, sh, F, mode, adj, st);
        case 1024: return launch_blue<1024>(a, sh, F, mode, adj, st);
        case 2048: return launch_blue<2048>(a, sh, F, mode, adj, st);
        case 4096: return launch_blue<4096>(a, sh, F, mode, adj, st);
        }
    }
    switch (nkx) {
    case 128: return launch_n<128>(a, sh, F, mode, adj, st);
    case 256: return launch_n<256>(a, sh, F, mode, adj, st);
    case 512: return launch_n<512>(a, sh, F, mode, adj, st);
    case 1024: return launch_n<1024>(a, sh, F, mode, adj, st);
    case 2048: return launch_n<2048>(a, sh, F, mode, adj, st);
    case 4096: return launch_n<4096>(a, sh, F, mode, adj, st);
    }
    return set_error(SWEM_EUNSUPPORTED, "2-D march: nkx=%d", nkx);
}

int angles_supported(int n) { return n >= 2 && (march2d_blue_len(n) || (n >= 128 && n <= 4096 && !(n & (n - 1)))); }

// The tables a launch needs for its transform length are present.
static bool len_tables(const March2DArgs& a, int kind)
{
    return kind == kLenPow2 || (is_mixed(kind) ? a.mr.n == a.nkx : a.chirp && a.bchirp);
}

int launch_angles(int which, const March2DArgs& ax, const March2DArgs& az, const AngleArgs& b, int F, hipStream_t st)
{
    const int n = which == 1 ? az.nkx : ax.nkx;
    const int m = march2d_blue_len(n);
    const int len = m ? m : n, kind = m ? march2d_kind(n) : kLenPow2;
    if (!angles_supported(n) || !len_tables(which == 1 ? az : ax, kind))
        return set_error(SWEM_EUNSUPPORTED, "angles: transform length %d", n);
    if (b.len < 1 || b.nz < 1 || b.nfc < 1 || (which > 0 && (b.inner < 1 || b.lines < 1)) ||
        (which == 2 && b.len != n) || (which == 1 && b.nz != n))
        return set_error(SWEM_EINVAL, "angles: inconsistent launch (len=%d nz=%d n=%d)", b.len, b.nz, n);
    switch (len) {
    case 128: return launch_angles_len<128>(which, kind, ax, az, b, F, st);
    case 256: return launch_angles_len<256>(which, kind, ax, az, b, F, st);
    case 512: return launch_angles_len<512>(which, kind, ax, az, b, F, st);
    case 1024: return launch_angles_len<1024>(which, kind, ax, az, b, F, st);
    case 2048: return launch_angles_len<2048>(which, kind, ax, az, b, F, st);
    case 4096: return launch_angles_len<4096>(which, kind, ax, az, b, F, st);
    }
    return set_error(SWEM_EUNSUPPORTED, "angles: transform length %d", n);
}

int launch_ewem(const March2DArgs& ap, const March2DArgs& as, const EwemArgs& e, int adj, hipStream_t st)
{
    const int n = ap.nkx, m = march2d_blue_len(n), len = m ? m : n, kind = m ? march2d_kind(n) : kLenPow2;
    if (!angles_supported(n) || as.nkx != n || !len_tables(ap, kind) || !len_tables(as, kind) || ap.nshot < 1 ||
        ap.ngroups != ap.nfc || ap.nmx > n)
        return set_error(SWEM_EINVAL, "ewem: inconsistent launch (nkx=%d nmx=%d)", n, ap.nmx);
    switch (len) {
    case 128: return launch_ewem_len<128>(kind, ap, as, e, adj, st);
    case 256: return launch_ewem_len<256>(kind, ap, as, e, adj, st);
    case 512: return launch_ewem_len<512>(kind, ap, as, e, adj, st);
    case 1024: return launch_ewem_len<1024>(kind, ap, as, e, adj, st);
    case 2048: return launch_ewem_len<2048>(kind, ap, as, e, adj, st);
    case 4096: return launch_ewem_len<4096>(kind, ap, as, e, adj, st);
    }
    return set_error(SWEM_EUNSUPPORTED, "ewem: transform length %d", n);
}

}  // namespace swem
