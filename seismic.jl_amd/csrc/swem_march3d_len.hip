// swem_march3d_len.hip -- the 3-D march and elastic kernels of one transform array length (SWEM_LEN, a
// power of two 128..1024), every length kind: one object per length, compiled in parallel.
#include "swem_march3d.hpp"

namespace swem {

#define SWEM_KIND(K)                                                                                               \
    template int launch_ewem3d_n<SWEM_LEN, K>(int, const March3DArgs&, const March3DArgs&, const Ewem3DArgs&, int, \
                                              int, hipStream_t);                                                   \
    template int launch3_n<SWEM_LEN, K>(int, const March3DArgs&, int, int, hipStream_t);
SWEM_KIND(kLenPow2)
SWEM_KIND(kLenMixed)
#if SWEM_LEN <= 512
SWEM_KIND(kLenMixedPrime)
#endif
SWEM_KIND(kLenBluestein)
#undef SWEM_KIND

}  // namespace swem
