// swem_march2d_len.hip -- the 2-D march, angle and elastic kernels of one transform array length
// (SWEM_LEN, a power of two 128..4096): one object per length, compiled in parallel.
#include "swem_march2d.hpp"

namespace swem {

template int launch_n<SWEM_LEN>(const March2DArgs&, const March2DShape&, int, int, int, hipStream_t);
template int launch_blue<SWEM_LEN>(const March2DArgs&, const March2DShape&, int, int, int, hipStream_t);
template int launch_angles_len<SWEM_LEN>(int, int, const March2DArgs&, const March2DArgs&, const AngleArgs&, int, hipStream_t);
template int launch_ewem_len<SWEM_LEN>(int, const March2DArgs&, const March2DArgs&, const EwemArgs&, int, hipStream_t);

}  // namespace swem
