// plane32.hip -- FP32 instances of the plane-per-lane operator kernel.
#include "plane_kernel.hpp"

namespace mfx {

template bool plane_instance<float>(int, int, bool, bool);
template void launch_plane<float>(const PlaneOp<float> &, const float *, float *, bool, hipStream_t,
                                  double *, const int *);

}  // namespace mfx
