// Run-time-length z passes, FP32.
#include "poisson_any_launch.h"

namespace pmgpu {
template int any_z<float>(ZArgs, const AnyPlan &, int, const float2 *, hipStream_t);
}  // namespace pmgpu
