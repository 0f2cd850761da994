// Run-time-length inverse x passes.
#include "poisson_any_launch.h"

namespace pmgpu {
template int any_xinv<float>(XInvArgs, const AnyPlan &, const float2 *, hipStream_t);
template int any_xinv<double>(XInvArgs, const AnyPlan &, const double2 *, hipStream_t);
}  // namespace pmgpu
