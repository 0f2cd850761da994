// Run-time-length strided passes.
#include "poisson_any_launch.h"

namespace pmgpu {
template int any_strided<float>(int, StridedArgs, const AnyPlan &, int, int, const float2 *, hipStream_t);
template int any_strided<double>(int, StridedArgs, const AnyPlan &, int, int, const double2 *, hipStream_t);
}  // namespace pmgpu
