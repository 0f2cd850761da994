// Run-time-length forward x passes.
#include "poisson_any_launch.h"

namespace pmgpu {
template int any_xfwd<float>(XFwdArgs, const AnyPlan &, const float2 *, hipStream_t);
template int any_xfwd<double>(XFwdArgs, const AnyPlan &, const double2 *, hipStream_t);
}  // namespace pmgpu
