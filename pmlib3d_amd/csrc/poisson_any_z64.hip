// Run-time-length z passes, FP64.
#include "poisson_any_launch.h"

namespace pmgpu {
template int any_z<double>(ZArgs, const AnyPlan &, int, const double2 *, hipStream_t);
}  // namespace pmgpu
