// Launchers of the run-time-length Poisson passes.  Each returns 1 when it
// launched, 0 when a line does not fit a block (the caller then uses the
// kernels of poisson_kernels.h), -1 on an error.  Included by the
// poisson_any_*.hip units, which instantiate them (they compile in parallel).
#pragma once
#include "poisson_any.h"
#include "poisson_any_ops.h"

namespace pmgpu {

using namespace any;

// the rows of one step of the first stage within a 32-bit byte offset
static inline bool any_rows_ok(const AnyPlan &pl, int64_t rsb) {
  const int nbf = pl.n > 1 ? pl.first.nbf : pl.last.nbf;
  return (double)(nbf + 1) * (double)rsb < (double)kMostRecords;
}

template <typename R>
int any_strided(int S, StridedArgs a, const AnyPlan &pl, int nb_y, int nb_z, const cplx_t<R> *tw, hipStream_t st) {
  AnyFit f;
  if (!any_rows_ok(pl, a.rs_in * (int64_t)sizeof(cplx_t<R>))) return 0;
  if (!any_fit(pl, sizeof(R) == 4 ? 16 : 8, 1, sizeof(cplx_t<R>), true, f)) return 0;
  const dim3 grid((a.ncols + f.T - 1) / f.T, nb_y, nb_z), block(f.T, f.P);
  if (S < 0)
    hipLaunchKernelGGL((k_strided_a<R, -1>), grid, block, f.lds, st, a, pl, tw);
  else
    hipLaunchKernelGGL((k_strided_a<R, 1>), grid, block, f.lds, st, a, pl, tw);
  return hipGetLastError() == hipSuccess ? 1 : -1;
}
template <typename R> int any_xfwd(XFwdArgs a, const AnyPlan &pl, const cplx_t<R> *tw, hipStream_t st) {
  AnyFit f;
  if (!any_fit(pl, 4, a.ncomp, sizeof(cplx_t<R>), false, f)) return 0;
  hipLaunchKernelGGL(k_x_fwd_a<R>, dim3((a.My + f.T - 1) / f.T, a.Mz), dim3(a.ncomp, f.P, f.T), f.lds, st, a, pl, tw);
  return hipGetLastError() == hipSuccess ? 1 : -1;
}
template <typename R> int any_xinv(XInvArgs a, const AnyPlan &pl, const cplx_t<R> *tw, hipStream_t st) {
  AnyFit f;
  if (!any_fit(pl, 4, a.ncomp, sizeof(cplx_t<R>), false, f)) return 0;
  hipLaunchKernelGGL(k_x_inv_a<R>, dim3((a.My + f.T - 1) / f.T, a.Mz), dim3(a.ncomp, f.P, f.T), f.lds, st, a, pl, tw);
  return hipGetLastError() == hipSuccess ? 1 : -1;
}
// one launch per field, the velocity, in place, last: a launch of its own
// transforms forward again, but keeps one set of lines in LDS and a field's
// registers (all fields in one kernel: 1157 against 700 us at 160 x 100 x 125)
template <typename R> int any_z(ZArgs a, const AnyPlan &pl, int Ly, const cplx_t<R> *tw, hipStream_t st) {
  AnyFit f;
  if (!any_rows_ok(pl, a.rs * (int64_t)sizeof(cplx_t<R>))) return 0;
  if (!any_fit(pl, 8, 3, sizeof(cplx_t<R>), false, f)) return 0;
  const dim3 grid((a.Hx + f.T - 1) / f.T, Ly), block(3 * f.T, f.P);
  if (a.want_psi) hipLaunchKernelGGL(k_z3_a<R>, grid, block, f.lds, st, a, pl, tw, 1, a.Bpsi);
  if (a.want_vort) hipLaunchKernelGGL(k_z3_a<R>, grid, block, f.lds, st, a, pl, tw, 2, a.Bvort);
  hipLaunchKernelGGL(k_z3_a<R>, grid, block, f.lds, st, a, pl, tw, 0, a.B);
  return hipGetLastError() == hipSuccess ? 1 : -1;
}

}  // namespace pmgpu
