// Entry points of the run-time-length Poisson passes (poisson_any.hip).
#pragma once
#include "pm_fft_any.h"
#include "poisson_kernels.h"

namespace pmgpu {

void make_any_plan(int L, int tw_off, any::AnyPlan &pl);
// block shape of a pass: units (rows, columns) per block, threads per line, LDS bytes
struct AnyFit {
  int T = 0, P = 0;
  size_t lds = 0;
};
constexpr int kAnyLds = 160 * 1024;
bool any_fit(const any::AnyPlan &pl, int most, int lines, int word, bool aligned, AnyFit &f);
template <typename R>
int any_strided(int S, StridedArgs a, const any::AnyPlan &pl, int nb_y, int nb_z, const cplx_t<R> *tw,
                hipStream_t st);
template <typename R> int any_xfwd(XFwdArgs a, const any::AnyPlan &pl, const cplx_t<R> *tw, hipStream_t st);
template <typename R> int any_xinv(XInvArgs a, const any::AnyPlan &pl, const cplx_t<R> *tw, hipStream_t st);
template <typename R> int any_z(ZArgs a, const any::AnyPlan &pl, int Ly, const cplx_t<R> *tw, hipStream_t st);

}  // namespace pmgpu
