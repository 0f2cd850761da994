// Plans of the run-time-length Poisson passes (poisson_any.h).
#include <algorithm>
#include <cstdlib>

#include "poisson_any_ops.h"

namespace pmgpu {
namespace any {

// Radices and the cost of one butterfly (real operations without twiddles).
struct RadixCost {
  int R, ops;
};
static const RadixCost kRadices[] = {{13, 300}, {12, 108}, {11, 216}, {10, 108}, {9, 96}, {8, 60},
                                     {7, 88},   {6, 44},   {5, 44},   {4, 16},   {3, 16},   {2, 4}};
static int radix_ops(int R) {
  for (const RadixCost &c : kRadices)
    if (c.R == R) return c.ops;
  return 0;
}

// Vector instructions of one butterfly of stage i: the transform, its
// twiddles, and per element the addresses and accesses of two trips (LDS or
// memory).
static double stage_ops(int R, int i) { return radix_ops(R) + (i > 0 ? 7.0 * (R - 1) : 0.0) + 6.0 * R; }

// barrier, LDS latency and twiddle address of a stage, in the same unit
constexpr double kStageOps = 60.0;

struct Search {
  int L, n = 0, best_n = 0;
  int R[kAnyStages], best[kAnyStages];
  double cost = 1e300;
  void leaf() {
    // the best thread count's instructions, idle threads of a stage included,
    // and the stage's barrier and LDS latency
    double c = 1e300;
    for (int i = 0; i < n; ++i)
      for (int m = 1; m <= any_mb(R[i]); ++m) {
        const int P = (L / R[i] + m - 1) / m;
        double cp = 0.0;
        for (int k = 0; k < n && cp >= 0.0; ++k) {
          const int mb = (L / R[k] + P - 1) / P;
          cp = mb > any_mb(R[k]) ? -1.0 : cp + P * (mb * stage_ops(R[k], k) + kStageOps);
        }
        if (cp >= 0.0 && cp < c) c = cp;
      }
    if (c < cost) {
      cost = c;
      best_n = n;
      std::copy(R, R + n, best);
    }
  }
  void go(int left, size_t from) {
    if (left == 1) {
      if (n > 0) leaf();
      return;
    }
    if (n == kAnyStages) return;
    for (size_t k = from; k < sizeof(kRadices) / sizeof(kRadices[0]); ++k)
      if (left % kRadices[k].R == 0) {
        R[n++] = kRadices[k].R;
        go(left / kRadices[k].R, k);
        --n;
      }
  }
};

// wave-instructions of a block of `lines` lines with P threads each (idle
// lanes and idle threads of a stage count); negative when a stage does not
// fit the threads' registers
static double block_cost(const AnyPlan &pl, int lines, int P) {
  const int waves = (lines * P + 63) / 64;
  double c = 0.0;
  const AnyStage *s[kAnyStages] = {&pl.first, &pl.m1, &pl.m2, &pl.m3, &pl.last};
  int i = 0;
  for (const AnyStage *t : s) {
    if (t->R == 0) continue;
    const int mb = (t->nbf + P - 1) / P;
    if (mb > any_mb(t->R)) return -1.0;
    c += mb * stage_ops(t->R, i++) + kStageOps;
  }
  return c * waves;
}

}  // namespace any

using namespace any;

// The cheapest factorisation into at most kAnyStages radices; pl.L = 0 when
// there is none (a prime factor above 13, or L > kAnyMostL).
void make_any_plan(int L, int tw_off, AnyPlan &pl) {
  pl = AnyPlan{};
  Search s;
  s.L = L;
  if (L > 1 && L <= kAnyMostL) s.go(L, 0);
  if (s.best_n == 0) return;
  pl.L = L;
  pl.n = s.best_n;
  pl.tw_off = tw_off;
  AnyStage *t[kAnyStages] = {&pl.first, &pl.m1, &pl.m2, &pl.m3, &pl.last};
  int Ns = 1;
  for (int i = 0; i < pl.n; ++i) {
    AnyStage &q = i + 1 == pl.n ? pl.last : *t[i];
    q.R = s.best[i];
    q.nbf = L / q.R;
    q.Ns = Ns;
    q.ts = L / (Ns * q.R);
    q.magic = Ns > 1 ? ((1u << 24) / (uint32_t)Ns) + 1 : 0u;
    Ns *= q.R;
  }
}

// Units of `lines` lines per block (at most `most`) and threads per line, a
// unit's LDS being `lines` strides of `word`-byte words: the cheapest block
// per unit.  `aligned`: `most` units are a row of whole cache lines, and fewer
// are taken only where they do not fit (half the LDS of a CU, kAnyThreads).
// Otherwise narrow rows pay a few per cent (a partial cache line each), and a
// block pays for the wavefront slots that it leaves empty: past four
// wavefronts a number that is no multiple of the four SIMDs, or blocks (by
// LDS and registers) that do not fill the CU (length 250 FP64, 25 threads a
// line: 225 threads 224 us, 300 292, 375 265, 450 227; length 252, 36 threads:
// 216 threads 260 us, 324 331, 648 335).  Returns false when not even one
// unit fits.
bool any_fit(const AnyPlan &pl, int most, int lines, int word, bool aligned, AnyFit &f) {
  f = AnyFit{};
  if (pl.L == 0) return false;
  const size_t unit = (size_t)lines * any_stride(pl.L) * word, cu = 160 * 1024;
  const int slots = word == 8 ? 24 : 16;   // resident wavefronts of a CU by registers (77 and 127)
  double best = 1e300;
  const AnyStage *s[kAnyStages] = {&pl.first, &pl.m1, &pl.m2, &pl.m3, &pl.last};
  for (int T = most; T >= 1; T = aligned ? T / 2 : T - 1) {
    if ((T > 1 && T * unit > cu / 2) || T * unit > (size_t)kAnyLds) continue;
    if (aligned && f.T > 0) break;
    for (const AnyStage *t : s)
      for (int m = 1; t->R && m <= any_mb(t->R); ++m) {
        const int P = (t->nbf + m - 1) / m;
        if (T * lines * P > kAnyThreads) continue;
        double c = block_cost(pl, T * lines, P);
        if (c < 0.0) continue;
        const int waves = (T * lines * P + 63) / 64;
        const int fit = (int)std::min<size_t>(cu / (T * unit), (size_t)std::max(1, slots / waves));
        const double round = waves <= 4 ? 1.0 : (double)((waves + 3) / 4 * 4) / waves;
        c *= std::max(round, (double)slots / (fit * waves)) * (1.0 + 4.0 / (T * lines * word)) / T;
        if (c < best) {
          best = c;
          f.T = T;
          f.P = P;
          f.lds = T * unit;
        }
      }
  }
  return f.T > 0;
}

}  // namespace pmgpu
