// Mixed-radix FFT engine for lengths without a compile-time specialisation
// (pm_fft_fixed.h): the length and the radix sequence are run-time values,
// the butterflies are compile-time.
//
// A block transforms n lines together, n = blockDim.x, with P = blockDim.y
// threads per line (line index fastest across the lanes, so that lanes that
// read or write one row of a tile touch consecutive words).  Stockham
// autosort stages: a thread takes its butterflies j = p, p + P, ... of radix
// R as a whole into registers (at most kAnyRegs complex words), the block
// synchronises, and the outputs go back to the same line, so a line needs one
// buffer.  The first stage of a transform reads through a loader (global
// memory, or a spectral product of other lines) and the last one writes
// through a storer, so that a line makes nstage - 1 trips through LDS rather
// than nstage + 1.  Radices 2 .. 13: most lengths up to 1000 need
// three stages, against five to eight with prime radices, and every radix is
// one switch case, uniform over the block.
// Twiddles w^k are products of the table's w, w^2, w^4, w^8 (at most three
// factors), loaded per butterfly.
// What bounds it: the vector units.  At length 250 (10, 5, 5) the fused FP32 z
// pass spends about 110 vector instructions per complex element on both
// transforms and the product, 65 of them arithmetic, against 70 with the
// length known at compile time; 120 us at 161 x 200 columns, 1.6 TB/s, where
// the run-time-planned kernels of pm_fft.h (prime radices up to 5, index
// divisions per element, registers spilled) took 1.4 ms.
#pragma once
#include "pm_fft.h"

namespace pmgpu {
namespace any {

constexpr int kAnyStages = 5;
constexpr int kAnyThreads = 1024;  // threads per block at most
constexpr int kAnyMostL = 4096;   // the stages' index arithmetic is 24-bit
// complex words a thread holds in a stage (13: with 16 the butterflies spill),
// and the wavefronts per SIMD that its registers are held to
constexpr int kAnyRegs = 13;
constexpr int any_waves(int word) { return word == 8 ? 5 : 4; }

struct AnyStage {
  int R, nbf;      // radix; butterflies of the line, L / R
  int Ns, ts;      // sub-transform length before the stage; L / (Ns R)
  uint32_t magic;  // floor(2^24 / Ns) + 1: j / Ns = (j magic) >> 24, exact for j Ns < 2^24
};
// The stages are separate members: an array of them, indexed at run time,
// would be copied to every thread's scratch.
struct AnyPlan {
  int L, n;        // length, stages (n = 1: `last` alone)
  int tw_off;      // offset of the length-L table
  AnyStage first, m1, m2, m3, last;
};
// LDS line stride in complex words (odd: neighbouring lines start on
// different banks)
__host__ __device__ inline int any_stride(int L) { return L | 1; }

// ------------------------------------------------------ composite butterflies
// cos / sin (2 pi k / R) of the odd radices
template <int R> struct Roots;
template <> struct Roots<7> {
  static constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
  static constexpr double s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};
template <> struct Roots<11> {
  static constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                  -0.65486073394528506406, -0.95949297361449738989};
  static constexpr double s[6] = {0.0, 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                  0.75574957435425828377, 0.28173255684142969771};
};
template <> struct Roots<13> {
  static constexpr double c[7] = {1.0, 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                  -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
  static constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                  0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};

template <int R, int S, typename V> struct DftC {
  static __device__ __forceinline__ void run(V *v) { Dft<R, S, V>::run(v); }
};
// odd prime radix: X_m = x_0 + sum_k c_{mk} (x_k + x_{R-k}) + S i sum_k s_{mk} (x_k - x_{R-k})
template <int R, int S, typename V> __device__ __forceinline__ void dft_odd(V *v) {
  using T = decltype(V::x);
  constexpr int H = (R - 1) / 2;
  V a[H], b[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    a[k] = cadd(v[k + 1], v[R - 1 - k]);
    b[k] = csub(v[k + 1], v[R - 1 - k]);
  }
  const V x0 = v[0];
#pragma unroll
  for (int k = 0; k < H; ++k) v[0] = cadd(v[0], a[k]);
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    V r = x0, q = cmake<V>(0, 0);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      const int e = (m * k) % R;
      const T c = (T)Roots<R>::c[e <= H ? e : R - e], s = (T)(e <= H ? Roots<R>::s[e] : -Roots<R>::s[R - e]);
      r = cadd(r, cscale(a[k - 1], c));
      q = cadd(q, cscale(b[k - 1], s));
    }
    q = cmul_i<S>(q);
    v[m] = cadd(r, q);
    v[R - m] = csub(r, q);
  }
}
template <int S, typename V> struct DftC<7, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_odd<7, S>(v); }
};
template <int S, typename V> struct DftC<11, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_odd<11, S>(v); }
};
template <int S, typename V> struct DftC<13, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_odd<13, S>(v); }
};
// coprime factors A B = R (no twiddles): input A-index a, B-index b is
// x[(a B + b A) mod R], output (c, d) is X[(c B (B^-1 mod A) + d A (A^-1 mod B)) mod R]
constexpr int inv_mod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if ((a * x) % m == 1) return x;
  return 1;
}
template <int A, int B, int S, typename V> __device__ __forceinline__ void dft_pfa(V *v) {
  constexpr int R = A * B;
  V t[B][A];
#pragma unroll
  for (int b = 0; b < B; ++b) {
#pragma unroll
    for (int a = 0; a < A; ++a) t[b][a] = v[(a * B + b * A) % R];
    Dft<A, S, V>::run(t[b]);
  }
#pragma unroll
  for (int c = 0; c < A; ++c) {
    V u[B];
#pragma unroll
    for (int b = 0; b < B; ++b) u[b] = t[b][c];
    Dft<B, S, V>::run(u);
#pragma unroll
    for (int d = 0; d < B; ++d) v[(c * B * inv_mod(B % A, A) + d * A * inv_mod(A % B, B)) % R] = u[d];
  }
}
template <int S, typename V> struct DftC<6, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_pfa<2, 3, S>(v); }
};
template <int S, typename V> struct DftC<10, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_pfa<2, 5, S>(v); }
};
template <int S, typename V> struct DftC<12, S, V> {
  static __device__ __forceinline__ void run(V *v) { dft_pfa<4, 3, S>(v); }
};
// A A = R: two passes with the constant twiddles exp(S 2 pi i b c / R)
template <int S, typename V> struct DftC<9, S, V> {
  static __device__ __forceinline__ void run(V *v) {
    using T = decltype(V::x);
    constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
    constexpr double s[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                             0.34202014332566873304};
    V t[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
#pragma unroll
      for (int a = 0; a < 3; ++a) t[b][a] = v[3 * a + b];
      Dft<3, S, V>::run(t[b]);
#pragma unroll
      for (int k = 1; k < 3; ++k)
        if (b > 0) t[b][k] = cmul(t[b][k], cmake<V>((T)c[b * k], (T)(S * s[b * k])));
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      V u[3] = {t[0][k], t[1][k], t[2][k]};
      Dft<3, S, V>::run(u);
#pragma unroll
      for (int d = 0; d < 3; ++d) v[k + 3 * d] = u[d];
    }
  }
};
// ------------------------------------------------------------------- stages
// butterflies of a radix that a thread takes at most
constexpr int any_mb(int R) { return kAnyRegs / R; }
// j / Ns with the full-rate 24-bit multiplier
__device__ __forceinline__ int any_div(int j, uint32_t magic) {
  return (int)(((uint64_t)((uint32_t)(j << 8) & 0xFFFFFFu) * (uint64_t)(magic & 0xFFFFFFu)) >> 32);
}

// v[r] *= w^r, w = tw[t] (conjugated for S > 0): the powers of two from the
// table, the others as products of them
template <int R, int S, typename V> __device__ __forceinline__ void twiddle_any(V *v, const V *tw, int t) {
  V w[R];
#pragma unroll
  for (int r = 1; r < R; ++r) {
    if ((r & (r - 1)) == 0) {
      w[r] = tw[r * t];
      if (S > 0) w[r].y = -w[r].y;
    } else {
      const int hi = r >= 8 ? 8 : (r >= 4 ? 4 : 2);
      w[r] = cmul(w[hi], w[r - hi]);
    }
    v[r] = cmul(v[r], w[r]);
  }
}

// one stage of radix R; SYNC: the loader reads lines that the storer writes.
// ld.at(j) / st.at(n, step) give an accessor of the elements j + r nbf / n +
// r step, so that the address of a butterfly is formed once.  A thread past
// the line's P threads passes p >= nbf and only synchronises.
template <int R, int S, bool SYNC, typename V, typename LD, typename ST>
__device__ __forceinline__ void stage_any(const AnyStage &s, int p, int P, const V *tw, const LD &ld, const ST &st) {
  constexpr int MB = any_mb(R);
  V v[MB][R];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j = p + m * P;
    if (j < s.nbf) {
      auto q = ld.at(j, s.nbf);
#pragma unroll
      for (int r = 0; r < R; ++r) v[m][r] = q(r);
    }
  }
  if (SYNC) __syncthreads();
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j = p + m * P;
    if (j < s.nbf) {
      int k = 0;
      if (s.Ns > 1) {
        k = j - (int)__umul24(any_div(j, s.magic), s.Ns);
        twiddle_any<R, S>(v[m], tw, (int)__umul24(k, s.ts));
      }
      DftC<R, S, V>::run(v[m]);
      auto q = st.at((j - k) * R + k, s.Ns);
#pragma unroll
      for (int r = 0; r < R; ++r) q(r, v[m][r]);
    }
  }
}
template <int S, bool SYNC, typename V, typename LD, typename ST>
__device__ __forceinline__ void stage_switch(const AnyStage &s, int p, int P, const V *tw, const LD &ld,
                                             const ST &st) {
  switch (s.R) {
    case 2: stage_any<2, S, SYNC>(s, p, P, tw, ld, st); break;
    case 3: stage_any<3, S, SYNC>(s, p, P, tw, ld, st); break;
    case 4: stage_any<4, S, SYNC>(s, p, P, tw, ld, st); break;
    case 5: stage_any<5, S, SYNC>(s, p, P, tw, ld, st); break;
    case 6: stage_any<6, S, SYNC>(s, p, P, tw, ld, st); break;
    case 7: stage_any<7, S, SYNC>(s, p, P, tw, ld, st); break;
    case 8: stage_any<8, S, SYNC>(s, p, P, tw, ld, st); break;
    case 9: stage_any<9, S, SYNC>(s, p, P, tw, ld, st); break;
    case 10: stage_any<10, S, SYNC>(s, p, P, tw, ld, st); break;
    case 11: stage_any<11, S, SYNC>(s, p, P, tw, ld, st); break;
    case 12: stage_any<12, S, SYNC>(s, p, P, tw, ld, st); break;
    default: stage_any<13, S, SYNC>(s, p, P, tw, ld, st); break;
  }
}

// a line in LDS as loader and as storer
template <typename V> struct LineIn {
  const V *line;
  __device__ __forceinline__ auto at(int j, int step) const {
    const V *q = line + j;
    return [q, step](int r) { return q[r * step]; };
  }
};
template <typename V> struct LineOut {
  V *line;
  __device__ __forceinline__ auto at(int n, int step) const {
    V *q = line + n;
    return [q, step](int r, const V &v) { q[r * step] = v; };
  }
};
// rows < lim of one column in global memory, through one buffer resource per
// r: its base is moved to row r step (scalar arithmetic), so that a thread has
// one 32-bit offset for the whole butterfly; a row past the resource's end
// reads as zero by its own bounds check, without a branch, and so does every
// row of a column that is off (kOffColumn).  The host keeps the bytes of step
// rows within kMostRecords (any_rows_ok), which `most` rows do not pass.
constexpr uint32_t kMostRecords = 0xFFFFF000u, kOffColumn = 0xFFFFFF00u;
__device__ __forceinline__ float2 rows_load(__amdgpu_buffer_rsrc_t r, uint32_t off, float2) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
__device__ __forceinline__ double2 rows_load(__amdgpu_buffer_rsrc_t r, uint32_t off, double2) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
template <typename V> struct RowsIn {
  const V *base;   // first row of the block's columns (uniform)
  int64_t rsb;     // bytes per row (its words past the thread's column are not read)
  int lim, most;   // rows; rows that one resource covers
  uint32_t off;    // the thread's column, in bytes, or kOffColumn
  __device__ __forceinline__ auto at(int j, int step) const {
    const uint32_t o = off == kOffColumn ? kOffColumn : off + (uint32_t)j * (uint32_t)rsb;
    const int64_t sb = step * rsb, b = rsb;
    const int l = lim, t = step, k = most;
    const char *p = reinterpret_cast<const char *>(base);
    return [p, sb, b, l, t, k, o](int r) {
      const int rows = min(max(l - r * t, 0), k);
      const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char *>(p + r * sb), (short)0, (int)((uint32_t)rows * (uint32_t)b), 0x00020000);
      return rows_load(rr, o, V{});
    };
  }
};
// rows < lim of one column in global memory, scaled, as the last stage writes
// them (rows n + r step, n < step: whole steps are decided for the block)
template <typename V> struct RowsOut {
  V *base;
  int64_t rs;
  int lim;
  bool on;   // false: the column is off
  decltype(V::x) sc;
  __device__ __forceinline__ auto at(int n, int step) const {
    V *q = base + (int64_t)n * rs;
    const int64_t s = step * rs;
    const int l = lim;
    const bool g = on;
    const auto c = sc;
    return [q, s, n, step, l, g, c](int r, const V &v) {
      if (r * step >= l) return;
      if (g && ((r + 1) * step <= l || n + r * step < l)) q[r * s] = cscale(v, c);
    };
  }
};

// Transform of one line: first stage through ld, last through st, the stages
// between in `line`.  LSYNC: ld reads lines in LDS that this transform
// overwrites.  Every thread of the block calls it; on return the stores of
// the last stage are not yet synchronised.  One-stage plans go from ld to st.
template <int S, bool LSYNC, typename V, typename LD, typename ST>
__device__ __forceinline__ void fft_any(const AnyPlan &pl, V *line, int p, int P, const V *tw_all, const LD &ld,
                                        const ST &st) {
  const V *tw = tw_all + pl.tw_off;
  if (pl.n == 1) {
    stage_switch<S, true>(pl.last, p, P, tw, ld, st);
    return;
  }
  stage_switch<S, LSYNC>(pl.first, p, P, tw, ld, LineOut<V>{line});
  __syncthreads();
#pragma unroll 1
  for (int i = 1; i + 1 < pl.n; ++i) {
    const AnyStage m = i == 1 ? pl.m1 : (i == 2 ? pl.m2 : pl.m3);
    stage_switch<S, true>(m, p, P, tw, LineIn<V>{line}, LineOut<V>{line});
    __syncthreads();
  }
  stage_switch<S, true>(pl.last, p, P, tw, LineIn<V>{line}, st);
}

}  // namespace any
}  // namespace pmgpu
