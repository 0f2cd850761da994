// Multiresolution coupling on one rank (HIP, gfx950): the parent topology of
// a refinement patch and the mesh-to-mesh interpolation between a patch and
// its parent, both directions, M'4 and M6*
// (interpolation/pmlib_interp_mesh_mesh.f:5-2078,
// topology/pmlib_topology_parent.f:5-100).
//
// Patch -> parent (the source is finer, reldx = dx_from / dx_to < 1) is a
// deposit in the reference: every source cell, ghosts included, spreads
// reldx W_x W_y W_z of its value over the target stencil; parent -> patch
// gathers W_x W_y W_z-weighted source values per target cell.  Both are
// tensor products of per-axis operators, so the default form sums one axis
// after the other, tile by tile in one kernel (no atomics).  The bit-identical forms (PMGPU_M2M_EXACT=1) keep the
// reference's term order: the deposit as a gather in which each target cell
// sums the terms of the source cells whose stencils cover it in the
// reference's source-cell order (k, j, i ascending), a block of 64 target
// cells of one (y, z) row staging the per-axis bases and weights it needs in
// LDS; the interpolation per target cell in the reference's term order.
// Compiled without multiply-add contraction.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "../../include/pmgpu.h"
// (the particle kernels of the header that this file does not launch)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wunused-function"
#include "particles_kernels.h"
#pragma clang diagnostic pop

namespace pmgpu {
namespace {

struct MGeom {
  int ncell[3], ng[3], E[3], bc[3];
  double xmin[3], xmax[3], dx[3], c1dx[3];
};

int make_mgeom(const pmgpu_geom *g, MGeom &m, const char *who) {
  PM_CHECK(g->interp_order == 3 || g->interp_order == 4,
           std::string(who) + ": interp_order must be 3 (M'4) or 4 (M6*)");
  for (int d = 0; d < 3; ++d) {
    PM_CHECK(g->ncell[d] > 0 && g->dx[d] > 0 && (g->bound_cond[d] == 0 || g->bound_cond[d] == 1),
             std::string(who) + ": bad geometry");
    m.ncell[d] = g->ncell[d];
    m.bc[d] = g->bound_cond[d];
    m.ng[d] = g->bound_cond[d] == 0 ? g->nghost : (g->interp_order == 4 ? 3 : 2);
    PM_CHECK(m.ng[d] >= 0, std::string(who) + ": negative ghost count");
    m.E[d] = m.ncell[d] + 2 * m.ng[d];
    m.xmin[d] = g->xmin[d];
    m.xmax[d] = g->xmax[d];
    m.dx[d] = g->dx[d];
    m.c1dx[d] = 1.0 / g->dx[d];
  }
  return 0;
}

constexpr int kTX = 64;       // target cells per deposit block along x
constexpr int kMaxRatio = 8;  // finest-to-coarsest cell ratio the deposit stages
// source candidates staged per block: x covers kTX + NS target bases at up to
// kMaxRatio source cells each, y and z one row's NS bases, plus margins
template <int NS> constexpr int cap_x() { return (kTX + NS + 2) * kMaxRatio + 8; }
template <int NS> constexpr int cap_yz() { return (NS + 2) * kMaxRatio + 8; }

// Conservative range of source indices (1-ng .. N+ng numbering) whose base
// index NINT((p - xmin_t) / dx_t) may fall in [blo, bhi]; the exact test is
// made on the staged bases.
__device__ __forceinline__ void src_range(const MGeom &f, const MGeom &t, int d, int blo, int bhi, int &ilo,
                                          int &ihi) {
  const double a = (t.xmin[d] - f.xmin[d] + ((double)blo - 1.0) * t.dx[d]) / f.dx[d];
  const double b = (t.xmin[d] - f.xmin[d] + ((double)bhi + 1.0) * t.dx[d]) / f.dx[d];
  ilo = (int)floor(a) - 1;
  ihi = (int)ceil(b) + 2;
  if (ilo < 1 - f.ng[d]) ilo = 1 - f.ng[d];
  if (ihi > f.ncell[d] + f.ng[d]) ihi = f.ncell[d] + f.ng[d];
}

// Base index, live flag and the NS weights reldx W_s of source index i on
// axis d (:93-158 (M'4), :520-640 (M6*)): the cell centre x_i, its target
// base b = NINT((x_i - xmin_t) / dx_t), the normalised offset and the kernel
// weights, rounded step by step as the reference evaluates them.  On a
// periodic target axis a source cell outside [xmin_t, xmax_t] deposits
// nothing (:174-195).
template <int NS>
__device__ __forceinline__ void stage_src(const MGeom &f, const MGeom &t, int d, int i, double reldx, int &b,
                                          unsigned char &live, double *w) {
  const double p = __dadd_rn(f.xmin[d], __dmul_rn(__dadd_rn((double)(i - 1), 0.5), f.dx[d]));
  b = cell_index(p, t.xmin[d], t.c1dx[d]);
  live = !(t.bc[d] != 0 && (p < t.xmin[d] || p > t.xmax[d]));
  const double dd = stencil_offset(p, t.xmin[d], t.dx[d], b, t.c1dx[d]);
#pragma unroll
  for (int s = 0; s < NS; ++s) w[s] = __dmul_rn(reldx, weight(NS == 6, s, dd));
}

// first staged entry with base >= v (bases are non-decreasing in i)
__device__ __forceinline__ int lower_bound_b(const int *bs, int n, int v) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (bs[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

struct DepArgs {
  MGeom f, t;
  double reldx;
  int clear;
};

// Patch -> parent: grid (ceil(Ex_t / kTX), Ey_t, Ez_t), kTX threads.
template <typename T, int NS>
__global__ void __launch_bounds__(kTX) k_m2m_deposit(const T *__restrict__ from, T *__restrict__ to, DepArgs a) {
  constexpr int off = NS == 6 ? 2 : 1;
  constexpr int CX = cap_x<NS>(), CY = cap_yz<NS>();
  __shared__ int xb[CX], yb[CY], zb[CY];
  __shared__ unsigned char xl[CX], yl[CY], zl[CY];
  __shared__ double xw[CX][NS], yw[CY][NS], zw[CY][NS];
  const MGeom &f = a.f, &t = a.t;
  // target indices in the reference's numbering (1 - ng .. N + ng)
  const int tx0 = (int)blockIdx.x * kTX + 1 - t.ng[0];
  const int txe = min(tx0 + kTX - 1, t.ncell[0] + t.ng[0]);
  const int ty = (int)blockIdx.y + 1 - t.ng[1], tz = (int)blockIdx.z + 1 - t.ng[2];
  // a source cell of base b covers target indices b - off .. b - off + NS - 1
  int ix0, ix1, iy0, iy1, iz0, iz1;
  src_range(f, t, 0, tx0 + off - NS + 1, txe + off, ix0, ix1);
  src_range(f, t, 1, ty + off - NS + 1, ty + off, iy0, iy1);
  src_range(f, t, 2, tz + off - NS + 1, tz + off, iz0, iz1);
  // (the host admits cell ratios up to kMaxRatio, for which the ranges fit
  // the staging arrays; the bounds are enforced here all the same)
  const int nx = min(ix1 - ix0 + 1, CX), ny = min(iy1 - iy0 + 1, CY), nz = min(iz1 - iz0 + 1, CY);
  for (int q = threadIdx.x; q < nx; q += blockDim.x) stage_src<NS>(f, t, 0, ix0 + q, a.reldx, xb[q], xl[q], xw[q]);
  for (int q = threadIdx.x; q < ny; q += blockDim.x) stage_src<NS>(f, t, 1, iy0 + q, a.reldx, yb[q], yl[q], yw[q]);
  for (int q = threadIdx.x; q < nz; q += blockDim.x) stage_src<NS>(f, t, 2, iz0 + q, a.reldx, zb[q], zl[q], zw[q]);
  __syncthreads();
  const int tx = tx0 + (int)threadIdx.x;
  if (tx > txe) return;
  // the staged entries whose stencil covers this target cell, per axis
  const int qx0 = lower_bound_b(xb, nx, tx + off - NS + 1), qx1 = lower_bound_b(xb, nx, tx + off + 1);
  const int qy0 = lower_bound_b(yb, ny, ty + off - NS + 1), qy1 = lower_bound_b(yb, ny, ty + off + 1);
  const int qz0 = lower_bound_b(zb, nz, tz + off - NS + 1), qz1 = lower_bound_b(zb, nz, tz + off + 1);
  const int64_t fsx = 3, fsy = 3 * (int64_t)f.E[0], fsz = fsy * f.E[1];
  const int64_t o = 3 * ((int64_t)(tx - 1 + t.ng[0]) +
                         (int64_t)t.E[0] * ((int64_t)(ty - 1 + t.ng[1]) + (int64_t)t.E[1] * (tz - 1 + t.ng[2])));
  double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
  if (!a.clear) {
    acc0 = (double)to[o];
    acc1 = (double)to[o + 1];
    acc2 = (double)to[o + 2];
  }
  for (int qz = qz0; qz < qz1; ++qz) {
    if (!zl[qz]) continue;
    const double wz = zw[qz][tz - zb[qz] + off];
    const int64_t oz = (int64_t)(iz0 + qz - 1 + f.ng[2]) * fsz;
    for (int qy = qy0; qy < qy1; ++qy) {
      if (!yl[qy]) continue;
      const double wy = yw[qy][ty - yb[qy] + off];
      const int64_t oy = oz + (int64_t)(iy0 + qy - 1 + f.ng[1]) * fsy;
      for (int qx = qx0; qx < qx1; ++qx) {
        if (!xl[qx]) continue;
        const double wx = xw[qx][tx - xb[qx] + off];
        const double ww = __dmul_rn(__dmul_rn(wx, wy), wz);
        const T *m = from + oy + (int64_t)(ix0 + qx - 1 + f.ng[0]) * fsx;
        acc0 = __dadd_rn(acc0, __dmul_rn(ww, (double)m[0]));
        acc1 = __dadd_rn(acc1, __dmul_rn(ww, (double)m[1]));
        acc2 = __dadd_rn(acc2, __dmul_rn(ww, (double)m[2]));
      }
    }
  }
  to[o] = (T)acc0;
  to[o + 1] = (T)acc1;
  to[o + 2] = (T)acc2;
}

// Parent -> patch (:1395-2062): every target cell (interior cells only on
// periodic axes) adds sum ((W_x W_y) W_z) m over the source stencil, the
// terms in i-fastest order, stencil indices outside the source mesh clamped
// to its last layer with weight 0.  clear writes 0 to the cells it skips.
template <typename T, int NS>
__global__ void k_m2m_interp(const T *__restrict__ from, T *__restrict__ to, MGeom f, MGeom t, int clear) {
  constexpr int off = NS == 6 ? 2 : 1;
  const int64_t n = (int64_t)t.E[0] * t.E[1] * t.E[2];
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
    const int ii[3] = {(int)(c % t.E[0]) + 1 - t.ng[0], (int)((c / t.E[0]) % t.E[1]) + 1 - t.ng[1],
                       (int)(c / ((int64_t)t.E[0] * t.E[1])) + 1 - t.ng[2]};
    bool skip = false;
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (t.bc[d] != 0 && (ii[d] < 1 || ii[d] > t.ncell[d])) skip = true;
    if (skip) {
      if (clear) to[3 * c] = to[3 * c + 1] = to[3 * c + 2] = (T)0;
      continue;
    }
    double w[3][NS];
    int64_t idx[3][NS];
    const int64_t st[3] = {3, 3 * (int64_t)f.E[0], 3 * (int64_t)f.E[0] * f.E[1]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double p = __dadd_rn(t.xmin[d], __dmul_rn(__dadd_rn((double)(ii[d] - 1), 0.5), t.dx[d]));
      const int b = cell_index(p, f.xmin[d], f.c1dx[d]);
      const double dd = stencil_offset(p, f.xmin[d], f.dx[d], b, f.c1dx[d]);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        int q = b - off + s;
        double ws = weight(NS == 6, s, dd);
        if (q < 1 - f.ng[d]) { ws = 0.0; q = 1 - f.ng[d]; }
        if (q > f.ncell[d] + f.ng[d]) { ws = 0.0; q = f.ncell[d] + f.ng[d]; }
        w[d][s] = ws;
        idx[d][s] = (int64_t)(q - 1 + f.ng[d]) * st[d];
      }
    }
    double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
    if (!clear) {
      acc0 = (double)to[3 * c];
      acc1 = (double)to[3 * c + 1];
      acc2 = (double)to[3 * c + 2];
    }
#pragma unroll
    for (int sz = 0; sz < NS; ++sz)
#pragma unroll
      for (int sy = 0; sy < NS; ++sy)
#pragma unroll
        for (int sx = 0; sx < NS; ++sx) {
          const double ww = __dmul_rn(__dmul_rn(w[0][sx], w[1][sy]), w[2][sz]);
          const T *m = from + idx[0][sx] + idx[1][sy] + idx[2][sz];
          acc0 = __dadd_rn(acc0, __dmul_rn(ww, (double)m[0]));
          acc1 = __dadd_rn(acc1, __dmul_rn(ww, (double)m[1]));
          acc2 = __dadd_rn(acc2, __dmul_rn(ww, (double)m[2]));
        }
    to[3 * c] = (T)acc0;
    to[3 * c + 1] = (T)acc1;
    to[3 * c + 2] = (T)acc2;
  }
}

// ---------------------------------------------------------------------------
// Separable form (the default).  Both directions are tensor products of
// per-axis operators: the deposit weight of a source cell onto a target cell
// is (reldx W_x)(reldx W_y)(reldx W_z), a cell outside a periodic axis is
// dropped on that axis, and the interpolation weight is W_x W_y W_z over the
// stencil cells inside the source mesh.  So the sums run one axis after the
// other: for an interpolation in one kernel, tile by tile with the
// intermediate sums in LDS (the mesh's type); for a deposit, whose tiles would
// have wide halos, in a kernel that streams the patch along z and one for x
// and y.  A workgroup tabulates its tile's weights in LDS.
// One direction with a kernel per axis and a table kernel per axis, and now,
// us: 256^3 FP32 ratio 2 M'4 deposit 225, 137, interpolation 225, 97; FP64
// 400, 247 and 404, 172; 192^3 FP32 ratio 4 M6* 177, 79 and 108, 59; 64^3 FP32
// ratio 2 36, 19 and 25, 8.
// The sums are regrouped against the reference's sequential loop (which
// adds ((W_x W_y) W_z) m term by term), so the result agrees to rounding
// (~1e-16 relative) rather than bit for bit; PMGPU_M2M_EXACT=1 selects the
// bit-identical gathers above.

constexpr int kMThreads = 512;
constexpr int kDownSeg = 320;   // words of a source row staged (deposit)
// source rows staged at a time (16 and 32 FP32 rows measure the same; fewer leave LDS for more workgroups)
template <typename T> constexpr int down_rows() { return sizeof(T) == 4 ? 16 : 8; }
constexpr int kUpCells = 4;     // target cells per thread and plane (interpolation)
constexpr int kMLds = 64 * 1024;

struct M2MArgs {
  MGeom f, t;
  double reldx;
  int clear;
  int W, H, D;        // target cells of a tile along x, y and of a march along z
  int nx, ny, nz;     // tiles
  int cap[3];         // staged source indices per axis (deposit: candidates; interpolation: source cells)
  int taps[2];        // most taps of a target index along x, y (deposit)
  int rows;           // source rows per pass (deposit)
  int stage_bytes;    // LDS of the rows and, before, of the staged indices
};

// a tile's position: workgroups of one XCD take neighbouring tiles (x fastest,
// then y, then z), whose source cells they share in that XCD's L2
__device__ __forceinline__ void m2m_tile(const M2MArgs &a, int *o, int *n) {
  const int64_t lt = xcd_tile(blockIdx.x, gridDim.x);
  o[0] = (int)(lt % a.nx) * a.W;
  o[1] = (int)((lt / a.nx) % a.ny) * a.H;
  o[2] = (int)(lt / ((int64_t)a.nx * a.ny)) * a.D;
  n[0] = min(a.W, a.t.E[0] - o[0]);
  n[1] = min(a.H, a.t.E[1] - o[1]);
  n[2] = min(a.D, a.t.E[2] - o[2]);
}

// i / n of the items of a tile, with inv = 1 / n (exact: i < 2^16, n < 2^10,
// and (i + 1/2) / n is 1 / 2n away from a whole number)
__device__ __forceinline__ int quot(int i, float inv) { return (int)(((float)i + 0.5f) * inv); }

// the three components of a cell
template <typename T> struct Cell3 {
  T x, y, z;
};

// words of a mesh line at a time (a line starts at any word)
template <typename T, int V> struct alignas(sizeof(T)) Words {
  T v[V];
};

// Patch -> parent, the sums along z: a thread owns V words of the mesh's planes
// and marches up the source planes that reach its D target planes, adding each
// to the NS target planes it reaches (a window in registers, stored as the
// planes leave it), four planes' loads in flight.  Reads the patch once but for
// the NS - 1 planes on either side of a march, and writes 1 / ratio of it:
// bound by memory, 256^3 FP32 70 us for 317 MB.
template <typename T, int NS, int V>
__global__ void __launch_bounds__(256) k_m2m_down_z(const T *__restrict__ from, T *__restrict__ mid, M2MArgs a) {
  constexpr int off = NS == 6 ? 2 : 1;
  extern __shared__ double m2m_lds[];
  const MGeom &f = a.f, &t = a.t;
  const int64_t words = 3 * (int64_t)f.E[0] * f.E[1];
  const int o = (int)blockIdx.y * a.D, n = min(a.D, t.E[2] - o);
  double *const zw = m2m_lds;
  int *const zb = reinterpret_cast<int *>(zw + (size_t)a.cap[2] * NS), *const zl = zb + a.cap[2];
  const int T0 = o + 1 - t.ng[2], T1 = T0 + n - 1;
  int zlo, zhi;
  src_range(f, t, 2, T0 + off - NS + 1, T1 + off, zlo, zhi);
  const int nzs = max(min(zhi - zlo + 1, a.cap[2]), 0);
  for (int q = threadIdx.x; q < nzs; q += blockDim.x) {
    unsigned char live;
    stage_src<NS>(f, t, 2, zlo + q, a.reldx, zb[q], live, zw + (size_t)q * NS);
    zl[q] = live;
  }
  __syncthreads();
  // (the last thread's words may be its neighbour's too: the same values)
  const int64_t w0 = min(V * (blockIdx.x * (int64_t)blockDim.x + threadIdx.x), words - V);
  if (V * (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >= words) return;
  const int q0 = lower_bound_b(zb, nzs, T0 + off - NS + 1), q1 = lower_bound_b(zb, nzs, T1 + off + 1);
  const T *src = from + w0 + words * (zlo - 1 + f.ng[2]);
  double acc[NS][V];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int c = 0; c < V; ++c) acc[s][c] = 0.0;
  int cur = T0 - NS + 1;   // target plane of acc[0]
  auto advance = [&] {
    if (cur >= T0) {
      Words<T, V> r;
#pragma unroll
      for (int c = 0; c < V; ++c) r.v[c] = (T)acc[0][c];
      *reinterpret_cast<Words<T, V> *>(mid + w0 + words * (cur - 1 + t.ng[2])) = r;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int c = 0; c < V; ++c) acc[s][c] = s + 1 < NS ? acc[s + 1][c] : 0.0;
    ++cur;
  };
  for (int q = q0; q < q1; q += 4) {
    Words<T, V> v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = *reinterpret_cast<const Words<T, V> *>(src + words * min(q + u, q1 - 1));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (q + u < q1 && zl[q + u]) {
        const int b = __builtin_amdgcn_readfirstlane(zb[q + u]);
        while (cur < b - off) advance();
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const double w = zw[(size_t)(q + u) * NS + s];
#pragma unroll
          for (int c = 0; c < V; ++c) acc[s][c] = __fma_rn(w, (double)v[u].v[c], acc[s][c]);
        }
      }
  }
  while (cur <= T1) advance();
}

// Patch -> parent, the sums along x and y of the planes summed along z.  A
// workgroup owns W x H target columns; a plane's source rows under them are
// copied into LDS (a wavefront per row, the next rows' loads in flight while
// these are summed), summed along x into LDS again, and along y in registers.
// What bounds it: LDS, NS ratio words per sum on both axes: 256^3 FP32 79 us.
// (Rows summed along x straight from memory, their loads waited for tap by tap,
// and all three axes in one march: 164 us against 149 for both kernels at 256^3
// FP32, 621 against 77 at 192^3 ratio 4 M6*.)
template <typename T, int NS>
__global__ void __launch_bounds__(kMThreads) k_m2m_down_xy(const T *__restrict__ mid, T *__restrict__ to, M2MArgs a) {
  constexpr int off = NS == 6 ? 2 : 1, kWaves = kMThreads / 64, RK = down_rows<T>() / kWaves, SK = kDownSeg / 64;
  extern __shared__ double m2m_lds[];
  const MGeom &f = a.f, &t = a.t;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int o[3], n[3];
  m2m_tile(a, o, n);
  // LDS: source rows and x sums (first the staged indices of one axis: weights,
  // bases, live flags), tap weights of x and y; first taps and counts
  double *const st_w = m2m_lds;
  T *const raw = reinterpret_cast<T *>(m2m_lds), *const X = raw + down_rows<T>() * kDownSeg;
  double *const wx = m2m_lds + a.stage_bytes / 8, *const wy = wx + a.taps[0] * a.W;
  int *const fx = reinterpret_cast<int *>(wy + a.taps[1] * a.H), *const cx = fx + a.W;
  int *const fy = cx + a.W, *const cy = fy + a.H;

  int lo[2], len[2];   // source cells under the tile
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int T0 = o[d] + 1 - t.ng[d], nt = n[d], cap = a.cap[d], w0 = d == 0 ? a.W : a.H;
    int *const sb = reinterpret_cast<int *>(st_w + (size_t)cap * NS), *const sl = sb + cap;
    int *const first = d == 0 ? fx : fy, *const count = d == 0 ? cx : cy;
    double *const wt = d == 0 ? wx : wy;
    int ilo, ihi;
    src_range(f, t, d, T0 + off - NS + 1, T0 + nt - 1 + off, ilo, ihi);
    const int ns = max(min(ihi - ilo + 1, cap), 0), i0 = ilo - 1 + f.ng[d];
    for (int q = tid; q < ns; q += kMThreads) {
      unsigned char live;
      stage_src<NS>(f, t, d, ilo + q, a.reldx, sb[q], live, st_w + (size_t)q * NS);
      sl[q] = live;
    }
    __syncthreads();
    const int b0 = lower_bound_b(sb, ns, T0 + off - NS + 1), b1 = lower_bound_b(sb, ns, T0 + nt + off);
    lo[d] = __builtin_amdgcn_readfirstlane(i0 + b0);
    len[d] = __builtin_amdgcn_readfirstlane(d == 0 ? min(b1 - b0, kDownSeg / 3) : b1 - b0);
    for (int q = tid; q < nt; q += kMThreads) {
      int q0 = lower_bound_b(sb, ns, T0 + q + off - NS + 1), q1 = lower_bound_b(sb, ns, T0 + q + off + 1);
      while (q0 < q1 && !sl[q0]) ++q0;
      while (q0 < q1 && !sl[q1 - 1]) --q1;
      first[q] = q0 - b0;
      count[q] = max(min(min(q1 - q0, a.taps[d]), len[d] - (q0 - b0)), 0);
    }
    __syncthreads();
    for (int i = tid; i < a.taps[d] * nt; i += kMThreads) {
      const int k = i / nt, q = i - k * nt;
      if (k < count[q]) {
        const int e = first[q] + b0 + k;
        wt[k * w0 + q] = st_w[(size_t)e * NS + (T0 + q - sb[e] + off)];
      }
    }
    __syncthreads();
  }
  const int ty = tid / n[0], tx = tid - ty * n[0];
  const bool mine = ty < n[1];
  const int my0 = mine ? fy[ty] : 0, my1 = my0 + (mine ? cy[ty] : 0);
  const int seg = 3 * len[0], rows = len[1], chunk = min(a.rows, down_rows<T>());
  const int plane = a.rows * a.W;   // LDS words of an x sum's component
  const int64_t sy = 3 * (int64_t)f.E[0], sz = sy * f.E[1];
  const T *src = mid + sy * lo[1] + 3 * (int64_t)lo[0] + sz * o[2];
  auto put = [&](int q, double v0, double v1, double v2) {
    if (!mine) return;
    Cell3<T> *p = reinterpret_cast<Cell3<T> *>(to) + (int64_t)(o[0] + tx) +
                  (int64_t)t.E[0] * ((o[1] + ty) + (int64_t)t.E[1] * (o[2] + q));
    if (!a.clear) {
      const Cell3<T> v = *p;
      v0 += (double)v.x;
      v1 += (double)v.y;
      v2 += (double)v.z;
    }
    *p = Cell3<T>{(T)v0, (T)v1, (T)v2};
  };
  if (seg <= 0 || rows <= 0) {   // no source cell reaches the tile
    for (int q = 0; q < n[2]; ++q) put(q, 0.0, 0.0, 0.0);
    return;
  }
  T reg[RK][SK];
  auto load = [&](int q, int r0) {
#pragma unroll
    for (int i = 0; i < RK; ++i) {
      const T *p = src + sz * q + sy * min(r0 + wave + kWaves * i, rows - 1);
#pragma unroll
      for (int k = 0; k < SK; ++k) reg[i][k] = p[min(lane + 64 * k, seg - 1)];
    }
  };
  const float inv = 1.0f / (float)n[0];
  load(0, 0);
  double v0 = 0.0, v1 = 0.0, v2 = 0.0;
  for (int q = 0, r0 = 0; q < n[2];) {
    const int m = min(chunk, rows - r0);
#pragma unroll
    for (int i = 0; i < RK; ++i)
#pragma unroll
      for (int k = 0; k < SK; ++k) raw[(wave + kWaves * i) * kDownSeg + lane + 64 * k] = reg[i][k];
    __syncthreads();
    const bool last = r0 + m >= rows;
    const int qn = last ? q + 1 : q, rn = last ? 0 : r0 + m;
    if (qn < n[2]) load(qn, rn);
    for (int i = tid; i < m * n[0]; i += kMThreads) {
      const int r = quot(i, inv), x = i - r * n[0];
      const T *p = raw + r * kDownSeg + 3 * fx[x];
      const double *w = wx + x;
      const int cnt = cx[x];
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
      for (int e = 0; e < cnt; ++e) {
        const double wt = w[e * a.W];
        s0 = __fma_rn(wt, (double)p[3 * e], s0);
        s1 = __fma_rn(wt, (double)p[3 * e + 1], s1);
        s2 = __fma_rn(wt, (double)p[3 * e + 2], s2);
      }
      T *xs = X + r * a.W + x;
      xs[0] = (T)s0;
      xs[plane] = (T)s1;
      xs[2 * plane] = (T)s2;
    }
    __syncthreads();
    const int e1 = min(my1, r0 + m);
    for (int e = max(my0, r0); e < e1; ++e) {
      const double wt = wy[(e - my0) * a.H + ty];
      const T *xs = X + (e - r0) * a.W + tx;
      v0 = __fma_rn(wt, (double)xs[0], v0);
      v1 = __fma_rn(wt, (double)xs[plane], v1);
      v2 = __fma_rn(wt, (double)xs[2 * plane], v2);
    }
    if (last) {
      put(q, v0, v1, v2);
      v0 = v1 = v2 = 0.0;
    }
    q = qn;
    r0 = rn;
  }
}

// Parent -> patch.  A workgroup owns W x H target columns and D target planes:
// for each plane the source cells under it are summed along z into LDS, those
// along y into LDS again, and those along x stored.
// What bounds it: the patch's store (256^3 FP32 211 MB, 41 us at the card's
// copy rate) and the sums along x, 6 NS conversions and multiply-adds per
// target cell and as many LDS reads: 97 us.
template <typename T, int NS>
__global__ void __launch_bounds__(kMThreads) k_m2m_up(const T *__restrict__ from, T *__restrict__ to, M2MArgs a) {
  constexpr int off = NS == 6 ? 2 : 1;
  extern __shared__ double m2m_lds[];
  const MGeom &f = a.f, &t = a.t;
  const int tid = threadIdx.x;
  int o[3], n[3];
  m2m_tile(a, o, n);
  // LDS: weights per target index, z sums, y sums, first source cells
  const int len[3] = {a.W, a.H, a.D};
  double *const wx = m2m_lds, *const wy = wx + NS * len[0], *const zw = wy + NS * len[1];
  T *const A = reinterpret_cast<T *>(zw + NS * len[2]);
  const int ca = a.cap[0] * a.cap[1], cb = a.cap[0] * a.H;
  T *const B = A + 3 * ca;
  int *const bx = reinterpret_cast<int *>(m2m_lds) + a.stage_bytes / 4, *const by = bx + len[0], *const zb = by + len[1];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double *const w = d == 0 ? wx : d == 1 ? wy : zw;
    int *const base = d == 0 ? bx : d == 1 ? by : zb;
    for (int q = tid; q < n[d]; q += kMThreads) {
      const double p = __dadd_rn(t.xmin[d], __dmul_rn(__dadd_rn((double)(o[d] + q - t.ng[d]), 0.5), t.dx[d]));
      const int b = cell_index(p, f.xmin[d], f.c1dx[d]);
      const double dd = stencil_offset(p, f.xmin[d], f.dx[d], b, f.c1dx[d]);
#pragma unroll
      for (int s = 0; s < NS; ++s) w[s * len[d] + q] = weight(NS == 6, s, dd);
      base[q] = b - off - 1 + f.ng[d];   // (0-based; the stencil may leave the source mesh)
    }
  }
  __syncthreads();
  // source cells under the tile (bases are non-decreasing)
  const int cx0 = bx[0], cy0 = by[0];
  const int cw = min(bx[n[0] - 1] - cx0 + NS, a.cap[0]), ch = min(by[n[1] - 1] - cy0 + NS, a.cap[1]);
  const float inv = 1.0f / (float)cw;
  const int64_t sy = 3 * (int64_t)f.E[0], sz = sy * f.E[1];
  auto skips = [&](int d, int x) { return t.bc[d] != 0 && (x < t.ng[d] || x >= t.ng[d] + t.ncell[d]); };
  // the thread's target cells
  int off_b[kUpCells], tx[kUpCells], ty[kUpCells];
#pragma unroll
  for (int k = 0; k < kUpCells; ++k) {
    const int i = tid + k * kMThreads;
    ty[k] = i / n[0];
    tx[k] = i - ty[k] * n[0];
    if (ty[k] >= n[1]) ty[k] = -1;
    off_b[k] = ty[k] < 0 ? 0 : ty[k] * a.cap[0] + bx[tx[k]] - cx0;
  }
  for (int q = 0; q < n[2]; ++q) {
    const int z = o[2] + q;
    const int z0 = __builtin_amdgcn_readfirstlane(zb[q]);
    double w[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) w[s] = zw[s * len[2] + q];
    for (int i = tid; i < cw * ch; i += kMThreads) {
      const int y = quot(i, inv), x = i - y * cw;
      const int gx = cx0 + x, gy = cy0 + y;
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
      if (gx >= 0 && gx < f.E[0] && gy >= 0 && gy < f.E[1]) {
        Cell3<T> v[NS];
        const T *p = from + sy * gy + 3 * (int64_t)gx;
#pragma unroll
        for (int s = 0; s < NS; ++s)
          v[s] = *reinterpret_cast<const Cell3<T> *>(p + sz * min(max(z0 + s, 0), f.E[2] - 1));
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (z0 + s >= 0 && z0 + s < f.E[2]) {
            s0 = __fma_rn(w[s], (double)v[s].x, s0);
            s1 = __fma_rn(w[s], (double)v[s].y, s1);
            s2 = __fma_rn(w[s], (double)v[s].z, s2);
          }
      }
      T *p = A + y * a.cap[0] + x;
      p[0] = (T)s0;
      p[ca] = (T)s1;
      p[2 * ca] = (T)s2;
    }
    __syncthreads();
    for (int i = tid; i < cw * n[1]; i += kMThreads) {
      const int y = quot(i, inv), x = i - y * cw;
      const T *p = A + (by[y] - cy0) * a.cap[0] + x;
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const double wt = wy[s * len[1] + y];
        s0 = __fma_rn(wt, (double)p[s * a.cap[0]], s0);
        s1 = __fma_rn(wt, (double)p[s * a.cap[0] + ca], s1);
        s2 = __fma_rn(wt, (double)p[s * a.cap[0] + 2 * ca], s2);
      }
      T *r = B + y * a.cap[0] + x;
      r[0] = (T)s0;
      r[cb] = (T)s1;
      r[2 * cb] = (T)s2;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kUpCells; ++k)
      if (ty[k] >= 0) {
        const bool skip = skips(0, o[0] + tx[k]) || skips(1, o[1] + ty[k]) || skips(2, z);
        const T *p = B + off_b[k];
        Cell3<T> *r = reinterpret_cast<Cell3<T> *>(to) + (int64_t)(o[0] + tx[k]) +
                      (int64_t)t.E[0] * ((o[1] + ty[k]) + (int64_t)t.E[1] * z);
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const double wt = wx[s * len[0] + tx[k]];
          s0 = __fma_rn(wt, (double)p[s], s0);
          s1 = __fma_rn(wt, (double)p[s + cb], s1);
          s2 = __fma_rn(wt, (double)p[s + 2 * cb], s2);
        }
        if (a.clear) {
          *r = skip ? Cell3<T>{0, 0, 0} : Cell3<T>{(T)s0, (T)s1, (T)s2};
        } else if (!skip) {
          const Cell3<T> v = *r;
          *r = Cell3<T>{(T)(s0 + (double)v.x), (T)(s1 + (double)v.y), (T)(s2 + (double)v.z)};
        }
      }
  }
}

// Tile of a deposit or an interpolation: W x H target columns, W at most
// most_w, W H at most `most` and equal along each axis, the ones that sum the
// fewest source cells (their halos count) and leave the fewest lanes without a
// column; D target planes so that the chip has kMTiles workgroups.
constexpr int kMTiles = 1024;
void m2m_tiles(M2MArgs &a, int most, int most_w, int halo) {
  double best = 0.0;
  for (int nx = 1; nx <= a.t.E[0]; ++nx) {
    const int W = (a.t.E[0] + nx - 1) / nx;
    if (W > std::min(most, most_w)) continue;
    if (W < 8 && best > 0.0) break;
    int H = std::min(std::min(most / W, a.t.E[1]), 64);
    const int ny = (a.t.E[1] + H - 1) / H;
    H = (a.t.E[1] + ny - 1) / ny;
    const double cost = (double)nx * ny * ((double)(H + halo) * (W + halo) + most);
    if (best == 0.0 || cost < best) {
      best = cost;
      a.W = W;
      a.H = H;
    }
  }
  a.nx = (a.t.E[0] + a.W - 1) / a.W;
  a.ny = (a.t.E[1] + a.H - 1) / a.H;
  const int64_t want = std::max<int64_t>(1, kMTiles / ((int64_t)a.nx * a.ny));
  a.D = (int)std::min<int64_t>((a.t.E[2] + want - 1) / want, 32);
  a.nz = (a.t.E[2] + a.D - 1) / a.D;
}

// Intermediate mesh of the deposit, grown on demand, kept until
// pmgpu_finalize (one per process: calls that overlap race).
struct M2MWS {
  void *a = nullptr;
  size_t na = 0;
};
M2MWS g_m2m;
std::mutex g_m2m_mu;

int grow(void *&p, size_t &have, size_t want) {
  if (have >= want) return 0;
  if (p) (void)hipFree(p);
  p = nullptr;
  have = 0;
  PM_HIP(hipMalloc(&p, want));
  have = want;
  return 0;
}

// 1: not a mesh for these kernels
template <typename T, int NS> int m2m_down(M2MArgs &a, const T *src, T *dst, hipStream_t st) {
  int ratio[3];
  for (int d = 0; d < 3; ++d) ratio[d] = std::max(1, (int)std::ceil(a.t.dx[d] / a.f.dx[d] - 1e-6));
  // z: V words per thread, D planes per march
  constexpr int V = 16 / sizeof(T);
  const int64_t words = 3 * (int64_t)a.f.E[0] * a.f.E[1];
  if (words < V) return 1;
  const size_t bytes = sizeof(T) * (size_t)words * a.t.E[2];
  std::lock_guard<std::mutex> lock(g_m2m_mu);
  if (grow(g_m2m.a, g_m2m.na, bytes)) return -1;
  T *mid = static_cast<T *>(g_m2m.a);
  const int64_t bx = (words + V * 256 - 1) / (V * 256);
  const int64_t marches = std::max<int64_t>(1, kMTiles / bx);
  a.D = (int)std::min<int64_t>((a.t.E[2] + marches - 1) / marches, 32);
  a.cap[2] = (a.D + NS + 2) * ratio[2] + 8;
  const dim3 zgrid((unsigned)bx, (a.t.E[2] + a.D - 1) / a.D);
  hipLaunchKernelGGL((k_m2m_down_z<T, NS, V>), zgrid, dim3(256),
                     a.cap[2] * (sizeof(double) * NS + 2 * sizeof(int)), st, src, mid, a);
  PM_HIP(hipGetLastError());
  // x and y: the widest tile whose source cells ((W + NS - 1) ratio and one for
  // the ends) fit the staged rows, and its sums LDS
  size_t lds = 0;
  for (int mw = (kDownSeg / 3 - 2) / ratio[0] - (NS - 1); mw > 0; --mw) {
    m2m_tiles(a, kMThreads, mw, NS - 1);
    const int n[2] = {a.W, a.H};
    for (int d = 0; d < 2; ++d) {
      a.cap[d] = (n[d] + NS + 2) * ratio[d] + 8;
      a.taps[d] = NS * ratio[d] + 2;
    }
    a.rows = std::min(down_rows<T>(), a.cap[1]);
    const size_t stage = std::max(a.cap[0], a.cap[1]) * (sizeof(double) * NS + 2 * sizeof(int));
    a.stage_bytes =
        (int)((std::max(sizeof(T) * (down_rows<T>() * kDownSeg + 3 * (size_t)a.rows * a.W), stage) + 7) / 8 * 8);
    lds = a.stage_bytes + sizeof(double) * ((size_t)a.taps[0] * a.W + (size_t)a.taps[1] * a.H) +
          sizeof(int) * 2 * ((size_t)a.W + a.H);
    if (lds <= kMLds) break;
  }
  if (lds == 0 || lds > kMLds) return 1;
  const int64_t tiles = (int64_t)a.nx * a.ny * a.nz;
  PM_CHECK(tiles < ((int64_t)1 << 31), "pmgpu_interp_mesh_mesh: mesh too large");
  hipLaunchKernelGGL((k_m2m_down_xy<T, NS>), dim3((unsigned)tiles), dim3(kMThreads), lds, st, (const T *)mid, dst, a);
  PM_HIP(hipGetLastError());
  return 0;
}

template <typename T, int NS> int m2m_up(M2MArgs &a, const T *src, T *dst, hipStream_t st) {
  // the largest tile whose sums fit in LDS; none for a mesh much finer along
  // another axis than along x
  size_t lds = 0;
  for (int most = kMThreads * kUpCells; most >= 64; most /= 2) {
    m2m_tiles(a, most, 128, 0);
    const int n[2] = {a.W, a.H};
    // (bases n - 1 spacings apart differ by that many source cells, rounded up)
    double c[2];
    for (int d = 0; d < 2; ++d) c[d] = std::ceil(n[d] * a.t.dx[d] / a.f.dx[d] * (1.0 + 1e-9)) + NS + 1;
    const double w = sizeof(double) * NS * ((double)a.W + a.H + a.D);
    lds = 0;
    if (w + 3.0 * sizeof(T) * c[0] * (c[1] + a.H) > kMLds) continue;
    for (int d = 0; d < 2; ++d) a.cap[d] = (int)c[d];
    a.stage_bytes = (int)(w + 3 * sizeof(T) * a.cap[0] * (a.cap[1] + a.H) + 7) / 8 * 8;
    lds = a.stage_bytes + sizeof(int) * ((size_t)a.W + a.H + a.D);
    break;
  }
  if (lds == 0) return 1;
  const int64_t tiles = (int64_t)a.nx * a.ny * a.nz;
  PM_CHECK(tiles < ((int64_t)1 << 31), "pmgpu_interp_mesh_mesh: mesh too large");
  hipLaunchKernelGGL((k_m2m_up<T, NS>), dim3((unsigned)tiles), dim3(kMThreads), lds, st, src, dst, a);
  PM_HIP(hipGetLastError());
  return 0;
}

// the ghost layers of periodic axes after a deposit (added onto their images,
// :1380-1386, pmlib_mesh_map_ghost with incl_edges, op add) or an
// interpolation (copied from their images, :2057-2063, op replace)
template <typename T> int m2m_periodic(const MGeom &t, bool deposit, T *dst, hipStream_t st) {
  PGeom pg{};
  for (int d = 0; d < 3; ++d) {
    pg.ncell[d] = t.ncell[d];
    pg.ngl[d] = t.ng[d];
    pg.E[d] = t.E[d];
  }
  for (int d = 0; d < 3; ++d)
    if (t.bc[d] != 0) {
      if (deposit)
        hipLaunchKernelGGL(k_halo_add<T>, dim3(256), dim3(256), 0, st, dst, pg, d);
      else
        hipLaunchKernelGGL(k_ghost_fill<T>, dim3(1024), dim3(256), 0, st, dst, t.E[0], t.E[1], t.E[2], d, t.ncell[d],
                           t.ng[d], 3);
      PM_HIP(hipGetLastError());
    }
  return 0;
}

template <typename T>
int m2m_exact(const MGeom &f, const MGeom &t, int ns, const void *from, void *to, int clear, hipStream_t st);

template <typename T>
int m2m_separable(const MGeom &f, const MGeom &t, int ns, const void *from, void *to, int clear, hipStream_t st) {
  const bool deposit = f.dx[0] / t.dx[0] <= 0.9999;
  for (int d = 0; d < 3; ++d)
    PM_CHECK(!deposit || t.dx[d] / f.dx[d] <= (double)kMaxRatio + 1e-9,
             "pmgpu_interp_mesh_mesh: cell size ratios above 8 are not supported");
  M2MArgs a{};
  a.f = f;
  a.t = t;
  a.reldx = f.dx[0] / t.dx[0];
  a.clear = clear;
  const T *src = static_cast<const T *>(from);
  T *dst = static_cast<T *>(to);
  const int e = deposit ? (ns == 6 ? m2m_down<T, 6>(a, src, dst, st) : m2m_down<T, 4>(a, src, dst, st))
                        : (ns == 6 ? m2m_up<T, 6>(a, src, dst, st) : m2m_up<T, 4>(a, src, dst, st));
  if (e > 0) return m2m_exact<T>(f, t, ns, from, to, clear, st);
  if (e) return -1;
  return m2m_periodic(t, deposit, dst, st);
}

// ---------------------------------------------------------------------------
// Bit-identical gathers (PMGPU_M2M_EXACT=1)
template <typename T>
int m2m_exact(const MGeom &f, const MGeom &t, int ns, const void *from, void *to, int clear, hipStream_t st) {
  const double reldx = f.dx[0] / t.dx[0];
  const T *src = static_cast<const T *>(from);
  T *dst = static_cast<T *>(to);
  if (reldx <= 0.9999) {
    for (int d = 0; d < 3; ++d)
      PM_CHECK(t.dx[d] / f.dx[d] <= (double)kMaxRatio + 1e-9,
               "pmgpu_interp_mesh_mesh: cell size ratios above 8 are not supported");
    DepArgs a{f, t, reldx, clear};
    dim3 grid((t.E[0] + kTX - 1) / kTX, t.E[1], t.E[2]);
    if (ns == 6) hipLaunchKernelGGL((k_m2m_deposit<T, 6>), grid, dim3(kTX), 0, st, src, dst, a);
    else hipLaunchKernelGGL((k_m2m_deposit<T, 4>), grid, dim3(kTX), 0, st, src, dst, a);
    PM_HIP(hipGetLastError());
  } else {
    const int64_t n = (int64_t)t.E[0] * t.E[1] * t.E[2];
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    if (ns == 6) hipLaunchKernelGGL((k_m2m_interp<T, 6>), dim3(blocks), dim3(256), 0, st, src, dst, f, t, clear);
    else hipLaunchKernelGGL((k_m2m_interp<T, 4>), dim3(blocks), dim3(256), 0, st, src, dst, f, t, clear);
    PM_HIP(hipGetLastError());
  }
  return m2m_periodic(t, reldx <= 0.9999, dst, st);
}

int m2m_check(const pmgpu_geom *gf, const pmgpu_geom *gt, MGeom &f, MGeom &t) {
  PM_CHECK(gf && gt, "pmgpu_interp_mesh_mesh: null geometry");
  if (make_mgeom(gf, f, "pmgpu_interp_mesh_mesh") || make_mgeom(gt, t, "pmgpu_interp_mesh_mesh")) return -1;
  PM_CHECK(gf->interp_order == gt->interp_order,
           "pmgpu_interp_mesh_mesh: both meshes must use the same interpolation order");
  for (int d = 0; d < 3; ++d)
    PM_CHECK(t.bc[d] == 0 || t.ncell[d] >= 2 * t.ng[d],
             "pmgpu_interp_mesh_mesh: a periodic target axis needs at least twice its ghost count in cells");
  return 0;
}

}  // namespace

void m2m_release() {
  std::lock_guard<std::mutex> lock(g_m2m_mu);
  if (g_m2m.a) (void)hipFree(g_m2m.a);
  g_m2m = M2MWS{};
}
}  // namespace pmgpu

using namespace pmgpu;

extern "C" {

int pmgpu_topology_parent(const pmgpu_geom *g, int32_t level, int32_t parent_level, pmgpu_geom *out) {
  PM_CHECK(g && out, "pmgpu_topology_parent: null argument");
  PM_CHECK(parent_level != 0, "pmlib_topology_parent: Cannot create parent topology on level 0");
  PM_CHECK(g->interp_order == 3 || g->interp_order == 4,
           "pmlib_topology_parent: Can not define number of ghost cells.");
  const double reldx = std::pow(2.0, (double)(level - parent_level));
  const long r = std::lround(reldx);
  PM_CHECK(r >= 1, "pmgpu_topology_parent: the parent level must not be finer than the patch");
  pmgpu_geom p = *g;
  for (int d = 0; d < 3; ++d) {
    PM_CHECK(g->ncell[d] % r == 0, "pmlib_topology_parent: Number mesh cells does not match");
    p.ncell[d] = (int32_t)std::lround((double)g->ncell[d] / reldx);
    p.dx[d] = reldx * g->dx[d];
  }
  p.nghost = g->interp_order == 4 ? 3 : 2;
  *out = p;
  return 0;
}

int pmgpu_interp_mesh_mesh_device(const pmgpu_geom *g_from, const pmgpu_geom *g_to, int32_t precision,
                                  const void *d_from, void *d_to, int32_t clear, void *stream) {
  MGeom f, t;
  if (m2m_check(g_from, g_to, f, t)) return -1;
  PM_CHECK(d_from && d_to, "pmgpu_interp_mesh_mesh: null mesh");
  PM_CHECK(precision == PMGPU_FP64 || precision == PMGPU_FP32, "pmgpu_interp_mesh_mesh: bad precision");
  const int ns = g_to->interp_order == 4 ? 6 : 4;
  hipStream_t st = (hipStream_t)stream;
  const char *ex = getenv("PMGPU_M2M_EXACT");
  if (ex && atoi(ex) != 0)
    return precision == PMGPU_FP64 ? m2m_exact<double>(f, t, ns, d_from, d_to, clear, st)
                                   : m2m_exact<float>(f, t, ns, d_from, d_to, clear, st);
  return precision == PMGPU_FP64 ? m2m_separable<double>(f, t, ns, d_from, d_to, clear, st)
                                 : m2m_separable<float>(f, t, ns, d_from, d_to, clear, st);
}

int pmgpu_interp_mesh_mesh(const pmgpu_geom *g_from, const pmgpu_geom *g_to, const double *from, double *to,
                           int32_t clear) {
  MGeom f, t;
  if (m2m_check(g_from, g_to, f, t)) return -1;
  PM_CHECK(from && to, "pmgpu_interp_mesh_mesh: null mesh");
  const size_t bf = sizeof(double) * 3 * (size_t)f.E[0] * f.E[1] * f.E[2];
  const size_t bt = sizeof(double) * 3 * (size_t)t.E[0] * t.E[1] * t.E[2];
  void *df = nullptr, *dt = nullptr;
  int e = 0;
  if (hipMalloc(&df, bf) != hipSuccess || hipMalloc(&dt, bt) != hipSuccess) {
    set_error("pmgpu_interp_mesh_mesh: device allocation failed");
    e = -1;
  }
  if (!e && (hipMemcpy(df, from, bf, hipMemcpyHostToDevice) != hipSuccess ||
             hipMemcpy(dt, to, bt, hipMemcpyHostToDevice) != hipSuccess)) {
    set_error("pmgpu_interp_mesh_mesh: host to device copy failed");
    e = -1;
  }
  if (!e) e = pmgpu_interp_mesh_mesh_device(g_from, g_to, PMGPU_FP64, df, dt, clear, nullptr);
  if (!e && hipMemcpy(to, dt, bt, hipMemcpyDeviceToHost) != hipSuccess) {
    set_error("pmgpu_interp_mesh_mesh: device to host copy failed");
    e = -1;
  }
  if (df) (void)hipFree(df);
  if (dt) (void)hipFree(dt);
  return e;
}

}  // extern "C"
