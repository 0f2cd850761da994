// Particle <-> mesh kernels (HIP, gfx950): M'4 / M6* deposition and gather,
// remeshing and the low-storage RK update with one-rank migration.
//
// Deposition is a gather, not a scatter: particles are binned by the cell of
// their stencil base index (bit-exact NINT) and counting-sorted by bin and,
// inside a bin, by particle id, and every mesh node sums the particles of the
// ns^2 stencil rows that cover it (each row one contiguous range), in a fixed
// order: wavefronts that march over columns of nodes (k_p2m_march), or on a
// small mesh a wavefront per line of nodes over records of each particle's
// kernel weights and strength (k_p2m_stage, k_p2m_rows).  No atomics touch
// the mesh, so the result is deterministic run to run.
#pragma once
#include <type_traits>

#include "pm_common.h"

namespace pmgpu {

struct PGeom {
  int ncell[3], ngl[3], bc[3];
  int E[3];           // mesh extent incl. ghosts
  int lo[3], hi[3];   // node index range 1-ng .. N+ng
  double xmin[3], xmax[3], dx[3], c1dx[3];
  int ns, off;        // stencil width and base offset (M'4: 4,1; M6*: 6,2)
  int m6;
  int nb[3];          // bins per axis: base index b in [lo + off - ns + 1, hi + off]
  int blo[3];         // b of bin 0
};

// NINT((x - xmin) * c_1_dx): correctly rounded subtract and multiply (no
// contraction), then round half away from zero, done by hand: trunc is exact
// and so is t - trunc(t), so the half-way test is exact too.
__device__ __forceinline__ int cell_index(double x, double xmin, double c1) {
  const double t = __dmul_rn(__dsub_rn(x, xmin), c1);
  if (!(fabs(t) < 1073741824.0)) return t > 0 ? 1073741824 : (t < 0 ? -1073741824 : 0);  // far off the mesh
  double r = trunc(t);
  const double f = __dsub_rn(t, r);
  if (f >= 0.5) r = __dadd_rn(r, 1.0);
  else if (f <= -0.5) r = __dsub_rn(r, 1.0);
  return (int)r;
}

// the same without the bound, for a position known to be near the mesh
__device__ __forceinline__ int cell_index_near(double x, double xmin, double c1) {
  const double t = __dmul_rn(__dsub_rn(x, xmin), c1);
  const double r = trunc(t), f = __dsub_rn(t, r);
  return (int)r + (f >= 0.5 ? 1 : 0) - (f <= -0.5 ? 1 : 0);
}

// normalised offset d = (x - xmin - h (b - 1/2)) * nrm
__device__ __forceinline__ double stencil_offset(double x, double xmin, double h, int b, double nrm) {
  double t = __dmul_rn(h, __dsub_rn((double)b, 0.5));
  return __dmul_rn(__dsub_rn(__dsub_rn(x, xmin), t), nrm);
}

// weight of stencil slot s for offset d (interp_particle_mesh.f:182-214, :565-602)
__device__ __forceinline__ double weight(int m6, int s, double d) {
  if (!m6) {
    switch (s) {
      case 0: { double u = __dadd_rn(d, 1.0), a = __dsub_rn(2.0, u);
                return __dmul_rn(__dmul_rn(0.5, __dmul_rn(a, a)), __dsub_rn(1.0, u)); }
      case 1: { double d2 = __dmul_rn(d, d), d3 = __dmul_rn(d2, d);
                return __dadd_rn(__dsub_rn(1.0, __dmul_rn(2.5, d2)), __dmul_rn(1.5, d3)); }
      case 2: { double u = __dsub_rn(1.0, d), u2 = __dmul_rn(u, u), u3 = __dmul_rn(u2, u);
                return __dadd_rn(__dsub_rn(1.0, __dmul_rn(2.5, u2)), __dmul_rn(1.5, u3)); }
      default: { double u = __dsub_rn(2.0, d), a = __dsub_rn(2.0, u);
                 return __dmul_rn(__dmul_rn(0.5, __dmul_rn(a, a)), __dsub_rn(1.0, u)); }
    }
  }
  const double c1 = -1.0 / 24.0, c2 = 1.0 / 24.0, c3 = -1.0 / 12.0;
  double x;
  switch (s) {
    case 0: x = __dadd_rn(d, 2.0); break;
    case 1: x = __dadd_rn(d, 1.0); break;
    case 2: x = d; break;
    case 3: x = __dsub_rn(1.0, d); break;
    case 4: x = __dsub_rn(2.0, d); break;
    default: x = __dsub_rn(3.0, d); break;
  }
  double x2 = __dmul_rn(x, x), x3 = __dmul_rn(x2, x), x4 = __dmul_rn(x3, x);
  if (s == 0 || s == 5) {
    double t = __dsub_rn(x, 3.0);
    double t3 = __dmul_rn(__dmul_rn(t, t), t);
    return __dmul_rn(__dmul_rn(__dmul_rn(c1, __dsub_rn(x, 2.0)), t3), __dsub_rn(__dmul_rn(5.0, x), 8.0));
  }
  if (s == 1 || s == 4) {
    double p = __dsub_rn(__dadd_rn(__dsub_rn(__dmul_rn(25.0, x3), __dmul_rn(114.0, x2)), __dmul_rn(153.0, x)), 48.0);
    return __dmul_rn(__dmul_rn(__dmul_rn(c2, __dsub_rn(x, 1.0)), __dsub_rn(x, 2.0)), p);
  }
  double p = __dadd_rn(__dadd_rn(__dsub_rn(__dsub_rn(__dmul_rn(25.0, x4), __dmul_rn(38.0, x3)), __dmul_rn(3.0, x2)),
                                 __dmul_rn(12.0, x)), 12.0);
  return __dmul_rn(__dmul_rn(c3, __dsub_rn(x, 1.0)), p);
}

// FP32 form of the kernel weights (same polynomials, single precision)
__device__ __forceinline__ float weight_f(int m6, int s, float d) {
  if (!m6) {
    switch (s) {
      case 0: { float u = d + 1.0f, a = 2.0f - u; return 0.5f * (a * a) * (1.0f - u); }
      case 1: return 1.0f - 2.5f * (d * d) + 1.5f * (d * d * d);
      case 2: { float u = 1.0f - d; return 1.0f - 2.5f * (u * u) + 1.5f * (u * u * u); }
      default: { float u = 2.0f - d, a = 2.0f - u; return 0.5f * (a * a) * (1.0f - u); }
    }
  }
  const float c1 = -1.0f / 24.0f, c2 = 1.0f / 24.0f, c3 = -1.0f / 12.0f;
  const float x = s == 0 ? d + 2.0f : (s == 1 ? d + 1.0f : (s == 2 ? d : (s == 3 ? 1.0f - d : (s == 4 ? 2.0f - d
                                                                                                      : 3.0f - d))));
  const float x2 = x * x, x3 = x2 * x, x4 = x3 * x;
  if (s == 0 || s == 5) {
    const float t = x - 3.0f;
    return c1 * (x - 2.0f) * (t * t * t) * (5.0f * x - 8.0f);
  }
  if (s == 1 || s == 4) return c2 * (x - 1.0f) * (x - 2.0f) * (25.0f * x3 - 114.0f * x2 + 153.0f * x - 48.0f);
  return c3 * (x - 1.0f) * (25.0f * x4 - 38.0f * x3 - 3.0f * x2 + 12.0f * x + 12.0f);
}

// Particle count of a launch: a host value, or, in a step recorded once
// and replayed (HIP graph), the count in device memory that earlier kernels
// of the same step wrote; the grid then covers the capacity and threads past
// the count do nothing.
struct NCount {
  int64_t n;
  const int *dev;
  __host__ __device__ NCount(int64_t v = 0) : n(v), dev(nullptr) {}
  __host__ __device__ NCount(int64_t cap, const int *d) : n(cap), dev(d) {}
  __device__ __forceinline__ int64_t get() const { return dev ? (int64_t)*dev : n; }
};

// compensated (Kahan) accumulation: sum + c carries the low-order bits the
// float sum drops (this file is compiled without contraction, so the
// compensation survives)
struct Kahan {
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ void add(float v) {
    const float y = v - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
};

// bin key of a particle (nbins: no stencil node touches the mesh, or the
// particle lies outside a periodic axis, where the reference zeroes every
// weight) and its arrival rank in the bin (an atomic count: the order within a
// bin is restored by particle id when the bin is staged)
// Particles near the cell centres have neighbours in one bin, whose atomics on
// one word wait for each other, so a run of neighbouring lanes of one bin adds
// its length once.  What bounds it: the atomics' round trips.  56.6M particles,
// 384^3: 727 us on average of a step's three calls and 1180 on the cell centres
// with an atomic per particle, 444 and 458 so (32 B a particle, 1.8 GB); 2.1M
// 34 -> 21 us.  (Four particles of a thread under way together: 549 us.)
__device__ __forceinline__ int p2m_key(const PGeom &g, const double *x, int nbins) {
  int b[3];
  bool ok = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    b[d] = cell_index(x[d], g.xmin[d], g.c1dx[d]);
    const int64_t bb = b[d];
    if (bb - g.off + g.ns - 1 < g.lo[d] || bb - g.off > g.hi[d]) ok = false;
    if (g.bc[d] != 0 && (x[d] < g.xmin[d] || x[d] > g.xmax[d])) ok = false;
  }
  return ok ? (b[0] - g.blo[0]) + g.nb[0] * ((b[1] - g.blo[1]) + g.nb[1] * (b[2] - g.blo[2])) : nbins;
}
// count[nbins + 1], the parts of the mesh that hold particles (k_p2m_binsort), is cleared.
static __global__ void k_p2m_keys(PGeom g, const double *__restrict__ pos, NCount npc, int nbins,
                                  int *__restrict__ key, int *__restrict__ rank, int *__restrict__ count) {
  const int64_t np = npc.get();
  if (blockIdx.x == 0 && threadIdx.x == 0) count[nbins + 1] = 0;
  const int lane = threadIdx.x & 63;
  // whole wavefronts: a lane past the end has no bin and stores nothing
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q - lane < np; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = q < np ? q : np - 1;
    const double x[3] = {pos[3 * p], pos[3 * p + 1], pos[3 * p + 2]};
    const int k = q < np ? p2m_key(g, x, nbins) : nbins;
    // neighbouring lanes of one bin as one count, that of the first of them
    const int before = __shfl_up(k, 1);
    const uint64_t heads = __ballot(lane == 0 || before != k);
    const uint64_t after = lane == 63 ? 0 : heads >> (lane + 1);
    const int run = after ? __ffsll((unsigned long long)after) : 64 - lane;
    int r = 0;
    if (k < nbins && (heads >> lane & 1)) r = atomicAdd(&count[k], run);
    const int head = lane - __clzll((long long)(heads << (63 - lane)));
    r = __shfl(r, head) + lane - head;
    if (q < np) {
      key[q] = k;
      rank[q] = r;
    }
  }
}

// counting-sort scatter: particle q to slot start[key] + rank of its bin
// clear (or null): the bin counts, set to zero for the next deposition
static __global__ void k_p2m_scatter(NCount npc, int nbins, const int *key, const int *rank, const int *start, int *ids,
                                     int *clear) {
  const int64_t np = npc.get();
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < np; q += (int64_t)gridDim.x * blockDim.x) {
    const int k = key[q];
    if (k < nbins) ids[start[k] + rank[q]] = (int)q;
  }
  if (clear)
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k <= nbins; k += (int64_t)gridDim.x * blockDim.x)
      clear[k] = 0;
}

// ascending order of ids[0, n) in place: insertion sort for the usual bins of
// a few particles, heap sort (n log n, no extra memory) for crowded ones
__device__ inline void sort_ids(int *ids, int n) {
  if (n <= 16) {
    for (int i = 1; i < n; ++i) {
      const int v = ids[i];
      int j = i - 1;
      while (j >= 0 && ids[j] > v) {
        ids[j + 1] = ids[j];
        --j;
      }
      ids[j + 1] = v;
    }
    return;
  }
  auto sift = [&](int root, int end) {
    while (2 * root + 1 < end) {
      int c = 2 * root + 1;
      if (c + 1 < end && ids[c + 1] > ids[c]) ++c;
      if (ids[root] >= ids[c]) return;
      const int t = ids[root];
      ids[root] = ids[c];
      ids[c] = t;
      root = c;
    }
  };
  for (int i = n / 2 - 1; i >= 0; --i) sift(i, n);
  for (int end = n - 1; end > 0; --end) {
    const int t = ids[0];
    ids[0] = ids[end];
    ids[end] = t;
    sift(0, end);
  }
}

// Staged particle record, in bin order: the 3 x ns kernel weights in slots
// [d * ns + s], the 3 strength components in slots 3 ns .. 3 ns + 2 and the
// base cell along x (a T-typed copy of the int) in slot 3 ns + 3.  For M'4
// (ns = 4) a record is 16 slots: one 128-byte line in FP64; for M6* 24.
template <typename T, int NS> struct PRec {
  static constexpr int kSlots = NS == 4 ? 16 : 24;
  static constexpr int kVal = 3 * NS, kBx = 3 * NS + 3;
};

// z nodes per marching wavefront (k_p2m_march).  More share a row's staging but
// take registers: 167 for 3 (M'4), three wavefronts per SIMD; 231 for M6*, two.
// 128^3 FP64 with 2, 3, 4: 216, 218, 220 us at each one's best chunk; M6*
// 112 x 96 x 80 373 us with 2, 346 with 3.
constexpr int kMarchQz = 3;
constexpr int kPartY = 4, kPartsOfBlock = 256 / kPartY, kPartBlocks = 256;
constexpr int kMarchRuns = 8;   // march_block

// The tiles of a march: nx segments of `width` x nodes, nz groups of kMarchQz z
// nodes, and y chunks of ylow to yhigh nodes.  How much of the mesh holds
// particles is counted in parts of one segment, kPartY bin rows along y and
// kMarchQz along z (py, pz of them).  A set that fills 40 % of them or more takes
// chunks of yhigh, the shortest with which all tiles are `resident` at most, the
// wavefronts that the chip holds (a second, nearly empty round of wavefronts
// costs most: 160^3 FP32 chunks of 8 nodes 313 us, of 9 266 us, of 12 290 us).
// For one that fills less, and would leave most of those wavefronts without
// particles, the chunks are so short that the tiles with particles are about
// three quarters of `resident`.  A node's sums do not depend on its chunk.
// Whole depositions, us, with chunks of yhigh for every set and now (a wavefront
// per line of nodes: FP64, then FP32 M'4): a cube of 2 % of 256^3 FP64 680, 283
// (980), FP32 655, 266 (525), of 10 % FP32 747, 432 (830); two rings on 128^3
// FP32 188, 146 (180), 256^3 911, 530 (1250), 384^3 2445, 1550 (3617).
struct MarchTiles {
  int width, nx, nz, py, pz, resident, ylow, yhigh;
  __host__ __device__ int parts() const { return nx * py * pz; }
  __host__ __device__ int part_blocks() const {
    const int n = (parts() + kPartsOfBlock - 1) / kPartsOfBlock;
    return n < kPartBlocks ? n : kPartBlocks;
  }
  __host__ __device__ bool fills(int filled) const { return 5 * filled >= 2 * parts(); }
  __host__ __device__ int64_t tiles(int ey, int yc) const { return (int64_t)nx * nz * ((ey + yc - 1) / yc); }
  // y chunk with which `used` columns of tiles are `most` tiles at most
  __host__ __device__ int chunk(int ey, int64_t used, int most) const {
    const int n = used > 0 && used < most ? (int)(most / used) : 1, yc = (ey + n - 1) / n;
    return yc < ylow ? ylow : (yc > yhigh ? yhigh : yc);
  }
  // (below ns / 2 nodes a chunk's ns - 1 further rows cost more than the chip's
  // idle SIMDs, unless there are as many of these as tiles)
  __host__ __device__ int chunk_of(int ey, int ns, int filled) const {
    if (fills(filled)) return yhigh;
    const int64_t used = ((int64_t)nx * nz * filled + parts() - 1) / parts();
    const int yc = chunk(ey, used, resident * 3 / 4), least = ns / 2 < yhigh ? ns / 2 : yhigh;
    return yc < least && used * ey > 1024 * (int64_t)yc ? least : yc;
  }
  __device__ int runs(int filled) const { return min(parts() / max(filled, 1), kMarchRuns); }
};

// One thread per bin: order the bin's particles by id (the order a stable
// sort by bin would give); bins of one particle, the usual case, do nothing.
// filled (or null): the first part_blocks() blocks count the parts of the mesh
// (MarchTiles) that hold a particle, for the march that follows, while the
// others sort (16 launches of up to 131^3 bins, on average 9.1 us, without the
// count 8.4; counted by the same blocks after the sort 10.7).
static __global__ void __launch_bounds__(256) k_p2m_binsort(PGeom g, const int *start, int nbins, int *ids,
                                                            MarchTiles mt, int *filled) {
  const int nblk = filled ? mt.part_blocks() : 0;
  if ((int)blockIdx.x >= nblk) {
    const int stride = ((int)gridDim.x - nblk) * (int)blockDim.x;
    for (int k = ((int)blockIdx.x - nblk) * (int)blockDim.x + (int)threadIdx.x; k < nbins; k += stride) {
      const int t0 = start[k], n = start[k + 1] - t0;
      if (n > 1) sort_ids(ids + t0, n);
    }
    return;
  }
  __shared__ int sum;
  if (threadIdx.x == 0) sum = 0;
  __syncthreads();
  int n = 0;
  // (a lane per bin row of a part's kPartY)
  const int row = threadIdx.x % kPartY;
  for (int p = (blockIdx.x * blockDim.x + threadIdx.x) / kPartY; p < mt.parts(); p += nblk * kPartsOfBlock) {
    const int seg = p % mt.nx, r = p / mt.nx, by = r % mt.py * kPartY, bz = r / mt.py * kMarchQz;
    const int x0 = seg * mt.width, xe = min(x0 + mt.width + g.ns - 1, g.nb[0]);
    int any = 0;
#pragma unroll
    for (int i = 0; i < kMarchQz; ++i) {
      const int k = g.nb[0] * (min(by + row, g.nb[1] - 1) + g.nb[1] * min(bz + i, g.nb[2] - 1));
      any |= start[k + xe] ^ start[k + x0];
    }
#pragma unroll
    for (int o = 1; o < kPartY; o *= 2) any |= __shfl_xor(any, o, 64);
    n += row == 0 && any != 0;
  }
  for (int o = 32; o > 0; o >>= 1) n += __shfl_down(n, o, 64);
  if ((threadIdx.x & 63) == 0 && n) atomicAdd(&sum, n);
  __syncthreads();
  if (threadIdx.x == 0 && sum) atomicAdd(filled, sum);
}

// One thread per sorted particle t < start[nbins]: its record at slot t
// (weights from the FP64 offsets; FP64: the reference's arithmetic; FP32:
// weights in single precision from the FP64 offset).
template <typename T, int NS>
__global__ void __launch_bounds__(256) k_p2m_stage(PGeom g, const double *pos, const double *val, const int *ids,
                                                   const int *start, int nbins, T *rec, int64_t rs) {
  const int nvalid = start[nbins];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nvalid; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = ids[t];   // (3 q passes 2^31 from 715,827,883 particles on)
    T wt[3 * NS];
    int bx = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double x = pos[3 * q + d];
      const int b = cell_index(x, g.xmin[d], g.c1dx[d]);
      if (d == 0) bx = b;
      const double dd = stencil_offset(x, g.xmin[d], g.dx[d], b, g.c1dx[d]);
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        if constexpr (sizeof(T) == sizeof(double))
          wt[d * NS + s2] = weight(NS == 6, s2, dd);
        else
          wt[d * NS + s2] = weight_f(NS == 6, s2, (float)dd);
      }
    }
    // planar records: field i of record t at rec[i * rs + t], so that the
    // stores of consecutive threads, and the gather's loads of one field of
    // consecutive records, are contiguous
    T *r = rec + t;
#pragma unroll
    for (int i = 0; i < 3 * NS; ++i) r[i * rs] = wt[i];
    r[PRec<T, NS>::kVal * rs] = (T)val[3 * q];
    r[(PRec<T, NS>::kVal + 1) * rs] = (T)val[3 * q + 1];
    r[(PRec<T, NS>::kVal + 2) * rs] = (T)val[3 * q + 2];
    r[PRec<T, NS>::kBx * rs] = (T)bx;
  }
}

// Row-staged gather.  A workgroup is one wavefront and owns a line of 64
// consecutive mesh nodes along x (node ix = 64 blockIdx.x + lane at node
// row iy = blockIdx.y, iz = blockIdx.z); each lane sums its own node.  The
// node line is reached by the ns x ns stencil rows (ky, kz) = (iy + a, iz + b),
// a, b < ns, and within a row by the bins [64 blockIdx.x, 64 blockIdx.x + 63
// + ns - 1], one contiguous range of records.  Row by row the wavefront
// copies those records into LDS with coalesced loads (only the values the
// row needs: the ns x weights, the row's y and z weights, the strength and
// the bin), and each lane then sums the records of its own bins [ix, ix + ns)
// from LDS.  The next row's records are loaded into registers while the
// current row is summed.  Per node the terms arrive in the order kz
// ascending (sz descending), ky ascending (sy descending), records
// ascending (bins ascending, particles by id within a bin); FP64 terms are
// ((wx wy) wz) v rounded per operation as the reference does; FP32 terms
// are wx (wy wz) v, fused into one partial sum per stencil row, and the ns^2
// row partials are Kahan-added.
constexpr int kRowCap = 128;   // records staged per row pass (two per lane)

template <typename T, int NS> struct RowStage {
  static constexpr int NV = NS + 5;   // wx[ns], wy, wz, v0, v1, v2
  T val[kRowCap / 64][NV];
  int xs[kRowCap / 64];               // x slot base
};

template <typename T, int NS>
__device__ __forceinline__ void row_fetch(RowStage<T, NS> &st, const T *rec, int64_t rs, int t0, int n, int lane,
                                          int sy, int sz, int x0, int blo0) {
  constexpr int KV = PRec<T, NS>::kVal, KB = PRec<T, NS>::kBx;
#pragma unroll
  for (int h = 0; h < kRowCap / 64; ++h) {
    const int i = lane + 64 * h;
    // unconditional loads (no branch for the wait counters to merge over):
    // an empty row reads record t0 <= np, inside the allocation of np + 1.
    // FP32: field f of record t0 + li is read as (rec + f rs + t0)[li], a
    // wave-uniform base (t0 is) and a 32-bit byte offset, so that no load
    // needs per-lane 64-bit address arithmetic (gather 193 -> 188 us at 2.1M
    // particles); FP64 keeps per-lane addresses (measured faster there)
    const int li = i < n ? i : (n > 0 ? n - 1 : 0);
    const T *rb = rec + t0, *r = rb + li;
    const uint32_t lb = (uint32_t)li * (uint32_t)sizeof(T);
    auto fld = [&](int f) -> T {
      if constexpr (sizeof(T) == sizeof(float))
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(rb + (int64_t)f * rs) + lb);
      else
        return r[f * rs];
    };
#pragma unroll
    for (int s = 0; s < NS; ++s) st.val[h][s] = fld(s);
    if constexpr (sizeof(T) == sizeof(double)) {
      st.val[h][NS] = fld(NS + sy);
      st.val[h][NS + 1] = fld(2 * NS + sz);
    } else {
      // FP32: the record's y-z weight product, formed once for its ns lanes
      st.val[h][NS] = fld(NS + sy) * fld(2 * NS + sz);
      st.val[h][NS + 1] = (T)0;
    }
    st.val[h][NS + 2] = fld(KV);
    st.val[h][NS + 3] = fld(KV + 1);
    st.val[h][NS + 4] = fld(KV + 2);
    const T bx = fld(KB);
    // x slot of lane 0: sx = lane + (x0 + ns - 1 - kx)
    st.xs[h] = x0 + NS - 1 - ((int)bx - blo0);
  }
}

template <typename T, int NS>
__global__ void __launch_bounds__(64) k_p2m_rows(PGeom g, const int *start, const T *rec, int64_t rs, T *mesh,
                                                 int accumulate) {
  constexpr int NV = RowStage<T, NS>::NV, NR = NS * NS;
  constexpr bool F64 = sizeof(T) == sizeof(double);
  __shared__ T lds[NV][kRowCap];
  __shared__ int ldsx[kRowCap];
  const int lane = threadIdx.x;
  // XCD-aware line order: the workgroups of one XCD take consecutive lines
  // (x fastest, then y, then z), so that the record rows neighbouring lines
  // share are fetched into that XCD's L2 once rather than into every XCD's
  const int64_t lt = xcd_tile(block_linear(), (int64_t)gridDim.x * gridDim.y * gridDim.z);
  const int x0 = (int)(lt % gridDim.x) * 64, iy = (int)((lt / gridDim.x) % gridDim.y),
            iz = (int)(lt / ((int64_t)gridDim.x * gridDim.y));
  const int ix = x0 + lane;
  const bool node_ok = ix < g.E[0];
  const int x1 = min(x0 + 64 + NS - 2, g.nb[0] - 1);
  const int blo0 = g.blo[0];
  // start[] offset of stencil row r: (ky, kz) = (iy + r % ns, iz + r / ns)
  auto krow = [&](int r) { return g.nb[0] * ((iy + r % NS) + g.nb[1] * (iz + r / NS)); };
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  Kahan f0, f1, f2;
  float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f;
  auto to_lds = [&](const RowStage<T, NS> &st, int m) {
#pragma unroll
    for (int h = 0; h < kRowCap / 64; ++h) {
      const int i = lane + 64 * h;
      if (i < m) {
#pragma unroll
        for (int v = 0; v < NV; ++v) lds[v][i] = st.val[h][v];
        ldsx[i] = st.xs[h];
      }
    }
  };
  // sum the lane's records t in [lo, hi) staged from record `base` on: the
  // first 8 as straight-line predicated code (no loop for the wait counters
  // to drain pending loads in front of), the rest in a loop
  auto term = [&](int i) {
    const int sx = lane + ldsx[i];   // in [0, ns) for the lane's bins
    const T wx = lds[sx][i];
    if constexpr (F64) {
      const double w = __dmul_rn(__dmul_rn(wx, lds[NS][i]), lds[NS + 1][i]);
      d0 = __dadd_rn(d0, __dmul_rn(w, lds[NS + 2][i]));
      d1 = __dadd_rn(d1, __dmul_rn(w, lds[NS + 3][i]));
      d2 = __dadd_rn(d2, __dmul_rn(w, lds[NS + 4][i]));
    } else {
      const float w = wx * lds[NS][i];
      r0 = __fmaf_rn(w, lds[NS + 2][i], r0);
      r1 = __fmaf_rn(w, lds[NS + 3][i], r1);
      r2 = __fmaf_rn(w, lds[NS + 4][i], r2);
    }
  };
  // FP32: a stencil row's terms (at most ns records per lane on a remeshed
  // set) go into one partial sum, and the row partials are Kahan-added
  auto row_done = [&]() {
    if constexpr (!F64) {
      f0.add(r0);
      f1.add(r1);
      f2.add(r2);
      r0 = r1 = r2 = 0.0f;
    }
  };
  auto sum = [&](int lo, int hi, int base) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (lo + u < hi) term(lo + u - base);
    for (int t = lo + 8; t < hi; ++t) term(t - base);
  };
  // every row's record range, loaded up front: uniform [rt0, rt1) over the
  // line's bins, per lane [ra0, ra1) over the lane's bins [ix, ix + ns)
  int rt0[NR], rt1[NR], ra0[NR], ra1[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int k = krow(r);
    // the line's range is the same for every lane: keep it in scalar registers
    rt0[r] = __builtin_amdgcn_readfirstlane(start[k + x0]);
    rt1[r] = __builtin_amdgcn_readfirstlane(start[k + x1 + 1]);
    ra0[r] = node_ok ? start[k + ix] : 0;
    ra1[r] = node_ok ? start[k + ix + NS] : 0;
  }
  int total = 0;
#pragma unroll
  for (int r = 0; r < NR; ++r) total += rt1[r] - rt0[r];
  if (total > 0) {
    // rows in order (the loop is unrolled: every index is static); row r + 1's
    // first pass loads while row r is summed
    RowStage<T, NS> cur, nxt;
    row_fetch<T, NS>(cur, rec, rs, rt0[0], min(rt1[0] - rt0[0], kRowCap), lane, NS - 1, NS - 1, x0, blo0);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int T0 = rt0[r], n = rt1[r] - rt0[r], a0 = ra0[r], a1 = ra1[r];
      const int sy = NS - 1 - r % NS, sz = NS - 1 - r / NS;
      if (n > 0) {
        to_lds(cur, min(n, kRowCap));
        __syncthreads();
      }
      if (r + 1 < NR)
        row_fetch<T, NS>(nxt, rec, rs, rt0[min(r + 1, NR - 1)], min(rt1[min(r + 1, NR - 1)] - rt0[min(r + 1, NR - 1)], kRowCap),
                         lane, NS - 1 - (r + 1) % NS, NS - 1 - (r + 1) / NS, x0, blo0);
      if (n > 0) {
        sum(a0, min(a1, T0 + kRowCap), T0);
        __syncthreads();
        for (int p = kRowCap; p < n; p += kRowCap) {   // rows of more than kRowCap records
          const int m = min(n - p, kRowCap);
          row_fetch<T, NS>(cur, rec, rs, T0 + p, m, lane, sy, sz, x0, blo0);
          to_lds(cur, m);
          __syncthreads();
          sum(max(a0, T0 + p), min(a1, T0 + p + m), T0 + p);
          __syncthreads();
        }
        row_done();
      }
      cur = nxt;
    }
  }
  if (node_ok) {
    T *m = mesh + 3 * ((int64_t)ix + (int64_t)g.E[0] * (iy + (int64_t)g.E[1] * iz));
    const T a[3] = {F64 ? (T)d0 : (T)f0.s, F64 ? (T)d1 : (T)f1.s, F64 ? (T)d2 : (T)f2.s};
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c] = accumulate ? m[c] + a[c] : a[c];
  }
}

// Deposition gather: one wavefront marches along y over a column of 64 x nodes
// (node ix = x0 + lane) and QZ z nodes, with no other wavefront's help.
//
// A node is reached by the ns x ns bin rows (by, bz) = (iy + a, iz + b), a, b
// < ns, and in a row by the bins [ix, ix + ns), one contiguous range of the
// sorted particles.  At step by the wavefront takes the QZ + ns - 1 bin rows
// of its z nodes one after the other: the row's particles (read through the
// sorted ids) are turned into kernel weights once, a lane per particle, and
// put into LDS; then each lane adds the particles of its own bins to its
// column's ns y nodes by the row's (static, 1 to ns) z nodes, ns nz FP64
// triples in registers.  The y node that no later row reaches is stored and
// the window shifted.  A particle's x weight and z products are thus formed
// once for ns y nodes, and a row is staged (QZ + ns - 1) / QZ times rather
// than ns^2 times as in k_p2m_rows, which LDS reads bound.  Whole depositions
// of 2.1M particles on 128^3: FP64 531 us with line wavefronts (the records
// 100, the lines 385 of them), 222 with this; M6* FP32 160^3 2142, 604.
// The loads of a row run ahead of it: row bounds three rows, ids two,
// positions and strengths one.
// Sums and weights are FP64 for both mesh precisions, in a fixed order (rows
// ascending in by, then bz; particles by bin, then id): deterministic, no
// atomics on the mesh.
// What bounds it: vector issue, about 3 + 3 nz + 3 ns nz operations per
// particle and row, is half of it (128^3 M'4: 60 M wavefront instructions on
// 1,024 SIMDs, 97 us on average and 108 on a SIMD with three wavefronts, of
// 187); the rest is latency, since one round of two or three wavefronts per
// SIMD leaves nothing to fill a stalled or finished one, and lanes that wait
// for the fullest of their row.
constexpr int kMarchWaves = 4;   // per block, one for each SIMD of a CU (they share nothing; 128^3 one: 243 us, four: 218)
constexpr int kMarchCap = 96;   // particles of a row staged at a time (lanes below 32 take two)

// kernel weights at offset d in [0, 1) (interp_particle_mesh.f:182-214, :565-602)
// in fused form, ns = 4 (e = 1 - d): -d e^2 / 2, 1 + d^2 (3/2 d - 5/2),
// 1 + e^2 (3/2 e - 5/2), -d^2 e / 2
template <int NS> __device__ __forceinline__ void p2m_weights(double d, double *w) {
  if constexpr (NS == 4) {
    const double e = 1.0 - d, d2 = d * d, e2 = e * e;
    w[0] = -0.5 * d * e2;
    w[1] = __fma_rn(d2, __fma_rn(1.5, d, -2.5), 1.0);
    w[2] = __fma_rn(e2, __fma_rn(1.5, e, -2.5), 1.0);
    w[3] = -0.5 * d2 * e;
  } else {
#pragma unroll
    for (int s = 0; s < NS; ++s) w[s] = weight(1, s, d);
  }
}

// the particles lane and 64 + lane of a bin row's segment
struct RowData {
  double x[2][3], v[2][3];
};

// Tile block of workgroup b, n in all: one run of consecutive blocks on each
// XCD, whose rows they share in its L2, or, for particles in a part of the mesh,
// up to kMarchRuns shorter ones, so that the part is work for every XCD.  Reaches
// every block of [0, n) once for b < n + 8 kMarchRuns.
__device__ __forceinline__ int64_t march_block(int64_t b, int64_t n, int runs) {
  const int64_t len = (n + 8 * runs - 1) / (8 * runs), x = b % 8, k = b / 8;
  return (k / len * 8 + x) * len + k % len;
}

template <typename T, int NS>
__global__ void __launch_bounds__(64 * kMarchWaves)
    k_p2m_march(PGeom g, const int *__restrict__ start, const int *__restrict__ ids, const double *__restrict__ pos,
                const double *__restrict__ val, MarchTiles mt, const int *__restrict__ filled, T *__restrict__ mesh,
                int accumulate) {
  constexpr int QZ = kMarchQz, NR = QZ + NS - 1;   // bin rows per step
  constexpr int NF = 3 * NS + 3;    // staged fields: x, y, z weights, strength
  __shared__ double lds_all[kMarchWaves][NF][kMarchCap];
  __shared__ int wxo_all[kMarchWaves][kMarchCap];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double (*lds)[kMarchCap] = lds_all[wave];
  // lane 0's x weight (a slot the particle may not have), in words from its column
  int *wxo = wxo_all[wave];
  // neighbouring columns, x fastest, then y, then z
  const int width = mt.width, nx = mt.nx;
  const int ychunk = mt.chunk_of(g.E[1], NS, *filled), ny = (g.E[1] + ychunk - 1) / ychunk;
  const int64_t tiles = mt.tiles(g.E[1], ychunk);
  const int64_t lt =
      march_block(blockIdx.x, (tiles + kMarchWaves - 1) / kMarchWaves, mt.runs(*filled)) * kMarchWaves +
      __builtin_amdgcn_readfirstlane(wave);
  if (lt >= tiles) return;
  const int x0 = (int)(lt % nx) * width;
  const int y0 = (int)((lt / nx) % ny) * ychunk, iz0 = (int)(lt / ((int64_t)nx * ny)) * QZ;
  const int y1 = min(y0 + ychunk, g.E[1]);
  const int ix = x0 + lane;
  const bool node_ok = lane < width && ix < g.E[0];
  const int xe = min(x0 + width + NS - 1, g.nb[0]);   // one past the segment's last bin
  // start[] offset of bin row bzr of step by; a row outside the mesh's bins or
  // past the march takes that of the first row (and is not used: no_row)
  auto no_row = [&](int by, int bzr) { return by >= y1 + NS - 1 || iz0 + bzr >= g.nb[2]; };
  auto row_key = [&](int by, int bzr) {
    return no_row(by, bzr) ? 0 : g.nb[0] * (by + g.nb[1] * (iz0 + bzr));
  };
  // no particle reaches the tile: its nodes take zeros, without a march (not
  // looked for in a set that fills the mesh)
  bool some = mt.fills(*filled);
  if (!some)
    for (int i = lane; i < (y1 - y0 + NS - 1) * NR; i += 64) {
      const int k = row_key(y0 + i / NR, i % NR);
      some = some || (!no_row(y0 + i / NR, i % NR) && start[k + xe] != start[k + x0]);
    }
  if (!__any(some)) {
    const int words = 3 * min(width, g.E[0] - x0);
    for (int r = 0; r < (y1 - y0) * QZ; ++r) {
      const int iy = y0 + r / QZ, iz = iz0 + r % QZ;
      if (iz >= g.E[2]) continue;
      T *m = mesh + 3 * ((int64_t)x0 + (int64_t)g.E[0] * (iy + (int64_t)g.E[1] * iz));
      for (int c = lane; c < words; c += 64) m[c] = accumulate ? (T)((double)m[c] + 0.0) : (T)0;
    }
    return;
  }
  double acc[NS][QZ][3];
#pragma unroll
  for (int j = 0; j < NS; ++j)
#pragma unroll
    for (int q = 0; q < QZ; ++q)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[j][q][c] = 0.0;

  // The loads have no branches (a load behind one is waited for where its
  // paths join).  Particle p + lane and p + 64 + lane of a segment of n from
  // t0: the sorted slot, slot 0 past the segment's end; its id as loaded; the
  // particle, number 0 where the slot was past the end (it exists, and what is
  // staged for it is never read).
  auto in_row = [&](int n, int p, int h) {
    return p + 64 * h + lane < n && (h == 0 || lane < kMarchCap - 64);
  };
  auto load_ids = [&](int t0, int n, int p, int *id) {
#pragma unroll
    for (int h = 0; h < 2; ++h) id[h] = ids[in_row(n, p, h) ? t0 + p + 64 * h + lane : 0];
  };
  auto load_data = [&](const int *id, int n, int p, RowData &r) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t q = in_row(n, p, h) ? id[h] : 0;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        r.x[h][c] = pos[3 * q + c];
        r.v[h][c] = val[3 * q + c];
      }
    }
  };
  // the range of the lane's own bins [ix, ix + ns)
  auto load_bins = [&](int k, int *a) {
    a[0] = start[k + (node_ok ? ix : 0)];
    a[1] = start[k + (node_ok ? ix + NS : 0)];
  };
  auto fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // weights of m particles into LDS
  auto stage = [&](const RowData &r, int m) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h == 1 && m <= 64) break;
      const int i = lane + 64 * h;
      if (h == 0 || lane < kMarchCap - 64) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double x = r.x[h][d];
          const int b = cell_index_near(x, g.xmin[d], g.c1dx[d]);
          double w[NS];
          p2m_weights<NS>(stencil_offset(x, g.xmin[d], g.dx[d], b, g.c1dx[d]), w);
#pragma unroll
          for (int s = 0; s < NS; ++s) lds[d * NS + s][i] = w[s];
          if (d == 0) wxo[i] = (x0 + NS - 1 - (b - g.blo[0])) * kMarchCap;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) lds[3 * NS + c][i] = r.v[h][c];
      }
    }
  };

  // The rows' loads run ahead of their sums: the bounds of a row's segment by
  // three rows (raw until they are used, so that nothing waits for them), its
  // ids by two, its particles and the lanes' bin ranges by one.
  auto raw = [&](int by, int bzr, int *r) {
    const int k = row_key(by, bzr);
    r[0] = start[k + x0];
    r[1] = start[no_row(by, bzr) ? x0 : k + xe];
  };
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  int rb[2];
  raw(y0, 0, rb);
  int t0 = uni(rb[0]), n0 = uni(rb[1]) - t0;   // the row to sum
  raw(y0 + 1 / NR, 1 % NR, rb);
  int t1 = uni(rb[0]), n1 = uni(rb[1]) - t1;   // the next row
  raw(y0 + 2 / NR, 2 % NR, rb);
  int id[2], idn[2], bins[2];
  RowData data;
  load_ids(t0, n0, 0, id);
  load_bins(row_key(y0, 0), bins);
  load_data(id, n0, 0, data);
  load_ids(t1, n1, 0, idn);
  for (int by = y0; by < y1 + NS - 1; ++by) {
#pragma unroll
    for (int bzr = 0; bzr < NR; ++bzr) {
      // z nodes of the row: q in [q0, q1], slot ns - 1 - (bzr - q)
      const int q0 = bzr - (NS - 1) > 0 ? bzr - (NS - 1) : 0, q1 = bzr < QZ - 1 ? bzr : QZ - 1;
      const int n = n0, tn = t0;
      const int a0 = bins[0] - tn, a1 = bins[1] - tn;
      if (n > 0) stage(data, min(n, kMarchCap));
      // run ahead
      t0 = t1;
      n0 = n1;
      t1 = uni(rb[0]);
      n1 = uni(rb[1]) - t1;
      id[0] = idn[0];
      id[1] = idn[1];
      load_data(id, n0, 0, data);
      load_bins(row_key(by + (bzr + 1) / NR, (bzr + 1) % NR), bins);
      load_ids(t1, n1, 0, idn);
      raw(by + (bzr + 3) / NR, (bzr + 3) % NR, rb);
      // the lane's particles i in [lo, hi) of the segment, staged from p on;
      // a particle's x slot is its own (wxo) plus the lane
      auto sum = [&](int lo, int hi, int p) {
        for (int i = lo - p; i < hi - p; ++i) {
          const double *r = &lds[0][i];
          const double wx = r[lane * kMarchCap + wxo[i]];
          const double v0 = wx * r[3 * NS * kMarchCap], v1 = wx * r[(3 * NS + 1) * kMarchCap],
                       v2 = wx * r[(3 * NS + 2) * kMarchCap];
          double wy[NS];
#pragma unroll
          for (int j = 0; j < NS; ++j) wy[j] = r[(NS + j) * kMarchCap];
#pragma unroll
          for (int q = 0; q < QZ; ++q)
            if (q >= q0 && q <= q1) {
              const double wz = r[(2 * NS + NS - 1 - (bzr - q)) * kMarchCap];
              const double u0 = wz * v0, u1 = wz * v1, u2 = wz * v2;
#pragma unroll
              for (int j = 0; j < NS; ++j) {
                acc[j][q][0] = __fma_rn(wy[j], u0, acc[j][q][0]);
                acc[j][q][1] = __fma_rn(wy[j], u1, acc[j][q][1]);
                acc[j][q][2] = __fma_rn(wy[j], u2, acc[j][q][2]);
              }
            }
        }
      };
      if (n > 0) {
        fence();
        sum(a0, min(a1, kMarchCap), 0);
        fence();
        // rows of more than kMarchCap particles: the rest, not run ahead
        for (int p = kMarchCap; p < n; p += kMarchCap) {
          int idp[2];
          RowData dp;
          const int m = min(n - p, kMarchCap);
          load_ids(tn, n, p, idp);
          load_data(idp, n, p, dp);
          stage(dp, m);
          fence();
          sum(max(a0, p), min(a1, p + m), p);
          fence();
        }
      }
    }
    // node iy = by - (ns - 1) has all its rows
    const int iy = by - (NS - 1);
    if (iy >= y0 && node_ok) {
#pragma unroll
      for (int q = 0; q < QZ; ++q)
        if (iz0 + q < g.E[2]) {
          T *m = mesh + 3 * ((int64_t)ix + (int64_t)g.E[0] * (iy + (int64_t)g.E[1] * (iz0 + q)));
#pragma unroll
          for (int c = 0; c < 3; ++c) m[c] = accumulate ? (T)((double)m[c] + acc[0][q][c]) : (T)acc[0][q][c];
        }
    }
#pragma unroll
    for (int j = 0; j + 1 < NS; ++j)
#pragma unroll
      for (int q = 0; q < QZ; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[j][q][c] = acc[j + 1][q][c];
#pragma unroll
    for (int q = 0; q < QZ; ++q)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[NS - 1][q][c] = 0.0;
  }
}

// Reverse periodic halo along axis d (mesh/pmlib_mesh_map_ghost.f with
// incl_edges = .TRUE., op = add): cells [0, 2ng) and [N, N + 2ng) exchange
// and add, both read before either is written.
template <typename T> __global__ void k_halo_add(T *m, PGeom g, int d) {
  const int E0 = g.E[0], E1 = g.E[1];
  int o1 = d == 0 ? 1 : 0, o2 = d == 2 ? 1 : 2;
  int64_t st[3] = {3, 3 * (int64_t)E0, 3 * (int64_t)E0 * E1};
  const int ng = g.ngl[d], N = g.ncell[d];
  int64_t n = (int64_t)g.E[o1] * g.E[o2] * 3 * 2 * ng;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int c = idx % 3;
    int64_t r = idx / 3;
    int t = r % (2 * ng);
    r /= 2 * ng;
    int a1 = r % g.E[o1];
    int a2 = r / g.E[o1];
    int64_t base = c + st[o1] * a1 + st[o2] * a2;
    T lo = m[base + st[d] * t], hi = m[base + st[d] * (N + t)];
    m[base + st[d] * t] = lo + hi;
    m[base + st[d] * (N + t)] = hi + lo;
  }
}

// M2P: one thread per particle, the reference's term order
// (interp_mesh_particle.f:87-409: sz, sy, sx ascending; the M'4 branch scales
// the y and z offsets by 1/dx(1), the M6* branch reproduces the k5/k6 quirk of
// :587-590), FP64 rounded per operation as the reference does; the FP32 form
// (FP32 mesh) takes FP32 weights, forms their product in FP64 and sums the
// weighted FP32 node values in FP64 (the output is FP64; one fused
// multiply-add per term and component, against four FP32 operations of a
// compensated FP32 sum).
// Stencil weights and indices live in registers (the stencil width is a
// template parameter).
//
// What bounds it: the L1, which takes about 16 cycles per load instruction of a
// wavefront, however narrow.  A stencil row's ns nodes lie side by side, so a
// row is read as the one run of 3 ns words they make (M'4: 6 dwordx4 in FP64, 3
// in FP32) instead of node by node (8 and 4 loads).  us before and now, a full
// set moved by a smooth flow of up to half a cell: 128^3 FP64 M'4 periodic 191,
// 149, free 189, 155; M6* free 572, 475; FP32 M'4 92, 75 and 104, 97; M6* free
// 322, 283; 384^3 FP32 2270, 2020.  The gathers of a two-ring step from
// jittered centres: 128^3 free FP64 244, 189, FP32 126, 118.
// (64^3 FP32 M6* free: 52, 56; its clamped lanes are a larger share.)
// Wavefronts with a stencil that leaves the mesh along x (clamped indices) move
// those lanes' runs inside and their x weights along.
// a stencil row: 3 ns words side by side, read 16 bytes at a time from any word
template <typename T, int NS> struct M2PRow {
  static constexpr int NW = 3 * NS * (int)sizeof(T) / 4, N4 = NW / 4, N1 = NW % 4;
  typedef unsigned Quad __attribute__((ext_vector_type(4), aligned(4)));
  typedef unsigned Pair __attribute__((ext_vector_type(2), aligned(4)));
  static_assert(N1 == 0 || N1 == 2);
  Quad q[N4];
  Pair p;
  __device__ __forceinline__ void load(const T *m) {
    const unsigned *u = reinterpret_cast<const unsigned *>(m);
#pragma unroll
    for (int i = 0; i < N4; ++i) q[i] = *reinterpret_cast<const Quad *>(u + 4 * i);
    if constexpr (N1 == 2) p = *reinterpret_cast<const Pair *>(u + 4 * N4);
  }
  __device__ __forceinline__ void get(T (&v)[NS][3]) const {
    auto word = [&](int i) { return i < 4 * N4 ? q[i / 4][i % 4] : p[i % 2]; };
#pragma unroll
    for (int i = 0; i < 3 * NS; ++i) {
      if constexpr (sizeof(T) == 8)
        v[i / 3][i % 3] = __builtin_bit_cast(double, ((uint64_t)word(2 * i + 1) << 32) | word(2 * i));
      else
        v[i / 3][i % 3] = __builtin_bit_cast(float, word(i));
    }
  }
};

template <typename T, int NS>
__global__ void __launch_bounds__(256) k_m2p(PGeom g, const T *mesh, const double *pos, NCount npc, double *out) {
  const int64_t np = npc.get();
  constexpr bool F64 = sizeof(T) == sizeof(double);
  constexpr bool M6 = NS == 6;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < np; q += (int64_t)gridDim.x * blockDim.x) {
    int idx[3][NS], i0x = 0;
    T w[3][NS];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double x = pos[3 * q + d];
      const int b = cell_index(x, g.xmin[d], g.c1dx[d]);
      // the reference normalises every axis by 1/dx of x for M'4
      const double nrm = M6 ? g.c1dx[d] : g.c1dx[0];
      const double dd = stencil_offset(x, g.xmin[d], g.dx[d], b, nrm);
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        if constexpr (F64)
          w[d][s2] = weight(M6, s2, dd);
        else
          w[d][s2] = weight_f(M6, s2, (float)dd);
        idx[d][s2] = b - g.off + s2;
      }
      if (d == 0) i0x = b - g.off;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        if (idx[d][s2] < g.lo[d]) {
          if (M6 && d == 2 && s2 >= 4) {   // the reference's M6* quirk on the y slots
            w[1][s2] = (T)0;
            idx[1][s2] = g.lo[2];
          }
          w[d][s2] = (T)0;
          idx[d][s2] = g.lo[d];
        }
        if (idx[d][s2] > g.hi[d]) {
          w[d][s2] = (T)0;
          idx[d][s2] = g.hi[d];
        }
      }
    // The quirk can leave a y index outside the y range (when the z axis has
    // more ghost layers); its weight is zero, so the read is clamped into the
    // mesh instead of leaving the allocation.
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2) idx[1][s2] = min(max(idx[1][s2], g.lo[1]), g.hi[1]);
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    // x run of the stencil: nodes xb .. xb + ns - 1 of the mesh, node j of it the
    // stencil's j - k0 (k0 = 0: no x index clamped)
    const int xb = min(max(i0x, g.lo[0]), g.hi[0] - NS + 1), k0 = i0x - xb;
    // one stencil row's sums
    auto add_row = [&](int r, const T (&mv)[NS][3]) {
      const int sy = r % NS, sz = r / NS;
      // FP32 form: the FP32 weights' product in FP64, y and z once per row
      const double wyz = F64 ? 0.0 : (double)w[1][sy] * (double)w[2][sz];
#pragma unroll
      for (int sx = 0; sx < NS; ++sx) {
        const T *m = mv[sx];
        if constexpr (F64) {
          const double wt = __dmul_rn(__dmul_rn(w[0][sx], w[1][sy]), w[2][sz]);
          const double t0 = __dmul_rn(wt, m[0]), t1 = __dmul_rn(wt, m[1]), t2 = __dmul_rn(wt, m[2]);
          if (r == 0 && sx == 0) {   // the first term starts the sums
            a0 = t0;
            a1 = t1;
            a2 = t2;
          } else {
            a0 = __dadd_rn(a0, t0);
            a1 = __dadd_rn(a1, t1);
            a2 = __dadd_rn(a2, t2);
          }
        } else {
          // weight times FP32 node value fused into the FP64 sum
          const double wt = (double)w[0][sx] * wyz;
          a0 = __fma_rn(wt, (double)m[0], a0);
          a1 = __fma_rn(wt, (double)m[1], a1);
          a2 = __fma_rn(wt, (double)m[2], a2);
        }
      }
    };
    // (indices and weights are hidden from the compiler in each of the two
    // forms: it would form the rows' addresses and products ahead of both)
    auto hide = [&] {
#pragma unroll
      for (int t = 0; t < NS; ++t)
        asm volatile("" : "+v"(idx[1][t]), "+v"(idx[2][t]), "+v"(w[1][t]), "+v"(w[2][t]));
    };
    auto row_at = [&](int r) {
      return 3 * ((int64_t)g.E[0] * ((idx[1][r % NS] - g.lo[1]) + (int64_t)g.E[1] * (idx[2][r / NS] - g.lo[2])));
    };
    // stencil rows r = (sz, sy) in order, G rows at a time: a group's rows are
    // all loaded before any is summed, and the scheduling barriers keep the
    // compiler from moving loads back beside their uses or hoisting the next
    // group's loads over this group's sums (register use stays bounded)
    constexpr int G = F64 ? (M6 ? 1 : 2) : 2;
    auto sum_rows = [&](auto clamped) {
      hide();
      constexpr bool CL = decltype(clamped)::value;
      const T *mx = mesh + 3 * (xb - g.lo[0]);
      bool in[NS];   // node j of the run is one of the stencil's
      if constexpr (CL) {
        T wx[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
          in[j] = j - k0 >= 0 && j - k0 < NS;
          wx[j] = (T)0;
#pragma unroll
          for (int t = 0; t < NS; ++t) wx[j] = j - k0 == t ? w[0][t] : wx[j];
        }
#pragma unroll
        for (int j = 0; j < NS; ++j) w[0][j] = wx[j];
      }
#pragma unroll
      for (int r0 = 0; r0 < NS * NS; r0 += G) {
        M2PRow<T, NS> mv[G];
#pragma unroll
        for (int k = 0; k < G; ++k) mv[k].load(mx + row_at(r0 + k));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < G; ++k) {
          T v[NS][3];
          mv[k].get(v);
          if constexpr (CL) {
            // the clamped nodes repeat the run's end with weight 0 (which an
            // infinity or NaN there turns into NaN); a node of the run that is
            // none of the stencil's adds nothing, whatever it holds
            T e[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) e[c] = k0 == 0 ? (T)0 : (k0 < 0 ? v[0][c] : v[NS - 1][c]);
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
              for (int c = 0; c < 3; ++c) v[j][c] = in[j] ? v[j][c] : (T)0;
            add_row(r0 + k, v);
            a0 += 0.0 * (double)e[0];
            a1 += 0.0 * (double)e[1];
            a2 += 0.0 * (double)e[2];
          } else {
            add_row(r0 + k, v);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto gather_rows = [&] {
      hide();
#pragma unroll
      for (int r0 = 0; r0 < NS * NS; r0 += G) {
        T mv[G][NS][3];
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const T *mrow = mesh + row_at(r0 + k);
#pragma unroll
          for (int sx = 0; sx < NS; ++sx)
#pragma unroll
            for (int c = 0; c < 3; ++c) mv[k][sx][c] = mrow[3 * (idx[0][sx] - g.lo[0]) + c];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < G; ++k) add_row(r0 + k, mv[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (g.E[0] < NS)
      gather_rows();
    else if (__any(k0 != 0))
      sum_rows(std::true_type());
    else
      sum_rows(std::false_type());
    out[3 * q] = a0;
    out[3 * q + 1] = a1;
    out[3 * q + 2] = a2;
  }
}

static __global__ void k_cell_index(PGeom g, const double *pos, int64_t np, int *out) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < 3 * np; q += (int64_t)gridDim.x * blockDim.x) {
    int d = q % 3;
    out[q] = cell_index(pos[q], g.xmin[d], g.c1dx[d]);
  }
}

// ------------------------------------------------------------ remesh
// flag of mesh cell idx (remesh/pmlib_remesh.f:104-125)
template <typename T>
__device__ __forceinline__ int remesh_flag(const PGeom &g, int64_t idx, const T *vort, const T *dvort,
                                           const uint8_t *mask, double min_vort, double min_dvort,
                                           int incl_ghost) {
  int ii[3];
  ii[0] = (int)(idx % g.E[0]) + g.lo[0];
  ii[1] = (int)((idx / g.E[0]) % g.E[1]) + g.lo[1];
  ii[2] = (int)(idx / ((int64_t)g.E[0] * g.E[1])) + g.lo[2];
  for (int d = 0; d < 3; ++d) {
    bool in = ii[d] >= 1 && ii[d] <= g.ncell[d];
    bool gh = incl_ghost && g.bc[d] == 0;
    if (!(in || gh)) return 0;
  }
  const T *v = vort + 3 * idx;
  T s = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  T ds = 0;
  if (dvort) {
    const T *u = dvort + 3 * idx;
    ds = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
  }
  if (!(s > min_vort || ds > min_dvort)) return 0;
  return mask ? (mask[idx] ? 1 : 0) : 1;
}

template <typename T>
__global__ void k_remesh_flags(PGeom g, const T *vort, const T *dvort, const uint8_t *mask,
                               double min_vort, double min_dvort, int incl_ghost, int *flag) {
  const int64_t nn = (int64_t)g.E[0] * g.E[1] * g.E[2];
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < nn;
       idx += (int64_t)gridDim.x * blockDim.x)
    flag[idx] = remesh_flag(g, idx, vort, dvort, mask, min_vort, min_dvort, incl_ghost);
}

// create particles at cell centres in (k, j, i) order from the scanned flags;
// vel / dvort are the fields copied (NULL: zero), per the vel / dvort flags.
// A workgroup takes 256 consecutive cells at a time: their particles are one
// contiguous range of the outputs, staged in LDS and then written with
// consecutive threads on consecutive words.  Launched with 256 threads.
// np (or null) takes the count, capped (err, bit 1: over capacity).
constexpr int kRemeshTile = 256;
template <typename T>
__global__ void __launch_bounds__(kRemeshTile) k_remesh_create(PGeom g, const int *flag, const int *offs,
                                                               const T *vort, const T *dvort, const T *vel,
                                                               double *pos, double *pvort, double *pvel,
                                                               double *pdvort, double *vel_rk, double *dvort_rk,
                                                               int64_t cap, int *np, int *err) {
  __shared__ double stage[4][3 * kRemeshTile];   // pos, vort, vel, dvort of the tile's particles
  const int64_t nn = (int64_t)g.E[0] * g.E[1] * g.E[2];
  const int64_t ntiles = (nn + kRemeshTile - 1) / kRemeshTile;
  const int tid = threadIdx.x;
  if (np && blockIdx.x == 0 && tid == 0) {
    const int64_t t = offs[nn];
    if (t > cap) atomicOr(err, 1);
    *np = (int)(t > cap ? cap : t);
  }
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t c0 = tile * kRemeshTile, idx = c0 + tid;
    const int64_t p0 = offs[c0], p1 = offs[min(c0 + kRemeshTile, nn)];
    if (idx < nn && flag[idx]) {
      const int s = (int)(offs[idx] - p0);
      int ii[3];
      ii[0] = (int)(idx % g.E[0]) + g.lo[0];
      ii[1] = (int)((idx / g.E[0]) % g.E[1]) + g.lo[1];
      ii[2] = (int)(idx / ((int64_t)g.E[0] * g.E[1])) + g.lo[2];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        stage[0][3 * s + d] = __dadd_rn(g.xmin[d], __dmul_rn(__dadd_rn((double)(ii[d] - 1), 0.5), g.dx[d]));
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        stage[1][3 * s + c] = (double)vort[3 * idx + c];
        stage[2][3 * s + c] = vel ? (double)vel[3 * idx + c] : 0.0;
        stage[3][3 * s + c] = dvort ? (double)dvort[3 * idx + c] : 0.0;
      }
    }
    __syncthreads();
    // words [3 p0, 3 p1) of every output, past the capacity dropped (the
    // caller reports an over-capacity count)
    const int64_t w0 = 3 * p0, w1 = 3 * (p1 < cap ? p1 : (p0 < cap ? cap : p0));
    for (int64_t wd = w0 + tid; wd < w1; wd += kRemeshTile) {
      const int k = (int)(wd - w0);
      pos[wd] = stage[0][k];
      pvort[wd] = stage[1][k];
      if (pvel) pvel[wd] = stage[2][k];
      if (pdvort) pdvort[wd] = stage[3][k];
      if (vel_rk) vel_rk[wd] = 0.0;
      if (dvort_rk) dvort_rk[wd] = 0.0;
    }
    __syncthreads();   // the stage is free for the next tile
  }
}

// ------------------------------------------------------------ advance
struct RkCoef {
  double a1, b1, c1, a2, b2, c2;
};

// the patch box [lo, hi) per axis; len: the period of a periodic axis, 0 on a
// free one (or where only outside or not is asked)
struct PBox {
  double lo[3], hi[3], len[3];
};

// the RK stage update of every particle word; with `outside` given, also
// flags a particle that the update leaves outside the box on any axis (bit 1),
// and one that is still outside after one wrap of a periodic axis (bit 2)
// dvort null: a zero right-hand side (dvort = dvort_rk = +0), dvort_rk is
// neither read nor written and vort takes the increment c2 dr that the full
// form rounds for those zeros, dr = a2 (+0) + (b2 dt) (+0)
static __global__ void k_rk_update(RkCoef k, double dt, NCount npc, double *pos, const double *vel, double *vort,
                                   const double *dvort, double *vel_rk, double *dvort_rk, PBox box, int *outside) {
  const int64_t np = npc.get();
  const bool rhs = dvort != nullptr;
  const double dinc = __dmul_rn(k.c2, __dadd_rn(__dmul_rn(k.a2, 0.0), __dmul_rn(__dmul_rn(k.b2, dt), 0.0)));
  // axis of word i, advanced with the grid stride (no 64-bit modulo)
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, s3 = (int)(((int64_t)gridDim.x * blockDim.x) % 3);
  int d = i0 % 3;
  for (int64_t i = i0; i < 3 * np; i += (int64_t)gridDim.x * blockDim.x, d = (d + s3) % 3) {
    double vr = __dadd_rn(__dmul_rn(k.a1, vel_rk[i]), __dmul_rn(__dmul_rn(k.b1, dt), vel[i]));
    vel_rk[i] = vr;
    const double x = __dadd_rn(pos[i], __dmul_rn(k.c1, vr));
    pos[i] = x;
    if (rhs) {
      double dr = __dadd_rn(__dmul_rn(k.a2, dvort_rk[i]), __dmul_rn(__dmul_rn(k.b2, dt), dvort[i]));
      dvort_rk[i] = dr;
      vort[i] = __dadd_rn(vort[i], __dmul_rn(k.c2, dr));
    } else {
      // (a zero increment changes -0 only: the store, 8 of 56 bytes per word,
      // falls away otherwise; 384^3 1.90 -> 1.56 ms)
      const double v = vort[i], w = __dadd_rn(v, dinc);
      if (__double_as_longlong(w) != __double_as_longlong(v)) vort[i] = w;
    }
    if (outside) {
      const bool o = x < box.lo[d] || x >= box.hi[d];
      const uint64_t m = __ballot(o);
      if (m) {
        const double y = x < box.lo[d] ? x + box.len[d] : x - box.len[d];
        const bool far = __any(o && box.len[d] != 0.0 && (y < box.lo[d] || y >= box.hi[d]));
        if ((threadIdx.x & 63) == __ffsll((unsigned long long)m) - 1) atomicOr(outside, far ? 3 : 1);
      }
    }
  }
}

}  // namespace pmgpu
