// Poisson passes for lengths without a compile-time specialisation, on the
// engine of pm_fft_any.h (see poisson_kernels.h for the data path and the
// argument structures).
#pragma once
#include "pm_fft_any.h"
#include "poisson_kernels.h"

namespace pmgpu {
namespace any {

// Strided complex pass: blockDim.x consecutive columns of one batch entry,
// each loaded and stored straight from and to global memory by the first and
// the last stage.
template <typename R, int S>
__global__ void __launch_bounds__(kAnyThreads, any_waves(2 * sizeof(R))) k_strided_a(StridedArgs a, AnyPlan pl, const cplx_t<R> *tw) {
  using V = cplx_t<R>;
  extern __shared__ unsigned char smem_raw[];
  V *lds = reinterpret_cast<V *>(smem_raw);
  const int T = blockDim.x, c = threadIdx.x, p = threadIdx.y;
  const int64_t lt = xcd_tile(block_linear(), (int64_t)gridDim.x * gridDim.y * gridDim.z);
  const int col0 = (int)(lt % gridDim.x) * T;
  const int64_t b = lt / gridDim.x;
  const bool ok = col0 + c < a.ncols;
  // rows [0, nin) of the columns from col0 on
  const V *in = reinterpret_cast<const V *>(a.in) + b * a.bs_in + col0;
  V *out = reinterpret_cast<V *>(a.out) + b * a.bs_out + col0 + c;
  const int64_t rsb = a.rs_in * (int64_t)sizeof(V);
  const RowsIn<V> ld{in, rsb, a.nin, (int)(kMostRecords / (uint32_t)rsb), ok ? c * (uint32_t)sizeof(V) : kOffColumn};
  const RowsOut<V> st{out, a.rs_out, a.nout, ok, (R)a.scale};
  fft_any<S, false>(pl, lds + c * any_stride(pl.L), p, blockDim.y, tw, ld, st);
}

// R2C along x: blockDim = (ncomp, P, T), T lines (y) of ncomp components.
// The first stage packs x[2n] + i x[2n+1]; the half-length spectrum stays in
// LDS for the pairing X[k] = (Z[k] + conj Z[Nh-k])/2 - i/2 W^k (Z[k] - conj Z[Nh-k]).
template <typename R> struct RealIn {
  const R *in;
  int64_t xs;
  int lim;   // reals of the line
  __device__ __forceinline__ auto at(int j, int step) const {
    const R *q = in + 2 * j * xs;
    const int64_t s = 2 * step * xs, x = xs;
    const int l = lim;
    return [q, s, x, j, step, l](int r) {
      cplx_t<R> v = cmake<cplx_t<R>>(0, 0);
      const int n2 = 2 * (j + r * step);
      if (n2 < l) v.x = q[r * s];
      if (n2 + 1 < l) v.y = q[r * s + x];
      return v;
    };
  }
};
template <typename R>
__global__ void __launch_bounds__(kAnyThreads, any_waves(2 * sizeof(R))) k_x_fwd_a(XFwdArgs a, AnyPlan pl, const cplx_t<R> *tw) {
  using V = cplx_t<R>;
  extern __shared__ unsigned char smem_raw[];
  V *lds = reinterpret_cast<V *>(smem_raw);
  const int Nh = pl.L, c = threadIdx.x, p = threadIdx.y, t = threadIdx.z;
  const int y = blockIdx.x * blockDim.z + t, z = blockIdx.y;
  const bool ok = y < a.My;
  V *line = lds + (t * blockDim.x + c) * any_stride(Nh);
  const R *in = reinterpret_cast<const R *>(a.in) + c * a.cs + (int64_t)y * a.ys + (int64_t)z * a.zs;
  fft_any<-1, false>(pl, line, p, blockDim.y, tw, RealIn<R>{in, a.xs, ok ? a.Min : 0}, LineOut<V>{line});
  __syncthreads();
  if (!ok) return;
  V *out = reinterpret_cast<V *>(a.out) + c * a.o_cs + (int64_t)y * a.o_ys + (int64_t)z * a.o_zs;
  const V *twL = tw + a.twL_off;
  for (int k = p; k <= Nh; k += blockDim.y) {
    const V zk = line[k == Nh ? 0 : k], zm = cconj(line[k == 0 ? 0 : Nh - k]);
    const V e = cscale(cadd(zk, zm), (R)0.5), wo = cmul(twL[k], cscale(csub(zk, zm), (R)0.5));
    out[k * a.o_ks] = cadd(e, cmake<V>(wo.y, -wo.x));
  }
}

// C2R along x, keeping x < Mout: the first stage forms Z[k] = (X[k] + conj
// X[Nh-k]) + i W^-k (X[k] - conj X[Nh-k]) from global memory (imaginary parts
// of X[0] and X[Nh] dropped), the last one stores the real pairs.
template <typename R> struct PairIn {
  const cplx_t<R> *xl, *twL;
  int64_t ks;
  int Nh;
  bool ok;
  __device__ __forceinline__ auto at(int j, int step) const {
    using V = cplx_t<R>;
    const V *qk = xl + j * ks, *qm = xl + (Nh - j) * ks, *w0 = twL + j;
    const int64_t s = step * ks;
    const bool g = ok;
    return [qk, qm, w0, s, j, step, g](int r) {
      if (!g) return cmake<V>(0, 0);
      V xk = qk[r * s], xm = qm[-(r * s)];
      if (j + r * step == 0) xk.y = xm.y = 0;
      const V e = cadd(xk, cconj(xm)), wd = cmul(cconj(w0[r * step]), csub(xk, cconj(xm)));
      return cadd(e, cmake<V>(-wd.y, wd.x));
    };
  }
};
template <typename R> struct RealOut {
  R *out;
  int64_t xs;
  int lim;
  R sc;
  __device__ __forceinline__ auto at(int n, int step) const {
    R *q = out + 2 * n * xs;
    const int64_t s = 2 * step * xs, x = xs;
    const int l = lim;
    const R c = sc;
    return [q, s, x, n, step, l, c](int r, const cplx_t<R> &v) {
      const int n2 = 2 * (n + r * step);
      if (n2 < l) q[r * s] = v.x * c;
      if (n2 + 1 < l) q[r * s + x] = v.y * c;
    };
  }
};
template <typename R>
__global__ void __launch_bounds__(kAnyThreads, any_waves(2 * sizeof(R))) k_x_inv_a(XInvArgs a, AnyPlan pl, const cplx_t<R> *tw) {
  using V = cplx_t<R>;
  extern __shared__ unsigned char smem_raw[];
  V *lds = reinterpret_cast<V *>(smem_raw);
  const int Nh = pl.L, c = threadIdx.x, p = threadIdx.y, t = threadIdx.z;
  const int y = blockIdx.x * blockDim.z + t, z = blockIdx.y;
  const bool ok = y < a.My;
  const V *xl = reinterpret_cast<const V *>(a.in) + c * a.i_cs + (int64_t)y * a.i_ys + (int64_t)z * a.i_zs;
  R *out = reinterpret_cast<R *>(a.out) + c * a.cs + (int64_t)y * a.ys + (int64_t)z * a.zs;
  fft_any<1, false>(pl, lds + (t * blockDim.x + c) * any_stride(Nh), p, blockDim.y, tw,
                    PairIn<R>{xl, tw + a.twL_off, a.i_ks, Nh, ok}, RealOut<R>{out, a.xs, ok ? a.Mout : 0, (R)a.scale});
}

// Fused z pass of one field (kind 0 velocity, 1 stream function, 2 filtered
// and, with reproj, reprojected vorticity): blockDim = (3 T, P), line l =
// 3 column + component, T consecutive kx columns of one ky row.  Forward
// transforms of the 3 T lines leave the spectra in LDS; each thread forms the
// three components of the field at wavenumbers of its own, so that G-hat and
// the wavenumbers are taken once per column and row; the lines are
// transformed back in place.
template <typename R>
__global__ void __launch_bounds__(kAnyThreads, 4)
    k_z3_a(ZArgs a, AnyPlan pl, const cplx_t<R> *tw, int kind, void *out) {
  using V = cplx_t<R>;
  extern __shared__ unsigned char smem_raw[];
  V *lds = reinterpret_cast<V *>(smem_raw);
  const int L = pl.L, st = any_stride(L), T = blockDim.x / 3;
  const int l = threadIdx.x, p = threadIdx.y, P = blockDim.y;
  const int col = l / 3, comp = l - 3 * col;
  const int64_t lt = xcd_tile(block_linear(), (int64_t)gridDim.x * gridDim.y);
  const int kx0 = (int)(lt % gridDim.x) * T, ky = (int)(lt / gridDim.x);
  const int kx = kx0 + col;
  const bool ok = kx < a.Hx;
  const int64_t tile = (int64_t)ky * a.kys + (int64_t)kx * a.kxs + comp * a.cs;
  // rows [0, Mz) of the tile's 3 T interleaved words (kxs = 3, cs = 1)
  const V *src = reinterpret_cast<const V *>(a.B) + (int64_t)ky * a.kys + (int64_t)kx0 * 3;
  const int64_t rsb = a.rs * (int64_t)sizeof(V);
  V *spec = lds + l * st;
  fft_any<-1, false>(pl, spec, p, P, tw,
                     RowsIn<V>{src, rsb, a.Mz, (int)(kMostRecords / (uint32_t)rsb),
                               ok ? l * (uint32_t)sizeof(V) : kOffColumn},
                     LineOut<V>{spec});
  __syncthreads();
  const R ki = wavenumber<R>(kx, a.Lx, a.dk[0], a.ksmp[0]);
  const R kj = wavenumber<R>(ky, a.Ly, a.dk[1], a.ksmp[1]);
  const bool nx = (2 * kx == a.Lx), ny = (2 * ky == a.Ly);
  const int kyf = ky <= a.Ly - ky ? ky : a.Ly - ky;
  const R pi = (R)3.14159265358979323846;
  const R twopi = (R)6.28318530717958647692;
  const int64_t gz = (int64_t)a.Hy * a.Hx, kz = (int64_t)a.Ly * a.Hx * 3;
  // a column past Hx reads column 0 (its lines are zero and not stored)
  const R *G = reinterpret_cast<const R *>(a.Ghat) + (int64_t)kyf * a.Hx + (ok ? kx : 0);
  const V *Kh = reinterpret_cast<const V *>(a.Ghat) + ((int64_t)ky * a.Hx + (ok ? kx : 0)) * 3;
  V *s0 = lds + 3 * col * st;
  const R kx_ = nx ? (R)0 : ki, ky_ = ny ? (R)0 : kj;
  // rows comp P + p + 3 P m of the column: one thread, three components
  for (int n = comp * P + p; n < L; n += 3 * P) {
    const R kk = wavenumber<R>(n, L, a.dk[2], a.ksmp[2]);
    const bool nz = (2 * n == L);
    const V w0 = s0[n], w1 = s0[st + n], w2 = s0[2 * st + n];
    R zeta = (R)1, g = (R)0;
    if (a.want_vort && (kind == 2 || a.allper))
      zeta = zeta_filter<R>(a.order, (R)a.eps2pi * sqrt(ki * ki + kj * kj + kk * kk));
    V r0, r1, r2;
    if (a.ker2) {
      // kernel 2: K = FFT(grad G) h^3, a complex half-spectrum
      const V *Kp = Kh + n * kz;
      const V K0 = cscale(Kp[0], (R)a.h3), K1 = cscale(Kp[1], (R)a.h3), K2 = cscale(Kp[2], (R)a.h3);
      if (kind == 0) {
        // u-hat = K x w-hat (poisson/pmlib_poisson_solve.f:898-900)
        r0 = csub(cmul(K1, w2), cmul(K2, w1));
        r1 = csub(cmul(K2, w0), cmul(K0, w2));
        r2 = csub(cmul(K0, w1), cmul(K1, w0));
      } else {
        r0 = cscale(w0, zeta);
        r1 = cscale(w1, zeta);
        r2 = cscale(w2, zeta);
        if (a.reproj) {
          // + K 2 pi i (k . w-hat) (:903-910); a Nyquist wavenumber drops
          // out of the Hermitian part
          V acc = cmake<V>(0, 0);
          if (!nx) acc = cadd(acc, cscale(w0, ki));
          if (!ny) acc = cadd(acc, cscale(w1, kj));
          if (!nz) acc = cadd(acc, cscale(w2, kk));
          const V d = cmake<V>(-twopi * acc.y, twopi * acc.x);
          r0 = cadd(r0, cmul(K0, d));
          r1 = cadd(r1, cmul(K1, d));
          r2 = cadd(r2, cmul(K2, d));
        }
      }
    } else {
      if (a.allper) {
        const R kmag = ki * ki + kj * kj + kk * kk;
        g = kmag > (R)0 ? zeta / ((R)4 * (pi * pi) * kmag) : (R)0;
      } else {
        g = G[(n <= L - n ? n : L - n) * gz] * (R)a.h3;
      }
      if (kind == 0) {
        // u-hat = G 2 pi i (k x w-hat); Nyquist wavenumbers drop out of
        // the real part of the inverse (Hermitian projection)
        const R kz_ = nz ? (R)0 : kk, f = g * twopi;
        const V c0 = csub(cscale(w2, ky_), cscale(w1, kz_));
        const V c1 = csub(cscale(w0, kz_), cscale(w2, kx_));
        const V c2 = csub(cscale(w1, kx_), cscale(w0, ky_));
        r0 = cmake<V>(-c0.y * f, c0.x * f);
        r1 = cmake<V>(-c1.y * f, c1.x * f);
        r2 = cmake<V>(-c2.y * f, c2.x * f);
      } else if (kind == 1) {
        r0 = cscale(w0, g);
        r1 = cscale(w1, g);
        r2 = cscale(w2, g);
      } else {
        r0 = cscale(w0, zeta);
        r1 = cscale(w1, zeta);
        r2 = cscale(w2, zeta);
        if (a.reproj) {
          // -4 pi^2 G k_c sum_d k_d w_d over pairs (c, d) of equal Nyquist
          // parity (:861-872)
          const V z0 = cscale(w0, ki), z1 = cscale(w1, kj), z2 = cscale(w2, kk);
          auto dot = [&](bool q) {
            V acc = cmake<V>(0, 0);
            if (nx == q) acc = cadd(acc, z0);
            if (ny == q) acc = cadd(acc, z1);
            if (nz == q) acc = cadd(acc, z2);
            return acc;
          };
          const R f = -(R)4 * (pi * pi) * g;
          r0 = cadd(r0, cscale(dot(nx), f * ki));
          r1 = cadd(r1, cscale(dot(ny), f * kj));
          r2 = cadd(r2, cscale(dot(nz), f * kk));
        }
      }
    }
    s0[n] = r0;
    s0[st + n] = r1;
    s0[2 * st + n] = r2;
  }
  __syncthreads();
  fft_any<1, true>(pl, spec, p, P, tw, LineIn<V>{spec},
                   RowsOut<V>{reinterpret_cast<V *>(out) + tile, a.rs, a.Mz, ok, (R)1 / (R)L});
}

}  // namespace any
}  // namespace pmgpu
