// Statements of k_z3_r (poisson_fixed.h): field F of the block's tile, from its
// names (a, tw, lds, rsrc, voff, rsb, kx, ky, kx0, col, p, col_ok, twd).
// Included into the kernel's body once for each field that it forms: as a
// function, inlined, the same statements take 16 more registers, and the FP64
// velocity of 512 points its third wavefront per SIMD.
V w[3][E];
#pragma unroll
for (int m = 0; m < E; ++m) {
  const bool ok = col_ok && (HALF ? m < E / 2 : p + P * m < a.Mz);
  const int soff = (int)((int64_t)P * m * rsb);
#pragma unroll
  for (int c = 0; c < 3; ++c)
    w[c][m] = ok ? buf_load(rsrc, voff + c * (int)sizeof(V), soff, V{}) : cmake<V>(0, 0);
}
V *line = lds + col * ST;
#pragma unroll
for (int c = 0; c < 3; ++c) fft_regs<K, -1, V, HALF, false, 1>(w[c], line, p, twd);
// u-hat = G 2 pi i (k x w-hat); Nyquist wavenumbers drop out (Hermitian
// projection of the real inverse); the 1 / L of the inverse transform
// rides on the same factor
const R ki = wavenumber<R>(kx, a.Lx, a.dk[0], a.ksmp[0]);
const R kj = wavenumber<R>(ky, a.Ly, a.dk[1], a.ksmp[1]);
const bool nx = 2 * kx == a.Lx, ny = 2 * ky == a.Ly;
const R kx_ = nx ? (R)0 : ki, ky_ = ny ? (R)0 : kj;
const int kyf = ky <= a.Ly - ky ? ky : a.Ly - ky;
const R pi = (R)3.14159265358979323846, inv_l = (R)1 / (R)L;
const R twopi = (R)6.28318530717958647692 / (R)L;
// G-hat of the thread's rows, all loads issued before any is used (a
// column past Hx reads column 0 and is masked)
const R *G = reinterpret_cast<const R *>(a.Ghat) + (int64_t)kyf * a.Hx + (col_ok ? kx : 0);
const int64_t gz = (int64_t)a.Hy * a.Hx;
R gv[E];
if constexpr (!ALLPER) {
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int n = p + P * m;
    const int kzf = n <= L - n ? n : L - n;
    gv[m] = G[kzf * gz];
  }
}
#pragma unroll
for (int m = 0; m < E; ++m) {
  const int n = p + P * m;
  const R kk = wavenumber<R>(n, L, a.dk[2], a.ksmp[2]);
  R zeta = (R)1, g;
  if (F == kVort || F == kVelFiltered || (F == kPsi && ALLPER && a.want_vort))
    zeta = zeta_filter<R>(a.order, (R)a.eps2pi * sqrt(ki * ki + kj * kj + kk * kk));
  if constexpr (ALLPER) {
    const R kmag = ki * ki + kj * kj + kk * kk;
    g = kmag > (R)0 ? zeta / ((R)4 * (pi * pi) * kmag) : (R)0;
  } else {
    g = col_ok ? gv[m] * (R)a.h3 : (R)0;
  }
  const bool nz = 2 * n == L;
  const V w0 = w[0][m], w1 = w[1][m], w2 = w[2][m];
  if constexpr (F == kVel || F == kVelFiltered) {
    const R kz_ = nz ? (R)0 : kk;
    const V c0 = csub(cscale(w2, ky_), cscale(w1, kz_));
    const V c1 = csub(cscale(w0, kz_), cscale(w2, kx_));
    const V c2 = csub(cscale(w1, kx_), cscale(w0, ky_));
    const R f = g * twopi;
    w[0][m] = cmake<V>(-c0.y * f, c0.x * f);
    w[1][m] = cmake<V>(-c1.y * f, c1.x * f);
    w[2][m] = cmake<V>(-c2.y * f, c2.x * f);
  } else if constexpr (F == kPsi) {
#pragma unroll
    for (int c = 0; c < 3; ++c) w[c][m] = cscale(w[c][m], g * inv_l);
  } else {
    // reprojection: -4 pi^2 G k_c sum_d k_d w_d over the pairs (c, d) of
    // equal Nyquist parity (:861-872)
    const R kd[3] = {ki, kj, kk};
    const bool nd[3] = {nx, ny, nz};
    const R f = a.reproj ? -(R)4 * (pi * pi) * g * inv_l : (R)0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const V wc = c == 0 ? w0 : (c == 1 ? w1 : w2);
      V q = cscale(wc, zeta * inv_l);
      if (a.reproj) {
        V acc = cmake<V>(0, 0);
        if (nd[0] == nd[c]) acc = cadd(acc, cscale(w0, ki));
        if (nd[1] == nd[c]) acc = cadd(acc, cscale(w1, kj));
        if (nd[2] == nd[c]) acc = cadd(acc, cscale(w2, kk));
        q = cadd(q, cscale(acc, f * kd[c]));
      }
      w[c][m] = q;
    }
  }
}
#pragma unroll
for (int c = 0; c < 3; ++c) fft_regs<K, 1, V, false, HALF, 1>(w[c], line, p, twd);
// Stores are plain global stores: buffer-resource stores of these
// 8-byte-aligned records, which the compiler merges into 16-byte stores
// across components, have returned corrupted first components.
if (col_ok) {
  V *out = reinterpret_cast<V *>(F == kPsi ? a.Bpsi : (F == kVort ? a.Bvort : a.B));
  V *dst = out + (int64_t)ky * a.kys + (int64_t)kx0 * 3 + (int64_t)p * a.rs + col * 3;
#pragma unroll
  for (int m = 0; m < E; ++m) {
    if (HALF ? m < E / 2 : p + P * m < a.Mz) {
#pragma unroll
      for (int c = 0; c < 3; ++c) dst[(int64_t)P * m * a.rs + c] = w[c][m];
    }
  }
}
