// Kernel bodies of the VPFP step.  Each body is written for one workgroup
// and a block context `Ctx` (vpfp_device.h); vpfp.hip, vpfp_row.hip and
// vpfp_drift.hip wrap them in __global__ kernels.
//
// Data layout (HBM): f is (nx, nv) row-major, v fastest, T = double or float.
// A row (fixed x) is contiguous; a column (fixed v) has stride nv.
//
//   row_body    one or more x-rows per workgroup.  Optional stages, in order:
//               kick A (v-advection by e(x) dt_a), collision (implicit LB/DG
//               solve along v), storage moments, kick B (v-advection by e(x)
//               dt_b).  One HBM read and one write of the row whatever the
//               stages.   [vlasov.py:113-140, collisions.py:26-160,222-265,
//               step.py:143-228]
//   drift_body  C v-columns per workgroup: x-advection of each column and the
//               per-column-tile partial trapz sums sum_v w_v f(x, v) feeding the
//               Poisson solve.   [vlasov.py:83-110, field.py:27-36]
//   field_body  one workgroup: density from the partial sums, pseudo-spectral
//               Poisson solve, driver added, E written (and <E^2>, <D^2>).
//               [field.py:39-88, step.py:215-216]
#pragma once
#include "vpfp_device.h"

namespace vp {

enum RowFlags { RK_KICK_A = 1, RK_COLLIDE = 2, RK_MOMENTS = 4, RK_KICK_B = 8 };
constexpr int kMoments = 8;  // n, j, T, q, fv4, vN, f^2, f log f

// trapz weight of sample m of an N-point row
VP_HD double trapw(int m, int N) { return (m == 0 || m == N - 1) ? 0.5 : 1.0; }

// ---------------------------------------------------------------------------
// spectral multiply along a length-2M real sequence held as M complex values:
// v in natural order in and out; buf serves the exchanges and ends free
// ---------------------------------------------------------------------------
template <class T, int M, int TPT, class Mul, class Ctx>
VP_HD void spectral_apply(Ctx& c, cx<T>* v, cx<T>* buf, const Tw<T>& tw, int t, Mul mult, bool act = true) {
  constexpr int Q = M / TPT;
  fft<T, M, TPT, false>(c, v, buf, tw, t, act);
  // only the partner bins cross threads
  if (act) {
#pragma unroll
    for (int i = 0; i < Q; ++i) buf[pidx(t + i * TPT)] = v[i];
  }
  cx<T> wk[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) wk[i] = at(tw.w + i * TPT, (unsigned)t);
  c.sync();
  cx<T> pz[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) pz[i] = buf[pidx((M - (t + i * TPT)) & (M - 1))];
  c.sync();
  couple<T, M, TPT>(v, pz, wk, t, mult);
  fft<T, M, TPT, true>(c, v, buf, tw, t, act);
}

// ---------------------------------------------------------------------------
// collision coefficients (collisions.py:67-79 LB, :138-156 DG)
//   l(m) = nu dt (-T/dv^2 + (v_{m-1} - vbar)/(2 dv)),  m >= 1
//   u(m) = nu dt (-T/dv^2 - (v_{m+1} - vbar)/(2 dv)),  m <= N-2
//   b    = 1 + nu dt (2 T / dv^2)
// ---------------------------------------------------------------------------
// With v_m = v0 + m dvv (the host checks that the grid is uniform to
// rounding) both off-diagonals are affine in m:
//   l(m) = nu dt (A0 + (v_{m-1} - vbar) H) = l0 + ls m
//   u(m) = nu dt (A0 - (v_{m+1} - vbar) H) = u0 - ls m
// with A0 = -T/dv^2, H = 1/(2 dv); one FMA per coefficient.
struct CollCoef {
  int N;
  double l0, u0, ls, bd;
  VP_HD void set(double ndt, double A0, double H, double v0, double dvv, double vbar, double bd_) {
    ls = ndt * (H * dvv);
    l0 = ndt * (A0 + ((v0 - dvv) - vbar) * H);
    u0 = ndt * (A0 - ((v0 + dvv) - vbar) * H);
    bd = bd_;
  }
  // rows m0 + i of one thread: l and u affine in the chunk index i (one FMA
  // each), the ends of the whole row zero
  template <int L>
  struct View {
    double lb, ub, ls, bd;
    bool first, last;
    VP_HD double l(int i) const { return (i == 0 && first) ? 0.0 : lb + ls * (double)i; }
    VP_HD double u(int i) const { return (i == L - 1 && last) ? 0.0 : ub - ls * (double)i; }
    VP_HD double b(int) const { return bd; }
  };
  template <int L>
  VP_HD View<L> view(int m0, bool first, bool last) const {
    return View<L>{l0 + ls * (double)m0, u0 - ls * (double)m0, ls, bd, first, last};
  }
};

// explicit diagonals a (nv-1), b (nv), c (nv-1) of one row
struct ArrCoef {
  const double* a;
  const double* bb;
  const double* cc;
  int N;
  template <int L>
  struct View {
    const double *a, *bb, *cc;
    int m0, N;
    bool first, last;
    // indices clamped into the arrays: the row ends are never read
    VP_HD double l(int i) const {
      const int k = m0 + i - 1;
      return (i == 0 && first) ? 0.0 : a[k > 0 ? k : 0];
    }
    VP_HD double u(int i) const {
      const int k = m0 + i;
      return (i == L - 1 && last) ? 0.0 : cc[k < N - 2 ? k : N - 2];
    }
    VP_HD double b(int i) const { return bb[m0 + i]; }
  };
  template <int L>
  VP_HD View<L> view(int m0, bool first, bool last) const {
    return View<L>{a, bb, cc, m0, N, first, last};
  }
};

// trapz weight of chunk element i of thread t (rows t L .. t L + L - 1 of a
// row of TPT L samples): 1/2 at the two ends of the row
template <int TPT, int L>
VP_HD double chunk_w(int i, int t) {
  return ((i == 0 && t == 0) || (i == L - 1 && t == TPT - 1)) ? 0.5 : 1.0;
}

// drift velocity and temperature of one row (un-normalised, trapz), chunk layout
template <int TPT, int L, class Ctx>
VP_HD void coll_moments(Ctx& c, const double* d, double v0, double dvv, int N, double dv, bool dg, int t,
                        double* rs, double& vbar, double& temp) {
  const int m0 = t * L;
  // v_{m0+i} = vb + i dvv
  const double vb = v0 + (double)m0 * dvv;
  double s[1] = {0.0};
  vbar = 0.0;
  if (dg) {
#pragma unroll
    for (int i = 0; i < L; ++i) s[0] += chunk_w<TPT, L>(i, t) * d[i] * (vb + (double)i * dvv);
    row_sum<TPT, 1>(c, s, rs);
    vbar = dv * s[0];
    s[0] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const double w = (vb + (double)i * dvv) - vbar;
    s[0] += chunk_w<TPT, L>(i, t) * d[i] * (w * w);
  }
  row_sum<TPT, 1>(c, s, rs);
  temp = dv * s[0];
}

// ---------------------------------------------------------------------------
// field kernel: n(x) = scale * sum_tiles part[tile][x];  E = Re ifft(i/kx fft(1 - n)) + driver
// ---------------------------------------------------------------------------
struct FieldArgs {
  const double* part;
  int ntiles;
  int nx;
  double scale;
  double* rho_g;          // [nx] global scratch when the grid has several workgroups
  unsigned int* counter;  // arrival counter (zero between launches)
  const double* okx;      // [nx]
  const cx<double>* tw;   // pow2 kernel: twiddle tables of nx (Tw); DFT kernel: exp(-2 pi i n / nx), n < nx
  const double* driver;   // [nx] or null
  double* e_out;          // [nx]
  double* series;         // [2] or null: mean(E^2), mean(driver^2)
  int series_stride;      // batched scan: doubles between consecutive instances' series entries
  const double* green;    // [nx] Green's function of the solve (single grids; field_rows, green_body)
};

// The view of instance inst of a batched field solve: every array is
// instance-major (part [inst][ntiles][nx], okx / driver / E [inst][nx],
// series [inst * series_stride], one 64-byte counter slot per instance).
// Instance 0 is the single-grid case itself.
VP_HD FieldArgs field_instance(const FieldArgs& a, int inst) {
  FieldArgs r = a;
  if (inst == 0) return r;
  const size_t xo = (size_t)inst * a.nx;
  r.part += (size_t)inst * a.ntiles * a.nx;
  if (r.rho_g) r.rho_g += xo;
  if (r.counter) r.counter += inst * 16;
  r.okx += xo;
  if (r.driver) r.driver += xo;
  r.e_out += xo;
  if (r.series) r.series += (size_t)inst * a.series_stride;
  return r;
}

// rho[x] = 1 - scale * sum_tiles part[tile][x] for x in [x0, x0 + XS)
// (all FT threads; XS divides FT or FT divides XS)
template <int FT, int U = 8, class Ctx>
VP_HD void field_density(Ctx& c, const FieldArgs& a, int x0, int XS, double* rho, double* tmp) {
  const int nx = a.nx;
  const int G = XS >= FT ? 1 : FT / XS;
  for (int l0 = c.tid; l0 < XS * G; l0 += FT) {
    const int xl = l0 % XS, g = l0 / XS;
    const double* p = a.part + x0 + xl;
    auto ld = [&](int tl) { return p[(size_t)tl * nx]; };
    // U independent partial sums keep U loads in flight per thread
    double acc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = 0.0;
    int tile = g;
    for (; tile + (U - 1) * G < a.ntiles; tile += U * G) {
#pragma unroll
      for (int u = 0; u < U; ++u) acc[u] += ld(tile + u * G);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (tile + u * G < a.ntiles) acc[u] += ld(tile + u * G);
#pragma unroll
    for (int h = U / 2; h >= 1; h >>= 1)
#pragma unroll
      for (int u = 0; u < h; ++u) acc[u] += acc[u + h];
    tmp[l0] = acc[0];
  }
  c.sync();
  for (int xl = c.tid; xl < XS; xl += FT) {
    double s = 0.0;
    for (int g = 0; g < G; ++g) s += tmp[g * XS + xl];
    rho[xl] = 1.0 - a.scale * s;
  }
  c.sync();
}

// Field at a workgroup's own rows (single grids): with the Green's function
//   g_d = (1/nx) sum_m Re(i okx_m exp(2 pi i m d / nx))
// of the solve, formed once per plan, E(x) = driver(x) + sum_j g_{x-j} rho_j is
// one dot product per row, so a row needs no field launch and no transform
// between the drift and its kick.  The partial density rows are summed here
// when they are few (kProSum values, nx <= kProNx: every workgroup reads them
// all), otherwise by k_rho into one row (ntiles = 1).  Every thread of a row
// gets E; thread t = 0 writes it.  64 x 1024 FP64 step: 21.2 us with the field
// launch, 18.2 with this; 1024 x 8192 (summed by k_rho): 187 -> 175.
// lds: rho [kProNx] | tmp [max(kProNx, FT)] | row_sum scratch [16]
constexpr int kProNx = 256;
constexpr int kProSum = 8192;
template <int FT>
struct ProCfg {
  static constexpr int tmp_n = kProNx > FT ? kProNx : FT;
  static constexpr int bytes = (kProNx + tmp_n + 16) * 8;
};

template <int FT, int TPT, class Ctx>
VP_HD double field_rows(Ctx& c, const FieldArgs& a, unsigned char* lds, int row, bool valid, int t) {
  double* rho = reinterpret_cast<double*>(lds);
  double* tmp = rho + kProNx;
  double* rs = tmp + ProCfg<FT>::tmp_n;
  const int nx = a.nx;
  double s[1] = {0.0};
  if (a.ntiles == 1) {
#pragma unroll 4
    for (int j = t; j < nx; j += TPT) s[0] += a.green[(row - j) & (nx - 1)] * (1.0 - a.scale * a.part[j]);
  } else {
    field_density<FT, 16>(c, a, 0, nx, rho, tmp);  // ends with a barrier
    for (int j = t; j < nx; j += TPT) s[0] += a.green[(row - j) & (nx - 1)] * rho[j];
  }
  row_sum<TPT, 1>(c, s, rs);
  if constexpr (TPT <= 64) c.sync();  // rho read before the transforms take the LDS
  const double e = s[0] + (a.driver ? a.driver[row] : 0.0);
  if (valid && t == 0) a.e_out[row] = e;
  return e;
}

// mean(E^2) and mean(driver^2) of a finished step (one workgroup of FT threads)
template <int FT, class Ctx>
VP_HD void series_body(Ctx& c, const double* e, const double* driver, int nx, double* out, double* rs) {
  double acc[2] = {0.0, 0.0};
  for (int x = c.tid; x < nx; x += FT) {
    const double ex = e[x], dr = driver ? driver[x] : 0.0;
    acc[0] += ex * ex;
    acc[1] += dr * dr;
  }
  row_sum<FT, 2>(c, acc, rs);
  if (c.tid == 0) {
    out[0] = acc[0] / nx;
    out[1] = acc[1] / nx;
  }
}

// E(x) = driver(x) + sum_j g_{x-j} rho_j at any nx, one wavefront per x
// (vpfp_field): nx = 100 2.7 us where the direct transform on one
// workgroup took 22.5
template <class Ctx>
VP_HD void green_body(Ctx& c, const FieldArgs& a) {
  const int lane = c.tid & 63;
  const int x0 = c.bid * (c.nthr / 64) + (c.tid >> 6);
  const int x = x0 < a.nx ? x0 : a.nx - 1;
  double s = 0.0;
#pragma unroll 4
  for (int j = lane; j < a.nx; j += 64) {
    const int d = x - j;
    s += a.green[d < 0 ? d + a.nx : d] * (1.0 - a.scale * a.part[j]);
  }
  s = lane_sum<64>(c, s);
  if (x0 < a.nx && lane == 0) a.e_out[x] = s + (a.driver ? a.driver[x] : 0.0);
}

// g_d, one wavefront per d: the bins m and nx - m of the sum are equal (only the
// odd part (okx_m - okx_{nx-m}) / 2 of the multiplier reaches the real part), so
// g_d = -(2/nx) sum_{0 < m < nx/2} g_m sin(2 pi m d / nx); tw[n] = exp(-2 pi i n / nx)
template <class Ctx>
VP_HD void green_table_body(Ctx& c, const double* okx, const cx<double>* tw, int nx, double* green) {
  const int lane = c.tid & 63;
  const int d0 = c.bid * (c.nthr / 64) + (c.tid >> 6);
  const int d = d0 < nx ? d0 : nx - 1;
  double s = 0.0;
  for (int m = 1 + lane; 2 * m < nx; m += 64)
    s += 0.5 * (okx[m] - okx[nx - m]) * tw[(int)(((long long)m * d) % nx)].im;
  s = lane_sum<64>(c, s);
  if (d0 < nx && lane == 0) green[d] = 2.0 * s / nx;
}

// ---------------------------------------------------------------------------
// first nm Fourier modes along x of every v column:
//   out[m][v] = sum_x f(x, v) exp(-2 pi i m x / nx)     (step.py:130-135)
// one thread per (m, v); the x sum is sequential in x order
// ---------------------------------------------------------------------------
template <class T, class Ctx>
VP_HD void xmodes_body(Ctx& c, const T* f, int nx, int nv, int nm, const cx<double>* tw, cx<double>* out) {
  const int idx = c.bid * c.nthr + c.tid;
  if (idx >= nm * nv) return;
  const int m = idx / nv, col = idx % nv;
  double re = 0.0, im = 0.0;
  // r = m x mod nx by increments: the loads of f and of the twiddles do not
  // wait on an index division, so consecutive iterations overlap
  int r = 0;
#pragma unroll 16
  for (int x = 0; x < nx; ++x) {
    const cx<double> w = tw[r];
    const double fv = (double)f[(size_t)x * nv + col];
    re += fv * w.re;
    im += fv * w.im;
    r += m;
    if (r >= nx) r -= nx;
  }
  out[idx] = mk<double>(re, im);
}

// ---------------------------------------------------------------------------
// row kernel
// ---------------------------------------------------------------------------
template <class T>
struct RowArgs {
  const T* f_in;
  T* f_out;          // null: f is not written back (moments only)
  int nx, nv;
  const double* e;  // [nx] field for the kicks
  double dt_a, dt_b;
  double dk;         // kv[1] of the fftfreq table
  double v0, dvv;    // v_m = v0 + m dvv
  double dv;
  const cx<T>* tw;   // twiddle tables of nv (Tw)
  double nu_dt;
  int op_dg;
  double* moments;  // [kMoments][nx]
  T* f_copy;        // [nx][nv] or null: f after the collision and moments (f itself under delta-f storage)
  int flags;
  const double* nu_dt_inst;  // batched scan: nu*dt per instance (rows are instance-major), or null
  int rows_per_inst;         // x rows per instance in a batch
  // field in the prologue (field_rows): E of the workgroup's rows from the
  // drift's densities instead of e (single grid)
  int field_pro;
  FieldArgs fld;
  // extra workgroups after the rows' own, for a finished earlier step (single
  // grid): one for the series of its E and driver (prev_series), then
  // xm_n * xm_nv threads for the first xm_n x-modes of its f copy xm_f [nx][nv]
  const double* prev_e;
  const double* prev_drv;
  double* prev_series;
  const T* xm_f;
  int xm_n;
  const cx<double>* xm_tw;  // exp(-2 pi i r / nx)
  cx<double>* xm_out;       // [xm_n][nv]
  // delta-f storage: f holds f - B(v) for a fixed background B (bg [nv],
  // FP64; spectrum tables bg_hat [nv] of BgPhaseMul in the storage precision);
  // the kicks shift B spectrally as part of the deviation's multiply, the
  // collision and moments see B + (f - B) in FP64
  const double* bg;
  const cx<T>* bg_hat;
};

template <class T, int M, int Q>
struct RowCfg {
  static constexpr int TPT = M / Q;
  static constexpr int L = 2 * Q;
  static constexpr int fft_bytes = Padded<M>::size * (int)sizeof(cx<T>);
  static constexpr int red_bytes = 8 * TPT * 8 + (TPT > 64 ? TPT / 64 * 8 : 0);
  static constexpr int region = ((fft_bytes > red_bytes ? fft_bytes : red_bytes) + 15) & ~15;
  static constexpr int wg = TPT >= 64 ? TPT : 64;
  static constexpr int rows = wg / TPT;
  static constexpr int sum_bytes = (TPT > 64 ? TPT / 64 : 1) * kMoments * 8;
  // the field prologue (field_rows) runs before the row buffers are used and
  // overlays them from offset 0
  static constexpr int pro_bytes = ProCfg<wg>::bytes;
  static constexpr int main_bytes = rows * region + sum_bytes;
  static constexpr int lds = main_bytes > pro_bytes ? main_bytes : pro_bytes;
  // minimum waves per SIMD asked of the register allocator: 3 (168 VGPRs) for
  // 8 values per thread and M <= 1024, the scans' classes, which otherwise come
  // out at 170 now and then and run two waves (FP64 M = 1024, 512 instances: 153
  // against 174 us); 4 spills 100 to 260 bytes and is slower (FP32 delta-f
  // M = 1024, 4096 instances 1116 -> 1431 us; M = 4096 FP64, 1024 rows 115 -> 134)
  static constexpr int min_waves = (Q == 8 && M <= 1024) ? 3 : 1;
};

// BG: delta-f storage (a.bg, a.bg_hat set); a kernel of its own so that the
// plain step's register allocation is unchanged
template <class T, int M, int Q, class Ctx, bool BG = false>
VP_HD void row_body(Ctx& c, unsigned char* lds, const RowArgs<T>& a) {
  using Cfg = RowCfg<T, M, Q>;
  constexpr int TPT = Cfg::TPT;
  constexpr int L = Cfg::L;
  if (a.prev_series || a.xm_out) {
    int b = c.bid - (a.nx + Cfg::rows - 1) / Cfg::rows;
    if (b >= 0 && a.prev_series && b-- == 0) {
      series_body<Cfg::wg>(c, a.prev_e, a.prev_drv, a.nx, a.prev_series, reinterpret_cast<double*>(lds));
      return;
    }
    if (b >= 0) {
      Ctx x = c;
      x.bid = b;
      xmodes_body<T>(x, a.xm_f, a.nx, a.nv, a.xm_n, a.xm_tw, a.xm_out);
      return;
    }
  }
  const int t = c.tid % TPT;
  const int rl = c.tid / TPT;
  const int row = c.bid * Cfg::rows + rl;
  const bool valid = row < a.nx;
  const int rowc = valid ? row : a.nx - 1;
  cx<T>* buf = reinterpret_cast<cx<T>*>(lds + rl * Cfg::region);
  double* red = reinterpret_cast<double*>(lds + rl * Cfg::region);
  double* rs = reinterpret_cast<double*>(lds + Cfg::rows * Cfg::region);

  const cx<T>* src = reinterpret_cast<const cx<T>*>(a.f_in + (size_t)rowc * a.nv);
  cx<T> v[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) v[i] = at(src + i * TPT, (unsigned)t);
  double e = 0.0;
  if (a.field_pro) {
    e = field_rows<Cfg::wg, TPT>(c, a.fld, lds, rowc, valid, t);
  } else if (a.flags & (RK_KICK_A | RK_KICK_B)) {
    e = a.e[rowc];
  }
  const Tw<T> tw = tw_at<M, Q>(a.tw);

  // kick by shift a: f(v) -> f(v - a), spectrally (the background's shift too
  // under delta-f storage)
  auto phases = [&](double shift) {
    if constexpr (BG)
      return BgPhaseMul<T>(a.dk * shift, M, t, TPT, a.bg_hat);
    else
      return PhaseMul<T>(a.dk * shift, M, t, TPT);
  };
  const bool chunk = (a.flags & (RK_COLLIDE | RK_MOMENTS)) != 0;
  // two half kicks by the same field with nothing between them (no
  // collision, moments or f store: the collisionless fused step) are one
  // kick by the sum of the shifts: the phase factors multiply exactly, so
  // one transform pair replaces two
  const bool merged = (a.flags & RK_KICK_A) && (a.flags & RK_KICK_B) && !chunk && !a.f_copy;
  decltype(phases(0.0)) ph;
  if (a.flags & RK_KICK_A) {
    ph = phases((merged ? a.dt_a + a.dt_b : a.dt_a) * e);
    spectral_apply<T, M, TPT>(c, v, buf, tw, t, ph);
  }

  if (a.f_copy && !chunk && valid) {
    // copy only: natural order, one complex pair per value (coalesced)
    cx<T>* dst = reinterpret_cast<cx<T>*>(a.f_copy + (size_t)row * a.nv);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      cx<T> z = v[i];
      if constexpr (BG) {
        const int j = t + i * TPT;
        z = mk<T>((T)((double)z.re + a.bg[2 * j]), (T)((double)z.im + a.bg[2 * j + 1]));
      }
      dst[t + i * TPT] = z;
    }
  }
  if (chunk) {
    // natural order -> contiguous chunk of L samples per thread
#pragma unroll
    for (int i = 0; i < Q; ++i) buf[pidx(t + i * TPT)] = v[i];
    c.sync();
    double d[L];
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const cx<T> z = buf[pidx(t * Q + i)];
      d[2 * i] = (double)z.re;
      d[2 * i + 1] = (double)z.im;
    }
    c.sync();
    const int N = a.nv;
    const int m0 = t * L;
    if constexpr (BG) {
#pragma unroll
      for (int i = 0; i < L; ++i) d[i] += at(a.bg + i, (unsigned)m0);
    }
    const double nu_dt = a.nu_dt_inst ? a.nu_dt_inst[rowc / a.rows_per_inst] : a.nu_dt;
    if ((a.flags & RK_COLLIDE) && nu_dt > 0.0) {
      double vbar, temp;
      coll_moments<TPT, L>(c, d, a.v0, a.dvv, N, a.dv, a.op_dg != 0, t, rs, vbar, temp);
      const double dv2 = a.dv * a.dv;
      CollCoef cf;
      cf.N = N;
      cf.set(nu_dt, -temp / dv2, 0.5 / a.dv, a.v0, a.dvv, vbar, 1.0 + nu_dt * (2.0 * temp / dv2));
      tridiag<TPT, L, CollCoef, Ctx, sizeof(T) == 8>(c, d, cf, t, red);
    }
    if (a.flags & RK_MOMENTS) {
      double s[kMoments];
#pragma unroll
      for (int q = 0; q < kMoments; ++q) s[q] = 0.0;
      const double vb = a.v0 + (double)m0 * a.dvv;
#pragma unroll
      for (int i = 0; i < L; ++i) {
        const double wf = chunk_w<TPT, L>(i, t) * d[i];
        const double vm = vb + (double)i * a.dvv;
        double p = wf;
        s[0] += p;
        p *= vm;
        s[1] += p;
        p *= vm;
        s[2] += p;
        p *= vm;
        s[3] += p;
        p *= vm;
        s[4] += p;
        p *= vm;
        s[5] += p;
        s[6] += wf * d[i];
        // f log f: in the storage precision (FP32 log on the FP32 path)
        s[7] += wf * (sizeof(T) == 8 ? log_f64(d[i]) : (double)logf((float)d[i]));
      }
      // each wave folds its eight sums over its lanes; one lane per sum then
      // adds the waves' shares
      constexpr int W = TPT < 64 ? TPT : 64;
      lane_fold<W, kMoments>(c, s);
      const int lane = t & (W - 1);
      if constexpr (TPT <= 64) {
        if (valid && fold_writer<W, kMoments>(lane)) {
#pragma unroll
          for (int j = 0; j < fold_count<W, kMoments>(); ++j)
            a.moments[(size_t)(fold_index<W, kMoments>(lane) + j) * a.nx + row] = a.dv * s[j];
        }
      } else {
        if (fold_writer<W, kMoments>(lane)) rs[(t >> 6) * kMoments + fold_index<W, kMoments>(lane)] = s[0];
        c.sync();
        if (valid && t < kMoments) {
          double sum = 0.0;
#pragma unroll
          for (int w = 0; w < TPT / 64; ++w) sum += rs[w * kMoments + t];
          a.moments[(size_t)t * a.nx + row] = a.dv * sum;
        }
      }
    }
    if (a.f_copy && valid) {
      // f after the collision (the reference's per-step f store); d holds f
      // itself here also under delta-f storage
      T* dst = a.f_copy + (size_t)row * a.nv + m0;
#pragma unroll
      for (int i = 0; i < L; ++i) dst[i] = (T)d[i];
    }
    if constexpr (BG) {
#pragma unroll
      for (int i = 0; i < L; ++i) d[i] -= at(a.bg + i, (unsigned)m0);
    }
    // chunk -> natural order
#pragma unroll
    for (int i = 0; i < Q; ++i) buf[pidx(t * Q + i)] = mk<T>((T)d[2 * i], (T)d[2 * i + 1]);
    c.sync();
#pragma unroll
    for (int i = 0; i < Q; ++i) v[i] = buf[pidx(t + i * TPT)];
    c.sync();
  }

  if ((a.flags & RK_KICK_B) && !merged) {
    // the second half kick of a step shifts by the first's amount: its phases
    // are kept through the collision
    if (!(a.flags & RK_KICK_A) || a.dt_b != a.dt_a) ph = phases(a.dt_b * e);
    spectral_apply<T, M, TPT>(c, v, buf, tw, t, ph);
  }

  if (valid && a.f_out) {
    cx<T>* dst = reinterpret_cast<cx<T>*>(a.f_out + (size_t)row * a.nv);
#pragma unroll
    for (int i = 0; i < Q; ++i) at(dst + i * TPT, (unsigned)t) = v[i];
  }
}

// Several workgroups: each reduces an x slice into rho_g; the last one to
// arrive (device-scope counter) continues with the whole rho.  Returns false
// in the workgroups that are done.
template <int FT, class Ctx>
VP_HD bool field_gather(Ctx& c, const FieldArgs& a, double* rho, double* tmp, int* flag) {
  const int nx = a.nx;
  if (c.nblk == 1) {
    field_density<FT>(c, a, 0, nx, rho, tmp);
    return true;
  }
  const int XS = nx / c.nblk;
  const int x0 = c.bid * XS;
  field_density<FT>(c, a, x0, XS, rho, tmp);
  for (int xl = c.tid; xl < XS; xl += FT) a.rho_g[x0 + xl] = rho[xl];
  c.fence();
  c.sync();
  if (c.tid == 0) *flag = (c.arrive(a.counter) == (unsigned)(c.nblk - 1)) ? 1 : 0;
  c.sync();
  if (!*flag) return false;
  c.fence();
  for (int x = c.tid; x < nx; x += FT) rho[x] = a.rho_g[x];
  if (c.tid == 0) c.reset(a.counter);
  c.sync();
  return true;
}

template <int FT, class Ctx>
VP_HD void field_finish(Ctx& c, const FieldArgs& a, int x, double ex, double* rs, double* acc) {
  const double dr = a.driver ? a.driver[x] : 0.0;
  const double e = ex + dr;
  a.e_out[x] = e;
  acc[0] += e * e;
  acc[1] += dr * dr;
}

template <int M, int Q, int FT>
struct FieldCfg {
  static constexpr int TPT = M / Q;
  static constexpr int nx = 2 * M;
  static constexpr int tmp_n = (nx > FT ? nx : FT);
  static constexpr int work = (Padded<M>::size * 16 > tmp_n * 8) ? Padded<M>::size * 16 : tmp_n * 8;
  // [okx (nx) | rho (nx) | fft buffer / reduction scratch | row_sum scratch | flag]
  static constexpr int lds = 2 * nx * 8 + work + 64 + 16;
};

// TAIL: called by the last workgroup of the drift kernel, which reads every
// partial density row itself, behind its own acquire fence, instead of the slice
// hand-off
template <int M, int Q, int FT, bool TAIL = false, class Ctx>
VP_HD void field_body(Ctx& c, unsigned char* lds, const FieldArgs& a) {
  using Cfg = FieldCfg<M, Q, FT>;
  constexpr int TPT = Cfg::TPT;
  static_assert(TPT <= FT, "field transform needs at most FT threads");
  double* okx = reinterpret_cast<double*>(lds);
  double* rho = okx + Cfg::nx;
  cx<double>* buf = reinterpret_cast<cx<double>*>(rho + Cfg::nx);
  double* tmp = reinterpret_cast<double*>(buf);
  double* rs = reinterpret_cast<double*>(lds + Cfg::lds - 80);
  int* flag = reinterpret_cast<int*>(lds + Cfg::lds - 16);
  if constexpr (TAIL) {
    // the caller's acquire fence makes the other workgroups' rows visible
    field_density<FT>(c, a, 0, Cfg::nx, rho, tmp);
  } else {
    if (!field_gather<FT>(c, a, rho, tmp, flag)) return;
  }
  for (int x = c.tid; x < Cfg::nx; x += FT) okx[x] = a.okx[x];
  c.sync();
  static_assert(Q == M || Q == 8 || M > 2048, "the field (nx <= 4096) has the pass tables of Q = 8");
  const Tw<double> tw = tw_at<M, Q>(a.tw);
  const bool act = c.tid < TPT;
  const int t = act ? c.tid : 0;
  cx<double> v[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int j = t + i * TPT;
    v[i] = mk<double>(rho[2 * j], rho[2 * j + 1]);
  }
  PoissonMul<double> mul;
  mul.okx = okx;
  mul.M = M;
  spectral_apply<double, M, TPT>(c, v, buf, tw, t, mul, act);
  // the TPT threads of the transform hold 2 Q values each: through LDS to one
  // value per thread, so that the stores are one pass over all FT threads
  if (act) {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int j = t + i * TPT;
      rho[2 * j] = v[i].re;
      rho[2 * j + 1] = v[i].im;
    }
  }
  c.sync();
  double acc[2] = {0.0, 0.0};
  for (int x = c.tid; x < Cfg::nx; x += FT) field_finish<FT>(c, a, x, rho[x], rs, acc);
  if (a.series) {
    row_sum<FT, 2>(c, acc, rs);
    if (c.tid == 0) {
      a.series[0] = acc[0] / a.nx;
      a.series[1] = acc[1] / a.nx;
    }
  }
}

// direct-DFT field solve for any nx (used when nx is not a power of two)
template <int FT, class Ctx>
VP_HD void field_dft_body(Ctx& c, unsigned char* lds, const FieldArgs& a) {
  const int nx = a.nx;
  double* rho = reinterpret_cast<double*>(lds);
  cx<double>* F = reinterpret_cast<cx<double>*>(lds + ((nx * 8 + 15) & ~15));
  double* tmp = reinterpret_cast<double*>(F);
  double* rs = reinterpret_cast<double*>(reinterpret_cast<unsigned char*>(F) + (size_t)(nx > FT ? nx : FT) * 16);
  field_density<FT>(c, a, 0, nx, rho, tmp);
  for (int m = c.tid; m < nx; m += FT) {
    cx<double> s = mk<double>(0.0, 0.0);
    for (int j = 0; j < nx; ++j) {
      const cx<double> w = a.tw[(int)(((long long)m * j) % nx)];
      s.re += rho[j] * w.re;
      s.im += rho[j] * w.im;
    }
    // effective multiplier Re-projection: (G_m + conj G_{nx-m}) / 2, G = i okx
    const double g = 0.5 * (a.okx[m] - a.okx[(nx - m) % nx]);
    F[m] = mk<double>(-g * s.im, g * s.re);
  }
  c.sync();
  double acc[2] = {0.0, 0.0};
  for (int x = c.tid; x < nx; x += FT) {
    double s = 0.0;
    for (int m = 0; m < nx; ++m) {
      const cx<double> w = a.tw[(int)(((long long)m * x) % nx)];
      // Re(F_m conj(w))
      s += F[m].re * w.re + F[m].im * w.im;
    }
    field_finish<FT>(c, a, x, s / nx, rs, acc);
  }
  if (a.series) {
    row_sum<FT, 2>(c, acc, rs);
    if (c.tid == 0) {
      a.series[0] = acc[0] / a.nx;
      a.series[1] = acc[1] / a.nx;
    }
  }
}

// ---------------------------------------------------------------------------
// drift kernel (x-advection of C columns) + partial density sums
// ---------------------------------------------------------------------------
template <class T>
struct DriftArgs {
  const T* f_in;
  T* f_out;
  int nx, nv;
  double dt;
  double dk;         // kx[1] of the fftfreq table
  const double* v;   // [nv]
  const cx<T>* tw;   // twiddle tables of nx (Tw)
  double* dens;      // [gridDim][nx] partial sums (unscaled), or null
  int fuse_field;    // 1: the last workgroup to finish solves the field (fld)
  FieldArgs fld;     // field arguments for the fused tail (part = dens)
  // batched scan: grid y = instance; f and dens are offset per instance
  // (the fused field tail takes field_instance of fld); dk_inst[inst]
  // replaces dk
  const double* dk_inst;
  int xcd_order;  // 1: consecutive column tiles go to workgroups on one XCD
  // FP32, nx in {32, 64}: the x-transforms as dense real-DFT products on
  // MFMA (vpfp_drift.hip k_drift_dft) with these matrices, [2][nx][nx]:
  // forward rows k <= nx/2 cos(2 pi k x / nx), rows nx/2 + j -sin(2 pi j x / nx)
  // (0 < j < nx/2); inverse [x][k] the matching real synthesis / nx.
  // Null: the Stockham transform (drift_body).
  const float* dft;
};

// Workgroup b of n runs on XCD b % 8 (round-robin dispatch).  With
// xcd_order the workgroups of one XCD take consecutive tiles, so the two
// halves of a 128-byte line read by neighbouring tiles meet in one L2.
VP_HD int xcd_block(int b, int n) { return (n & 7) ? b : (b & 7) * (n >> 3) + (b >> 3); }

// values per thread of the x-advection transforms.  Short FP64 columns (M = 32,
// 64) take 8, two Stockham passes instead of three: scans of nx = 64 and 128
// 41 -> 38 and 75 -> 68 us.  FP32 ones, bound by VALU issue, gain nothing at
// nx = 64 and lose the occupancy at nx = 128 (436 -> 457 us).
template <class T>
VP_HD constexpr int drift_q(int M) {
  return M <= 16 || (sizeof(T) == 4 && M <= 64) ? (M < 4 ? M : 4) : 8;
}
constexpr int kDriftStageM = 128;

template <class T, int M, int Q, int C>
struct DriftCfg {
  static constexpr int TPT = M / Q;
  static constexpr int wg = TPT * C;
  // odd stride (in complex elements): the C column buffers of a tile start
  // on different LDS banks (an even multiple of 64 banks made the columns a
  // wave touches collide)
  static constexpr int stride = Padded<M>::size | 1;
  // the twiddle tables of short columns are staged in LDS (2 M entries for
  // the C columns that share them): read through L1 they took as many loads
  // as f itself (nx = 128 FP32 scan: 472 us, staged 436).  Longer columns
  // need the LDS for a second workgroup on the CU.
  static constexpr bool stage = Q < M && M <= kDriftStageM;
  static constexpr int tw_bytes = stage ? 2 * M * (int)sizeof(cx<T>) : 0;
  static constexpr int own = tw_bytes + C * stride * (int)sizeof(cx<T>);
  // fused field tail (small grids): M-point Poisson transform on the same workgroup
  static constexpr int fq = M < 8 ? M : 8;
  static constexpr bool tail = M <= 128 && (M / fq) <= wg;
  static constexpr int field_lds = tail ? FieldCfg<M, fq, wg>::lds : 0;
  static constexpr int lds = own > field_lds ? own : field_lds;
  // one tile per workgroup (ONE): without the next tile's values and the running
  // density in registers, two workgroups of eight waves fit a CU, and one loads
  // while the other transforms (nx = 1024, nv = 8192: FP32 36.2 -> 27.3 us; FP64,
  // which spills 88 bytes per lane for it, 46 MB of traffic each way, 55 -> 47)
  static constexpr int min_waves = wg == 512 && 2 * lds <= 160 * 1024 ? 4 : 1;
};

// ONE: one tile per workgroup.  Off: the type of an element's offset from the
// first row of a tile (32 bits where nx nv is known to allow it)
template <class T, int M, int Q, int C, bool ONE, class Off, class Ctx>
VP_HD void drift_body(Ctx& c, unsigned char* lds, const DriftArgs<T>& a) {
  using Cfg = DriftCfg<T, M, Q, C>;
  constexpr int TPT = Cfg::TPT;
  const int cc = c.tid % C;
  const int t = c.tid / C;
  cx<T>* buf = reinterpret_cast<cx<T>*>(lds + Cfg::tw_bytes) + cc * Cfg::stride;
  const size_t nv = (size_t)a.nv;
  const int inst = c.bidy;
  const size_t foff = (size_t)inst * (size_t)a.nx * nv;
  const double dk = a.dk_inst ? a.dk_inst[inst] : a.dk;
  const Off xo = (Off)(2 * t) * (Off)a.nv + (Off)cc;  // row 2t of a tile's column cc
  Tw<T> tw = tw_at<M, Q>(a.tw);
  if constexpr (Cfg::stage) {
    cx<T>* tl = reinterpret_cast<cx<T>*>(lds);
    for (int i = c.tid; i < 2 * M; i += c.nthr) tl[i] = i < M ? tw.w[i] : tw.p[i - M];
    tw = Tw<T>{tl, tl + M};
  }
  double acc[2 * Q];
  const int ntiles = a.nv / C;
  // workgroup b takes the run of `per` consecutive column tiles starting at
  // b per (per = ntiles / workgroups rounded up): neighbouring narrow tiles
  // share 128-byte lines, which one workgroup then fetches into one L2;
  // it accumulates the density of its tiles into one partial row dens[b][x]
  const int b0 = a.xcd_order ? xcd_block(c.bid, c.nblk) : c.bid;
  const int per = (ntiles + c.nblk - 1) / c.nblk;
  const int t0 = b0 * per, t1 = t0 + per < ntiles ? t0 + per : ntiles;
  auto load = [&](int tile, cx<T>* dst, double& vcol) {
    const T* fi = a.f_in + foff + tile * C;
#pragma unroll
    for (int i = 0; i < Q; ++i)
      dst[i] = mk<T>(at(fi + (size_t)(2 * i * TPT) * nv, xo), at(fi + (size_t)(2 * i * TPT + 1) * nv, xo));
    vcol = at(a.v + tile * C, (unsigned)cc);
  };
  auto advect = [&](int tile, cx<T>* v, double vc) {
    spectral_apply<T, M, TPT>(c, v, buf, tw, t, PhaseMul<T>((dk * a.dt) * vc, M, t, TPT));
    T* fo = a.f_out + foff + tile * C;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      at(fo + (size_t)(2 * i * TPT) * nv, xo) = v[i].re;
      at(fo + (size_t)(2 * i * TPT + 1) * nv, xo) = v[i].im;
    }
  };
  cx<T> v[Q];
  double vc = 0.0;
  if constexpr (ONE) {
    load(b0, v, vc);
    if constexpr (Cfg::stage) c.sync();
    advect(b0, v, vc);
    const double w = trapw(b0 * C + cc, a.nv);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      acc[2 * i] = w * (double)v[i].re;
      acc[2 * i + 1] = w * (double)v[i].im;
    }
  } else {
    // the next tile's columns are loaded before this tile's transforms, so
    // its reads are in flight during them
    cx<T> nxt[Q];
    double vc_next = 0.0;
#pragma unroll
    for (int i = 0; i < 2 * Q; ++i) acc[i] = 0.0;
    if (t0 < t1) load(t0, nxt, vc_next);
    if constexpr (Cfg::stage) c.sync();
    for (int tile = t0; tile < t1; ++tile) {
#pragma unroll
      for (int i = 0; i < Q; ++i) v[i] = nxt[i];
      vc = vc_next;
      if (tile + 1 < t1) load(tile + 1, nxt, vc_next);
      advect(tile, v, vc);
      const double w = trapw(tile * C + cc, a.nv);
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        acc[2 * i] += w * (double)v[i].re;
        acc[2 * i + 1] += w * (double)v[i].im;
      }
    }
  }
  if (a.dens) {
    double* out = a.dens + ((size_t)inst * c.nblk + c.bid) * a.nx;
    lane_fold<C, 2 * Q>(c, acc);
    if (fold_writer<C, 2 * Q>(cc)) {
      const int i0 = fold_index<C, 2 * Q>(cc);
#pragma unroll
      for (int j = 0; j < fold_count<C, 2 * Q>(); ++j) {
        const int i = i0 + j;  // sum i: x = 2 (t + (i / 2) TPT) + i % 2
        out[2 * (t + (i >> 1) * TPT) + (i & 1)] = acc[j];
      }
    }
  }
  if constexpr (Cfg::tail) {
    if (a.fuse_field) {
      // last workgroup to arrive reduces every partial row and solves Poisson
      int* flag = reinterpret_cast<int*>(lds + Cfg::lds - 16);
      const FieldArgs fa = field_instance(a.fld, inst);
      c.fence();
      c.sync();
      if (c.tid == 0) *flag = (c.arrive(fa.counter) == (unsigned)(c.nblk - 1)) ? 1 : 0;
      c.sync();
      if (!*flag) return;
      c.fence();
      field_body<M, Cfg::fq, Cfg::wg, true>(c, lds, fa);
      if (c.tid == 0) c.reset(fa.counter);
    }
  }
}

// ---------------------------------------------------------------------------
// x-advection of FP32 columns as two dense real-DFT products on MFMA
// (nx = NX in {32, 64}).  Each wave takes a tile of 16 columns:
//   Y = F X      (F: [NX][NX] forward real DFT, X: [NX][16] the columns)
//   phase        (Re_k, Im_k) of column c times exp(-i k phi_c)
//   X' = G Y'    (G: [NX][NX] inverse real DFT)
// through the context's 16 x 16 x 4 FP32 matrix product (c.mfma_16x16x4:
// D = A B + C, A 16x4, B 4x16; lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16], r < 4).  Rows of Y:
// Re_k for k <= NX/2 (row NX/2 the Nyquist bin), Im_k at row NX/2 + k
// (0 < k < NX/2), so a lane holds Re_k and Im_k of one column in tiles t and
// t + NX/32 at the same position.  The phase is the Stockham drift's:
// phi = (dk dt) v_c, exp(-i k phi) for 0 < k < NX/2 and cos((NX/2) phi) on
// the Nyquist bin (the real part the reference keeps).  The B operand of the
// second product is re-laid through a per-wave LDS tile.  W waves per
// workgroup; the workgroups stride over groups of W tiles (the tile count a
// multiple of W, so every wave makes the same number of passes).
// ---------------------------------------------------------------------------
struct f4 {
  float v[4];
};

template <int NX, int W>
struct DftCfg {
  static constexpr int T = NX / 16;   // 16-row tiles of the products
  static constexpr int KS = NX / 4;   // k-steps of 4
  static constexpr int GP = 17;       // pitch (floats) of a wave's Y' tile
  static constexpr int mat = 2 * NX * NX * 4;
  static constexpr int gt = NX * GP * 4;
  static constexpr int lds = mat + W * gt + W * NX * 8;
};

template <int NX, int W, class Ctx>
VP_HD void drift_dft_body(Ctx& c, unsigned char* lds, const DriftArgs<float>& a) {
  using Cfg = DftCfg<NX, W>;
  constexpr int T = Cfg::T, KS = Cfg::KS, GP = Cfg::GP;
  float* Fw = reinterpret_cast<float*>(lds);
  float* Iv = Fw + NX * NX;
  const int lane = c.tid & 63, w = c.tid >> 6;
  float* Y = reinterpret_cast<float*>(lds + Cfg::mat) + w * NX * GP;
  double* red = reinterpret_cast<double*>(lds + Cfg::mat + W * Cfg::gt);
  for (int i = c.tid; i < 2 * NX * NX; i += c.nthr) Fw[i] = a.dft[i];
  const int li = lane & 15, lk = lane >> 4;
  const size_t nv = (size_t)a.nv;
  const int inst = c.bidy;
  const size_t foff = (size_t)inst * NX * nv;
  const double dk = a.dk_inst ? a.dk_inst[inst] : a.dk;
  double dacc[T][4];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) dacc[t][r] = 0.0;
  // workgroup b takes a run of consecutive passes (neighbouring 16-column
  // tiles share 128-byte lines)
  const int groups = (a.nv / 16) / W;
  const int per = (groups + c.nblk - 1) / c.nblk;
  const int g0 = c.bid * per, g1 = g0 + per < groups ? g0 + per : groups;
  c.sync();  // matrices staged
  for (int gi = g0; gi < g1; ++gi) {
    const int col = (gi * W + w) * 16 + li;
    const float* fi = a.f_in + foff + col;
    f4 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = f4{{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float xb = fi[(size_t)(4 * s + lk) * nv];
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] = c.mfma_16x16x4(Fw[(16 * t + li) * NX + 4 * s + lk], xb, acc[t]);
    }
    // phase: bins k = 16 t + 4 lk + r (t < T/2) by a running product,
    // exp(-i k phi) = exp(-i 4 lk phi) exp(-i r phi) exp(-i 16 t phi)
    const double phi = (dk * a.dt) * a.v[col];
    cx<float> p0, p1, p16;
    cis_neg((double)(4 * lk) * phi, p0);
    cis_neg(phi, p1);
    cis_neg(16.0 * phi, p16);
    cx<float> pt = p0;
#pragma unroll
    for (int t = 0; t < T / 2; ++t) {
      cx<float> pk = pt;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float re = acc[t].v[r], im = acc[t + T / 2].v[r];
        if (t == 0 && r == 0 && lk == 0) {
          // DC unchanged; the partner row holds the real Nyquist bin
          cx<float> pn;
          cis_neg((double)(NX / 2) * phi, pn);
          acc[T / 2].v[0] = pn.re * im;
        } else {
          acc[t].v[r] = re * pk.re - im * pk.im;
          acc[t + T / 2].v[r] = im * pk.re + re * pk.im;
        }
        pk = mul(pk, p1);
      }
      pt = mul(pt, p16);
    }
    // Y' to the wave's LDS tile, rows 16 t + 4 lk + r, column li
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[(16 * t + 4 * lk + r) * GP + li] = acc[t].v[r];
    c.sync();
    f4 out[T];
#pragma unroll
    for (int t = 0; t < T; ++t) out[t] = f4{{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float yb = Y[(4 * s + lk) * GP + li];
#pragma unroll
      for (int t = 0; t < T; ++t) out[t] = c.mfma_16x16x4(Iv[(16 * t + li) * NX + 4 * s + lk], yb, out[t]);
    }
    c.sync();  // Y read by every lane before the next pass writes it
    float* fo = a.f_out + foff + col;
    const double wc = (col == 0 || col == a.nv - 1) ? 0.5 : 1.0;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        fo[(size_t)(16 * t + 4 * lk + r) * nv] = out[t].v[r];
        dacc[t][r] += wc * (double)out[t].v[r];
      }
  }
  if (!a.dens) return;
  // partial density of this workgroup: sum over the 16 columns of a lane
  // group, then over the waves
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double v = dacc[t][r];
      v = lane_sum<16>(c, v);
      if (li == 0) red[w * NX + 16 * t + 4 * lk + r] = v;
    }
  c.sync();
  double* out = a.dens + ((size_t)inst * c.nblk + c.bid) * NX;
  for (int x = c.tid; x < NX; x += c.nthr) {
    double sum = 0.0;
#pragma unroll
    for (int ww = 0; ww < W; ++ww) sum += red[ww * NX + x];
    out[x] = sum;
  }
}

// ---------------------------------------------------------------------------
// density rows: part[x] = scale * sum_v w_v f(x, v), W threads per row (64: one
// wavefront each, 256: one workgroup, for long rows), eight loads in flight
// per thread
// ---------------------------------------------------------------------------
template <class T, int W, class Ctx>
VP_HD void density_body(Ctx& c, const T* f, int nx, int nv, double scale, double* part, double* rs) {
  const int t = c.tid % W;
  const int row = c.bid * (c.nthr / W) + c.tid / W;
  const int rowc = row < nx ? row : nx - 1;
  const T* fr = f + (size_t)rowc * nv;
  double s[1] = {0.0};
  int m = t;
  for (; m + 7 * W < nv; m += 8 * W) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = (double)fr[m + u * W];
#pragma unroll
    for (int u = 0; u < 8; ++u) s[0] += trapw(m + u * W, nv) * x[u];
  }
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (m + u * W < nv) s[0] += trapw(m + u * W, nv) * (double)fr[m + u * W];
  row_sum<W, 1>(c, s, rs);
  if (row < nx && t == 0) part[row] = scale * s[0];
}

// ---------------------------------------------------------------------------
// collision diagonals a, b, c of every row (one wavefront per row)
// ---------------------------------------------------------------------------
template <class T, class Ctx>
VP_HD void diag_body(Ctx& c, const T* f, int nx, int nv, const double* v, double dv, double nu_dt, int op_dg,
                     double* A, double* B, double* Cc) {
  const int lane = c.tid & 63;
  const int row = c.bid * (c.nthr / 64) + (c.tid >> 6);
  const int rowc = row < nx ? row : nx - 1;
  const T* fr = f + (size_t)rowc * nv;
  double vbar = 0.0;
  double s[1] = {0.0};
  if (op_dg) {
    for (int m = lane; m < nv; m += 64) s[0] += trapw(m, nv) * (double)fr[m] * v[m];
    s[0] = lane_sum<64>(c, s[0]);
    vbar = dv * s[0];
    s[0] = 0.0;
  }
  for (int m = lane; m < nv; m += 64) {
    const double w = v[m] - vbar;
    s[0] += trapw(m, nv) * (double)fr[m] * (w * w);
  }
  s[0] = lane_sum<64>(c, s[0]);
  const double temp = dv * s[0];
  if (row >= nx) return;
  const double dv2 = dv * dv;
  const double A0 = -temp / dv2, H = 0.5 / dv;
  const double bd = 1.0 + nu_dt * (2.0 * temp / dv2);
  double* ar = A + (size_t)row * (nv - 1);
  double* cr = Cc + (size_t)row * (nv - 1);
  double* br = B + (size_t)row * nv;
  for (int m = lane; m < nv; m += 64) {
    br[m] = bd;
    if (m < nv - 1) {
      ar[m] = nu_dt * (A0 + (v[m] - vbar) * H);
      cr[m] = nu_dt * (A0 - (v[m + 1] - vbar) * H);
    }
  }
}

// ---------------------------------------------------------------------------
// tridiagonal solve with explicit diagonals (batched over rows)
// ---------------------------------------------------------------------------
template <class T>
struct TriArgs {
  const double* a;  // [nx][nv-1]
  const double* b;  // [nx][nv]
  const double* cc; // [nx][nv-1]
  const T* d;       // [nx][nv]
  T* x;             // [nx][nv]
  int nx, nv;
};

template <class T, int M, int Q, class Ctx>
VP_HD void tri_body(Ctx& c, unsigned char* lds, const TriArgs<T>& a) {
  using Cfg = RowCfg<T, M, Q>;
  constexpr int TPT = Cfg::TPT;
  constexpr int L = Cfg::L;
  const int t = c.tid % TPT;
  const int rl = c.tid / TPT;
  const int row = c.bid * Cfg::rows + rl;
  const bool valid = row < a.nx;
  const int rowc = valid ? row : a.nx - 1;
  double* red = reinterpret_cast<double*>(lds + rl * Cfg::region);
  const int N = a.nv;
  const T* dr = a.d + (size_t)rowc * N;
  double d[L];
#pragma unroll
  for (int i = 0; i < L; ++i) d[i] = (double)dr[t * L + i];
  ArrCoef cf;
  cf.a = a.a + (size_t)rowc * (N - 1);
  cf.bb = a.b + (size_t)rowc * N;
  cf.cc = a.cc + (size_t)rowc * (N - 1);
  cf.N = N;
  tridiag<TPT, L, ArrCoef, Ctx, sizeof(T) == 8>(c, d, cf, t, red);
  if (valid) {
    T* xr = a.x + (size_t)row * N;
#pragma unroll
    for (int i = 0; i < L; ++i) xr[t * L + i] = (T)d[i];
  }
}

// ---------------------------------------------------------------------------
// several batches in one launch (vpfp_group_*): each kernel takes a table of
// segments, one per batch, and its workgroups are numbered across them;
// segment s owns the workgroups [blk0, blk0 of segment s+1).  The wrapper
// picks the workgroup's segment, rebases the arguments and runs the body
// with the workgroup index local to the segment.
// ---------------------------------------------------------------------------
constexpr int kMaxSeg = 8;

template <class T>
struct RowSeg {
  T* f;  // read and written in place
  const double* e;
  const double* nu_dt;  // per instance
  int rows;             // x rows of the batch (instances * nx)
  int rows_per_inst;
  int blk0;
};
template <class T>
struct RowMulti {
  RowArgs<T> base;  // shared: flags, dt, v grid, tables (one nv)
  int nseg;
  RowSeg<T> seg[kMaxSeg];
};

template <class T>
struct DriftSeg {
  T* f;
  const double* v;
  const double* dk;  // per instance
  double* dens;
  int nv;
  int gx;            // workgroups per instance
  int n_inst;
  int blk0;
};
template <class T>
struct DriftMulti {
  DriftArgs<T> base;  // shared: nx, dt, twiddles
  int nseg;
  DriftSeg<T> seg[kMaxSeg];
};

struct FieldSeg {
  const double* part;
  double scale;  // dv of the batch's v grid
  int ntiles;
  const double* okx;
  double* e_out;
  double* series;
  int n_inst;
  int blk0;
};
struct FieldMulti {
  FieldArgs base;  // shared: nx, scale, twiddles
  int nseg;
  FieldSeg seg[kMaxSeg];
};

// segment of workgroup b (blk0 ascending, seg[0].blk0 == 0)
template <class S>
VP_HD int seg_of(const S* seg, int nseg, int b) {
  int s = 0;
  for (int i = 1; i < nseg; ++i)
    if (b >= seg[i].blk0) s = i;
  return s;
}

}  // namespace vp
