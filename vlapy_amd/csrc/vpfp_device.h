// Device building blocks for the VPFP kernels (gfx950, wave64).
//
// Everything here is written against a small block context `Ctx` that
// provides `tid`, `nthr` (thread index and count in the workgroup), `bid`,
// `nblk` (workgroup index and count along x), `bidy` (workgroup index along
// y: the instance of a batched scan), `sync()` (workgroup barrier),
// `add_lane<MASK>(v)` and `fold_lane<MASK>(lo, hi)` (sums of a lane pair),
// `any(p)` (over a wavefront) and, for the cross-workgroup hand-off of the field
// kernel, `fence()` (device-scope fence), `arrive(counter)` (device-scope atomic
// increment, returns the old value) and `reset(counter)`.  GpuCtx
// (vpfp_launch.h) provides it with the hardware primitives.
//
// Contents
//   * cx<T>        : complex value in registers / LDS (T = double or float)
//   * dft<R>       : R-point DFT in registers (radix-2 network, R <= 32)
//   * fft<M,TPT>   : M-point complex FFT of one sequence held by TPT threads,
//                    Q = M/TPT values per thread in registers, exchanged
//                    through a padded LDS buffer between Stockham passes
//   * couple()     : half-length real-FFT unpack, Fourier multiplier, repack
//   * row_sum<>    : sum over the TPT threads that own one sequence
//   * tridiag      : partition solver for one diagonally dominant
//                    tridiagonal system held by TPT threads (one elimination
//                    sweep per chunk, elimination of the even interface
//                    unknowns, parallel cyclic reduction of the TPT odd ones
//                    in LDS, back-substitution of the chunk interiors)
#pragma once

#if defined(__HIP__)
#include <hip/hip_runtime.h>
#define VP_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#define VP_HD inline
#endif

namespace vp {

// ---------------------------------------------------------------------------
// complex arithmetic
// ---------------------------------------------------------------------------
template <class T>
struct cx {
  T re, im;
};

template <class T>
VP_HD cx<T> mk(T r, T i) {
  cx<T> z;
  z.re = r;
  z.im = i;
  return z;
}
template <class T>
VP_HD cx<T> add(cx<T> a, cx<T> b) { return mk<T>(a.re + b.re, a.im + b.im); }
template <class T>
VP_HD cx<T> sub(cx<T> a, cx<T> b) { return mk<T>(a.re - b.re, a.im - b.im); }
template <class T>
VP_HD cx<T> mul(cx<T> a, cx<T> b) {
  return mk<T>(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
// a * conj(b)
template <class T>
VP_HD cx<T> mulc(cx<T> a, cx<T> b) {
  return mk<T>(a.re * b.re + a.im * b.im, a.im * b.re - a.re * b.im);
}

// base[i] with a base that is the same in all lanes and a 32-bit byte offset
// per lane (i * sizeof < 2^32): the address stays in scalar registers, where
// base[i] with an int takes a 64-bit one per load and lane (the drift of one
// tile per workgroup at nx = 1024: 117 -> 109 registers FP32, 152 -> 88 bytes
// spilled FP64; drift of nx = 64 FP32 scan columns 122 -> 112 us, rows of
// nv = 1024 224 -> 213 us)
template <class U>
VP_HD U& at(U* base, unsigned i) {
  using B = char;
  return *reinterpret_cast<U*>(const_cast<B*>(reinterpret_cast<const B*>(base)) + i * (unsigned)sizeof(U));
}

template <class U>
VP_HD U& at(U* base, unsigned long i) {
  return base[i];
}

// Padded LDS index: one spare slot every 16 elements keeps the strided
// writes of the first Stockham pass and the chunk reads of the tridiagonal
// solver spread over the LDS banks.
VP_HD constexpr int pidx(int i) { return i + (i >> 4); }
template <int M>
struct Padded {
  static constexpr int size = M + ((M - 1) >> 4) + 1;
};

// ---------------------------------------------------------------------------
// 1/x to double precision: hardware reciprocal estimate refined by two
// Newton steps (within an ulp of the correctly rounded quotient; cheaper
// than the IEEE division sequence in the tridiagonal sweeps)
// ---------------------------------------------------------------------------
VP_HD double rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
#else
  return 1.0 / x;
#endif
}
// The same with one Newton step: the estimate's ~23 correct bits doubled to
// ~46 (relative error ~2^-46), for the FP64 elimination of FP32-stored f,
// whose own rounding (2^-24) is ten orders of magnitude larger.
VP_HD double rcp46(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(x);
  return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
#else
  return 1.0 / x;
#endif
}
template <bool FULL>
VP_HD double rcpp(double x) {
  if constexpr (FULL)
    return rcp(x);
  else
    return rcp46(x);
}

// ---------------------------------------------------------------------------
// exp(-i theta) in the working precision
// ---------------------------------------------------------------------------
// sin and cos of |y| <= pi/2 in FP32 from their Taylor series, Horner in y^2
// with fma: sin to y^13, cos to y^14 (the first terms left out are below
// 1e-9 at pi/2); absolute error ~1 ulp of 1, and sin keeps its relative
// precision for small y (the y term is added last).  Cheaper than a general
// sincosf, which reduces the argument again and checks for large ones.
VP_HD void sincos_half(float y, float& s, float& c) {
  const float y2 = y * y;
  const float ps = fmaf(
      y2, fmaf(y2, fmaf(y2, fmaf(y2, fmaf(y2, 1.605904384e-10f, -2.505210839e-08f), 2.755731922e-06f), -1.984126984e-04f),
               8.333333333e-03f),
      -1.666666667e-01f);
  s = fmaf(y * y2, ps, y);
  const float pc = fmaf(
      y2,
      fmaf(y2, fmaf(y2, fmaf(y2, fmaf(y2, fmaf(y2, -1.147074560e-11f, 2.087675699e-09f), -2.755731922e-07f), 2.480158730e-05f),
                    -1.388888889e-03f),
           4.166666667e-02f),
      -0.5f);
  c = fmaf(y2, pc, 1.f);
}

VP_HD void cis_neg(double th, cx<float>& out) {
  // reduce in double so that large arguments keep float accuracy; then the
  // half angle (|r / 2| <= pi / 2): cos r = 1 - 2 s^2, sin r = 2 s c
  const double r = th - 6.283185307179586 * rint(th * 0.15915494309189535);
  float s, c;
  sincos_half((float)(0.5 * r), s, c);
  out = mk<float>(fmaf(-2.f * s, s, 1.f), -2.f * s * c);
}

// Natural log in FP64 for the f log f moment: x = m 2^e with m in
// [sqrt(1/2), sqrt(2)), f = m - 1 (exact), s = f / (2 + f) (|s| <= 0.1716),
// log(1 + f) = 2 atanh(s) = f - s (f - R), R = sum_k 2 s^(2k) / (2k + 1) for
// k = 1..11 (the first term left out is below 2e-19 relative), and
// log x = e ln 2 + log(1 + f) with ln 2 split in two; ~2 ulp.  x = 0 gives
// -inf, x < 0 and NaN give NaN, +inf gives +inf, as log does.  About half the
// instructions of the library log, which also covers the correctly rounded
// cases this moment does not need.
VP_HD double log_f64(double x) {
  int e;
  double m = frexp(x, &e);
  const bool lo = m < 0.70710678118654752;
  m = lo ? 2.0 * m : m;
  e -= lo ? 1 : 0;
  const double f = m - 1.0;
  const double s = f * rcp(2.0 + f);
  const double z = s * s;
  double r = 0.086956521739130432;  // 2/23
  r = fma(z, r, 0.095238095238095233);
  r = fma(z, r, 0.10526315789473684);
  r = fma(z, r, 0.11764705882352941);
  r = fma(z, r, 0.13333333333333333);
  r = fma(z, r, 0.15384615384615385);
  r = fma(z, r, 0.18181818181818182);
  r = fma(z, r, 0.22222222222222221);
  r = fma(z, r, 0.2857142857142857);
  r = fma(z, r, 0.40000000000000002);
  r = fma(z, r, 0.66666666666666663);  // 2/3
  r *= z;
  const double l1p = fma(-s, f - r, f);
  const double de = (double)e;
  const double v = fma(de, 0.6931471805599453, fma(de, 2.3190468138462996e-17, l1p));
  return x > 0.0 ? (x < __builtin_huge_val() ? v : x) : (x == 0.0 ? -__builtin_huge_val() : __builtin_nan(""));
}

// theta - 2 pi n with n = rint(theta / 2 pi), two-term Cody-Waite with fma
// (2 pi = C1 + C2, C1 its double rounding): |r| <= pi to a few ulp for the
// arguments of the kicks and drifts
VP_HD double reduce_2pi(double th) {
  const double n = rint(th * 0.15915494309189535);
  return fma(-n, 2.4492935982947064e-16, fma(-n, 6.283185307179586, th));
}

// sin and cos of |y| <= pi/2 in FP64 from their Taylor series, Horner in y^2
// with fma: sin to y^23, cos to y^24 (the first terms left out are below
// 1e-20 at pi/2); ~1 ulp, and sin keeps its relative precision for small y
VP_HD void sincos_half(double y, double& s, double& c) {
  const double y2 = y * y;
  double p = -3.86817017063068413e-23;
  p = fma(y2, p, 1.95729410633912626e-20);
  p = fma(y2, p, -8.22063524662432950e-18);
  p = fma(y2, p, 2.81145725434552060e-15);
  p = fma(y2, p, -7.64716373181981641e-13);
  p = fma(y2, p, 1.60590438368216133e-10);
  p = fma(y2, p, -2.50521083854417202e-08);
  p = fma(y2, p, 2.75573192239858925e-06);
  p = fma(y2, p, -1.98412698412698413e-04);
  p = fma(y2, p, 8.33333333333333322e-03);
  p = fma(y2, p, -1.66666666666666657e-01);
  s = fma(y * y2, p, y);
  double q = 1.61173757109611839e-24;
  q = fma(y2, q, -8.89679139245057408e-22);
  q = fma(y2, q, 4.11031762331216484e-19);
  q = fma(y2, q, -1.56192069685862253e-16);
  q = fma(y2, q, 4.77947733238738525e-14);
  q = fma(y2, q, -1.14707455977297245e-11);
  q = fma(y2, q, 2.08767569878681002e-09);
  q = fma(y2, q, -2.75573192239858883e-07);
  q = fma(y2, q, 2.48015873015873016e-05);
  q = fma(y2, q, -1.38888888888888894e-03);
  q = fma(y2, q, 4.16666666666666644e-02);
  q = fma(y2, q, -0.5);
  c = fma(y2, q, 1.0);
}

VP_HD void cis_neg(double th, cx<double>& out) {
  double s, c;
  sincos_half(0.5 * reduce_2pi(th), s, c);
  out = mk<double>(fma(-2.0 * s, s, 1.0), -2.0 * s * c);
}

// ---------------------------------------------------------------------------
// R-point DFT in registers (radix-2 decimation in time, R <= 32)
// ---------------------------------------------------------------------------
// cos(2 pi j / 32) for j = 0..8, correctly rounded
VP_HD constexpr double cos32q(int j) {
  return j == 0   ? 1.0
         : j == 1 ? 0.9807852804032304
         : j == 2 ? 0.9238795325112867
         : j == 3 ? 0.8314696123025452
         : j == 4 ? 0.7071067811865476
         : j == 5 ? 0.5555702330196022
         : j == 6 ? 0.3826834323650898
         : j == 7 ? 0.19509032201612828
                  : 0.0;
}
VP_HD constexpr double cos32(int J) {
  return (J & 31) <= 8    ? cos32q(J & 31)
         : (J & 31) <= 16 ? -cos32q(16 - (J & 31))
         : (J & 31) <= 24 ? -cos32q((J & 31) - 16)
                          : cos32q(32 - (J & 31));
}
VP_HD constexpr double sin32(int J) { return cos32(J - 8); }

// b * W_32^J for J = 0, 8, 16 or 24 (forward: W = exp(-2 pi i J / 32); inverse: conjugate)
template <bool INV, class T>
VP_HD cx<T> quarter_turns(cx<T> b, int J) {
  if (J == 0) return b;
  if (J == 16) return mk<T>(-b.re, -b.im);
  if (J == 8) return INV ? mk<T>(-b.im, b.re) : mk<T>(b.im, -b.re);
  return INV ? mk<T>(b.im, -b.re) : mk<T>(-b.im, b.re);
}

template <int R>
VP_HD constexpr int brev(int i) {
  int r = 0;
  for (int b = 1; b < R; b <<= 1) {
    r = (r << 1) | (i & 1);
    i >>= 1;
  }
  return r;
}

VP_HD float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
VP_HD double fma_t(double a, double b, double c) { return fma(a, b, c); }

// (a, b) <- (a + W b, a - W b) with W = W_32^J (inverse: its conjugate), in 6
// instructions at odd multiples of 45 degrees, whose factor goes into the two
// sums as their fma, instead of the 8 of a product and two sums.
//
// The other angles (radix 16) take 10, with the larger part of W as 1 - g: a
// rounded cos(pi/8) is the same 3e-8 off in every transform, so its error grows
// with the steps as nothing random does, and 1 - g with a rounded g is 2e-9 off.
// Rows of nv = 8192 in FP32 at 16 values, collisions, f after 4 and 12 steps:
// 8.05e-7 and 2.18e-6 off with tan(pi/8) and the rounded larger part factored out
// (6 instructions, four steps of 1024 rows 364 us), 5.9e-7 and 1.50e-6 so (366 to
// 368 us); 8 values, which have multiples of 45 degrees only, 6.6e-7 and 1.67e-6
// (with the half phase in FP64 since: 5.7e-7, 1.42e-6; 6.4e-7, 1.59e-6).
template <bool INV, class T>
VP_HD void butterfly(cx<T>& a, cx<T>& b, int J) {
  J &= 31;
  const cx<T> x = a;
  if ((J & 7) == 0) {
    const cx<T> w = quarter_turns<INV>(b, J);
    a = add(x, w);
    b = sub(x, w);
    return;
  }
  // W b = (b.re cd + b.im sd, b.im cd - b.re sd)
  const double cd = cos32(J), sd = INV ? -sin32(J) : sin32(J);
  if ((J & 3) == 0) {
    const T f = (T)cd;
    const bool same = (cd > 0) == (sd > 0);
    const T u = same ? b.re + b.im : b.re - b.im, w = same ? b.im - b.re : b.im + b.re;
    a = mk<T>(x.re + f * u, x.im + f * w);
    b = mk<T>(x.re - f * u, x.im - f * w);
    return;
  }
  // W b = sg (p - g p + h q), p the turn of b by the axis next to W, q by the other
  const bool cbig = cd * cd > sd * sd;
  const double big = cbig ? cd : sd, small = cbig ? sd : cd;
  const bool pos = big > 0;
  const T g = (T)(1.0 - (pos ? big : -big)), h = (T)(pos ? small : -small);
  const cx<T> r = mk<T>(b.im, -b.re), p = cbig ? b : r, q = cbig ? r : b;
  const T u = p.re + fma_t(h, q.re, -g * p.re), w = p.im + fma_t(h, q.im, -g * p.im);
  a = pos ? mk<T>(x.re + u, x.im + w) : mk<T>(x.re - u, x.im - w);
  b = pos ? mk<T>(x.re - u, x.im - w) : mk<T>(x.re + u, x.im + w);
}

template <int R, bool INV, class T>
VP_HD void dft(cx<T>* x) {
  static_assert(R >= 1 && R <= 32 && (R & (R - 1)) == 0, "radix must be a power of two <= 32");
  if constexpr (R == 1) return;
  cx<T> y[R];
#pragma unroll
  for (int i = 0; i < R; ++i) y[brev<R>(i)] = x[i];
#pragma unroll
  for (int h = 1; h < R; h <<= 1) {
#pragma unroll
    for (int g = 0; g < R; g += 2 * h) {
#pragma unroll
      for (int j = 0; j < h; ++j) butterfly<INV>(y[g + j], y[g + j + h], j * (16 / h));
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) x[i] = y[i];
}

// ---------------------------------------------------------------------------
// Twiddle tables of an N = 2M point real transform, in global memory:
//   [ W_N^k, k < M | passes for Q = 8 | passes for Q = 4 | passes for Q = 16 ],
// M entries each (the field's table ends after the second).  A pass of radix R
// after NS = R0 R1 ... points (R0 the first radix) reads W_{NS R}^{r k} from
// entry NS - R0 + (r - 1) NS + k of its Q's part, so that the lanes of a wave
// read consecutive entries.  They come through L1 while the passes exchange
// through LDS; each is loaded before the barrier ahead of its use.  Staged in
// LDS instead, the table limited the workgroups on a CU (16 KiB of 25 for an
// FP64 row of nv = 1024) and its strided reads conflicted on the banks: scan
// step of 512 FP64 instances 669 -> 594 us, 1024 x 8192 FP64 218 -> 195.
// ---------------------------------------------------------------------------
VP_HD constexpr int tw_slot(int Q) { return Q == 4 ? 2 : Q == 16 ? 3 : 1; }

template <class T>
struct Tw {
  const cx<T>* w;  // W_N^k
  const cx<T>* p;  // pass tables of the transform's Q
};

// the tables at `tab` for Q values per thread (Q = M < 8: one pass, no table)
template <int M, int Q, class T>
VP_HD Tw<T> tw_at(const cx<T>* tab) {
  return Tw<T>{tab, tab + M * (Q == M ? 0 : tw_slot(Q))};
}

// ---------------------------------------------------------------------------
// M-point complex FFT held by TPT threads (Stockham autosort, radix <= 16)
//
// Register layout: thread t holds element t + i*TPT in v[i], i < Q = M/TPT.
// A pass of radix R with NS = product of the earlier radices takes the
// butterfly j = t + q*TPT (inputs j + r*M/R = v[q + r*Q/R]), twiddles input r
// by W_{NS*R}^{r*(j mod NS)}, does an R-point DFT and sends output r to
// position (j - j mod NS)*R + j mod NS + r*NS.  In the last pass NS = M/R, so
// j mod NS = j and output r belongs at j + r*M/R: the place its register
// already has.  Only the passes before the last go through `buf`; the
// transform ends with the data in natural order in v and `buf` free.
//
// ---------------------------------------------------------------------------
template <int M, int TPT, int NS>
struct Pass {
  static constexpr int Q = M / TPT;
  static_assert(Q >= 2 && Q * TPT == M, "each thread must hold at least two values");
  static constexpr int RMAX = Q < 16 ? Q : 16;
  static constexpr int R0 = M < RMAX ? M : RMAX;
  static constexpr int R = (M / NS) < RMAX ? (M / NS) : RMAX;
  static constexpr int NB = Q / R;
  static_assert(NB * R == Q, "radix must divide the per-thread count");
  // j mod NS is the same for all of a thread's butterflies when NS divides TPT
  static constexpr int NK = NS > TPT ? NB : 1;
  static constexpr int NW = NK * (R - 1) > 0 ? NK * (R - 1) : 1;
};

template <class T, int M, int TPT, int NS>
VP_HD void load_twiddles(cx<T>* w, const Tw<T>& tw, int t) {
  using P = Pass<M, TPT, NS>;
#pragma unroll
  for (int q = 0; q < P::NK; ++q) {
    const cx<T>* p = tw.p + (NS - P::R0);
    const unsigned k = (unsigned)(t + q * TPT) & (NS - 1);
#pragma unroll
    for (int r = 1; r < P::R; ++r) w[q * (P::R - 1) + r - 1] = at(p + (r - 1) * NS, k);
  }
}

// passes from NS on; w: this pass's twiddles (NS > 1).  `act` false: the
// thread only takes part in the barriers (no LDS writes).
template <class T, int M, int TPT, bool INV, int NS, class Ctx>
VP_HD void fft_passes(Ctx& c, cx<T>* v, cx<T>* buf, const Tw<T>& tw, int t, bool act, const cx<T>* w) {
  using P = Pass<M, TPT, NS>;
  constexpr int Q = P::Q, R = P::R, NB = P::NB;
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const int j = t + q * TPT;
    const int k = j & (NS - 1);
    cx<T> u[R];
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = v[q + r * NB];
    if constexpr (NS > 1) {
      const cx<T>* wq = w + (P::NK > 1 ? q * (R - 1) : 0);
#pragma unroll
      for (int r = 1; r < R; ++r) u[r] = INV ? mulc(u[r], wq[r - 1]) : mul(u[r], wq[r - 1]);
    }
    dft<R, INV>(u);
    if constexpr (NS * R < M) {
      if (act) {
        const int base = (j - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[pidx(base + r * NS)] = u[r];
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) v[q + r * NB] = u[r];
    }
  }
  if constexpr (NS * R < M) {
    cx<T> wn[Pass<M, TPT, NS * R>::NW];
    load_twiddles<T, M, TPT, NS * R>(wn, tw, t);
    c.sync();
#pragma unroll
    for (int i = 0; i < Q; ++i) v[i] = buf[pidx(t + i * TPT)];
    c.sync();
    fft_passes<T, M, TPT, INV, NS * R>(c, v, buf, tw, t, act, wn);
  }
}

template <class T, int M, int TPT, bool INV, class Ctx>
VP_HD void fft(Ctx& c, cx<T>* v, cx<T>* buf, const Tw<T>& tw, int t, bool act = true) {
  fft_passes<T, M, TPT, INV, 1>(c, v, buf, tw, t, act, static_cast<const cx<T>*>(nullptr));
}

// ---------------------------------------------------------------------------
// Fourier multipliers for the half-length real transform
//
// For own bin k in [0, M) `pair` returns P_k and P_{M-k}; for k == 0 it
// returns the real factors applied to the DC and Nyquist bins (the real part
// of the multiplier, which is what taking Re() of the complex inverse leaves).
// ---------------------------------------------------------------------------

// s (C + i S) / (C^2 + S^2), with the rounding error of the norm taken to first
// order.  A spectrum with F_{k+M} = 0 (a resolved f) comes out of the
// expression below times (C - i S) (C + i S) / M: dividing by the rounded
// norm keeps the pushers from scaling every mode by the same rounding error
// step after step, and what is left of the error of C and S is one of P_M.
//
// Of FP32 C and S it is formed, and multiplied with a phase, in FP64: the low
// bins, where a resolved f lies, take no other product, so its roundings come back
// kick by kick, and an FP32 correction of the norm is lost below half an ulp of 1.
// Eight steps with collisions, 64 x 512: f 9.8e-7 off with FP32 products, 8.2e-7 so
// (7.9e-7 with unpack, multiply and repack apart); 64 x 1024: 8.9e-7, 7.6e-7
// (7.6e-7); 256 x 2048 delta-f: E 3.8e-7, 3.1e-7 (4.7e-7).  It takes no time.
VP_HD cx<double> half_phase(double C, double S, double s) {
  const double e = C * C > 0.5 ? fma(S, S, fma(C, C, -1.0)) : fma(C, C, fma(S, S, -1.0));
  const double w = s - s * e;
  return mk<double>(C * w, S * w);
}
VP_HD cx<float> mul(cx<float> a, cx<double> b) {
  const double x = a.re, y = a.im;
  return mk<float>((float)(x * b.re - y * b.im), (float)(x * b.im + y * b.re));
}

// Phase shift exp(-i theta_k) of the exponential pushers, theta_k = k phi
// with phi = (dk * dt) * s: dk is the first wavenumber of an fftfreq table
// (checked on the host to be linear in k to rounding), s the advection speed
// (e(x) for the v-kick, v for the x-drift).
//
// With P_{M-k} = P_M conj(P_k) the unpack, multiply and repack of couple()
// below collapse into one expression in Z_k and Z_{M-k}:
//   Z'_k = p_k [ (C + i S sin(pi k / M)) Z_k + S cos(pi k / M) conj(Z_{M-k}) ],
//   C + i S = exp(i M phi / 2),  p_k = exp(-i (k - M/2) phi) / M,
// for 0 < k < M (from E + i O = Z and W O + i conj(W) E =
// -sin Z + i cos conj(Z_{M-k}) with W = exp(-i pi k / M)); the DC bin keeps its
// value and the Nyquist bin gets cos(M phi) = 1 - 2 S^2.  16 instructions per
// bin instead of 44 for the three steps apart; with the last Stockham passes
// kept in registers: nv = 8192 FP64 kicks 69 -> 63 us (1024 rows), nx = 1024
// FP64 drift 66 -> 59 us, nx = 128 FP32 drift of a scan 503 -> 482 us.  Bins
// are visited in the order k = t, t + TPT, ..., so p_k is a running product, of
// at most 8 factors: with 16 bins per thread it starts anew at the 9th, whose
// rounding otherwise grows with them (one FP32 kick of nv = 8192 by 3 dk dt:
// 7.8e-7 off in f, with the new start 4.0e-7, with 8 bins per thread 5.9e-7).
template <class T>
struct PhaseMul {
  T C, S;
  cx<T> cur, step, mid;  // mid: cur of the 9th of 16 bins
  VP_HD PhaseMul() {}
  VP_HD PhaseMul(double phi, int M, int t, int TPT) {
    cx<T> h;
    cis_neg(-0.5 * (double)M * phi, h);
    C = h.re;
    S = h.im;
    cis_neg((double)t * phi, cur);
    cur = mul(cur, half_phase(C, S, 1.0 / M));
    cis_neg((double)TPT * phi, step);
    if (M / TPT == 16) {
      cis_neg((double)(t + 8 * TPT) * phi, mid);
      mid = mul(mid, half_phase(C, S, 1.0 / M));
    }
  }
};

// exp(-i theta) - 1 without cancellation: (-2 sin^2(theta/2), -2 sin(theta/2)
// cos(theta/2)), from one sincos of the half angle after reduction in double
// (FP32 sincos for FP32 results: both parts keep FP32 relative precision
// also for tiny theta)
template <class T>
VP_HD cx<T> cis_neg_m1(double th) {
  const double r = th - 6.283185307179586 * rint(th * 0.15915494309189535);
  if constexpr (sizeof(T) == 4) {
    float s, c;
    sincos_half((float)(0.5 * r), s, c);
    return mk<T>(-2.0f * s * s, -2.0f * s * c);
  } else {
    double s, c;
    sincos_half(0.5 * reduce_2pi(th), s, c);
    return mk<T>(-2.0 * s * s, -2.0 * s * c);
  }
}

// PhaseMul on a stored deviation f - B from a fixed background B with
// unnormalised spectrum B_k: the shift of B itself enters as
// F'_k += B_k (P_k - 1), F'_{k+M} += B_{k+M} (conj P_{M-k} - 1), in the repacked
// spectrum
//   Z'_k += b1_k (P_k - 1) + b2_k (conj P_{M-k} - 1),
//   b1_k = B_k (1 + i conj W_k) / N,  b2_k = B_{k+M} (1 - i conj W_k) / N,
// tables the host forms ([b1: M | b2: M], storage precision).  Both factors are
// carried without cancellation: c_k = P_k - 1 by c_{k+s} = c_k + c_s + c_k c_s
// upwards from the thread's first bin, and q_k = conj P_{M-k} - 1 =
// exp(i (M - k) phi) - 1 the same way downwards from its last bin, where it is
// smallest and b2 largest (formed from c_k and P_M instead, q_k keeps only the
// absolute rounding of P_M: FP32 scans at nv = 2048 were 7e-6 off in f
// after four steps, now 7e-7).  The data's phases are
// p_k = (1 + c_k) (C + i S) / M.
template <class T>
struct BgPhaseMul {
  T C, S;
  cx<T> cm, cs, qm;  // P_t - 1, P_TPT - 1, exp(i (TPT - t) phi) - 1
  cx<T> cm8, qm7;    // of 16 bins: P_k - 1 of the 9th, exp(i (M - k) phi) - 1 of the 8th
  const cx<T>* bhat;
  VP_HD BgPhaseMul() {}
  VP_HD BgPhaseMul(double phi, int M, int t, int TPT, const cx<T>* bhat_) : bhat(bhat_) {
    cx<T> h;
    cis_neg(-0.5 * (double)M * phi, h);
    C = h.re;
    S = h.im;
    cm = cis_neg_m1<T>((double)t * phi);
    cs = cis_neg_m1<T>((double)TPT * phi);
    qm = cis_neg_m1<T>((double)(t - TPT) * phi);
    if (M / TPT == 16) {
      cm8 = cis_neg_m1<T>((double)(t + 8 * TPT) * phi);
      qm7 = cis_neg_m1<T>((double)(t - 9 * TPT) * phi);
    }
  }
};

// Poisson multiplier i * one_over_kx (zero real part at DC and Nyquist);
// okx is an LDS copy of the one_over_kx table.
template <class T>
struct PoissonMul {
  const double* okx;
  int M;
  VP_HD void pair(int k, cx<T>& pk, cx<T>& pmk) {
    if (k == 0) {
      pk = mk<T>(T(0), T(0));
      pmk = mk<T>(T(0), T(0));
      return;
    }
    pk = mk<T>(T(0), (T)okx[k]);
    pmk = mk<T>(T(0), (T)okx[M - k]);
  }
};

// z_j = f_{2j} + i f_{2j+1} was transformed to Z (M points).  With
// E_k = (Z_k + conj Z_{M-k})/2, O_k = (Z_k - conj Z_{M-k})/(2i) and
// W = exp(-2 pi i k / N), the real N-point spectrum is F_k = E_k + W O_k and
// F_{k+M} = E_k - W O_k.  After F'_k = P_k F_k, F'_{k+M} = conj(P_{M-k}) F_{k+M}
// the repacked spectrum Z'_k = (F'_k + F'_{k+M} + i (F'_k - F'_{k+M}) conj W)/N
// inverse-transforms (unnormalised M-point) to f'_{2j} + i f'_{2j+1}.
// v[i] holds Z_k, pz[i] Z_{M-k} and wk[i] W^k for k = t + i*TPT.
template <class T, int M, int TPT>
VP_HD void couple(cx<T>* v, const cx<T>* pz, const cx<T>* wk, int t, PoissonMul<T>& mult) {
  constexpr int Q = M / TPT;
  const T invN = T(1) / T(2 * M);
  const T h = T(0.5);
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int k = t + i * TPT;
    const cx<T> a = v[i], p = pz[i];
    const cx<T> E = mk<T>((a.re + p.re) * h, (a.im - p.im) * h);
    const cx<T> O = mk<T>((a.im + p.im) * h, (p.re - a.re) * h);
    const cx<T> W = wk[i];
    const cx<T> WO = mul(W, O);
    const cx<T> Fk = add(E, WO), Fkm = sub(E, WO);
    cx<T> pk, pmk;
    mult.pair(k, pk, pmk);
    const cx<T> G1 = mul(pk, Fk);
    const cx<T> G2 = mulc(Fkm, pmk);
    const cx<T> S = add(G1, G2);
    const cx<T> D = mulc(sub(G1, G2), W);
    v[i] = mk<T>((S.re - D.im) * invN, (S.im + D.re) * invN);
  }
}

// (C + i S sin) a + S cos conj(p), W = (cos, -sin)
template <class T>
VP_HD cx<T> couple_bin(T C, T S, cx<T> W, cx<T> a, cx<T> p) {
  const T g = S * W.im, h = S * W.re;  // g = -S sin
  return mk<T>(C * a.re + g * a.im + h * p.re, C * a.im - g * a.re - h * p.im);
}

// DC unchanged, Nyquist times 1 + nyq
template <class T>
VP_HD cx<T> couple_dc(cx<T> a, T nyq, T invN) {
  const T f0 = a.re + a.im, fm = a.re - a.im;
  const T g2 = fm + nyq * fm;
  return mk<T>((f0 + g2) * invN, (f0 - g2) * invN);
}

template <class T, int M, int TPT>
VP_HD void couple(cx<T>* v, const cx<T>* pz, const cx<T>* wk, int t, PhaseMul<T>& m) {
  constexpr int Q = M / TPT;
  cx<T> cur = m.cur;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const cx<T> a = v[i];
    v[i] = mul(cur, couple_bin(m.C, m.S, wk[i], a, pz[i]));
    if (i == 0 && t == 0) v[0] = couple_dc(a, T(-2) * m.S * m.S, T(1) / T(2 * M));
    if (i + 1 < Q) cur = Q == 16 && i == 7 ? m.mid : mul(cur, m.step);
  }
}

template <class T, int M, int TPT>
VP_HD void couple(cx<T>* v, const cx<T>* pz, const cx<T>* wk, int t, BgPhaseMul<T>& m) {
  constexpr int Q = M / TPT;
  const cx<double> hp = half_phase(m.C, m.S, 1.0 / M);
  const cx<T> kap = mk<T>((T)hp.re, (T)hp.im);
  // a + b + a b
  auto m1_mul = [](cx<T> a, cx<T> b) {
    return mk<T>((a.re + b.re) + (a.re * b.re - a.im * b.im), (a.im + b.im) + (a.re * b.im + a.im * b.re));
  };
  const cx<T> csc = mk<T>(m.cs.re, -m.cs.im);
  cx<T> q[Q];
  q[Q - 1] = m.qm;
#pragma unroll
  for (int i = Q - 2; i >= 0; --i) q[i] = Q == 16 && i == 7 ? m.qm7 : m1_mul(q[i + 1], csc);
  cx<T> cm = m.cm;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const cx<T> B1 = at(m.bhat + i * TPT, (unsigned)t), B2 = at(m.bhat + i * TPT + M, (unsigned)t);
    const cx<T> a = v[i];
    const cx<T> pk = mk<T>(kap.re + (kap.re * cm.re - kap.im * cm.im), kap.im + (kap.re * cm.im + kap.im * cm.re));
    const cx<T> y = mul(pk, couple_bin(m.C, m.S, wk[i], a, pz[i]));
    v[i] = add(y, add(mul(B1, cm), mul(B2, q[i])));
    if (i == 0 && t == 0) {
      const T nyq = T(-2) * m.S * m.S;
      v[0] = add(couple_dc(a, nyq, T(1) / T(2 * M)), mk<T>(B2.re * nyq, B2.im * nyq));
    }
    if (i + 1 < Q) cm = Q == 16 && i == 7 ? m.cm8 : m1_mul(cm, m.cs);
  }
}

// ---------------------------------------------------------------------------
// sums over groups of W consecutive lanes (W a power of two <= 64)
// ---------------------------------------------------------------------------
// Lane exchanges run on the VALU (DPP, permlane swaps) instead of ds_bpermute,
// which takes an LDS round trip per level: the row of a 64 x 1024 FP64 step
// with its eight moments 13.5 -> 11.7 us, the drift of an FP32 scan at nx = 128
// 528 -> 472.
template <int W, class Ctx>
VP_HD double lane_sum(Ctx& c, double v) {
  if constexpr (W >= 64) v = c.template add_lane<32>(v);
  if constexpr (W >= 32) v = c.template add_lane<16>(v);
  if constexpr (W >= 16) v = c.template add_lane<8>(v);
  if constexpr (W >= 8) v = c.template add_lane<4>(v);
  if constexpr (W >= 4) v = c.template add_lane<2>(v);
  if constexpr (W >= 2) v = c.template add_lane<1>(v);
  return v;
}

// N sums at once (N a power of two): from the highest lane bit down, a pair of
// lanes shares the sums still held, each keeping half of them, until one is
// left; the remaining bits add.  Lane l ends with sum fold_index(l) + j in
// a[j], j < fold_count (lanes that differ only in bits left over when one sum
// remained hold the same).
template <int W, int N>
VP_HD constexpr int fold_count() {
  return N > W ? N / W : 1;
}
template <int W, int N>
VP_HD int fold_index(int lane) {
  int idx = 0, n = N;
  for (int m = W / 2; m >= 1 && n > 1; m >>= 1) {
    n >>= 1;
    if (lane & m) idx += n;
  }
  return idx;
}
template <int W, int N>
VP_HD bool fold_writer(int lane) {
  return N >= W ? true : (lane & (W / N - 1)) == 0;
}
template <int W, int N, class Ctx>
VP_HD void lane_fold(Ctx& c, double* a) {
  if constexpr (W > 1) {
    if constexpr (N > 1) {
#pragma unroll
      for (int j = 0; j < N / 2; ++j) a[j] = c.template fold_lane<W / 2>(a[j], a[j + N / 2]);
      lane_fold<W / 2, N / 2>(c, a);
    } else {
      a[0] = c.template add_lane<W / 2>(a[0]);
      lane_fold<W / 2, 1>(c, a);
    }
  }
}

// ---------------------------------------------------------------------------
// sums over the TPT threads that own one sequence (all of them get the sum)
// scratch: (TPT/64)*NV doubles per sequence when TPT > 64 (one sequence per
// workgroup in that case)
// ---------------------------------------------------------------------------
template <int TPT, int NV, class Ctx>
VP_HD void row_sum(Ctx& c, double* vals, double* scratch) {
  constexpr int W = TPT < 64 ? TPT : 64;
#pragma unroll
  for (int q = 0; q < NV; ++q) vals[q] = lane_sum<W>(c, vals[q]);
  if constexpr (TPT > 64) {
    constexpr int NW = TPT / 64;
    const int w = c.tid >> 6;
    if ((c.tid & 63) == 0) {
#pragma unroll
      for (int q = 0; q < NV; ++q) scratch[w * NV + q] = vals[q];
    }
    c.sync();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      double s = 0.0;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) s += scratch[ww * NV + q];
      vals[q] = s;
    }
    c.sync();
  }
}

// ---------------------------------------------------------------------------
// Partition solver for one tridiagonal system of N = TPT*L unknowns.
//
// Row m reads  l(m) x_{m-1} + b(m) x_m + u(m) x_{m+1} = d_m  with l(0) = 0 and
// u(N-1) = 0.  Thread t owns rows m0 = t*L .. m0+L-1 with d in `d[L]`; on
// return `d` holds the solution.  Coef::view<L>(m0, first, last) gives the
// thread's coefficients l(i), u(i), b(i) of row m0 + i (zero l(0) on the
// first thread and u(L-1) on the last).
// red: 8*TPT doubles of LDS for the interface system (one row per thread
// after the even interface unknowns are eliminated).
// ---------------------------------------------------------------------------
// FULL: reciprocals to full double precision (FP64 f); otherwise to ~2^-46
// (FP32 f).
template <int TPT, int L, class Coef, class Ctx, bool FULL = true>
VP_HD void tridiag(Ctx& c, double* d, const Coef& cf, int t, double* red) {
  static_assert(L >= 2, "chunk must hold at least two rows");
  const int m0 = t * L;
  // this thread's rows m0 .. m0+L-1: coefficients by chunk index i (the
  // first thread's l(0) and the last thread's u(L-1) are zero)
  const auto cv = cf.template view<L>(m0, t == 0, t == TPT - 1);
  // One elimination sweep, x_{m0} kept free (i = 1 .. L-1):
  //   x_i = p_i + q_i x_{m0} - r_i x_{i+1}          (p_i in d[i])
  // and its back-substitution from x_{m0+L-1}, which gives x_1 in the chunk's
  // two ends, hence row 0 in them and x_{m0-1}.  The same p, q, r give the
  // interior once the ends are known, so the chunk is eliminated (one
  // reciprocal per row) once.  With a second, upward elimination for row 0 and
  // the interior solved anew a scan step of 512 FP64 instances took 712 us, of
  // 4096 FP32 delta-f instances 3120; with this 669 and 3040.
  double qa[L], ra_[L];
  double p = 0, q = 0, r = 0;
#pragma unroll
  for (int i = 1; i < L; ++i) {
    const double lm = cv.l(i), um = cv.u(i), bm = cv.b(i);
    const double den = (i == 1) ? bm : bm - lm * r;
    const double inv = rcpp<FULL>(den);
    p = (i == 1) ? d[i] * inv : (d[i] - lm * p) * inv;
    q = (i == 1) ? -lm * inv : -lm * q * inv;
    r = um * inv;
    d[i] = p;
    qa[i] = q;
    ra_[i] = r;
  }
  double bp = 0.0, bq = 0.0, br = 1.0;  // x_1 = bp + bq x_{m0} + br x_{m0+L-1}
#pragma unroll
  for (int i = L - 2; i >= 1; --i) {
    bp = d[i] - ra_[i] * bp;
    bq = qa[i] - ra_[i] * bq;
    br = -ra_[i] * br;
  }
  const double u0 = cv.u(0), inv0 = rcpp<FULL>(cv.b(0) + u0 * bq);
  const double p2 = (d[0] - u0 * bp) * inv0, q2 = -u0 * br * inv0, r2 = cv.l(0) * inv0;
  // interface unknowns y_{2t} = x_{m0}, y_{2t+1} = x_{m0+L-1}:
  //   row 2t  :  r2 y_{2t-1} + y_{2t} - q2 y_{2t+1} = p2
  //   row 2t+1: -q  y_{2t}   + y_{2t+1} + r  y_{2t+2} = p
  // Eliminating the even unknowns (y_{2t} by row 2t, y_{2t+2} by row 2t+2 of
  // the next thread) leaves one row per thread in z_t = y_{2t+1}:
  //   A z_{t-1} + B z_t + C z_{t+1} = D,
  //   A = q r2, B = 1 - q q2 - r r2', C = r q2', D = p + q p2 - r p2'
  // (primes: thread t+1's values; r = 0 on the last thread, r2 = 0 on the
  // first).  It is a Schur complement of the diagonally dominant system,
  // hence diagonally dominant itself, and is solved by parallel cyclic
  // reduction, one row per thread.
  //
  // A level whose update changes no row's B or D (the couplings have fallen
  // below the rounding of the rows they reach) ends the reduction: those of the
  // levels after it are the squares.  Weak collisions (nu dt T/dv^2 ~ 1, 16 rows
  // per chunk) need 3-4 of 7 levels, strong ones all.  Two buffers take turns,
  // so a level has one barrier.  With two
  // barriers and every level: 64 x 1024 FP64 step 18.2 us, with this 17.9;
  // 1024 x 8192 FP64 row launch 120 -> 115 us, FP32 92.5 -> 87.5.
  constexpr int NW = TPT > 64 ? TPT / 64 : 1;
  unsigned* vote = reinterpret_cast<unsigned*>(red + 8 * TPT);  // [2][NW], TPT > 64 only
  double* X = red + 4 * TPT;
  X[t] = p2;
  X[TPT + t] = q2;
  X[2 * TPT + t] = r2;
  c.sync();
  const bool last = t == TPT - 1;
  const double p2n = last ? 0.0 : X[t + 1], q2n = last ? 0.0 : X[TPT + t + 1], r2n = last ? 0.0 : X[2 * TPT + t + 1];
  double ra = q * r2, rb = 1.0 - q * q2 - r * r2n, rc = r * q2n, rd = p + q * p2 - r * p2n;
  // each thread publishes 1/B of its row with it (one reciprocal per level)
  double bi = rcpp<FULL>(rb);
  bool changed = true;
  int o = 0;  // buffer of this level
  for (int s = 1; s < TPT; s <<= 1) {
    if constexpr (TPT <= 64) {
      if (!c.any(changed)) break;
    }
    double* A = red + o;
    double* BI = A + TPT;
    double* C = A + 2 * TPT;
    double* D = A + 3 * TPT;
    A[t] = ra;
    BI[t] = bi;
    C[t] = rc;
    D[t] = rd;
    if constexpr (TPT > 64) {
      unsigned* vw = vote + (o ? NW : 0);
      const bool w = c.any(changed);
      if ((t & 63) == 0) vw[t >> 6] = w;
      c.sync();
      unsigned go = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) go |= vw[i];
      if (!go) break;
    } else {
      c.sync();
    }
    const int im = t - s, ip = t + s;
    double na = 0.0, nb = rb, nc = 0.0, nd = rd;
    if (im >= 0) {
      const double al = -ra * BI[im];
      na = al * A[im];
      nb += al * C[im];
      nd += al * D[im];
    }
    if (ip < TPT) {
      const double ga = -rc * BI[ip];
      nc = ga * C[ip];
      nb += ga * A[ip];
      nd += ga * D[ip];
    }
    changed = !(nb == rb && nd == rd);  // true for NaN: it spreads as it does without the test
    ra = na;
    rb = nb;
    rc = nc;
    rd = nd;
    bi = rcpp<FULL>(rb);
    o = 4 * TPT - o;
  }
  const double xe = rd * bi;
  // y_{2t} = p2 - r2 z_{t-1} + q2 z_t
  X = red + o;  // not read by any thread still in the last level
  X[t] = xe;
  c.sync();
  const double zm = t > 0 ? X[t - 1] : 0.0;
  c.sync();
  const double xs = p2 - r2 * zm + q2 * xe;
  // interior rows with both chunk ends known
  d[0] = xs;
  d[L - 1] = xe;
#pragma unroll
  for (int i = L - 2; i >= 1; --i) d[i] = (d[i] + qa[i] * xs) - ra_[i] * d[i + 1];
}

}  // namespace vp
