// FP64 logarithm, reciprocal, reciprocal square root, sine and cosine for the
// pair kernels, written for the vector ALU.  The pair kernels are bound by the
// instructions they issue, and the FP64 multiply-add issues no slower than a
// 32-bit move, so what counts is the number of vector instructions of any kind.
//
// fma_k(a, b, k) = a b + k with a constant k.  For p = p z + k the compiler
// takes v_fmac_f64, whose addend is its destination, and so first copies the
// constant into vector registers, two moves a term; v_fma_f64 with k in scalar
// registers needs none (constants and table entries are loaded there by the
// scalar unit).  k must be the same for all lanes.
//
// fast_hlog: log(x) / 2.  x = 2^e m with m in [sqrt(1/2), sqrt(2)) by integer
//   arithmetic on the high word, log(m) / 2 = atanh(s), s = (m - 1) / (m + 1),
//   |s| <= 0.1716, as s + s^3 p(s^2), p of degree 6 the Chebyshev interpolant
//   (relative error 4e-18, computed with mpmath); e ln(2) / 2 is added with
//   ln(2) / 2 split into a head exact in its product with e and a tail.  s is the
//   product with the hardware's reciprocal and two residual corrections.
//   Relative error a few units in the last place; x must be positive and
//   normal (the pair kernels pass |z|^2 of pairs not excluded by the threshold).
// fast_rcp: 1/x from the hardware approximation and one step of third order,
//   fast_rsqrt: 1/sqrt(x) likewise; both within one unit in the last place for
//   normal x (fast_rsqrt takes subnormal x too).
// fast_sincos: x - n pi/2 by two multiply-adds with pi/2 in two parts (the first
//   product is exact in the multiply-add), then Chebyshev interpolants of
//   degree 5 of (sin r - r) / r^3 and (cos r - 1 + r^2/2) / r^4 in r^2 on
//   |r| <= pi/4 (2e-17, 1e-18; mpmath).  |x| < 2^50; the library beyond, out of line.
// The constants come from gen_fastmath.py.
//
// Against the forms before (degree-9 Taylor series, two Newton steps, the
// library's sincos and square root, constants through moves; and the Helmholtz
// pair in complex arithmetic throughout): 1e10 Laplace pairs with gradient 21.2
// -> 15.2 ms, 4e8 Helmholtz pairs of charges and dipoles with gradient 7.3 ->
// 3.3 ms.  Evaluating four Laplace pairs together without branches between them
// changed nothing: the issue slots are full.
#pragma once
#include "common.h"

namespace fmm2d {

FMM2D_HD double fma_k(double a, double b, double k) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(k));
  return r;
#else
  return fma(a, b, k);
#endif
}

FMM2D_HD double fast_rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(x);
#else
  const double r = 1.0 / x;
#endif
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

FMM2D_HD double fast_rsqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
#else
  const double y = 1.0 / sqrt(x);
#endif
  // 1/sqrt(1 - e) = 1 + e/2 + 3 e^2/8 + ...
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma_k(0.375, e, 0.5), y);
}

FMM2D_HD double fast_hlog(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  // -e = ceil((sqrt(1/2) - x) / 2^20) on the high words; ldexp keeps a NaN
  const int e = (0x3fe6a09f + 0xfffff - __double2hiint(x)) >> 20;
  const double m = __builtin_amdgcn_ldexp(x, e);
  const double t = m - 1.0;  // exact
  const double d = m + 1.0;
  const double r = __builtin_amdgcn_rcp(d);
  double s = t * r;
  s = fma(fma(-s, d, t), r, s);
  s = fma(fma(-s, d, t), r, s);
#else
  int e;
  double m = frexp(x, &e);  // x = m 2^e, m in [0.5, 1)
  e = -e;
  if (m < 0.70710678118654752440) {
    m = 2.0 * m;
    e += 1;
  }
  const double s = (m - 1.0) / (m + 1.0);
#endif
  const double z = s * s;
  double p = fma_k(z, 0.073083605831438, 0.07665849817321138);
  p = fma_k(p, z, 0.09091444893078995);
  p = fma_k(p, z, 0.11111105562861631);
  p = fma_k(p, z, 0.14285714313015532);
  p = fma_k(p, z, 0.1999999999994969);
  p = fma_k(p, z, 0.3333333333333335);
  const double lm = fma(s * z, p, s);
  const double de = (double)e;
  return fma(de, -0.3465735900681466, fma(de, -2.118260682904642e-10, lm));
}

static __host__ __device__ __noinline__ void sincos_large(double x, double* sn, double* cs) {
  sincos(x, sn, cs);
}

FMM2D_HD void fast_sincos(double x, double* sn, double* cs) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr double kMagic = 6755399441055744.0;  // 1.5 2^52: the sum's low word holds n
  const double tn = fma_k(x, 0.6366197723675814, kMagic);
  const double n = tn - kMagic;
  double r = fma(-n, 1.5707963267948966, x);
  r = fma(-n, 6.123233995736766e-17, r);
  const double z = r * r;
  double ps = fma_k(z, 1.591810123167728e-10, -2.5051131455447428e-08);
  ps = fma_k(ps, z, 2.755731610068312e-06);
  ps = fma_k(ps, z, -0.0001984126983675497);
  ps = fma_k(ps, z, 0.008333333333330946);
  ps = fma_k(ps, z, -0.16666666666666666);
  double pc = fma_k(z, -1.1382614869434128e-11, 2.087614602470193e-09);
  pc = fma_k(pc, z, -2.7557317270560385e-07);
  pc = fma_k(pc, z, 2.4801587298763433e-05);
  pc = fma_k(pc, z, -0.0013888888888887395);
  pc = fma_k(pc, z, 0.041666666666666664);
  const double s = fma(r * z, ps, r);
  const double c = fma(z * z, pc, fma(-0.5, z, 1.0));
  const unsigned q = (unsigned)__double2loint(tn);
  const double a = (q & 1u) ? c : s, b = (q & 1u) ? s : c;
  *sn = __hiloint2double(__double2hiint(a) ^ (int)((q << 30) & 0x80000000u), __double2loint(a));
  *cs = __hiloint2double(__double2hiint(b) ^ (int)(((q + 1u) << 30) & 0x80000000u),
                         __double2loint(b));
  if (!(fabs(x) < 1125899906842624.0)) sincos_large(x, sn, cs);
#else
  sincos(x, sn, cs);
#endif
}

}  // namespace fmm2d
