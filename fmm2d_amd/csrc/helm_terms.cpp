// Helmholtz expansion-order rule (h2dterms, helmholtz/h2dterms.f:35-96).
//
// nterms = j + 1 for the first j >= 2 with
//   (|J_j(z2) H_j(z1)| + |J_{j-1}(z2) H_{j-1}(z1)|) |H_0(z1)|
//       < eps (|J_0(z2) H_0(z1)| + |J_1(z2) H_1(z1)|),
// z1 = 1.5 k bs, z2 = k bs sqrt(2)/2, searched up to j = 50000 (else ier 13).
// H_n by upward recurrence from H0, H1 (stable for H); J_n by Miller's
// backward recurrence normalised with the Jacobi-Anger identity at theta = pi,
//   exp(-i z) = J_0(z) + 2 sum_{n>=1} (-i)^n J_n(z),
// (exp(+i z) with (+i)^n below the real axis), which does not cancel for
// complex z.  Long double keeps the unnormalised recurrences in range.
#include <cmath>
#include <complex>
#include <vector>

#include "hankel.h"
#include "helm_ops.h"

namespace fmm2d {

using lc = std::complex<long double>;

namespace {

// |a|, through the square root where the square is in range
inline long double abs_l(lx a) {
  const long double n = norm(a);
  return (n > 1e-4000L && n < 1e4000L) ? std::sqrt(n) : std::hypot(a.re, a.im);
}

}  // namespace

// J_0..J_n(z) for n >= 1
std::vector<lx> bessel_j(lx z, int n) {
  if (abs_l(z) < 1e-200L) {
    std::vector<lx> out(n + 1, lx{0, 0});
    out[0] = lx{1, 0};
    return out;
  }
  const lx zi = to_lx(1.0L / to_lc(z));
  // start index: forward recurrence from n until it has grown by 1e20
  int ntop = n + 1;
  {
    lx f0{0, 0}, f1{1, 0};
    for (int i = n; i < n + 100000; ++i) {
      const lx f2 = (2.0L * i) * zi * f1 - f0;
      f0 = f1;
      f1 = f2;
      if (norm(f2) > 1e40L) {
        ntop = i + 1;
        break;
      }
    }
  }
  std::vector<lx> f(ntop + 1, lx{0, 0});
  f[ntop - 1] = lx{1, 0};
  for (int i = ntop - 1; i >= 1; --i) {
    f[i - 1] = (2.0L * i) * zi * f[i] - f[i + 1];
    if (norm(f[i - 1]) > 1e300L) {  // rescale the tail
      for (int k = i - 1; k <= ntop; ++k) f[k] = 1e-150L * f[k];
    }
  }
  // sum of f_n (+-i)^n, n >= 1
  const bool below = z.im < 0;
  lx psi{0, 0};
  for (int i = 1; i <= ntop; ++i) {
    const lx v = f[i];
    switch (below ? i & 3 : -i & 3) {
      case 0: psi = psi + v; break;
      case 1: psi = psi + lx{-v.im, v.re}; break;
      case 2: psi = psi - v; break;
      default: psi = psi + lx{v.im, -v.re}; break;
    }
  }
  psi = 2.0L * psi + f[0];
  const lc ez = below ? std::exp(lc(0, 1) * to_lc(z)) : std::exp(lc(0, -1) * to_lc(z));
  const lx sc = to_lx(ez / to_lc(psi));
  f.resize(n + 1);
  for (int i = 0; i <= n; ++i) f[i] = f[i] * sc;
  return f;
}

int h2dterms(double bsize, cplx zk, double eps, int* ier) {
  *ier = 0;
  const lx k{zk.re, zk.im};
  const lx z1 = 1.5L * ((long double)bsize * k);
  const lx z2 = (std::sqrt(2.0L) / 2.0L) * ((long double)bsize * k);
  const int ntmax = 50000;
  cplx h0d, h1d;
  hank01(cplx{(double)z1.re, (double)z1.im}, &h0d, &h1d);
  const lx zi = to_lx(1.0L / to_lc(z1));
  // search in growing windows so that small problems stay cheap
  int nwin = std::min(ntmax, std::max(48, (int)abs_l(z1) + 48));
  for (;;) {
    const std::vector<lx> J = bessel_j(z2, nwin);
    lx hm1{h0d.re, h0d.im}, h{h1d.re, h1d.im};
    const long double absh0 = abs_l(hm1);
    long double last = abs_l(J[1] * h);  // |J_j H_j| of the j before
    const long double x0 = abs_l(J[0] * hm1) + last;
    for (int j = 2; j <= nwin; ++j) {
      const lx hn = (2.0L * (j - 1)) * zi * h - hm1;
      hm1 = h;
      h = hn;
      const long double cur = abs_l(J[j]) * abs_l(h);
      const long double x = (cur + last) * absh0;
      if (x < (long double)eps * x0) return j + 1;
      last = cur;
    }
    if (nwin >= ntmax) break;
    nwin = std::min(ntmax, 2 * nwin);
  }
  *ier = 13;
  return 10001;
}

}  // namespace fmm2d
