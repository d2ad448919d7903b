// The 15-significant-digit round trip of an eikonal table value: written with
// std::setprecision(15) and read back with std::stod (IArray1D::WriteArray / ReadArray,
// src/MEikonal.cc:404-485).
#pragma once

#include <cmath>
#include <cstdio>
#include <cstdlib>

#ifdef __HIPCC__
#define GRA_HD __host__ __device__
#else
#define GRA_HD
#endif

namespace gra_hip {

inline double round15_text(double v) {
  char buf[64];
  snprintf(buf, sizeof(buf), "%.15g", v);
  return std::strtod(buf, nullptr);
}

// The same value by arithmetic for 1e-7 <= |v| < 1e15. With k chosen so that v 10^k has 15
// digits before the point, 10^k is an exact double (k <= 22), and p + e = |v| 10^k holds
// exactly with e = fma(|v|, 10^k, -p). p is a multiple of its ulp, which divides 1/2, and
// |e| <= ulp / 2, so the nearest integer n to p + e (ties to even, as printf rounds) is
// decided exactly; n / 10^k, a quotient of two exact doubles, is the double nearest to the
// decimal number, which is what strtod returns. k stays within [0, 22] for these v, so
// device code needs no text path: the table kernel rounds its rows itself. 60006 values
// of two tables: 13 ms through text on the host, 1.0 ms by arithmetic there; a set-up took
// 2.27 ms with that and takes 1.32 with the kernel rounding.
GRA_HD inline bool round15_exact(double v) {
  const double a = fabs(v);
  return a >= 1e-7 && a < 1e15;
}
// round15 of a v with round15_exact(v)
GRA_HD inline double round15_arith(double v) {
  constexpr double p10[23] = {1e0,  1e1,  1e2,  1e3,  1e4,  1e5,  1e6,  1e7,
                              1e8,  1e9,  1e10, 1e11, 1e12, 1e13, 1e14, 1e15,
                              1e16, 1e17, 1e18, 1e19, 1e20, 1e21, 1e22};
  const double a = fabs(v);
  int b;
  (void)frexp(a, &b);
  // 10^(14 - k) <= a up to one step, which the loop takes
  int k = 14 - (int)floor((b - 1) * 0.30102999566398120);
  double p, e;
  for (;;) {
    p = a * p10[k];
    e = fma(a, p10[k], -p);
    if (p < 1e14 || (p == 1e14 && e < 0.0)) ++k;
    else if (p > 1e15 || (p == 1e15 && e >= 0.0)) --k;
    else break;
  }
  double n = floor(p);
  const double t = (p - n) - 0.5;
  if (t > 0.0 || (t == 0.0 && (e > 0.0 || (e == 0.0 && fmod(n, 2.0) != 0.0)))) n += 1.0;
  return copysign(n / p10[k], v);
}
inline double round15(double v) { return round15_exact(v) ? round15_arith(v) : round15_text(v); }

}  // namespace gra_hip
