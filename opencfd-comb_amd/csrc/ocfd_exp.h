// ocfd_exp.h -- the exponential of the chemistry and transport kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

// exp(x) = 2^e T[j] (1 + p(f)), x = (64 e + j) ln2/64 + f, |f| <= ln2/128: a
// table of 2^(j/64) in LDS (head and tail) and the Taylor polynomial of
// e^f - 1 to degree 5 (remainder below 2^-54).  About 17 vector instructions;
// the library's exp takes 60 to 70 here, half of them moves of its
// polynomial's constants.  Largest error on |x| <= 700 (4e6 points against
// 80-bit exp): 0.82 ulp.  (The scheme is P. T. P. Tang's table-driven
// exponential, ACM TOMS 15, 1989, with the Taylor polynomial.)  Beyond the
// range of a double the result is 0 or infinite up to |x| = 2e7, where k still
// is a 32-bit number; an infinite x gives NaN, so callers keep x finite.
constexpr int CH_EXPN = 64;
// w exp(x), scaled last: finite where the product is, though exp(x) by itself
// may overflow or w be subnormal; otherwise the same bits as w * exp(x)
__device__ __forceinline__ double chem_exp_times(const double2* tab, double w, double x) {
  const double n = __builtin_rint(x * 92.332482616893656877);  // 64 / ln 2
  // ln2 / 64 as a 32-bit head (its products with n are exact) and a tail
  double f = __builtin_fma(-n, 0x1.62e42fefp-7, x);
  f = __builtin_fma(-n, 0x1.473de6af278edp-40, f);
  const int k = (int)n;
  const double2 t = tab[k & (CH_EXPN - 1)];
  double p = __builtin_fma(f, 1.0 / 120.0, 1.0 / 24.0);
  p = __builtin_fma(f, p, 1.0 / 6.0);
  p = __builtin_fma(f, p, 0.5);
  p = __builtin_fma(f * f, p, f);
  return __builtin_amdgcn_ldexp(w * (t.x + __builtin_fma(t.x, p, t.y)), k >> 6);
}
__device__ __forceinline__ double chem_exp(const double2* tab, double x) { return chem_exp_times(tab, 1.0, x); }

// 2^(j/64) and its rounding
inline void chem_exp_table(double (*t)[2]) {
  for (int j = 0; j < CH_EXPN; j++) {
    const long double v = std::exp2((long double)j / CH_EXPN);
    t[j][0] = (double)v;
    t[j][1] = (double)(v - (long double)t[j][0]);
  }
}
