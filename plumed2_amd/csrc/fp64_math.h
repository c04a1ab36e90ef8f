// FP64 device functions of the inner loops that the library forms are too long
// for: no special cases beyond what the callers need.
#pragma once
#include <hip/hip_runtime.h>

namespace p2a {

#pragma clang fp contract(off)

// exp(x), |x| < 2^20: ln2 reduction and the
// Taylor polynomial of degree 13 on |r| <= ln2/2 (truncation 4e-18) in pairs,
// so that its depth is 6 multiply-adds instead of a dozen in a row.  The 1 is
// added last: within 1.04 ulp (with 1 + r as a partial sum 2.2).  The chain of heights keeps the constants in registers (a 64-bit
// literal costs two moves): ExpK, made opaque there.
struct ExpK {
  double log2e = 1.4426950408889634;
  // ln2 in two parts, the first of 32 bits (its product with n is exact)
  double hi = -0x1.62e42fee00000p-1, lo = -0x1.a39ef35793c76p-33;
  double m[6] = {1.0 / 6, 1.0 / 120, 1.0 / 5040, 1.0 / 362880, 1.0 / 39916800, 1.0 / 6227020800.0};
  double a[5] = {1.0 / 24, 1.0 / 720, 1.0 / 40320, 1.0 / 3628800, 1.0 / 479001600};
};
// exp(x) = 2^n (1 + p): p from x and n = rint(x log2e)
__device__ __forceinline__ double exp_part(double x, double n, const ExpK& C) {
  double r = fma(n, C.hi, x);
  r = fma(n, C.lo, r);
  const double r2 = r * r, r4 = r2 * r2, r8 = r4 * r4;
  const double p23 = fma(r, C.m[0], 0.5);
  const double p45 = fma(r, C.m[1], C.a[0]), p67 = fma(r, C.m[2], C.a[1]);
  const double p89 = fma(r, C.m[3], C.a[2]), pab = fma(r, C.m[4], C.a[3]), pcd = fma(r, C.m[5], C.a[4]);
  const double q0 = fma(r2, p45, p23), q1 = fma(r2, p89, p67), q2 = fma(r2, pcd, pab);
  return fma(r2, fma(r8, q2, fma(r4, q1, q0)), r);
}
__device__ __forceinline__ double exp_core(double x) {
  const ExpK C;
  const double n = rint(x * C.log2e);
  return ldexp(1.0 + exp_part(x, n, C), (int)n);
}

// 1/sqrt(x) for x > 0, to an ulp or two: v_rsq_f64 (2^-23) and two Newton steps
__device__ __forceinline__ double rsqrt64(double x) {
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const double h = 0.5 * y;
    y = fma(h, fma(-x * y, y, 1.0), y);
  }
  return y;
}

#pragma clang fp contract(fast)

}  // namespace p2a
