// gmc_arith.hpp -- divisions and square roots in fewer instructions than the
// compiler's sequences.  Everything but the hardware's estimates is host code
// as well: tests/test_div_rn.py runs it on the CPU.
#pragma once

#include <hip/hip_runtime.h>

namespace gmc {

// a / d from y = 1 / d correctly rounded: q0 = a y, the exact remainder e =
// a - d q0 (one fma), q = q0 + e y rounded once (Markstein's correction step,
// P. W. Markstein, IBM J. Res. Dev. 34 (1990) 111-119).  The value of the IEEE
// quotient for finite a and d with |a| >= 2^-969 or a = 0 (-0 may give +0) and
// y and a / d normal; the remainder of a smaller a is not exact, and the
// quotient then within a unit of it.
// Three FP64 operations instead of the scale / reciprocal / Newton / fixup
// sequence of a division, for denominators shared by a wavefront (metric terms
// of one row) or by several numerators.
__host__ __device__ __forceinline__ double div_rn(double a, double d, double y) {
  const double q0 = a * y;
  return __builtin_fma(__builtin_fma(-q0, d, a), y, q0);
}

// a / d for a, d and a / d well inside the normal range, from an estimate y of
// 1 / d that is within 2^-22 of it: two Newton steps leave y correctly rounded
// or the number next to that, which the correction step of div_rn then takes
// to the IEEE quotient (sampled by the test; the compiler's division has the
// same steps between its scaling and its fixup).
__host__ __device__ __forceinline__ double div_from(double a, double d, double y) {
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  return div_rn(a, d, y);
}
// ... from the hardware's estimate (2^29 units), and the fixup of zero, infinite
// and NaN operands (vanishing or overflowing depths and winds): 9 instructions.
// The compiler's division adds the scaling, which leaves such operands as they
// are, 11.
__device__ __forceinline__ double div_mid(double a, double d) {
  return __builtin_amdgcn_div_fixup(div_from(a, d, __builtin_amdgcn_rcp(d)), d, a);
}

// sqrt(x) correctly rounded for x = 0 and finite x >= 1e-290, from an estimate
// y of 1 / sqrt(max(x, 1e-290)) within 2^-22: the coupled Newton iteration of
// (sqrt, 1 / 2 sqrt) with two corrections of the root.  Smaller x gives a root
// below 1e-140, of no account where it is added to kEps.
__host__ __device__ __forceinline__ double sqrt_from(double x, double y) {
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
// a / (sqrt(x) + eps) of 0 <= a <= sqrt(x), eps^2 far above 1e-290: without the
// compiler's scaling of subnormal operands, and with one fixup for root and
// quotient, in which x stands for its root (an infinite x gives 0 or, with an
// infinite a, NaN; an a below 2^-1075 x gives 0)
__device__ __forceinline__ double div_root(double a, double x, double eps) {
  const double xm = __builtin_fmax(x, 1e-290), d = sqrt_from(x, __builtin_amdgcn_rsq(xm)) + eps;
  return __builtin_amdgcn_div_fixup(div_from(a, d, __builtin_amdgcn_rcp(d)), xm, a);
}

}  // namespace gmc
