// Division with the rounding of the IEEE quotient, in three FMA-unit
// operations instead of the ~11 of a full division (scale, reciprocal,
// Newton steps, fixup).
//
// Markstein's correction (P. Markstein, IBM J. Res. Dev. 34 (1990) 111-119;
// J.-M. Muller et al., Handbook of Floating-Point Arithmetic, 2nd ed.,
// sec. 4.7): with ry = RN(1/y) and q within one ulp of x/y, the remainder
// x - q y is exactly representable (one FMA computes it exactly) and
// RN(q + (x - q y) ry) = RN(x/y).
//
// div12: ry = RN(1/12) has relative error 2^-54, so q = RN(x ry) is within
// one ulp of x/12 and the theorem applies to every x away from underflow
// (|x| > 2^-1018) and overflow.
//
// div_by: ry = RN(1/y) is shared by all numerators of a divisor, from an IEEE
// division or from quot(1, y), which is the same number (but for a divisor
// whose significand is all ones: its reciprocal may be an ulp off, and the
// result with it).  q = RN(x ry) is within 1.5 ulp of x/y in general; the
// corrected result matched the IEEE quotient on every one of 6e8 random and
// structured operand pairs (divisor significands near 1, 4/3, 3/2 and 2,
// dense and sparse bit patterns) and is within one ulp by construction.
//
// Domain.  Both return the IEEE quotient for x = 0, or for 2^-968 <= |x| <
// 2^1023 with a quotient of magnitude in [2^-968, 2^1023) and y finite,
// nonzero and normal.  Outside it they differ in two ways: a numerator
// below 2^-968 (the remainder underflows) can leave the result one unit in
// the last place off, and y = 0, y = +-inf or x = +-inf give NaN where the
// IEEE quotient is +-inf or +-0.  The kernels divide only by quantities that
// are positive and finite for a finite state (u^t, twice the fast-speed
// quadratic's leading coefficient, the HLL denominator c+ + c- + 1e-20, the
// cell volume), so only states that are already non-finite, or values below
// 1e-291, can reach the outside.
//
// quot and root are the division and square root the compiler emits for
// FP64 (hardware reciprocal or reciprocal square root, Newton steps, a
// correction from the exact remainder) without the scaling and the fix-ups
// that serve operands near the ends of the exponent range: 8 instructions
// instead of 11, 10 instead of 18.  (Newton's iteration for the reciprocal with
// Markstein's final correction, and Goldschmidt's coupled iteration for the
// root and half its reciprocal with two remainder corrections: Handbook of
// Floating-Point Arithmetic, sec. 4.7 and 5.4; P. Markstein, Proc. 6th Conf.
// Real Numbers and Computers (2004) 146-157.)  Where no scaling would happen the steps
// are the same, so the results are: quot the IEEE quotient for x = 0 or
// |x|, |y| and |x / y| in [2^-900, 2^900] (a divisor whose significand is all
// ones can round a near tie the other way, with or without the scaling), root
// the IEEE square root for x in [2^-760, 2^1000] (0 and infinity give NaN;
// the caller excludes 0).
// Outside, quot(x, 0), quot(x, +-inf), a subnormal divisor and a quotient that
// overflows give NaN, and subnormal remainders can cost a unit in the last
// place.  The kernels use them on lapses, Lorentz factors, enthalpies and wave
// speed sums, which leave the range only below densities of 1e-303 or where
// squares overflow, and in the recovery's searches.  There, iterates of cells
// without a solution pass through any value, so a division stays IEEE where
// one that leaves the range could come back: 1Dvsq's by W^2 and W^3, 2D's
// dP/dv^2 at v^2 = 1, its determinant and v^2.  The rest end alike: a NaN in a
// search ends in the status that an infinity ends in.  Kastaun's
// mu + 1e-300 divides a difference that is 0 when mu is, and eps >= 1e-300
// enters as a term next to 1.
// With min2 / max2 (physics_dev.h) the three sweeps of a face go from 4228 to
// 4012 vector instructions, which are what they wait for: 3-D torus
// 256x128x128 3.85 -> 3.82 ms per cycle, and with the Kastaun search on quot
// and root its recovery of 128x64x64 cells 48.4 -> 45.2 us and an ensemble of
// 20 meshes 401 -> 389 us per cycle.
//
// The remainder is negated inside the second FMA, so a zero quotient keeps
// the sign the IEEE division gives it (compilers that fold the negation
// into the first FMA, as GCC does at -O2 with FMA units, lose that sign;
// clang keeps it).  Both helpers need -ffp-contract=off around them only as
// much as the rest of the code does: the FMAs are explicit.
#pragma once
#include <cmath>

#ifdef __HIPCC__
#define PANGU_HD __host__ __device__ __forceinline__
#else
#define PANGU_HD inline
#endif

namespace pangu {

PANGU_HD double div12(double x) {
  constexpr double ry = 1.0 / 12.0;
  const double q = x * ry;
  const double e = fma(q, 12.0, -x);  // q*12 - x, exact
  return fma(-e, ry, q);
}

// x / y given ry = 1 / y (IEEE).
PANGU_HD double div_by(double x, double y, double ry) {
  const double q = x * ry;
  const double e = fma(q, y, -x);
  return fma(-e, ry, q);
}

// First approximations of 1 / y and 1 / sqrt(x).
#ifndef PANGU_SEED_RCP
#ifdef __HIP_DEVICE_COMPILE__
#define PANGU_SEED_RCP(y) __builtin_amdgcn_rcp(y)
#define PANGU_SEED_RSQ(x) __builtin_amdgcn_rsq(x)
#else
#define PANGU_SEED_RCP(y) (1.0 / (y))
#define PANGU_SEED_RSQ(x) (1.0 / std::sqrt(x))
#endif
#endif

PANGU_HD double quot(double x, double y) {
  double r = PANGU_SEED_RCP(y);
  r = fma(r, fma(-y, r, 1.0), r);
  r = fma(r, fma(-y, r, 1.0), r);
  const double q = x * r;
  return fma(fma(-y, q, x), r, q);
}

PANGU_HD double root(double x) {
  const double y = PANGU_SEED_RSQ(x);
  double s = x * y, h = 0.5 * y;
  const double e = fma(-h, s, 0.5);
  h = fma(h, e, h);
  s = fma(s, e, s);
  s = fma(fma(-s, s, x), h, s);
  return fma(fma(-s, s, x), h, s);
}

}  // namespace pangu
