// Shorter division and square root sequences for the nonlinear momentum
// terms, equal to the IEEE operations wherever their results can matter.
//
// The IEEE single-precision division on gfx950 is eleven VALU operations:
// two operand scalings (V_DIV_SCALE), a reciprocal with one Newton step,
// the quotient with two residual corrections (the last one V_DIV_FMAS) and
// a special-case fix-up (V_DIV_FIXUP).  The momentum kernels spend about a
// fifth of their instructions on fourteen divisions per cell.
//
// div_inrange(a, b) is that sequence without the scalings, the fix-up and
// the first residual correction.  The refined reciprocal is 1/b correctly
// rounded for every divisor in range (gcomcot_reciprocal_check_ tries them all
// on the device), and then one correction q + (a - b q)/b rounds to the IEEE
// quotient: before that rounding it is within 2.3 * 2^-24 ulp of a/b, which
// leaves per divisor only the numerators whose quotient comes that close to a
// midpoint; they are all enumerated in tests/quotient_check.cpp, and none
// rounds wrongly.  V_DIV_SCALE leaves both operands unchanged, and V_DIV_FIXUP
// passes the quotient through, unless b is 0, denormal or so large that
// 1/b is, a is 0 or below 2^-103 in magnitude, a/b is below 2^-126 or the
// exponents differ by 96 or more; for the other (a, b) the result is the
// IEEE quotient bit for bit (div_inrange_applies states the range that the
// device self-check, gcomcot_division_check_, covers).
// At the call sites below the divisor is a total depth (>= 1e-5 where the
// result is used), a friction power of one (>= 1e-7) or 1 + FF (>= 1), so
// only a numerator below 2^-103 leaves that range.  The quotient is then
// below 2^-86, and every path from it ends in the flux, which is set to 0
// when below EPS = 1e-10 (moment.f90:565, 759, 1054, 1247): a change
// of that size cannot move a sum that survives the test, since it is far
// below half an ulp of 1e-10.  A zero numerator gives +0 for -0/b (IEEE:
// -0), which the same test turns into the same +0.
//
// div12(x) is x / 12 as RN(1/12) times x with one residual correction.
// Checked against IEEE division for every float (tests/test_fastdiv.py):
// equal for all |x| >= 2^-124 and for zeros; the only differences are
// denormal quotients.  Its argument at the call sites is a positive
// coefficient times a depth of at least 1e-5.
#pragma once

#if defined(__HIPCC__) || defined(__HIP__)
#define GC_FD_HD __host__ __device__ __forceinline__
#else
#define GC_FD_HD static inline
#include <math.h>
#endif

namespace gc {

// RN(1/12)
constexpr float kRcp12 = 1.0f / 12.0f;

GC_FD_HD float div12(float x) {
  const float q = x * kRcp12;
  const float r = fmaf(-12.0f, q, x);
  const float d = fmaf(r, kRcp12, q);
  return x == 0.0f ? q : d;  // q keeps the sign of a zero x
}

// The operands div_inrange is claimed for (with q = a / b): both normal,
// |b| within 2^+-kDivRange, |a| >= 2^-103, an exponent gap below 96 and a
// normal quotient.  The call sites stay far inside it.
constexpr int kDivRange = 120;
GC_FD_HD bool div_inrange_applies(float a, float b, float q) {
  const float lo = 0x1p-120f, hi = 0x1p120f;
  return fabsf(b) >= lo && fabsf(b) <= hi && fabsf(a) >= 0x1p-103f && fabsf(a) <= 0x1p127f &&
         fabsf(q) >= 0x1p-126f && fabsf(q) <= 0x1p95f;
}

// Whether Manning friction leaves a flux as it is: FF = KF sqrt(P^2 + Q^2) /
// DF^2.3333333 enters as X - FF P and as X / (1 + FF), and both are X where
// |FF P| <= 2^-26 |X| (a quarter of an ulp at most, also just above a power of
// two) and FF <= 2^-26.  sqrt(P^2 + Q^2) <= |P| + |Q|, and the power is at
// least DF^2 from a depth of 1 on and 8 DF^2 (short by 1e-7) from 512 on;
// kf26 = drag_scaled(KF) is 2^26 KF with 1e-3 to spare for every rounding
// here and there.  Where a product underflows so does FF P.  The exact terms
// give NaN where P^2 overflows, and no product here may overflow either: the
// power's bound ends at 2^40 (a depth of 370 km) and kf26 starts at 2^-23, so
// b <= w leaves fluxes of at most 2^63, and infinite and NaN ones fail.  In
// open water this holds for every flux of a wave (4000 m deep, steps of a
// second or two: up to 1000 m^2/s), which then needs no square root, power or
// quotient of it: 12 operations for 50.
// 4096x3072 spherical 115.5 -> 111.5 us per step (now bound by memory), 1024x768
// 18.3 -> 17.2.  Cartesian layers, metre grids on shallow water, almost never
// pass (1201x901 harbour with the test 18.3 -> 19.5): they go without it.
constexpr float kDragScale = 0x1p26f * 1.001f;
GC_FD_HD float drag_scaled(float kfric) {
  const float k = kDragScale * kfric;
  return k < 0x1p-23f ? 0x1p-23f : k;  // NaN passes
}
GC_FD_HD bool drag_vanishes(float kf26, float p, float q, float df, float x) {
  const float d2 = df * df, w = fminf(df >= 512.0f ? 8.0f * d2 : d2, 0x1p40f);
  const float b = kf26 * (fabsf(p) + fabsf(q));
  return (df >= 1.0f) & (b <= w) & (b * fabsf(p) <= w * fabsf(x));
}

#if defined(__HIPCC__) || defined(__HIP__)
// div_inrange split in two: the refined reciprocal of b (three operations
// that depend on b alone), and the quotient from it (three more).  div_by(a, b,
// recip_refined(b)) is div_inrange(a, b) bit for bit, so quotients with one
// divisor can share the first part.
__device__ __forceinline__ float recip_refined(float b) {
  const float y = __builtin_amdgcn_rcpf(b);
  const float e = fmaf(-b, y, 1.0f);
  return fmaf(e, y, y);
}
__device__ __forceinline__ float div_by(float a, float b, float y) {
  const float q = a * y;
  return fmaf(fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float div_inrange(float a, float b) {
  return div_by(a, b, recip_refined(b));
}

// sqrt(x) as the correctly rounded square root sequence computes it for
// x >= 2^-96: the hardware estimate, then the neighbour one ulp below or
// above where the residual says so.  That sequence first scales smaller x
// by 2^32 (and selects x itself for +-0 and +inf, which the steps below
// already return).  At the call sites x is g*D (D = 0 or >= 1e-5) or
// P^2 + Q^2 of the friction term; there a smaller x only feeds a friction
// numerator below 2^-48 into the quotient argument above.  Equal to IEEE
// sqrt for every float >= 2^-96 and for +-0 and +inf (device self-check
// over all floats, gcomcot_division_check_).
__device__ __forceinline__ float sqrt_inrange(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float sm = __uint_as_float(__float_as_uint(s) - 1u);
  const float rm = fmaf(-sm, s, x);
  const float sp = __uint_as_float(__float_as_uint(s) + 1u);
  const float rp = fmaf(-sp, s, x);
  const float t = rm <= 0.0f ? sm : s;
  return rp > 0.0f ? sp : t;
}

// WAVE_BREAKING's threshold on |Z2 - Z1| is DT * 0.08 * sqrt(g D); this times
// a hardware sqrt(D) is a safe lower bound of it (2^-12 below, against
// rounding errors of 2^-21), and 0 where D is.
__device__ __forceinline__ float breaking_floor(float dt) {
  return 0.08f * 3.1316129f * 0.99975586f * dt;  // 0.08 sqrt(g) (1 - 2^-12) DT
}
#endif

}  // namespace gc
