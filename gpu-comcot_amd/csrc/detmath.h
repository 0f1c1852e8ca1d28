// Deterministic float pow / exp for the nonlinear momentum terms.
//
// COMCOT's nonlinear momentum evaluates Manning friction as
//   FF = 0.5*dt*g * n^2 * sqrt(P^2 + Q^2) / D^(2.3333333)
// (moment.f90:459-460, 945-946, 656-657, 1139-1140, 207-208, 250-251) and the
// breaking damping as EXP(-REF) (moment.f90:1323).  The Fortran calls libm
// powf/expf on the host; a GPU math library gives different last bits.  To
// make the device result reproducible on any host, both functions here are
// computed in IEEE double using only +, -, *, explicit fma (each correctly
// rounded on CPU and GPU alike; FP contraction is disabled around them) and
// bit manipulation, then rounded once to float.  The double result is
// within ~1e-16 (relative) of the exact value, so the float result is the
// correctly rounded one except when the exact value lies that close to a
// float rounding midpoint.
//
// Method (table-driven, as in the usual libm designs), for x = 2^e m with m
// in [1,2), c_k the centre of m's interval and r = m/c_k - 1 computed exactly
// as fma(m, 1/c_k, -1) with 1/c_k rounded to 28 bits:
//   x^y, y = 2.3333333 (the Manning power): 2^(e y) * c_k^y * (1 + r)^y, the
//            first two factors from tables (64 intervals), the third its
//            binomial series to degree 6: one exponentiation without a
//            logarithm, 21 instructions against 42 for exp2(y log2 x), and
//            closer (each factor is within half an ulp, where y log2 x near
//            30 loses five bits);
//   log2 x = e + log2(c_k) + log2(1 + r) (128 intervals, degree 6);
//   2^t    = 2^(k/32) * 2^g,  k = round(32 t), |g| <= 1/64 (degree 6).
// The tables are built by constexpr code from series (atanh for ln, Taylor
// for exp) at compile time, those of the Manning power in double-double
// arithmetic, so host and device hold identical values.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__) || defined(__HIP__)
#define GC_HD __host__ __device__ __forceinline__
#define GC_TABLE __device__ __constant__
#else
#define GC_HD static inline
#define GC_TABLE static
#endif

namespace gcdet {

GC_HD double bits_to_double(uint64_t u) {
  union { uint64_t u; double d; } v; v.u = u; return v.d;
}
GC_HD uint64_t double_to_bits(double d) {
  union { uint64_t u; double d; } v; v.d = d; return v.u;
}

constexpr double kLn2 = 0.69314718055994530942;

// ---- compile-time table construction (plain IEEE double arithmetic)
constexpr double cx_ln(double x) {  // x in [0.5, 2]: 2*atanh((x-1)/(x+1))
  double s = (x - 1.0) / (x + 1.0), s2 = s * s, p = 0.0;
  for (int k = 40; k >= 0; --k) p = p * s2 + 1.0 / (2.0 * k + 1.0);
  return 2.0 * s * p;
}
constexpr double cx_exp(double r) {  // |r| <= 1
  double p = 0.0;
  for (int k = 30; k >= 1; --k) p = 1.0 + p * r / k;
  return p;
}
constexpr double cx_round28(double v) {  // v in (0.5, 1]: keep 28 significant bits
  double s = v * 268435456.0;               // 2^28
  long long q = (long long)(s + 0.5);
  return (double)q / 268435456.0;
}

// ---- double-double for the Manning tables (Dekker/Knuth exact sums and
// products)
struct cx_dd { double hi, lo; };
constexpr cx_dd cx_sum(double a, double b) {
  double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
constexpr cx_dd cx_prod(double a, double b) {
  double p = a * b, ca = 134217729.0 * a, cb = 134217729.0 * b;
  double ah = ca - (ca - a), al = a - ah, bh = cb - (cb - b), bl = b - bh;
  return {p, ((ah * bh - p) + ah * bl + al * bh) + al * bl};
}
constexpr cx_dd cx_add(cx_dd a, cx_dd b) {
  cx_dd s = cx_sum(a.hi, b.hi);
  return cx_sum(s.hi, s.lo + (a.lo + b.lo));
}
constexpr cx_dd cx_mul(cx_dd a, cx_dd b) {
  cx_dd p = cx_prod(a.hi, b.hi);
  return cx_sum(p.hi, p.lo + (a.hi * b.lo + a.lo * b.hi));
}
constexpr cx_dd cx_div(cx_dd a, double b) {
  double q = a.hi / b;
  cx_dd p = cx_prod(q, b);
  double r = ((a.hi - p.hi) - p.lo) + a.lo;
  return cx_sum(q, r / b);
}
constexpr cx_dd cx_lndd(double x) {  // ln of x in [0.5, 1]: 2 atanh((x-1)/(x+1))
  cx_dd n = cx_sum(x, -1.0), d = cx_sum(x, 1.0);
  double q = n.hi / d.hi;
  cx_dd p = cx_mul({q, 0.0}, d);
  double r = ((n.hi - p.hi) - p.lo) + n.lo;
  cx_dd s = cx_sum(q, r / d.hi), s2 = cx_mul(s, s), v = {0.0, 0.0};
  for (int k = 34; k >= 0; --k) v = cx_add(cx_mul(v, s2), cx_div({1.0, 0.0}, 2.0 * k + 1.0));
  return cx_mul({2.0 * s.hi, 2.0 * s.lo}, v);
}
constexpr double cx_expdd(cx_dd t) {  // e^t, 0 <= t < 2, rounded to double
  cx_dd x = {t.hi / 16.0, t.lo / 16.0}, v = {1.0, 0.0};
  for (int k = 18; k >= 1; --k) v = cx_add({1.0, 0.0}, cx_div(cx_mul(v, x), (double)k));
  for (int k = 0; k < 4; ++k) v = cx_mul(v, v);
  return v.hi;
}

// The Manning exponent, the Fortran's REAL 2.3333333
constexpr float kManningExp = 2.3333333f;
constexpr double kManY = (double)kManningExp;
// Exponents of the Manning table: 2^-17 < 1e-5, the smallest depth a caller
// passes, up to 2^56, whose power (and that of everything above) overflows
// a float.
constexpr int kManE0 = -17, kManE1 = 56, kManE = kManE1 - kManE0 + 1;

struct Tables {
  double mc[2 * 64];    // pairs 1/c_k, c_k^y of m's 64 intervals
  double me[kManE];     // 2^(e y), e = kManE0..kManE1
  double exp2j[32];     // 2^(j/32)
};

constexpr Tables make_tables() {
  Tables t{};
  for (int k = 0; k < 64; ++k) {
    double ic = cx_round28(1.0 / (1.0 + (k + 0.5) / 64.0));
    t.mc[2 * k] = ic;
    t.mc[2 * k + 1] = cx_expdd(cx_mul({-kManY, 0.0}, cx_lndd(ic)));
  }
  for (int e = kManE0; e <= kManE1; ++e) {
    double p = e * kManY;  // exact: 24 + 6 bits
    int n = (int)p;
    if (p < n) --n;        // floor
    double v = cx_expdd(cx_mul({p - n, 0.0}, {0.693147180559945309417, 2.319046813846299558e-17}));
    for (; n > 0; --n) v *= 2.0;
    for (; n < 0; ++n) v *= 0.5;
    t.me[e - kManE0] = v;
  }
  for (int j = 0; j < 32; ++j) t.exp2j[j] = cx_exp(j * (kLn2 / 32.0));
  return t;
}

GC_TABLE constexpr Tables kTab = make_tables();

#if !defined(__HIP_DEVICE_COMPILE__)
// log2 tables of the general power, host only
struct LogTables {
  double invc[128];
  double logc[128];  // log2(1/invc), of the stored invc
};
constexpr LogTables make_log_tables() {
  LogTables t{};
  for (int k = 0; k < 128; ++k) {
    double ic = cx_round28(1.0 / (1.0 + (k + 0.5) / 128.0));
    t.invc[k] = ic;
    t.logc[k] = -cx_ln(ic) / kLn2;
  }
  return t;
}
static constexpr LogTables kLogTab = make_log_tables();
#endif

// (1+r)^y = 1 + r (kB1 + r (kB2 + ...))
constexpr double kB1 = kManY, kB2 = kB1 * (kManY - 1.0) / 2.0, kB3 = kB2 * (kManY - 2.0) / 3.0,
                 kB4 = kB3 * (kManY - 3.0) / 4.0, kB5 = kB4 * (kManY - 4.0) / 5.0,
                 kB6 = kB5 * (kManY - 5.0) / 6.0;

// log2(1+r)/r and 2^g coefficients
constexpr double kL1 = 1.0 / kLn2, kL2 = -1.0 / (2.0 * kLn2), kL3 = 1.0 / (3.0 * kLn2),
                 kL4 = -1.0 / (4.0 * kLn2), kL5 = 1.0 / (5.0 * kLn2),
                 kL6 = -1.0 / (6.0 * kLn2);
constexpr double kE1 = kLn2, kE2 = kLn2 * kLn2 / 2.0, kE3 = kLn2 * kLn2 * kLn2 / 6.0,
                 kE4 = kLn2 * kLn2 * kLn2 * kLn2 / 24.0,
                 kE5 = kLn2 * kLn2 * kLn2 * kLn2 * kLn2 / 120.0,
                 kE6 = kLn2 * kLn2 * kLn2 * kLn2 * kLn2 * kLn2 / 720.0;

GC_HD double dfma(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_fma(a, b, c);
#else
  return __builtin_fma(a, b, c);  // correctly rounded (libm fma if no FMA unit)
#endif
}

// fma(a, b, c) for a constant addend c.  On the device it is one VOP3
// v_fma_f64 that reads c from a scalar register pair; left to itself the
// compiler writes the two-address v_fmac_f64 instead, which needs c copied
// into the accumulator first (an extra vector move per polynomial step) and
// keeps every coefficient in vector registers for the whole kernel.  The
// operation, and so the result, is the same IEEE double fma either way.
GC_HD double dfma_k(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r;
  __asm__("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
  return r;
#else
  return __builtin_fma(a, b, c);
#endif
}

// x * 2^e for a result in the normal range, where it is exact: one
// instruction on the device (the same value as multiplying by the power).
GC_HD double scale2(double x, int e) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ldexp(x, e);
#else
  return x * bits_to_double((uint64_t)(uint32_t)(e + 1023) << 52);
#endif
}

GC_HD float bits_to_float(uint32_t u) {
  union { uint32_t u; float f; } v; v.u = u; return v.f;
}
GC_HD uint32_t float_to_bits(float f) {
  union { uint32_t u; float f; } v; v.f = f; return v.u;
}

// 2^t; only ever rounded to float by the callers, so beyond |t| = 300 the
// result is 0 or +inf there, as libm's expf/powf give (WAVE_BREAKING meets
// t = -inf where the cell is dry: COEF = EXP(-(+inf)) = 0).  NaN passes.
template <class TAB>
GC_HD double exp2_core(double t, const TAB &T) {
  if (t != t) return t;
  if (t < -300.0) return 0.0;
  if (t > 300.0) return bits_to_double(0x7ff0000000000000ULL);
  const double s = t * 32.0;
  const int k = (int)(s + (s >= 0.0 ? 0.5 : -0.5));
  const double g = t - (double)k * (1.0 / 32.0);
  const int j = k & 31;
  const int e2 = k >> 5;  // floor(k / 32)
  double q = dfma(g, kE6, kE5);
  q = dfma_k(g, q, kE4);
  q = dfma_k(g, q, kE3);
  q = dfma_k(g, q, kE2);
  q = dfma_k(g, q, kE1);
  q = dfma(g, q, 1.0);
  return scale2(T.exp2j[j] * q, e2);
}

// x^2.3333333 for the depth terms of Manning friction, whose callers
// guarantee x >= 1e-5 (the momentum routines clamp or test the depth first).
// NaN passes, +inf and every depth whose power overflows give +inf.
template <class TAB>
GC_HD float powf_manning(float x, float, const TAB &T) {
  const uint32_t b = float_to_bits(x);
  const uint32_t ei = (b >> 23) - (uint32_t)(127 + kManE0);
  const uint32_t e = ei < (uint32_t)(kManE - 1) ? ei : (uint32_t)(kManE - 1);
  const uint32_t k = (b >> 17) & 63u;
  const double m = (double)bits_to_float((b & 0x007fffffu) | 0x3f800000u);
  const double r = dfma(m, T.mc[2 * k], -1.0);
  const double t = T.mc[2 * k + 1] * T.me[e];
  double p = dfma(r, kB6, kB5);
  p = dfma_k(r, p, kB4);
  p = dfma_k(r, p, kB3);
  p = dfma_k(r, p, kB2);
  p = dfma_k(r, p, kB1);
  const float v = (float)dfma(t, r * p, t);
  return x != x ? x : v;
}

// e^x
template <class TAB>
GC_HD float expf_det(float x, const TAB &T) {
  return (float)exp2_core((double)x * (1.0 / kLn2), T);
}

#if !defined(__HIP_DEVICE_COMPILE__)
// host entry points on the compile-time tables
// log2 of a positive, finite, normal float (32-bit decomposition)
static inline double log2_pos(float x, const LogTables &T) {
  const uint32_t b = float_to_bits(x);
  const int e = (int)(b >> 23) - 127;
  const int k = (int)((b >> 16) & 127);
  const double m = (double)bits_to_float((b & 0x007fffffu) | 0x3f800000u);
  const double r = dfma(m, T.invc[k], -1.0);
  double p = dfma(r, kL6, kL5);
  p = dfma_k(r, p, kL4);
  p = dfma_k(r, p, kL3);
  p = dfma_k(r, p, kL2);
  p = dfma_k(r, p, kL1);
  return (double)e + (T.logc[k] + r * p);
}

static inline float powf_manning(float x, float y) { return powf_manning(x, y, kTab); }

// x^y for the depths the momentum routines raise to 7/3: x > 0 finite
// (they bound it below by 1e-3 or 1e-5), where y = 2.3333333 takes the
// Manning form.  NaN, zero, negative and infinite x follow C's powf for
// y > 0: NaN, 0, NaN, +inf; subnormal x (whose power underflows for y > 1)
// gives 0.
static inline float powf_det(float x, float y) {
  if (x != x) return x;
  if (!(x > 0.0f)) return x == 0.0f ? 0.0f : (float)bits_to_double(0x7ff8000000000000ULL);
  if (x > 3.0e38f) return (float)bits_to_double(0x7ff0000000000000ULL);
  if (x < 1.17549435e-38f) return 0.0f;
  if (y == kManningExp && x >= 1.0e-5f) return powf_manning(x, y);
  return (float)exp2_core((double)y * log2_pos(x, kLogTab), kTab);
}
static inline float expf_det(float x) { return expf_det(x, kTab); }
#endif

}  // namespace gcdet
