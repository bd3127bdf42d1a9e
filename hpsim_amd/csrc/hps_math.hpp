// hps_math.hpp -- FP64 elementary functions for the tracking kernels.
//
// The reference kernels use the CUDA device math library (exp, log, sinh,
// cosh, sincos, rsqrt, fmod: simulation_kernel.cu:30,176-177,
// space_charge_kernel.cu:60, beam_kernel.cu:1520).  These functions follow
// published methods instead and are written so that a serial host build of
// the same method gives identical bits:
//   exp    Cody-Waite reduction by ln2 (two-part constant, fma), degree-13
//          Taylor polynomial, exact scaling by two powers of two;
//   log    x = 2^e m, m in [sqrt(1/2), sqrt(2)], 2*atanh((m-1)/(m+1)) series;
//   sincos Cody-Waite reduction by pi/2 (three-part constant, fma), Taylor
//          polynomials (sin to r^17, cos to r^18) on |r| <= pi/4;
//   sinh/cosh  Taylor series for |x| < 1, else (e^|x| -/+ e^-|x|)/2;
//   fmod   exact remainder by subtracting power-of-two multiples of the
//          divisor (each step exact by Sterbenz's lemma).
// Only correctly rounded primitives are used (+ - * /, sqrt, fma, floor);
// the library is compiled with -ffp-contract=off.  The exception is the
// second build of the tracking kernels (hps_push_fast.hip).  It serves
// batches held to error bounds, not to the oracle's bits.  Its maps, kick
// and deposit take psqrt, psincos and psinhcosh as sqrt_rsq (v_rsq_f64 and
// two refinement steps) and shorter Taylor polynomials.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define HPS_HD __host__ __device__ __forceinline__

namespace hps {

constexpr double kLn2Hi = 0x1.62e42fefa39efp-1;
constexpr double kLn2Lo = 0x1.abc9e3b39803fp-56;
constexpr double kInvLn2 = 0x1.71547652b82fep+0;
constexpr double kPio2A = 0x1.921fb54442d18p+0;
constexpr double kPio2B = 0x1.1a62633145c07p-54;
constexpr double kPio2C = -0x1.f1976b7ed8fbcp-110;
constexpr double kTwoOverPi = 0x1.45f306dc9c883p-1;
constexpr double kSqrt2 = 1.4142135623730951;
constexpr double kInf = __builtin_huge_val();

HPS_HD uint64_t bits_of(double v) { return __builtin_bit_cast(uint64_t, v); }
HPS_HD double double_of(uint64_t u) { return __builtin_bit_cast(double, u); }
HPS_HD double pow2i(int k) { return double_of((uint64_t)(k + 1023) << 52); }

// Quotients without exponent scaling.  The compiler spends eleven vector
// instructions on an FP64 quotient, several of which only scale operands near
// the ends of the exponent range.  This is its sequence without them: the
// reciprocal of v_rcp_f64 with two Newton steps, one corrected quotient (the
// residual is exact), v_div_fixup for zeros, infinities and NaN.  For a
// numerator that is 0 or of 2^-968 and up, a denominator between 2^-1000 and
// 2^1000 and a quotient between 2^-1000 and 2^1000 every step rounds the
// same, so the result is the correctly rounded one.  Past that it is not (a
// subnormal denominator gives NaN), so callers keep their operands in range:
// see Quick below.  Quotients by one denominator share its reciprocal: four
// instructions for each further one.
// The build of hps_push_fast.hip and host code divide as they are compiled.
static HPS_HD double recip(double d)
{
#if defined(__HIP_DEVICE_COMPILE__) && !defined(HPS_FAST_PUSH)
  double y = __builtin_amdgcn_rcp(d);
  y = ::fma(y, ::fma(-d, y, 1.0), y);
  return ::fma(y, ::fma(-d, y, 1.0), y);
#else
  return 1.0 / d;
#endif
}

// n / d with y = recip(d), or the rounded 1 / d
static HPS_HD double div_by(double n, double d, double y)
{
#if defined(__HIP_DEVICE_COMPILE__) && !defined(HPS_FAST_PUSH)
  const double q = n * y;
  return __builtin_amdgcn_div_fixup(::fma(::fma(-d, q, n), y, q), d, n);
#else
  (void)y;
  return n / d;
#endif
}

static HPS_HD double pdiv(double n, double d) { return div_by(n, d, recip(d)); }

// A polynomial coefficient in scalar registers.  The compiler turns a Horner
// step fma(p, z, c) into the two-operand v_fmac, whose addend must first be
// moved into a vector register pair: two vector instructions more per step
// (37 steps in a half quad, 15 in each sine and cosine of a gap).  The empty
// asm is not volatile: a volatile one keeps the compiler from merging blocks,
// and the build of hps_push_fast.hip then shares other reciprocals.
static HPS_HD double uconst(double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(c));
#endif
  return c;
}

HPS_HD double exp(double x)
{
  if (x != x) return x;
  if (x > 709.79) return kInf;
  if (x < -745.2) return 0.0;
  const double kd = ::floor(x * kInvLn2 + 0.5);
  double r = ::fma(-kd, kLn2Hi, x);
  r = ::fma(-kd, kLn2Lo, r);
  // Taylor coefficients 1/13! ... 1/2!, then 1, 1.
  double p = 1.6059043836821613e-10;
  p = ::fma(p, r, uconst(2.08767569878681e-09));
  p = ::fma(p, r, uconst(2.505210838544172e-08));
  p = ::fma(p, r, uconst(2.755731922398589e-07));
  p = ::fma(p, r, uconst(2.7557319223985893e-06));
  p = ::fma(p, r, uconst(2.48015873015873e-05));
  p = ::fma(p, r, uconst(0.0001984126984126984));
  p = ::fma(p, r, uconst(0.001388888888888889));
  p = ::fma(p, r, uconst(0.008333333333333333));
  p = ::fma(p, r, uconst(0.041666666666666664));
  p = ::fma(p, r, uconst(0.16666666666666666));
  p = ::fma(p, r, uconst(0.5));
  p = ::fma(p, r, uconst(1.0));
  p = ::fma(p, r, uconst(1.0));
  const int k = (int)kd;
  const int k1 = k / 2;
  return (p * pow2i(k1)) * pow2i(k - k1);
}

HPS_HD double log(double x)
{
  if (x != x) return x;
  if (x < 0.0) return __builtin_nan("");
  if (x == 0.0) return -kInf;
  if (x == kInf) return x;
  uint64_t u = bits_of(x);
  int e = (int)((u >> 52) & 0x7ff);
  if (e == 0) {               // subnormal: renormalise
    x = x * 0x1p54;
    u = bits_of(x);
    e = (int)((u >> 52) & 0x7ff) - 54;
  }
  e -= 1023;
  double m = double_of((u & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL);
  if (m > kSqrt2) { m = m * 0.5; e += 1; }
  const double s = pdiv(m - 1.0, m + 1.0);
  const double z = s * s;
  // 1/23, 1/21, ..., 1/3
  double p = 0.043478260869565216;
  p = ::fma(p, z, uconst(0.047619047619047616));
  p = ::fma(p, z, uconst(0.05263157894736842));
  p = ::fma(p, z, uconst(0.058823529411764705));
  p = ::fma(p, z, uconst(0.06666666666666667));
  p = ::fma(p, z, uconst(0.07692307692307693));
  p = ::fma(p, z, uconst(0.09090909090909091));
  p = ::fma(p, z, uconst(0.1111111111111111));
  p = ::fma(p, z, uconst(0.14285714285714285));
  p = ::fma(p, z, uconst(0.2));
  p = ::fma(p, z, uconst(0.3333333333333333));
  const double s2 = 2.0 * s;
  const double lm = ::fma(s2 * z, p, s2);
  const double ed = (double)e;
  return ::fma(ed, kLn2Hi, ::fma(ed, kLn2Lo, lm));
}

// kd mod 4 of a whole kd: four instructions where a conversion to 64-bit
// integers takes nine
HPS_HD int quadrant(double kd) { return (int)::fma(-4.0, ::floor(kd * 0.25), kd); }

// sine and cosine turned by q quarter turns
HPS_HD void turn(int q, double s, double c, double* sp, double* cp)
{
  const uint64_t ns = (uint64_t)(q & 2) << 62, nc = (uint64_t)((q + 1) & 2) << 62;
  *sp = double_of(bits_of(q & 1 ? c : s) ^ ns);
  *cp = double_of(bits_of(q & 1 ? s : c) ^ nc);
}

HPS_HD void sincos(double x, double* sp, double* cp)
{
  if (!(__builtin_fabs(x) < kInf)) { *sp = x - x; *cp = x - x; return; }
  const double kd = ::floor(x * kTwoOverPi + 0.5);
  double r = ::fma(-kd, kPio2A, x);
  r = ::fma(-kd, kPio2B, r);
  r = ::fma(-kd, kPio2C, r);
  const int q = quadrant(kd);
  const double z = r * r;
  // sin: 1/17!, -1/15!, ..., -1/3!
  double ps = 2.8114572543455206e-15;
  ps = ::fma(ps, z, uconst(-7.647163731819816e-13));
  ps = ::fma(ps, z, uconst(1.6059043836821613e-10));
  ps = ::fma(ps, z, uconst(-2.505210838544172e-08));
  ps = ::fma(ps, z, uconst(2.7557319223985893e-06));
  ps = ::fma(ps, z, uconst(-0.0001984126984126984));
  ps = ::fma(ps, z, uconst(0.008333333333333333));
  ps = ::fma(ps, z, uconst(-0.16666666666666666));
  const double s = ::fma(r * z, ps, r);
  // cos: -1/18!, 1/16!, ..., -1/2!
  double pc = -1.5619206968586225e-16;
  pc = ::fma(pc, z, uconst(4.779477332387385e-14));
  pc = ::fma(pc, z, uconst(-1.1470745597729725e-11));
  pc = ::fma(pc, z, uconst(2.08767569878681e-09));
  pc = ::fma(pc, z, uconst(-2.755731922398589e-07));
  pc = ::fma(pc, z, uconst(2.48015873015873e-05));
  pc = ::fma(pc, z, uconst(-0.001388888888888889));
  pc = ::fma(pc, z, uconst(0.041666666666666664));
  pc = ::fma(pc, z, uconst(-0.5));
  const double c = ::fma(z, pc, 1.0);
  turn(q, s, c, sp, cp);
}

HPS_HD double sinh(double x)
{
  const double ax = __builtin_fabs(x);
  if (ax < 1.0) {
    const double z = x * x;
    double p = 1.9572941063391263e-20;   // 1/21!
    p = ::fma(p, z, uconst(8.22063524662433e-18));
    p = ::fma(p, z, uconst(2.8114572543455206e-15));
    p = ::fma(p, z, uconst(7.647163731819816e-13));
    p = ::fma(p, z, uconst(1.6059043836821613e-10));
    p = ::fma(p, z, uconst(2.505210838544172e-08));
    p = ::fma(p, z, uconst(2.7557319223985893e-06));
    p = ::fma(p, z, uconst(0.0001984126984126984));
    p = ::fma(p, z, uconst(0.008333333333333333));
    p = ::fma(p, z, uconst(0.16666666666666666));
    return ::fma(x * z, p, x);
  }
  const double e = hps::exp(ax);
  const double h = 0.5 * e - 0.5 / e;
  return x < 0.0 ? -h : h;
}

HPS_HD double cosh(double x)
{
  const double ax = __builtin_fabs(x);
  if (ax < 1.0) {
    const double z = x * x;
    double p = 4.110317623312165e-19;    // 1/20!
    p = ::fma(p, z, uconst(1.5619206968586225e-16));
    p = ::fma(p, z, uconst(4.779477332387385e-14));
    p = ::fma(p, z, uconst(1.1470745597729725e-11));
    p = ::fma(p, z, uconst(2.08767569878681e-09));
    p = ::fma(p, z, uconst(2.755731922398589e-07));
    p = ::fma(p, z, uconst(2.48015873015873e-05));
    p = ::fma(p, z, uconst(0.001388888888888889));
    p = ::fma(p, z, uconst(0.041666666666666664));
    p = ::fma(p, z, uconst(0.5));
    return ::fma(z, p, 1.0);
  }
  const double e = hps::exp(ax);
  return 0.5 * e + 0.5 / e;
}

// sinh and cosh of one argument with a single exp: the same two results as
// sinh(x) and cosh(x) above, bit for bit.
HPS_HD void sinhcosh(double x, double* shp, double* chp)
{
  const double ax = __builtin_fabs(x);
  if (ax < 1.0) {
    *shp = hps::sinh(x);
    *chp = hps::cosh(x);
    return;
  }
  const double e = hps::exp(ax);
  const double h = 0.5 * e - 0.5 / e;
  *shp = x < 0.0 ? -h : h;
  *chp = 0.5 * e + 0.5 / e;
}

// tan(x) = sin(x) / cos(x) from sincos.
HPS_HD double tan(double x)
{
  double s, c;
  sincos(x, &s, &c);
  return s / c;
}

// Square root from v_rsq_f64.  One Goldschmidt step refines g ~ sqrt(x)
// and h ~ 1 / (2 sqrt(x)); one Newton correction of g follows.  For
// 2^-767 <= x < inf the result is within about one unit in the last place.
// The correctly rounded ::sqrt adds a second correction, scales x below
// 2^-767, and costs 21 instructions against 12.  +-0 and +inf are returned
// as they are; negative x and NaN give NaN.  Positive x below 2^-767 is
// outside its range.  Device code only.
__device__ __forceinline__ double sqrt_rsq(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = ::fma(-h, g, 0.5);
  g = ::fma(g, r, g);
  h = ::fma(h, r, h);
  const double d = ::fma(-g, g, x);
  g = ::fma(d, h, g);
  return (x == 0.0 || x == kInf) ? x : g;
}

// sincos with the Taylor polynomials cut at r^13 (sin) and r^14 (cos) after
// the same reduction: on |r| <= pi/4 the first omitted terms are below
// 2.1e-14 and 1.1e-15.  Device code only.
__device__ __forceinline__ void sincos_short(double x, double* sp, double* cp)
{
  if (!(__builtin_fabs(x) < kInf)) { *sp = x - x; *cp = x - x; return; }
  const double kd = ::floor(x * kTwoOverPi + 0.5);
  double r = ::fma(-kd, kPio2A, x);
  r = ::fma(-kd, kPio2B, r);
  r = ::fma(-kd, kPio2C, r);
  const int q = quadrant(kd);
  const double z = r * r;
  // sin: 1/13!, -1/11!, ..., -1/3!
  double ps = 1.6059043836821613e-10;
  ps = ::fma(ps, z, uconst(-2.505210838544172e-08));
  ps = ::fma(ps, z, uconst(2.7557319223985893e-06));
  ps = ::fma(ps, z, uconst(-0.0001984126984126984));
  ps = ::fma(ps, z, uconst(0.008333333333333333));
  ps = ::fma(ps, z, uconst(-0.16666666666666666));
  const double s = ::fma(r * z, ps, r);
  // cos: 1/14!, -1/12!, ..., -1/2!
  double pc = -1.1470745597729725e-11;
  pc = ::fma(pc, z, uconst(2.08767569878681e-09));
  pc = ::fma(pc, z, uconst(-2.755731922398589e-07));
  pc = ::fma(pc, z, uconst(2.48015873015873e-05));
  pc = ::fma(pc, z, uconst(-0.001388888888888889));
  pc = ::fma(pc, z, uconst(0.041666666666666664));
  pc = ::fma(pc, z, uconst(-0.5));
  const double c = ::fma(z, pc, 1.0);
  turn(q, s, c, sp, cp);
}

// sinhcosh with the Taylor series for |x| < 1 cut at x^15 (sinh) and x^16
// (cosh): the first omitted terms at |x| = 1 are 2.8e-15 and 1.6e-16 of the
// results.  |x| >= 1 as sinhcosh.  Device code only.
__device__ __forceinline__ void sinhcosh_short(double x, double* shp, double* chp)
{
  const double ax = __builtin_fabs(x);
  if (ax < 1.0) {
    const double z = x * x;
    double p = 7.647163731819816e-13;    // 1/15!
    p = ::fma(p, z, uconst(1.6059043836821613e-10));
    p = ::fma(p, z, uconst(2.505210838544172e-08));
    p = ::fma(p, z, uconst(2.7557319223985893e-06));
    p = ::fma(p, z, uconst(0.0001984126984126984));
    p = ::fma(p, z, uconst(0.008333333333333333));
    p = ::fma(p, z, uconst(0.16666666666666666));
    *shp = ::fma(x * z, p, x);
    double c = 4.779477332387385e-14;     // 1/16!
    c = ::fma(c, z, uconst(1.1470745597729725e-11));
    c = ::fma(c, z, uconst(2.08767569878681e-09));
    c = ::fma(c, z, uconst(2.755731922398589e-07));
    c = ::fma(c, z, uconst(2.48015873015873e-05));
    c = ::fma(c, z, uconst(0.001388888888888889));
    c = ::fma(c, z, uconst(0.041666666666666664));
    c = ::fma(c, z, uconst(0.5));
    *chp = ::fma(z, c, 1.0);
    return;
  }
  sinhcosh(x, shp, chp);
}

// sincos and sinhcosh of the per-particle maps: the full polynomials, or the
// short ones in the build of hps_push_fast.hip (see psqrt below).
static __device__ __forceinline__ void psincos(double x, double* sp, double* cp)
{
#ifdef HPS_FAST_PUSH
  sincos_short(x, sp, cp);
#else
  sincos(x, sp, cp);
#endif
}

static __device__ __forceinline__ void psinhcosh(double x, double* shp, double* chp)
{
#ifdef HPS_FAST_PUSH
  sinhcosh_short(x, shp, chp);
#else
  sinhcosh(x, shp, chp);
#endif
}

// The square root of the per-particle maps, the kick and the deposit: the
// correctly rounded ::sqrt, or sqrt_rsq in the build of hps_push_fast.hip,
// which serves batches whose results are held to error bounds, not to the
// oracle's bits.  Internal to each translation unit, so the two builds keep
// their own.
static __device__ __forceinline__ double psqrt(double x)
{
#ifdef HPS_FAST_PUSH
  return sqrt_rsq(x);
#else
  return ::sqrt(x);
#endif
}

// The root of v_rsq_f64 with one Goldschmidt step and two corrections, ten
// instructions where ::sqrt takes twenty-one: correctly rounded from 2^-960 to
// 2^1000, NaN for 0 and infinity.
static __device__ __forceinline__ double sqrt_unscaled(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = ::fma(-h, g, 0.5);
  g = ::fma(g, r, g);
  h = ::fma(h, r, h);
  g = ::fma(::fma(-g, g, x), h, g);
  return ::fma(::fma(-g, g, x), h, g);
}

// Quotients and roots of the maps, the kick, the deposit and the Green's
// table, which take one of these as a template argument.
//
// Any takes every operand: the compiler's own sequences.
//
// Quick leaves out the exponent scaling (recip, div_by, sqrt_unscaled) and
// gives the same bits while all operands stay in the range stated there.  A
// function that takes it marks the few values of the particle that every
// quotient and root of it follows from; where one of them lies outside
// 2^-64 .. 2^64 or is 0, infinite or NaN (off), the particle goes through Any
// instead.  The element's or mesh's constants are held to the same range (or
// 0 where they are only numerators) once, before the particles (usual).  A sum
// of such values is 0 or at least an ulp of the smaller one, so cancellation
// stays far above 2^-968.
// The tracking kernels are bound by vector instructions (k_segment 88 % of its
// waves' time); a mark costs two, the zero and infinity cases that its roots
// need not treat three each.  1,048,576 particles on 32 x 128, 800 elements,
// a step: 60.8 ms, with Any alone 65.7.
#if defined(HPS_FAST_PUSH) || !defined(__HIP_DEVICE_COMPILE__)
constexpr bool kBounded = false;
#else
constexpr bool kBounded = true;
#endif

namespace {

struct Any {
  // Its quotients are not moved past each other: it is seldom run, and side by
  // side they would take the kernels from 65 to 79 VGPRs.
  static HPS_HD void order()
  {
#if defined(__HIP_DEVICE_COMPILE__) && !defined(HPS_FAST_PUSH)
    __builtin_amdgcn_sched_barrier(0);
#endif
  }
  static HPS_HD double recip(double) { return 0.0; }
  static HPS_HD double div(double n, double d)
  {
    order();
    const double q = n / d;
    order();
    return q;
  }
  static HPS_HD double div_by(double n, double d, double) { return div(n, d); }
  static __device__ __forceinline__ double sqrt(double x)
  {
    order();
    const double q = psqrt(x);
    order();
    return q;
  }
  static __device__ __forceinline__ double sqrt0(double x) { return psqrt(x); }
  static HPS_HD uint32_t mark(double) { return 0; }
  static HPS_HD uint32_t mark0(double) { return 0; }
  static HPS_HD bool off(uint32_t) { return false; }
};

struct Quick {
  static HPS_HD double recip(double d) { return hps::recip(d); }
  static HPS_HD double div(double n, double d) { return hps::pdiv(n, d); }
  static HPS_HD double div_by(double n, double d, double y) { return hps::div_by(n, d, y); }
  static __device__ __forceinline__ double sqrt(double x) { return sqrt_unscaled(x); }
  static __device__ __forceinline__ double sqrt0(double x) { return x > 0.0 ? sqrt(x) : x; }
  // bits 27 to 30 of a mark are 0 if and only if |v| is in [2^-64, 2^64):
  // the biased exponent less that of 2^-64, modulo 2^11.  Marks are or'ed.
  static HPS_HD uint32_t mark(double v) { return (uint32_t)(bits_of(v) >> 32) - 0x3bf00000u; }
  // The same with 0 in range (a particle on the axis).  Infinities and NaN
  // pass too: for the RF gap, which loses such a particle in either form.
  static __device__ __forceinline__ uint32_t mark0(double v)
  {
#ifdef __HIP_DEVICE_COMPILE__
    return (uint32_t)(__builtin_amdgcn_frexp_exp(v) + 63) << 20;
#else
    return 0;
#endif
  }
  static constexpr uint32_t kOff = 0x78000000u;
  static HPS_HD bool off(uint32_t m) { return (m & kOff) != 0; }
};

typedef std::conditional<kBounded, Quick, Any>::type Usual;

// |v| in [2^-64, 2^64)
HPS_HD bool in_range(double v) { return !Quick::off(Quick::mark(v)); }
// |v| < 2^64
HPS_HD bool below_range_end(double v)
{
  return (uint32_t)(bits_of(v) >> 32 & 0x7fffffffu) < 0x43f00000u;
}
HPS_HD bool zero_or_in_range(double v) { return bits_of(v) << 1 == 0 || in_range(v); }

}  // namespace

// Remainder of x >= 0 by y > 0 (finite), exact.
HPS_HD double fmod_pos(double x, double y)
{
  if (!(x < kInf)) return __builtin_nan("");
  if (x < y) return x;
  double yy = y;
  while (yy * 2.0 <= x) yy = yy * 2.0;
  while (yy >= y) {
    if (x >= yy) x = x - yy;
    yy = yy * 0.5;
  }
  return x;
}

// double -> int: NaN -> 0, saturating at the int range.
HPS_HD int to_int(double v)
{
  if (v != v) return 0;
  if (v >= 2147483647.0) return 2147483647;
  if (v <= -2147483648.0) return -2147483647 - 1;
  return (int)v;
}

}  // namespace hps
