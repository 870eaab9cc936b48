// Deterministic single-precision elementary functions shared by the gfx950
// transport kernels and their CPU replay.
//
// Vendor libm / device math libraries differ between host and device, so the
// mixed-precision engine uses only these routines, built from IEEE-754 +, -,
// *, /, sqrt and fused multiply-add, all correctly rounded on both sides.
// Every translation unit that includes this header is compiled with
// -ffp-contract=off, so the compiler forms no FMA of its own; the polynomial
// steps below ask for one explicitly (fma_f: v_fma_f32 on the device, the
// correctly rounded fmaf of the C library on the host).
// Methods:
//   log   : exponent/mantissa split with m in [sqrt(1/2), sqrt(2)), then
//           log(m) = 2 atanh(s), s = (m-1)/(m+1), atanh series to s^9;
//           ln2 split in two parts (Cody & Waite, "Software Manual for the
//           Elementary Functions", 1980).
//   exp   : Cody-Waite reduction y = k ln2 + r, |r| <= ln2/2, Taylor series
//           of e^r to r^8, scaling by 2^k through the exponent field.
//   expm1 : Taylor series to y^9 for |y| < ln2/2, exp(y) - 1 otherwise.
//   sincos of 2*pi*u : exact quadrant reduction of 4u, Taylor series of sin
//           and cos on [-pi/4, pi/4].
//   1/x, sqrt, a/b (recip_f, sqrt_f, div_f): the hardware's 1 ulp estimate
//           and one Newton step with a fused remainder, which rounds as IEEE
//           does over the ranges stated at each (on gfx950 1/x and sqrt are
//           checked for every float of the range; a/b, whose rounding follows
//           from the theorem named there, for 2^28 pairs); the host uses the
//           IEEE operators.
// Accuracy is a few ulp, far below Monte Carlo noise; what matters is that
// host and device produce the same bits.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>
#include "hd.h"

namespace storm {
namespace fpm {

STORM_HD uint32_t f2u(float x) {
  uint32_t u;
  memcpy(&u, &x, sizeof(u));
  return u;
}
STORM_HD float u2f(uint32_t u) {
  float x;
  memcpy(&x, &u, sizeof(x));
  return x;
}
STORM_HD uint64_t d2u(double x) {
  uint64_t u;
  memcpy(&u, &x, sizeof(u));
  return u;
}
STORM_HD double u2d(uint64_t u) {
  double x;
  memcpy(&x, &u, sizeof(x));
  return x;
}

// a * b + c with one rounding
STORM_HD float fma_f(float a, float b, float c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_fmaf(a, b, c);
#else
  return ::fmaf(a, b, c);
#endif
}

// 1 / x as IEEE rounds it, for 2^-126 <= |x| <= 2^126 (3 instructions; the
// compiler's full-range division takes 10).
STORM_HD float recip_f(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
#else
  return 1.0f / x;
#endif
}

// sqrt(x) as IEEE rounds it, for 2^-100 <= x <= 2^100 and for 0.
STORM_HD float sqrt_f(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = x * y;
  const float q = __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
  return x > 0.0f ? q : 0.0f;
#else
  return ::sqrtf(x);
#endif
}

// a / b as IEEE rounds it, for |b| within [2^-60, 2^60] and a +0 or |a| within
// [2^-60, 2^60]: with the correctly rounded reciprocal the
// quotient corrected by its exact remainder is correctly rounded (Markstein
// 1990).
STORM_HD float div_f(float a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float y = recip_f(b);
  const float q = a * y;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
#else
  return a / b;
#endif
}

constexpr float kLn2Hi = 0.693115234375f;          // 12 significant bits
constexpr float kLn2Lo = 3.194618329871446e-05f;   // ln2 - kLn2Hi
constexpr float kLog2e = 1.4426950216293335f;
constexpr float kHalfPi = 1.5707963705062866f;
constexpr float kSqrt2 = 1.4142135381698608f;

// Natural log for finite x > 0 (normal or subnormal).  Returns -inf for 0.
STORM_HD float logf_d(float x) {
  if (!(x > 0.0f)) return x == 0.0f ? -u2f(0x7f800000u) : u2f(0x7fc00000u);
  uint32_t b = f2u(x);
  int e = 0;
  if (b < 0x00800000u) {  // subnormal: scale by 2^24 first
    x = x * 16777216.0f;
    b = f2u(x);
    e = -24;
  }
  e += static_cast<int>((b >> 23) & 0xffu) - 127;
  float m = u2f((b & 0x007fffffu) | 0x3f800000u);  // [1, 2)
  if (m > kSqrt2) {
    m = m * 0.5f;
    e += 1;
  }
  float f = m - 1.0f;
  float s = f / (2.0f + f);
  float z = s * s;
  float p = 1.0f / 9.0f;
  p = fma_f(z, p, 1.0f / 7.0f);
  p = fma_f(z, p, 1.0f / 5.0f);
  p = fma_f(z, p, 1.0f / 3.0f);
  p = fma_f(z, p, 1.0f);
  float lm = 2.0f * s * p;
  float ef = static_cast<float>(e);
  return fma_f(ef, kLn2Hi, fma_f(ef, kLn2Lo, lm));
}

// logf_d for the uniforms: the same bits for normal x in (0, 1], without the
// cases logf_d tells apart first (0, negative, NaN and subnormal arguments;
// some finite value for 0).  The quotient (m - 1) / (m + 1) needs no reciprocal
// step: the corrected estimate is the IEEE quotient for every m.
STORM_HD float log_unit(float x) {
  const uint32_t b = f2u(x);
  int e = static_cast<int>(b >> 23) - 127;
  float m = u2f((b & 0x007fffffu) | 0x3f800000u);  // [1, 2)
  const bool up = m > kSqrt2;
  m = up ? m * 0.5f : m;
  e = up ? e + 1 : e;
  const float f = m - 1.0f;
#if defined(__HIP_DEVICE_COMPILE__)
  const float d = 2.0f + f;
  const float y = __builtin_amdgcn_rcpf(d);
  const float q = f * y;
  const float s = __builtin_fmaf(__builtin_fmaf(-d, q, f), y, q);
#else
  const float s = f / (2.0f + f);
#endif
  const float z = s * s;
  float p = 1.0f / 9.0f;
  p = fma_f(z, p, 1.0f / 7.0f);
  p = fma_f(z, p, 1.0f / 5.0f);
  p = fma_f(z, p, 1.0f / 3.0f);
  p = fma_f(z, p, 1.0f);
  const float lm = 2.0f * s * p;
  const float ef = static_cast<float>(e);
  return fma_f(ef, kLn2Hi, fma_f(ef, kLn2Lo, lm));
}

// e^y.  Flushes to 0 below -87 and saturates to +inf above 88.
STORM_HD float expf_d(float y) {
  if (y < -87.0f) return 0.0f;
  if (y > 88.0f) return u2f(0x7f800000u);
  float kf = y * kLog2e;
  int k = static_cast<int>(kf + (kf >= 0.0f ? 0.5f : -0.5f));
  float fk = static_cast<float>(k);
  float r = fma_f(-fk, kLn2Lo, fma_f(-fk, kLn2Hi, y));
  float p = 1.0f / 40320.0f;
  p = fma_f(r, p, 1.0f / 5040.0f);
  p = fma_f(r, p, 1.0f / 720.0f);
  p = fma_f(r, p, 1.0f / 120.0f);
  p = fma_f(r, p, 1.0f / 24.0f);
  p = fma_f(r, p, 1.0f / 6.0f);
  p = fma_f(r, p, 0.5f);
  p = fma_f(r, p, 1.0f);
  p = fma_f(r, p, 1.0f);
  // scale by 2^k in two halves so that k down to -126-ish stays representable
  int k1 = k / 2;
  int k2 = k - k1;
  float s1 = u2f(static_cast<uint32_t>(k1 + 127) << 23);
  float s2 = u2f(static_cast<uint32_t>(k2 + 127) << 23);
  return (p * s1) * s2;
}

// e^y - 1.
STORM_HD float expm1f_d(float y) {
  float ay = y < 0.0f ? -y : y;
  if (ay < 0.34657359f) {
    float p = 1.0f / 362880.0f;
    p = fma_f(y, p, 1.0f / 40320.0f);
    p = fma_f(y, p, 1.0f / 5040.0f);
    p = fma_f(y, p, 1.0f / 720.0f);
    p = fma_f(y, p, 1.0f / 120.0f);
    p = fma_f(y, p, 1.0f / 24.0f);
    p = fma_f(y, p, 1.0f / 6.0f);
    p = fma_f(y, p, 0.5f);
    return fma_f(y * y, p, y);
  }
  return expf_d(y) - 1.0f;
}

// expm1f_d for y <= 0, the same bits in one straight line: near 0 and away
// from it share the middle of their series (the terms from y^2/2 down to
// y^8/8!), so lanes of both kinds run it once.
STORM_HD float expm1_neg(float y) {
  const bool near = y > -0.34657359f;
  const float yc = y < -87.0f ? -87.0f : y;  // e^-87 - 1 rounds to -1
  const float kf = yc * kLog2e;
  const int k = near ? 0 : static_cast<int>(kf - 0.5f);
  const float fk = static_cast<float>(k);
  const float r = fma_f(-fk, kLn2Lo, fma_f(-fk, kLn2Hi, yc));  // y itself for k = 0
  const float p9 = fma_f(r, 1.0f / 362880.0f, 1.0f / 40320.0f);
  float p = near ? p9 : 1.0f / 40320.0f;
  p = fma_f(r, p, 1.0f / 5040.0f);
  p = fma_f(r, p, 1.0f / 720.0f);
  p = fma_f(r, p, 1.0f / 120.0f);
  p = fma_f(r, p, 1.0f / 24.0f);
  p = fma_f(r, p, 1.0f / 6.0f);
  p = fma_f(r, p, 0.5f);
  const float small = fma_f(r * r, p, r);
  const float q = fma_f(r, fma_f(r, p, 1.0f), 1.0f);
  // 2^k is normal for k >= -126, and what is lost below 1 does not matter
  const float big = q * u2f(static_cast<uint32_t>(k + 127) << 23) - 1.0f;
  return near ? small : big;
}

// sin and cos of 2*pi*u for u in [0, 1].
STORM_HD void sincos2pi(float u, float &s_out, float &c_out) {
  float v = 4.0f * u;  // quadrant coordinate, exact
  int q = static_cast<int>(v + 0.5f);
  float t = v - static_cast<float>(q);  // [-0.5, 0.5], exact
  float a = t * kHalfPi;
  float a2 = a * a;
  float sp = 1.0f / 362880.0f;
  sp = fma_f(a2, sp, -1.0f / 5040.0f);
  sp = fma_f(a2, sp, 1.0f / 120.0f);
  sp = fma_f(a2, sp, -1.0f / 6.0f);
  float s = fma_f(a * a2, sp, a);
  float cp = -1.0f / 3628800.0f;
  cp = fma_f(a2, cp, 1.0f / 40320.0f);
  cp = fma_f(a2, cp, -1.0f / 720.0f);
  cp = fma_f(a2, cp, 1.0f / 24.0f);
  cp = fma_f(a2, cp, -0.5f);
  float c = fma_f(a2, cp, 1.0f);
  switch (q & 3) {
    case 0: s_out = s; c_out = c; break;
    case 1: s_out = c; c_out = -s; break;
    case 2: s_out = -s; c_out = -c; break;
    default: s_out = -c; c_out = s; break;
  }
}

// Exact power of two as a double, 2^k; k is clamped to the normal range
// [-1022, 1023].
STORM_HD double pow2d(int k) {
  k = k < -1022 ? -1022 : (k > 1023 ? 1023 : k);
  return u2d(static_cast<uint64_t>(k + 1023) << 52);
}

}  // namespace fpm
}  // namespace storm
