// Arithmetic policy of the two engines, host/device.
//   float  : the deterministic own routines of fpmath.h (mixed engine; the CPU
//            replay reproduces them bit for bit)
//   double : the platform libm (plain FP64 engine)
#pragma once

#include <stdint.h>
#include <math.h>
#include "fpmath.h"
#include "hd.h"
#include "philox.h"

namespace storm {

template <typename Real>
struct MathPolicy;

template <>
struct MathPolicy<float> {
  STORM_HD static float log(float x) { return fpm::logf_d(x); }
  STORM_HD static float exp(float x) { return fpm::expf_d(x); }
  STORM_HD static float expm1_neg(float x) { return fpm::expm1_neg(x); }  // x <= 0
  STORM_HD static float log_unit(float x) { return fpm::log_unit(x); }    // x a uniform or 1 minus one
  STORM_HD static float recip(float x) { return fpm::recip_f(x); }        // |x| in [2^-126, 2^126]
  STORM_HD static float recip_any(float x) {
    return (x >= 0x1p-126f && x <= 0x1p126f) ? fpm::recip_f(x) : 1.0f / x;
  }
  // a / b, rounded as IEEE does for b within [2^-60, 2^60] and a +0 or within
  // [2^-60, 2^60]; elsewhere about it, or no number
  STORM_HD static float div_tame(float a, float b) { return fpm::div_f(a, b); }
  // the middle one of three, the smaller of the others if one is no number
  STORM_HD static float median(float a, float b, float c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_fmed3f(a, b, c);
#else
    const float lo = a < b ? a : b, hi = a < b ? b : a;
    return c < lo ? lo : (c > hi ? hi : c);
#endif
  }
  STORM_HD static float sqrt_unit(float x) { return fpm::sqrt_f(x); }     // x 0 or in [2^-100, 2^100]
  STORM_HD static void sincos2pi(float u, float &s, float &c) { fpm::sincos2pi(u, s, c); }
  STORM_HD static float sqrt(float x) { return ::sqrtf(x); }
  STORM_HD static float uniform(uint32_t x) { return u01_f32(x); }
  STORM_HD static float inf() { return fpm::u2f(0x7f800000u); }
};

template <>
struct MathPolicy<double> {
  STORM_HD static double log(double x) { return ::log(x); }
  STORM_HD static double exp(double x) { return ::exp(x); }
  STORM_HD static double expm1_neg(double x) { return ::expm1(x); }
  STORM_HD static double log_unit(double x) { return ::log(x); }
  STORM_HD static double recip(double x) { return 1.0 / x; }
  STORM_HD static double recip_any(double x) { return 1.0 / x; }
  STORM_HD static double div_tame(double a, double b) { return a / b; }
  STORM_HD static double median(double a, double b, double c) {
    const double lo = a < b ? a : b, hi = a < b ? b : a;
    return c < lo ? lo : (c > hi ? hi : c);
  }
  STORM_HD static double sqrt_unit(double x) { return ::sqrt(x); }
  STORM_HD static void sincos2pi(double u, double &s, double &c) {
#if defined(__HIP_DEVICE_COMPILE__)
    // of pi times 2 u: the quadrant is exact and 2 pi u is not rounded, and
    // there is no reduction of large arguments to carry along
    ::sincospi(2.0 * u, &s, &c);
    return;
#endif
    double a = 6.283185307179586476925286766559 * u;
    s = ::sin(a);
    c = ::cos(a);
  }
  STORM_HD static double sqrt(double x) { return ::sqrt(x); }
  STORM_HD static double uniform(uint32_t x) { return (static_cast<double>(x) + 0.5) * 2.3283064365386963e-10; }
  STORM_HD static double inf() { return fpm::u2d(0x7ff0000000000000ull); }
};

// Isotropic unit vector from two uniforms: mu = 2 u0 - 1, phi = 2 pi u1
// (isotropicVelocity, radiation/RadiationOpacityModel.hpp:139-150).
template <typename Real>
STORM_HD void isotropic_dir(Real u0, Real u1, Real o[3]) {
  Real mu = Real(2) * u0 - Real(1);
  Real st2 = Real(1) - mu * mu;
  Real st = MathPolicy<Real>::sqrt(st2 > Real(0) ? st2 : Real(0));
  Real sp, cp;
  MathPolicy<Real>::sincos2pi(u1, sp, cp);
  o[0] = st * cp;
  o[1] = st * sp;
  o[2] = mu;
}

}  // namespace storm
