// Angle bins, radii and the rotation's division for the TurboQuant encoder
// without the full IEEE / fdlibm sequences, for the values where that is
// proven to give the same result.
//
// The codes are defined by float32 atan2 with the C library's steps
// (vrm_fdlibm_atan2f.h), two IEEE operations and a truncation.  Only the
// truncated bin leaves the encoder, so the angle is needed to the distance of
// the nearest sector edge, not to the last bit: fast_bin computes the position
// t in [0, 2^bits] of the angle with a polynomial and reports whether t is
// within kMargin * 2^bits of an edge.  Off the edges its bin is the defined
// one; a row with an angle at an edge is encoded again by the defining path.
// Multiples of pi / 4, which are edges and fill rows of zeros, signs or small
// integers, are decided here all the same, or such rows would be encoded twice,
// one after another on their wavefront (2048 rows of zeros 47 us against 12,
// of the integers -2 .. 2 59 against 15, with the row kernel 13 and 14).
//
// Bound (fractions of the full range, 2 pi at level 0 and pi / 2 above):
//   defining path: atan2 within 1 ulp, theta - lo and the division rounded,
//   the constants' own rounding: 1.8e-7 (level 0), 1.6e-7 (above);
//   fast_bin: polynomial 2.5e-7 rad, quotient 1.5 ulp (v_rcp_f32 is within 1
//   ulp), products and the folds rounded: 2.2e-7 (level 0), 4.1e-7 (above).
// Their sum stays below 5.7e-7; kMargin is 1e-6.  Plain C++, so that the host
// tests run the same code.
#pragma once
#include <math.h>
#include <stdint.h>

#ifndef VRM_HD
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define VRM_HD __host__ __device__ __forceinline__
#else
#define VRM_HD static inline
#endif
#endif

namespace vrm_tq_bin {

#define VRM_TQ_BIN_MARGIN 1.0e-6f

// Bin of atan2(y, x) over 2^BITS sectors of [-pi, pi] (LEVEL0) or [0, pi / 2]
// (x, y > 0, normal).  rcp is the reciprocal of max(|x|, |y|) to 1 ulp.  `edge`
// is true when the angle is too near a sector edge, other than those below, or
// the reciprocal overflowed.  NaN and infinite inputs are the caller's.
// Fused operations are wanted here; the polynomial is the minimax odd
// polynomial of degree 13 of atan on [0, 1], coefficients found by Remez
// exchange, scaled to sectors at compile time.
//
// No edges, in the sense that the defined bin is known (t is moved off them by
// kOff, far more than its error and far less than a sector):
//   level 0: multiples of pi / 4, which operands of one magnitude and zeros
//     (with their signs) give exactly; the defining path floors there;
//   above: the middle, pi / 4, where the defining path floors from y / x
//     rounded to 1 on, and the ends, where it stays within the range.
template <int BITS, bool LEVEL0>
VRM_HD int fast_bin(float x, float y, float rcp, bool& edge) {
  constexpr float kOff = 0x1p-10f;
  const float nb = (float)(1 << BITS);
  const double k = (double)(1 << BITS) / (LEVEL0 ? 6.283185307179586 : 1.5707963267948966);
  const float ax = fabsf(x), ay = fabsf(y), mn = fminf(ax, ay);
  const float q = mn * rcp;
  const float z = q * q;
  float p = (float)(0.006811792962253094 * k);
  p = fmaf(p, z, (float)(-0.0336042195558548 * k));
  p = fmaf(p, z, (float)(0.07962366938591003 * k));
  p = fmaf(p, z, (float)(-0.1323334276676178 * k));
  p = fmaf(p, z, (float)(0.19807815551757812 * k));
  p = fmaf(p, z, (float)(-0.3331736922264099 * k));
  p = fmaf(p, z, (float)(0.9999961256980896 * k));
  float t = q * p;
  if (LEVEL0) {
    const bool axis = mn == 0.f;
    t = axis ? 0.f : t;
    t = ay > ax ? 0.25f * nb - t : t;
    t = copysignf(1.f, x) < 0.f ? 0.5f * nb - t : t;
    t = 0.5f * nb + copysignf(t, y);
    t = axis || ax == ay ? t + kOff : t;
  } else {
    t = fminf(fmaxf(t, kOff), 0.5f * nb - kOff);
    t = ay >= ax ? nb - t : t;
  }
#ifdef __HIP_DEVICE_COMPILE__
  const float f = __builtin_amdgcn_fractf(t);
#else
  const float f = t - floorf(t);
#endif
  edge = !(fabsf(f - 0.5f) < 0.5f - VRM_TQ_BIN_MARGIN * nb);
  const int b = (int)t;
  return LEVEL0 && b > (1 << BITS) - 1 ? (1 << BITS) - 1 : b;
}

// x / (float)sqrt(128): with y the correctly rounded reciprocal of the
// divisor, one residual correction of x * y is the correctly rounded quotient
// (Markstein 1990) for every x whose residual does not underflow; checked for
// every significand in the host tests (2^-100 <= |x|, and both zeros: the
// residual is taken negated, since fma(-q, root, x) would turn -0 into +0).
VRM_HD float div_sqrt128(float x) {
  const float root = 11.313708305358887f, y = 0.08838834613561630249f;
  const float q = x * y;
  return fmaf(fmaf(q, root, -x), -y, q);
}

}  // namespace vrm_tq_bin
