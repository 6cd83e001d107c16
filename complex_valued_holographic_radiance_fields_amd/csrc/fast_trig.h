// fast_trig.h — sine and cosine of large float arguments for the transfer
// function of the propagation kernels.
//
// The phase d*kz is formed in float exactly as the reference forms it and
// reaches ~1e4-1e5 rad.  Its sine and cosine are taken here by reducing the
// float argument modulo 2*pi in double precision (x is exact as a double and
// x/(2*pi) keeps 53 bits, so the fractional revolution is accurate to ~1e-12)
// and evaluating the hardware sin/cos of that fraction in revolutions
// (v_sin_f32 / v_cos_f32 compute sin(2*pi*r)).  Absolute error is a few 1e-7,
// checked against float64 sin/cos by the GPU tests.
#pragma once

#include <hip/hip_runtime.h>

namespace hrf {

__device__ __forceinline__ void sincos_big(float x, float* s, float* c) {
  constexpr double kInvTwoPi = 0.15915494309189533577;  // 1 / (2 pi)
  const double t = static_cast<double>(x) * kInvTwoPi;
  const float rev = static_cast<float>(t - __builtin_rint(t));  // in [-0.5, 0.5]
  *s = __builtin_amdgcn_sinf(rev);
  *c = __builtin_amdgcn_cosf(rev);
}

// The same reduction without double precision, for the propagation's
// inner loops: 1/(2 pi) split into a float head kHi and tail kLo, the
// product x kHi rounded to hi with its exact rounding error
// e = fma(x, kHi, -hi), hi - rint(hi) exact (Sterbenz), and the revolution
// r = (hi - rint(hi)) + fma(x, kLo, e): for |x| below 2^21 revolutions'
// worth its error is the final rounding (2^-25 of a revolution) plus
// ~|x| 2^-48, the double-precision version's accuracy with six single-rate
// instructions instead of five at double rate.
__device__ __forceinline__ void sincos_big_ff(float x, float* s, float* c) {
  constexpr float kHi = 0.15915493667125701904f;        // float(1 / (2 pi))
  constexpr float kLo = 6.4206383167313347657e-09f;     // 1 / (2 pi) - kHi
  const float hi = x * kHi;
  const float e = fmaf(x, kHi, -hi);
  const float rev = (hi - __builtin_rintf(hi)) + fmaf(x, kLo, e);  // in [-0.5, 0.5]
  *s = __builtin_amdgcn_sinf(rev);
  *c = __builtin_amdgcn_cosf(rev);
}

// The same reduction down to a quadrant, and polynomials instead of the
// hardware functions: with rev = q / 4 + f, |f| <= 1/8, the remainder keeps
// two more bits than a half revolution does, and sin(2 pi f) = f S(f^2),
// cos(2 pi f) = 1 + f^2 C(f^2) with cubic S and C (interpolated at Chebyshev
// nodes of f^2 in [0, 1/64], rounded to float).  2.1e-8 rms off float64 in
// each, where the hardware functions of a rounded half revolution leave about
// 6e-8: for the transforms that replace ones whose transfer function called
// sincosf (1.5e-8).
__device__ __forceinline__ void sincos_big_quad(float x, float* s, float* c) {
  constexpr float kHi = 0.15915493667125701904f;
  constexpr float kLo = 6.4206383167313347657e-09f;
  const float hi = x * kHi;
  const float lo = fmaf(x, kLo, fmaf(x, kHi, -hi));
  const float r = hi - __builtin_rintf(hi);       // exact, in [-0.5, 0.5]
  const float q4 = __builtin_rintf(4.0f * r);     // -2 .. 2
  const float f = fmaf(q4, -0.25f, r) + lo;       // the fma is exact
  const float g = f * f;
  const float sn =
      f * fmaf(g, fmaf(g, fmaf(g, -75.40184020996094f, 81.59254455566406f), -41.3416633605957f),
               6.2831854820251465f);
  const float cs =
      fmaf(g, fmaf(g, fmaf(g, fmaf(g, 59.42423629760742f, -85.44882202148438f),
                           64.93936920166016f), -19.739208221435547f), 1.0f);
  const int q = static_cast<int>(q4);
  const float a = (q & 1) ? cs : sn, b = (q & 1) ? sn : cs;
  // quadrants 2, 3 negate the sine, 1, 2 the cosine (q mod 4)
  *s = (q & 2) ? -a : a;
  *c = ((q + 1) & 2) ? -b : b;
}

}  // namespace hrf
