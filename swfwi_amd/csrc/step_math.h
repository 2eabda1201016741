// The arithmetic of one 4t10s step, shared by the per-step kernels (tiles and
// strips) and the resident time loop.  kExact reproduces the reference's
// expression trees (fd4t10s-damp-zjh.c:44-54,85-88; fd4t10s-zjh.c:28-38,49-52):
// float ring sums, float coefficient products, double accumulation of
// -4.0*a0*p and the (2-2d+d^2)p / 2p terms, one rounding to float on store.  A
// product that is exact in its type (two 24-bit significands in a double, a
// power of two times a float) is folded into the following addition as an fma:
// the same bits, one instruction less.  kFp32 is pure FP32 with explicit fmaf.
#pragma once
#include <type_traits>

#include "kernels.h"

namespace swfwi {

// Zhang Jinhai coefficients as float, as the reference stores them.
constexpr float A0 = 1.53400796f, A1 = 1.78858721f, A2 = -0.31660756f;
constexpr float A3 = 0.07612173f, A4 = -0.01626042f, A5 = 0.00216736f;
constexpr double M4A0 = -4.0 * (double)A0;
constexpr float C12 = 1.0f / 12;

// u2 from the centre value and the five ring sums r_k = ((z-k + z+k) + x-k)
// + x+k, summed as the reference does.
template <int P>
__device__ __forceinline__ float u2_sum(float s0, float r1, float r2, float r3, float r4, float r5) {
  if constexpr (P == kExact) {
    double acc = __builtin_fma(M4A0, (double)s0, (double)(A1 * r1));  // M4A0 * s0 is exact
    acc = acc + (double)(A2 * r2);
    acc = acc + (double)(A3 * r3);
    acc = acc + (double)(A4 * r4);
    acc = acc + (double)(A5 * r5);
    return (float)acc;
  } else {
    float acc = (-4.0f * A0) * s0;
    acc = __builtin_fmaf(A1, r1, acc);
    acc = __builtin_fmaf(A2, r2, acc);
    acc = __builtin_fmaf(A3, r3, acc);
    acc = __builtin_fmaf(A4, r4, acc);
    acc = __builtin_fmaf(A5, r5, acc);
    return acc;
  }
}

// The damped update's coefficients of cur and prev for a damping delta.
template <int P>
struct Damp {
  using A = typename std::conditional<P == kExact, double, float>::type;
  A a;
  float b;
};
template <int P>
__device__ __forceinline__ Damp<P> damp_coeffs(float delta) {
  Damp<P> d;
  if constexpr (P == kExact)
    d.a = (2. - (double)(2 * delta)) + (double)(delta * delta);
  else
    d.a = (2.0f - 2 * delta) + delta * delta;
  d.b = 1 - 2 * delta;
  return d;
}

// The 4th-order-in-time coefficient of the point.
__device__ __forceinline__ float cc_of(float rv) { return (C12 * rv) * rv; }

// The 5-point Laplacian of u2 at a point of value u0, from its z (zm, zp) and
// x (xm, xp) neighbours.  4 * u0 is exact, so fused or not gives the same
// bits; in FP32 the fused form makes the forward tiles 1% slower (11 entries
// of 301x201, 16 wide: 5.89 us a step against 5.82).
template <int P>
__device__ __forceinline__ float lap_of(float u0, float zm, float zp, float xm, float xp) {
  const float lap = ((zm + zp) + xm) + xp;
  if constexpr (P == kExact) return __builtin_fmaf(-4.0f, u0, lap);
  return lap - 4 * u0;
}

// next from cur c, prev p, reciprocal model rv, cc = cc_of(rv), u2 at the
// point u0 and its Laplacian lap, and the damping coefficients (ignored when
// !DAMPED).
template <bool DAMPED, int P>
__device__ __forceinline__ float update_lap(float c, float p, float rv, float cc, float u0, float lap,
                                            const Damp<P>& d) {
  if constexpr (P == kExact) {
    double acc;
    if constexpr (DAMPED) {
      acc = d.a * (double)c;
      acc = acc - (double)(d.b * p);
    } else {
      acc = __builtin_fma(2., (double)c, -(double)p);  // 2 * c is exact
    }
    acc = acc + (double)(rv * u0);
    acc = acc + (double)(cc * lap);
    return (float)acc;
  } else {
    float acc;
    if constexpr (DAMPED)
      acc = __builtin_fmaf(d.a, c, -(d.b * p));
    else
      acc = __builtin_fmaf(2.0f, c, -(1.0f * p));
    acc = __builtin_fmaf(rv, u0, acc);
    return __builtin_fmaf(cc, lap, acc);
  }
}
template <bool DAMPED, int P>
__device__ __forceinline__ float update_coeffs(float c, float p, float rv, float cc, float u0, float zm, float zp,
                                               float xm, float xp, const Damp<P>& d) {
  return update_lap<DAMPED, P>(c, p, rv, cc, u0, lap_of<P>(u0, zm, zp, xm, xp), d);
}

}  // namespace swfwi
