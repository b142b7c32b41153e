// ostc_weno.hpp -- the WENO face reconstructions of every scheme, air and
// mixtures, and the reciprocal and square root that they and the flux
// splitting use.
//
// These evaluations fill most of the inviscid kernels' FP64 issue slots, so
// they are written for the instruction count: an IEEE division costs 11
// instructions, and the textbook form of one side of WENO-Z5 has four of them
// and 75 other operations.  Here a side is formed from the differences of its
// points.  With second differences s_k, the indicators times 4 are
// 13/3 s^2 + t^2 (t = 4 x the first derivative's weight, a combination of two
// first differences), and the face value is the upwind cell's value plus the
// central candidate's offset plus the weighted offsets of the other candidates
// from the central one, which are multiples of differences of the s_k:
//
//   f = f2 + [b + 2c + (3 G0 (s1 - s0) - 2 G2 (s1 - s2)) / (3 G0 + 6 G1 + G2)] / 6
//
// The weights are those of the reference (src/WENO.cu:1582-1693) up to the
// common factor; they multiply only the small offsets, so their rounding does
// not reach the leading digits, and the differences of neighbouring points are
// exact or nearly so.  49 operations and four reciprocals a side, a reciprocal
// being one estimate and three FMAs.
// By itself, in the tile kernels that then did every scheme: a step of 24 air
// blocks (12.5 M nodes, WENO-Z5) 16.25 -> 14.42 ms, WENO-Z7 on 101x75x49 nodes
// 688 -> 603 us, characteristic 1.91 -> 1.78 ms, a reacting 256x128x64 block
// 20.3 -> 19.5 ms.  The error of a step against 64-bit whole-array arithmetic
// in another order (mean of 6 seeds) is no larger: w on 16^3 nodes 6.85e-15 ->
// 6.52e-15, on 64^3 (WENO5-JS) 5.38e-15 -> 5.04e-15, v on 101x75x49 (WENO-Z7)
// 4.31e-14 -> 4.31e-14.
#pragma once
#include <hip/hip_runtime.h>

namespace ostc {

// 1 / x for normal x whose reciprocal is normal: the hardware's estimate
// (relative error measured 2^-24.4) and one cubic step.  Measured over
// 2^+-300: within 1.0 * 2^-53 of the exact value, as a correctly rounded
// quotient is.  A zero or infinite x gives NaN: only for operands that are
// neither, or whose result is NaN by the divisions of the textbook form as
// well (the smoothness indicators: eps and squares of flux differences, zero
// only where eps is, infinite only beyond differences of 10^153).
__device__ __forceinline__ double rcp64_normal(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// The same with the result of a division for a zero, infinite or NaN x (one
// instruction more).
__device__ __forceinline__ double rcp64(double x) { return __builtin_amdgcn_div_fixup(rcp64_normal(x), x, 1.0); }

// sqrt(x) for x that is no subnormal number: estimate (2^-24.2), one coupled
// step for the root and half its reciprocal, one residual correction; 0 and
// infinity are their own roots.  Measured over 2^+-300: within 1.0 * 2^-53 of
// the exact value.
__device__ __forceinline__ double sqrt64(double x) {
  constexpr int zero_or_inf = 0x020 | 0x040 | 0x200;  // -0, +0, +infinity
  const double s = __builtin_amdgcn_rsq(x);
  const double h = x * s, g = 0.5 * s;
  const double d = __builtin_fma(-h, g, 0.5);
  const double h1 = __builtin_fma(h, d, h), g1 = __builtin_fma(g, d, g);
  const double root = __builtin_fma(__builtin_fma(-h1, h1, x), g1, h1);
  return __builtin_amdgcn_class(x, zero_or_inf) ? x : root;
}

// n / d as an IEEE division rounds it, for d and quotient that are no
// subnormal numbers: the compiler's own sequence for a division without its
// scaling and condition-code steps (estimate, two Newton steps, quotient and
// one correction, fix-up of zeros, infinities and NaN).
__device__ __forceinline__ double div64(double n, double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, q, n), r, q), d, n);
}

// n / d of a finite n with r the correctly rounded 1 / d of a normal d at hand:
// correctly rounded (Markstein 1990) in three instructions.
__device__ __forceinline__ double div64(double n, double d, double r) {
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// One side of WENO-Z5 (Z) or WENO5-JS from five points, upwind first, in the
// form above: the face value is f2 + the return value / 6.  eps4 = 4 eps.
template <bool Z>
__device__ __forceinline__ double weno5_side(double f0, double f1, double f2, double f3, double f4, double eps4) {
  constexpr double c133{13.0 / 3.0};
  const double a = f1 - f0, b = f2 - f1, c = f3 - f2, d = f4 - f3;
  const double s2 = b - a, s1 = c - b, s0 = d - c;
  const double t2 = __builtin_fma(3.0, b, -a), t1 = b + c, t0 = __builtin_fma(-3.0, c, d);
  const double b0 = __builtin_fma(t0, t0, __builtin_fma(c133 * s0, s0, eps4));
  const double b1 = __builtin_fma(t1, t1, __builtin_fma(c133 * s1, s1, eps4));
  const double b2 = __builtin_fma(t2, t2, __builtin_fma(c133 * s2, s2, eps4));
  double g0 = rcp64_normal(b0), g1 = rcp64_normal(b1), g2 = rcp64_normal(b2);
  if constexpr (Z) {  // 1 + (tau / (eps + beta))^2
    const double tau = b0 - b2;
    g0 *= tau;
    g1 *= tau;
    g2 *= tau;
    g0 = __builtin_fma(g0, g0, 1.0);
    g1 = __builtin_fma(g1, g1, 1.0);
    g2 = __builtin_fma(g2, g2, 1.0);
  } else {  // 1 / (eps + beta)^2
    g0 *= g0;
    g1 *= g1;
    g2 *= g2;
  }
  const double a0 = 3.0 * g0;
  const double num = __builtin_fma(a0, s1 - s0, -2.0 * (g2 * (s1 - s2)));
  const double sum = __builtin_fma(6.0, g1, a0 + g2);
  return __builtin_fma(num, rcp64_normal(sum), __builtin_fma(2.0, c, b));
}

// One side of WENO-Z7 from seven points, upwind first: the face value is
// f3 + the return value / 12.  eps36 = 36 eps.  With second differences q_k,
// third differences r_k and fourth differences p_k, 36 beta_k =
// S (S + r / 2) + 39 s^2 + 1043/960 36 r^2 with S = 6 s1 of the reference,
// and the candidates' offsets from the second one are -3 p0, -p1 and p2 - p1.
__device__ __forceinline__ double weno7_side(double f0, double f1, double f2, double f3, double f4, double f5,
                                             double f6, double eps36) {
  constexpr double c3{1043.0 / 960 * 36};
  const double d0 = f1 - f0, d1 = f2 - f1, d2 = f3 - f2, d3 = f4 - f3, d4 = f5 - f4, d5 = f6 - f5;
  const double q0 = d1 - d0, q1 = d2 - d1, q2 = d3 - d2, q3 = d4 - d3, q4 = d5 - d4;
  const double r0 = q1 - q0, r1 = q2 - q1, r2 = q3 - q2, r3 = q4 - q3;
  auto beta = [&](double S, double s, double r) {
    const double tail = __builtin_fma(c3 * r, r, __builtin_fma(39.0 * s, s, eps36));
    return __builtin_fma(S, __builtin_fma(0.5, r, S), tail);
  };
  const double b0 = beta(__builtin_fma(6.0, d2, __builtin_fma(3.0, q1, 2.0 * r0)), q1 + r0, r0);
  const double b1 = beta(__builtin_fma(6.0, d2, __builtin_fma(2.0, q2, q1)), q2, r1);
  const double b2 = beta(__builtin_fma(6.0, d3, -__builtin_fma(2.0, q2, q3)), q2, r2);
  const double b3 = beta(__builtin_fma(6.0, d3, __builtin_fma(-5.0, q3, 2.0 * q4)), __builtin_fma(2.0, q3, -q4), r3);
  const double tau = b0 - b3;
  double g0 = tau * rcp64_normal(b0), g1 = tau * rcp64_normal(b1), g2 = tau * rcp64_normal(b2), g3 = tau * rcp64_normal(b3);
  g0 = __builtin_fma(g0, g0, 1.0);
  g1 = __builtin_fma(g1, g1, 1.0);
  g2 = __builtin_fma(g2, g2, 1.0);
  g3 = __builtin_fma(g3, g3, 1.0);
  const double p0 = r1 - r0, p1 = r2 - r1, p2 = r3 - r2;
  const double a2 = 18.0 * g2, a3 = 4.0 * g3;
  const double num = __builtin_fma(-3.0 * g0, p0, __builtin_fma(-a2, p1, a3 * (p2 - p1)));
  const double sum = __builtin_fma(12.0, g1, g0 + a2) + a3;
  const double base = __builtin_fma(6.0, d2, __builtin_fma(4.0, q1, 3.0 * r1));
  return __builtin_fma(num, rcp64_normal(sum), base);
}

// Face value of F+ plus face value of F-.  5-point schemes: vp = F+ at
// i-2..i+2, vm = F- at i-1..i+3 (the reference's WENO5, src/WENO.cu:1582-1617;
// WENO5-JS has no counterpart there, scheme 50 here); WENO-Z7: vp at
// i-3..i+3, vm at i-2..i+4 (src/WENO.cu:1619-1693).
__device__ __forceinline__ double weno5z(const double* vp, const double* vm, double eps) {
  const double e = 4.0 * eps;
  const double c = weno5_side<true>(vp[0], vp[1], vp[2], vp[3], vp[4], e) +
                   weno5_side<true>(vm[4], vm[3], vm[2], vm[1], vm[0], e);
  return __builtin_fma(1.0 / 6, c, vp[2] + vm[2]);
}

__device__ __forceinline__ double weno5js(const double* vp, const double* vm, double eps) {
  const double e = 4.0 * eps;
  const double c = weno5_side<false>(vp[0], vp[1], vp[2], vp[3], vp[4], e) +
                   weno5_side<false>(vm[4], vm[3], vm[2], vm[1], vm[0], e);
  return __builtin_fma(1.0 / 6, c, vp[2] + vm[2]);
}

__device__ __forceinline__ double weno7z(const double* vp, const double* vm, double eps) {
  const double e = 36.0 * eps;
  const double c = weno7_side(vp[0], vp[1], vp[2], vp[3], vp[4], vp[5], vp[6], e) +
                   weno7_side(vm[6], vm[5], vm[4], vm[3], vm[2], vm[1], vm[0], e);
  return __builtin_fma(1.0 / 12, c, vp[3] + vm[3]);
}

}  // namespace ostc
