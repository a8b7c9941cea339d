// spss_pairs64.hpp -- the pair sums of the FP64 kernels through the neighbours' phasors.
//
// The reference adds sin(phi_j - phi_i - alpha) pair by pair.  With psi = phi - phi_ref for one
// reference phase phi_ref per group of particles,
//   sum sin(phi_j - phi_i - alpha) = cos(alpha) (c_i S - s_i C) - sin(alpha) (c_i C + s_i S),
//   S = sum sin psi_j, C = sum cos psi_j,
// so a pair costs two additions and the trigonometry is paid once per particle.  phi - phi_ref
// rounds like phi_j - phi_i does, and near synchrony (all psi small) S, s_i and every rounding
// error scale with the spread of the phases, so the sums keep the relative accuracy of the direct
// form there as well.  The complementary force's sum of (omega_j - omega_i) cos(phi_j - phi_i -
// alpha) goes through the sums of (omega_j - omega_i) sin psi_j and (omega_j - omega_i) cos psi_j: the differences
// are taken pair by pair (an operation of some twenty), since no frame's omega would do for all, where one is
// far off the others.
//
// Neighbour sets are the reference's bit for bit: the cheap distance test decides only outside a
// guard band around rho^2 that covers its rounding, pairs inside it go through the reference's own
// expressions on the stored positions (pair_in_range).
#pragma once

#include <math.h>

#include "spss_device.hpp"

namespace spss {

// sums over the neighbours of one particle, in the frame of the reference phase
struct PhasorSums {
  double S = 0.0, C = 0.0, card = 0.0;
  double TS = 0.0, TC = 0.0;  // of omega_j - omega_i times the phasors
};

// sin and cos of x + e for |x| <= 2^30 and a correction |e| <= 2^-22: reduction to |r| <= pi/4 by
// multiples of pi/2 (pi/2 in two parts, Cody and Waite, Software Manual for the Elementary Functions;
// the first difference is exact, the multiples' low bits are 2^-52; the second part and the correction go into r
// together, which leaves 2^-54 for what r lacks: that much may be taken to first order), then the Taylor
// polynomials to r^17 and r^16, whose next terms are below 2^-60.  Branch-free and about a fifth of the instructions of the general sincos.
__device__ __forceinline__ void small_sincos(double x, double e, double &sn, double &cs) {
  const double k = rint(x * 0x1.45f306dc9c883p-1);  // 2 / pi
  const double r0 = __builtin_fma(-k, 0x1.921fb54442d18p+0, x);
  const double t = __builtin_fma(-k, 0x1.1a62633145c07p-54, e);
  const double r = r0 + t;
  e = (r0 - r) + t;  // what r lacks
  const double z = r * r;
  double p = __builtin_fma(z, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
  p = __builtin_fma(z, p, 1.0 / 6227020800.0);
  p = __builtin_fma(z, p, -1.0 / 39916800.0);
  p = __builtin_fma(z, p, 1.0 / 362880.0);
  p = __builtin_fma(z, p, -1.0 / 5040.0);
  p = __builtin_fma(z, p, 1.0 / 120.0);
  p = __builtin_fma(z, p, -1.0 / 6.0);
  const double h = 0.5 * z, w = 1.0 - h;
  const double s = r + __builtin_fma(r * z, p, __builtin_fma(-h, e, e));
  double q = __builtin_fma(z, 1.0 / 20922789888000.0, -1.0 / 87178291200.0);
  q = __builtin_fma(z, q, 1.0 / 479001600.0);
  q = __builtin_fma(z, q, -1.0 / 3628800.0);
  q = __builtin_fma(z, q, 1.0 / 40320.0);
  q = __builtin_fma(z, q, -1.0 / 720.0);
  q = __builtin_fma(z, q, 1.0 / 24.0);
  // 1 - z/2 + z^2 q with the rounding of 1 - z/2 put back
  const double c = w + __builtin_fma(-e, r, __builtin_fma(z * z, q, (1.0 - w) - h));
  const int n = (int)k;
  const double a = (n & 1) ? c : s, b = (n & 1) ? s : c;
  sn = (n & 2) ? -a : a;
  cs = ((n + 1) & 2) ? -b : b;
}

// sin and cos of any phase
__device__ __forceinline__ void phasor_of(double phi, double &sn, double &cs) {
  if (fabs(phi) <= 0x1p30)
    small_sincos(phi, 0.0, sn, cs);
  else
    sincos(phi, &sn, &cs);
}

// a - b and its rounding error
__device__ __forceinline__ double two_diff(double a, double b, double &err) {
  const double d = a - b, c = d - a;
  err = (a - (d - c)) - (b + c);
  return d;
}

// sin, cos of phi - ref; the difference's rounding error (up to 2^-51 for phases a turn apart) is
// carried along, which keeps the phasors within an ulp of those of the exact difference
// (phases and references up to kPhase64)
constexpr double kPhase64 = 0x1p29;
__device__ __forceinline__ void frame_phasor(double phi, double ref, double &sn, double &cs) {
  double err;
  const double d = two_diff(phi, ref, err);
  small_sincos(d, err, sn, cs);
}

// the same for any phase
__device__ __forceinline__ void frame_phasor_any(double phi, double ref, double &sn, double &cs) {
  double err;
  const double d = two_diff(phi, ref, err);
  if (fabs(d) <= 0x1p30) {
    small_sincos(d, err, sn, cs);
  } else {
    double s, c, se, ce;  // the error is of order one from 2^53 on
    sincos(d, &s, &c);
    sincos(err, &se, &ce);
    sn = __builtin_fma(se, c, ce * s);
    cs = __builtin_fma(-se, s, ce * c);
  }
}

// a reference phase: any value of an ordinary size serves
__device__ __forceinline__ double frame_ref(double v) { return fabs(v) <= kPhase64 ? v : 0.0; }

// |t| of a pair below which its distance test goes to pair_in_range.  Coordinates up to
// kFar64 boxes from the origin, wrapped and shifted, put |dx| off by at most ~2^-40 of the box;
// t = d^2 - rho^2 by 2 rho times that, and the rounding of t itself is far below rho^2 2^-30.
constexpr double kFar64 = 4096.0;
inline double pair_band(double rho2, double xs, double ys) {
  return rho2 * 0x1p-30 + sqrt(rho2) * (xs > ys ? xs : ys) * 0x1p-33;
}

// the weight of a pair at t = d^2 - rho^2: 1 within the radius, 0 beyond it (and for NaN), one VALU
// operation with the output clamp.  -slope is a power of two with slope * band > 2, so it is exact
// outside the guard band.
__device__ __forceinline__ double pair_weight(double t, double neg_slope) { return fmin(fmax(t * neg_slope, 0.0), 1.0); }
inline double pair_neg_slope(double band) { return -ldexp(1.0, ilogb(2.0 / band) + 1); }

// the reference's own distance test: models 3 and 4 ClassC on the wrapped x_i and stored x_j
// (ParticleSystemFirstOrderPtr.cpp:285-289), model 6 ClassA (ParticleSystemSecondOrderPtr.cpp:208-212)
template <int S>
__device__ __forceinline__ bool pair_in_range(const DevParams &P, double x_i, double y_i, double x_j, double y_j) {
  double dx, dy;
  if (S == 6)
    class_a(P, x_i, y_i, x_j, y_j, dx, dy);
  else
    class_c_unsigned(P, x_i, y_i, x_j, y_j, dx, dy);
  return dx * dx + dy * dy <= P.rho2;
}

// a b - c d, the rounding of c d put back
__device__ __forceinline__ double cross(double a, double b, double c, double d) {
  const double p = c * d;
  return __builtin_fma(a, b, -p) - __builtin_fma(c, d, -p);
}

// the coupling sums of the reference (PairAcc) from the phasor sums: s_i, c_i the particle's own
// phasor
template <int S>
__device__ __forceinline__ PairAcc pair_acc(const DevParams &P, const PhasorSums &q, double s_i, double c_i) {
  PairAcc a{0.0, 0.0, 0.0};
  if (q.card == 0.0) return a;
  // sums of sin, cos (phi_j - phi_i)
  const double sn = cross(c_i, q.S, s_i, q.C), cs = __builtin_fma(c_i, q.C, s_i * q.S);
  a.align = sn * P.cos_a - cs * P.sin_a;
  a.card = q.card;
  if (S == 4 && P.higher_order) {
    const double tsn = cross(c_i, q.TS, s_i, q.TC), tcs = __builtin_fma(c_i, q.TC, s_i * q.TS);
    a.compl_f = tcs * P.cos_a + tsn * P.sin_a;
  }
  return a;
}

}  // namespace spss
