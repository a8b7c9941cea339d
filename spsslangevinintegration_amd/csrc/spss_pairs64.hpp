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
// alpha) goes through sum omega' sin psi and sum omega' cos psi with omega' = omega - omega_ref.
//
// Neighbour sets are the reference's bit for bit: the cheap distance test decides only outside a
// guard band around rho^2 that covers its rounding, pairs inside it go through the reference's own
// expressions on the stored positions (pair_in_range).
#pragma once

#include "spss_device.hpp"

namespace spss {

// sums over the neighbours of one particle, in the frame of the reference phase
struct PhasorSums {
  double S = 0.0, C = 0.0, card = 0.0, TS = 0.0, TC = 0.0;
};

// a reference phase or phase velocity: any finite value serves
__device__ __forceinline__ double frame_ref(double v) { return fabs(v) < 1e300 ? v : 0.0; }

// |t| of a pair below which its distance test goes to pair_in_range.  Coordinates up to
// kFar64 boxes from the origin, wrapped and shifted, put |dx| off by at most ~2^-40 of the box;
// t = d^2 - rho^2 by 2 rho times that, and the rounding of t itself is far below rho^2 2^-30.
constexpr double kFar64 = 4096.0;
inline double pair_band(double rho2, double xs, double ys) {
  return rho2 * 0x1p-30 + sqrt(rho2) * (xs > ys ? xs : ys) * 0x1p-33;
}

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

// the coupling sums of the reference (PairAcc) from the phasor sums: psi_i, om_i relative to the
// frame's references
template <int S>
__device__ __forceinline__ PairAcc pair_acc(const DevParams &P, const PhasorSums &q, double psi_i, double om_i) {
  PairAcc a{0.0, 0.0, 0.0};
  if (q.card == 0.0) return a;
  double s_i, c_i;
  sincos(psi_i, &s_i, &c_i);
  const double sn = c_i * q.S - s_i * q.C, cs = c_i * q.C + s_i * q.S;  // sums of sin, cos (phi_j - phi_i)
  a.align = sn * P.cos_a - cs * P.sin_a;
  a.card = q.card;
  if (S == 4 && P.higher_order) {
    const double tsn = c_i * q.TS - s_i * q.TC, tcs = c_i * q.TC + s_i * q.TS;
    a.compl_f = (tcs - om_i * cs) * P.cos_a + (tsn - om_i * sn) * P.sin_a;
  }
  return a;
}

}  // namespace spss
