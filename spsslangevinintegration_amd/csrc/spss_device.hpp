// spss_device.hpp -- device-side building blocks shared by the HIP kernels.
//
// FP64 helpers restate the reference's expressions operation by operation;
// the library is compiled with -ffp-contract=off so each one rounds as the
// separate IEEE operation the reference performs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace spss {

constexpr int kBlock = 256;

// Scalars every RHS kernel needs, computed once on the host in FP64.
struct DevParams {
  int n;
  int s;
  double v0;
  double xi;       // model 4: xi; model 6: xi_phi
  double sigma;
  double rho2;     // rho * rho (ParticleSystemFirstOrderPtr.cpp:26)
  double alpha;
  double cos_a;    // std::cos(alpha) (ParticleSystemFirstOrderPtr.cpp:28)
  double sin_a;    // std::sin(alpha)
  double xi_r;     // model 6
  double xs, ys;   // PeriodicBoundaryConditions x_size_, y_size_
  double xrs, yrs; // 1.0 / x_size (the constructor, PeriodicBoundaryConditions.cpp:7-21)
  int natfreq_local;
  int higher_order;
  int fresh_k;     // the derivative starts from zero: entries the local branches leave alone are written as 0
};

// ---- periodic boundary conditions (BoundaryConfiguration/PeriodicBoundaryConditions.cpp)

// ClassCEffectiveParticleDistanceUnsigned, PeriodicBoundaryConditions.cpp:107-119
__device__ __forceinline__ void class_c_unsigned(const DevParams &P, double xi, double yi, double xj,
                                                 double yj, double &dx, double &dy) {
  dx = fabs(xj - xi);
  dx -= (double)((int)(dx * P.xrs + 0.5)) * P.xs;
  dy = fabs(yj - yi);
  dy -= (double)((int)(dy * P.yrs + 0.5)) * P.ys;
}

// ClassAEffectiveParticleDistance, PeriodicBoundaryConditions.cpp:26-38
__device__ __forceinline__ void class_a(const DevParams &P, double xi, double yi, double xj, double yj,
                                        double &dx, double &dy) {
  dx = xj - xi;
  dx -= (double)((int)(dx * 2.0 * P.xrs)) * P.xs;
  dy = yj - yi;
  dy -= (double)((int)(dy * 2.0 * P.yrs)) * P.ys;
}

// ApplyPeriodicBoundaryConditions(x, y, x_pbc, y_pbc), PeriodicBoundaryConditions.cpp:121-125
__device__ __forceinline__ void apply_pbc(const DevParams &P, double x, double y, double &xw, double &yw) {
  xw = x - floor(x * P.xrs) * P.xs;
  yw = y - floor(y * P.yrs) * P.ys;
}

// The wrap applied before cell keys: unconditional for models 3/4
// (ParticleSystemFirstOrderPtr.cpp:374), only outside the box for model 6
// (ParticleSystemSecondOrderPtr.cpp:292-295).
template <int S>
__device__ __forceinline__ void key_wrap(const DevParams &P, double x, double y, double &xw, double &yw) {
  if (S == 6) {
    if (x < 0.0 || x >= 1.0 || y < 0.0 || y >= 1.0) {
      apply_pbc(P, x, y, xw, yw);
    } else {
      xw = x;
      yw = y;
    }
  } else {
    apply_pbc(P, x, y, xw, yw);
  }
}

// int(x / x_size_ * nc) with x_size_ = 1.0 (ParticleSystemFirstOrderPtr.cpp:377-379).  The
// reference leaves x - floor(x) == 1.0 (tiny negative x) unguarded; clamp to the last cell.
__device__ __forceinline__ int cell_coord(double xw, int nc) {
  int c = (int)(xw / 1.0 * (double)nc);
  c = c < 0 ? 0 : c;
  return c >= nc ? nc - 1 : c;
}

// AdjustNeighboringCellToPeriodicBoundaries, ParticleSystemFirstOrderPtr.cpp:817-834
__device__ __forceinline__ int adjust_cell(int c, int nc) { return c < 0 ? nc - 1 : (c >= nc ? 0 : c); }

template <int S>
struct Slots {
  static constexpr int phi = (S == 6) ? 4 : 2;
  static constexpr int omega = (S == 6) ? 5 : 3;
};

// ---- pair term of every local branch
// model 4/3: ParticleSystemFirstOrderPtr.cpp:285-299; model 6: ParticleSystemSecondOrderPtr.cpp:208-215
struct PairAcc {
  double align;
  double card;
  double compl_f;
};

template <int S>
__device__ __forceinline__ void pair_term(const DevParams &P, double x_i, double y_i, double phi_i,
                                          double omega_i, double x_j, double y_j, double phi_j,
                                          double omega_j, PairAcc &a) {
  double dx, dy;
  if (S == 6)
    class_a(P, x_i, y_i, x_j, y_j, dx, dy);
  else
    class_c_unsigned(P, x_i, y_i, x_j, y_j, dx, dy);
  double dr2 = dx * dx + dy * dy;
  if (dr2 <= P.rho2) {
    if (S == 6) {
      a.align += sin(phi_j - phi_i - P.alpha);
      a.card += 1.0;
    } else {
      a.align += sin(phi_j - phi_i) * P.cos_a - cos(phi_j - phi_i) * P.sin_a;
      a.card += 1.0;
      if (S == 4 && P.higher_order) {
        a.compl_f += (omega_j - omega_i) * (cos(phi_j - phi_i) * P.cos_a + sin(phi_j - phi_i) * P.sin_a);
      }
    }
  }
}

// ---- output row of the local branches
// model 4: ParticleSystemFirstOrderPtr.cpp:303-313; model 6: ParticleSystemSecondOrderPtr.cpp:219-227;
// model 3 (m = 0): k = (v0 cos phi, v0 sin phi, w_i + sigma A / n)
// (sin_i, cos_i: of the particle's phase)
template <int S>
__device__ __forceinline__ void write_k(const DevParams &P, const double *st, int i, const PairAcc &a,
                                        double nat_i, double sin_i, double cos_i, double *k_next,
                                        double *compl_out) {
  const long ii = (long)i * S;
  if (S == 4) {
    const double omega_i = st[3];
    k_next[ii] = P.v0 * cos_i;
    k_next[ii + 1] = P.v0 * sin_i;
    k_next[ii + 2] = omega_i;
    if (P.natfreq_local) {
      if (a.card != 0.0)
        k_next[ii + 3] = -P.xi * omega_i + nat_i + P.sigma * a.align / a.card;
      else
        k_next[ii + 3] = -P.xi * omega_i + nat_i;
    } else if (a.card != 0.0) {
      k_next[ii + 3] = -P.xi * omega_i + P.sigma * a.align / a.card;
    } else if (P.fresh_k) {
      k_next[ii + 3] = 0.0;
    }
    if (P.higher_order && compl_out) {
      double c = a.compl_f;
      if (a.card != 0.0) c *= P.sigma / a.card;
      compl_out[i] = c;
    }
  } else if (S == 6) {
    const double vx = st[2], vy = st[3], omega_i = st[5];
    k_next[ii] = vx;
    k_next[ii + 1] = vy;
    k_next[ii + 2] = -P.xi_r * vx + P.v0 * cos_i;
    k_next[ii + 3] = -P.xi_r * vy + P.v0 * sin_i;
    k_next[ii + 4] = omega_i;
    if (a.card != 0.0)
      k_next[ii + 5] = -P.xi * omega_i + P.sigma * a.align / a.card;
    else if (P.fresh_k)
      k_next[ii + 5] = 0.0;
  } else {
    k_next[ii] = P.v0 * cos_i;
    k_next[ii + 1] = P.v0 * sin_i;
    if (a.card != 0.0)
      k_next[ii + 2] = nat_i + P.sigma * a.align / a.card;
    else
      k_next[ii + 2] = nat_i;
  }
}

template <int S>
__device__ __forceinline__ void write_k(const DevParams &P, const double *st, int i, const PairAcc &a,
                                        double nat_i, double *k_next, double *compl_out) {
  write_k<S>(P, st, i, a, nat_i, sin(st[Slots<S>::phi]), cos(st[Slots<S>::phi]), k_next, compl_out);
}

// ---- counter-based RNG: Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) written from the
// published round function: two 32x32->64 multiplies per round, Weyl key schedule.
struct U4 {
  uint32_t x, y, z, w;
};

__host__ __device__ __forceinline__ U4 philox4x32_10(U4 c, uint32_t k0, uint32_t k1) {
  const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
  const uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    uint64_t p0 = (uint64_t)M0 * c.x;
    uint64_t p1 = (uint64_t)M1 * c.z;
    U4 n;
    n.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
    n.y = (uint32_t)p1;
    n.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
    n.w = (uint32_t)p0;
    c = n;
    k0 += W0;
    k1 += W1;
  }
  return c;
}

// ln u for u in (0, 1], a normal number: u = 2^e m with m in [sqrt(1/2), sqrt(2)), ln m = 2 artanh(s) with
// s = (m - 1) / (m + 1) and what s lacks, by the Taylor series to s^21 (|s| < 0.172: the next term is
// below 2^-55 of the sum), ln 2 in two parts.  Within 0.55 ulp, and about 40 instructions where the
// general logarithm takes a hundred.
__device__ __forceinline__ double log_unit(double u) {
  double m = __builtin_amdgcn_frexp_mant(u);
  int e = __builtin_amdgcn_frexp_exp(u);
  if (m < 0x1.6a09e667f3bcdp-1) {
    m += m;
    --e;
  }
  const double r = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);
  double y = __builtin_amdgcn_rcp(d);
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  const double s = r * y, sl = __builtin_fma(-s, dl, __builtin_fma(-d, s, r)) * y, z = s * s;
  double p = __builtin_fma(z, 1.0 / 21.0, 1.0 / 19.0);
  p = __builtin_fma(z, p, 1.0 / 17.0);
  p = __builtin_fma(z, p, 1.0 / 15.0);
  p = __builtin_fma(z, p, 1.0 / 13.0);
  p = __builtin_fma(z, p, 1.0 / 11.0);
  p = __builtin_fma(z, p, 1.0 / 9.0);
  p = __builtin_fma(z, p, 1.0 / 7.0);
  p = __builtin_fma(z, p, 1.0 / 5.0);
  p = __builtin_fma(z, p, 1.0 / 3.0);
  const double a = (double)e * 0x1.62e42fefa38p-1, b = s + s, h = a + b, l = b - (h - a);
  return h + (l + __builtin_fma(b * z, p, __builtin_fma((double)e, 0x1.ef35793c7673p-45, sl + sl)));
}

// n / d and the remainder for 0 <= n < 2^31, d > 0, quotients below 2^22: FP32, off by one at most, put right
__device__ __forceinline__ int div_small(int n, int d, int &rem) {
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)d));
  int r = n - q * d;
  if (r < 0) {
    --q;
    r += d;
  } else if (r >= d) {
    ++q;
    r -= d;
  }
  rem = r;
  return q;
}

// two FP64 standard normals from one Philox block: 53-bit uniforms u1 in (0,1], u2 in [0,1),
// Box-Muller (r = sqrt(-2 ln u1), angle 2 pi u2)
__device__ __forceinline__ void philox_normal2(uint64_t seed, uint32_t particle, uint32_t block,
                                               uint64_t step, double &z0, double &z1) {
  U4 c{particle, block, (uint32_t)step, (uint32_t)(step >> 32)};
  U4 r = philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  uint64_t a = ((uint64_t)r.x << 21) ^ (uint64_t)(r.y >> 11);
  uint64_t b = ((uint64_t)r.z << 21) ^ (uint64_t)(r.w >> 11);
  const double inv53 = 1.0 / 9007199254740992.0;
  double u1 = ((double)(a & ((1ull << 53) - 1)) + 1.0) * inv53;
  double u2 = (double)(b & ((1ull << 53) - 1)) * inv53;
  double rad = sqrt(-2.0 * log_unit(u1));
  double sn, cs;
  sincospi(2.0 * u2, &sn, &cs);
  z0 = rad * cs;
  z1 = rad * sn;
}

}  // namespace spss
