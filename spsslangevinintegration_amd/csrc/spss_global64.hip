// spss_global64.hip -- the FP64 global polar order field, ParticleSystemFirstOrderPtr.cpp:155-223:
// right-hand side, the three steppers and the stages of the Dormand-Prince integrator on it.
//
// An evaluation needs Z = <e^{i phi}> (and W = <omega e^{i phi}> for the complementary force) of its
// stage state before any particle's derivative.  So a launch takes the block sums that the launch
// before it left, forms Z, evaluates its particles, and, since a stage state is known where its
// derivative is, goes on to the next stage state and leaves that one's block sums: one launch per
// stage, no stage pass, no launch for the reduction.  A small system stays in the registers of one
// workgroup for whole steps.
//
// What bounds it: small systems the chain phasor - sums - derivative (n = 1,000: 1.2 us per stage; a
// Runge-Kutta step took 55 us in 17 launches and takes 4.7), systems up to about 100,000 the latency of a
// launch (4 us; a step of 16,384: 56 -> 17 us), large ones memory: a Dormand-Prince trial of 1,048,576 470 ->
// 214 us, an Euler step 75 -> 25 us.
//
// |Z| sin(arg Z - phi) is Im(Z e^{-i phi}): no arc tangent, no second pair of sine and cosine.
#pragma clang fp contract(off)

#include "spss_launch.hpp"
#include "spss_pairs64.hpp"

namespace spss {

namespace {

constexpr int kMaxBlocks = 1024;  // every workgroup reads the sums of all of them

__device__ __forceinline__ void two_sum(double a, double b, double &s, double &e) {
  s = a + b;
  const double bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

// x of the lane that a DPP control names, 0 where there is none
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp(double x) {
  union { double d; int w[2]; } u, v;
  u.d = x;
  v.w[0] = __builtin_amdgcn_update_dpp(0, u.w[0], CTRL, ROWS, 0xf, false);
  v.w[1] = __builtin_amdgcn_update_dpp(0, u.w[1], CTRL, ROWS, 0xf, false);
  return v.d;
}

// sum over a wave in a fixed tree of register moves (row shifts, then row broadcasts); in lane 63
__device__ __forceinline__ double wave_sum63(double x) {
  x += dpp<0x111, 0xf>(x);  // row_shr:1
  x += dpp<0x112, 0xf>(x);
  x += dpp<0x114, 0xf>(x);
  x += dpp<0x118, 0xf>(x);
  x += dpp<0x142, 0xa>(x);  // row_bcast:15
  x += dpp<0x143, 0xc>(x);  // row_bcast:31
  return x;
}

template <int CTRL>
__device__ __forceinline__ void pair_level(double &s, double &c) {
  const double s2 = dpp<CTRL, 0xf>(s), c2 = dpp<CTRL, 0xf>(c);
  double t, e;
  two_sum(s, s2, t, e);
  s = t;
  c = c + c2 + e;
}

// sum of the compensated pairs (s, c) of lanes 0..15, for every lane
__device__ __forceinline__ double row_total(double s, double c) {
  pair_level<0x111>(s, c);
  pair_level<0x112>(s, c);
  pair_level<0x114>(s, c);
  pair_level<0x118>(s, c);
  union { double d; int w[2]; } u;
  u.d = s + c;
  u.w[0] = __builtin_amdgcn_readlane(u.w[0], 15);
  u.w[1] = __builtin_amdgcn_readlane(u.w[1], 15);
  return u.d;
}

// the field as its users need it
struct Field {
  double zx, zy, wx, wy, absz, ux, uy;  // Z, W, |Z|, W / |W|
};

template <bool HO>
__device__ __forceinline__ void finish_field(Field &f) {
  if (!HO) return;
  f.absz = hypot(f.zx, f.zy);
  const double w = hypot(f.wx, f.wy);
  f.ux = w > 0.0 ? f.wx / w : 1.0;  // arg(0) = 0
  f.uy = w > 0.0 ? f.wy / w : 0.0;
}

// the derivative of one particle of state st and phasor (c, s), and the complementary force (with
// arg(W) in its last sine, as the reference has it, :215-219)
template <int S, bool HO>
__device__ __forceinline__ void derivative(const DevParams &P, const Field &f, const double *st, double s, double c,
                                           double nat_i, double *k, double &compl_f) {
  const double A = f.zy * c - f.zx * s, B = f.zx * c + f.zy * s;  // |Z| sin, cos (arg Z - phi)
  const double force = P.sigma * (A * P.cos_a - B * P.sin_a);
  k[0] = P.v0 * c;
  k[1] = P.v0 * s;
  compl_f = 0.0;
  if (S == 4) {
    k[2] = st[3];
    k[3] = -P.xi * st[3] + nat_i + force;
    if (HO) {
      const double wc = f.wx * c + f.wy * s, ws = f.wy * c - f.wx * s;
      compl_f = P.sigma * ((wc * P.cos_a + ws * P.sin_a) -
                           st[3] * (B * P.cos_a + f.absz * (f.uy * c - f.ux * s) * P.sin_a));
    }
  } else {
    k[2] = nat_i + force;
  }
}

// the sums a stage state adds to: cos, sin, omega cos, omega sin
template <int S, bool HO>
__device__ __forceinline__ void field_terms(const double *st, double *v) {
  phasor_of(st[2], v[1], v[0]);
  if (HO) {
    v[2] = st[S - 1] * v[0];
    v[3] = st[S - 1] * v[1];
  }
}

// sums of one workgroup of 256 threads, a compensated pair per column, to out[column][2]
template <int COLS>
__device__ __forceinline__ void block_sums(const double *s, const double *c, double *__restrict__ out) {
  __shared__ double sh[4][COLS][2];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < COLS; ++q) {
    const double ws = wave_sum63(s[q]), wc = wave_sum63(c[q]);
    if (lane == 63) {
      sh[wv][q][0] = ws;
      sh[wv][q][1] = wc;
    }
  }
  __syncthreads();
  if (threadIdx.x < COLS) {
    double t = 0.0, e = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      double r, d;
      two_sum(t, sh[w][threadIdx.x][0], r, d);
      t = r;
      e += d + sh[w][threadIdx.x][1];
    }
    out[2 * threadIdx.x] = t;
    out[2 * threadIdx.x + 1] = e;
  }
}

// Z (and W) from the block sums of nb workgroups, by every workgroup for itself: a thread per block,
// then the compensated pairs in fixed trees.  COLS pairs per block.
template <bool HO>
__device__ __forceinline__ void field_of(const double *__restrict__ part, int nb, double n, Field &f) {
  constexpr int COLS = HO ? 4 : 2;
  __shared__ double fs[16][COLS][2];
  double s[COLS] = {}, c[COLS] = {};
  for (int b = threadIdx.x; b < nb; b += 256)
#pragma unroll
    for (int q = 0; q < COLS; ++q) {
      const double x = part[((long)b * COLS + q) * 2], y = part[((long)b * COLS + q) * 2 + 1];
      double t, e;
      two_sum(s[q], x, t, e);
      s[q] = t;
      c[q] += e + y;
    }
  // rows of 16 lanes first: lane 15 of each holds its pair
  const int row = threadIdx.x >> 4;
#pragma unroll
  for (int q = 0; q < COLS; ++q) {
    pair_level<0x111>(s[q], c[q]);
    pair_level<0x112>(s[q], c[q]);
    pair_level<0x114>(s[q], c[q]);
    pair_level<0x118>(s[q], c[q]);
    if ((threadIdx.x & 15) == 15) {
      fs[row][q][0] = s[q];
      fs[row][q][1] = c[q];
    }
  }
  __syncthreads();
  double v[COLS];
#pragma unroll
  for (int q = 0; q < COLS; ++q) v[q] = row_total(fs[threadIdx.x & 15][q][0], fs[threadIdx.x & 15][q][1]) / n;
  f.zx = v[0];
  f.zy = v[1];
  if (HO) {
    f.wx = v[COLS - 2];
    f.wy = v[COLS - 1];
  }
  finish_field<HO>(f);
}

template <int S>
__device__ __forceinline__ void load_row(const double *__restrict__ p, long i, double *v) {
#pragma unroll
  for (int q = 0; q < S; ++q) v[q] = p[i * S + q];
}
template <int S>
__device__ __forceinline__ void store_row(double *__restrict__ p, long i, const double *v) {
#pragma unroll
  for (int q = 0; q < S; ++q) p[i * S + q] = v[q];
}

// what a thread adds up over its particles, with the rounding errors
template <int COLS>
__device__ __forceinline__ void add_terms(const double *w, double *s, double *c) {
#pragma unroll
  for (int q = 0; q < COLS; ++q) {
    double t, e;
    two_sum(s[q], w[q], t, e);
    s[q] = t;
    c[q] += e;
  }
}

// the block sums of a first stage x + c0 * k0 (k0 may be null)
template <int S, bool HO, int PER>
__global__ __launch_bounds__(256) void gf_first(int n, const double *__restrict__ x, const double *__restrict__ k0,
                                                double c0, double *__restrict__ part) {
  constexpr int COLS = HO ? 4 : 2, kPart = 256 * PER;
  double s[COLS] = {}, c[COLS] = {};
  for (long b = (long)blockIdx.x * kPart; b < n; b += (long)gridDim.x * kPart) {
    double v[PER][S];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= n) continue;
      load_row<S>(x, i, v[p]);
      if (k0) {
        double k[S];
        load_row<S>(k0, i, k);
#pragma unroll
        for (int q = 0; q < S; ++q) v[p][q] = v[p][q] + c0 * k[q];
      }
    }
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= n) continue;
      double w[COLS];
      field_terms<S, HO>(v[p], w);
      add_terms<COLS>(w, s, c);
    }
  }
  block_sums<COLS>(s, c, part + (long)blockIdx.x * COLS * 2);
}

// what follows the derivative k of a particle
enum GfThen {
  kThenNothing,  // a right-hand side
  kThenNext,     // the next stage state base + c k, and its block sums
  kThenRk4,      // the step: state += (k1 + 2 k2 + 2 k3 + k) dt / 6, and its block sums
  kThenEuler,    // the stochastic steps (StochasticEulerStepperPtr.hpp:40-73,
  kThenSrk       // StochasticRungeKuttaStepperPtr.hpp:50-76) and the block sums of the new state
};

struct GfStep {
  const double *x = nullptr, *kprev = nullptr;  // stage state x + kc * kprev (kprev may be null)
  double kc = 0.0;
  const double *in = nullptr;  // its block sums
  int nb = 0;                  // from that many workgroups
  const double *nat = nullptr;
  double *k = nullptr, *compl_out = nullptr;  // the derivative, the complementary force (may be null)
  const double *base = nullptr;
  double c = 0.0;                  // the coefficient of k in the next stage state
  const double *k1 = nullptr, *k2 = nullptr, *k3 = nullptr;
  double *next = nullptr, *out = nullptr;  // the state written and its block sums
  GfNoise noise{};
  double dt = 0.0;
};

__device__ __forceinline__ double gf_draw(const GfNoise &z, long idx, uint32_t particle, int which) {
  if (z.mode == 1) return z.array[idx];
  if (z.mode != 3) return 0.0;
  double z0, z1;
  philox_normal2(z.seed, particle, 0, z.step, z0, z1);
  return which ? z1 : z0;
}

// the step of a stochastic stepper from the derivative f
template <int S, bool SRK>
__device__ __forceinline__ void stochastic_update(const GfNoise &z, double dt, int i, const double *f, double compl_f,
                                                  double *st) {
  if (!SRK) {
    const double dW = z.sqrt_dt * gf_draw(z, i, i, 0);
#pragma unroll
    for (int q = 0; q < S - 1; ++q) st[q] += f[q] * dt;
    st[S - 1] += f[S - 1] * dt + z.amp * dW;
  } else {
    double U1 = 0.0, U2 = 0.0;
    if (z.mode == 1) {
      U1 = z.array[2L * i];
      U2 = z.array[2L * i + 1];
    } else if (z.mode == 3) {
      philox_normal2(z.seed, (uint32_t)i, 0, z.step, U1, U2);
    }
    const double dW = U1 * z.sqrt_dt, dZ = z.c15 * (U1 + z.is3 * U2);
    const double t0 = f[0] * dt - 0.5 * f[2] * f[1] * dt * dt;
    const double t1 = f[1] * dt + 0.5 * f[2] * f[0] * dt * dt;
    const double t2 = f[2] * dt + 0.5 * f[S - 1] * dt * dt + z.amp * dZ;
    const double t3 = f[S - 1] * dt + 0.5 * (compl_f - z.friction * f[S - 1]) * dt * dt + z.amp * (dW - z.friction * dZ);
    st[0] += t0;
    st[1] += t1;
    st[2] += t2;
    st[S - 1] += t3;
  }
}

// PER: particles per thread and pass
template <int S, bool HO, int THEN, int PER>
__global__ __launch_bounds__(256) void gf_stage(DevParams P, GfStep G) {
  constexpr int COLS = HO ? 4 : 2, kPart = 256 * PER;
  constexpr bool kSums = THEN != kThenNothing;
  Field F{};
  double s[COLS] = {}, c[COLS] = {};
  for (long b = (long)blockIdx.x * kPart; b < P.n; b += (long)gridDim.x * kPart) {
    double st[PER][S];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= P.n) continue;
      load_row<S>(G.x, i, st[p]);
      if (G.kprev) {
        double kp[S];
        load_row<S>(G.kprev, i, kp);
#pragma unroll
        for (int q = 0; q < S; ++q) st[p][q] = st[p][q] + G.kc * kp[q];
      }
    }
    if (b == (long)blockIdx.x * kPart) field_of<HO>(G.in, G.nb, (double)P.n, F);  // over the first loads
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= P.n) continue;
      double v[S], d[3][S], k[S], cf;
      if (THEN == kThenNext || THEN == kThenRk4) load_row<S>(G.base, i, v);
      if (THEN == kThenRk4) {
        load_row<S>(G.k1, i, d[0]);
        load_row<S>(G.k2, i, d[1]);
        load_row<S>(G.k3, i, d[2]);
      }
      double sn, cs;
      phasor_of(st[p][2], sn, cs);
      derivative<S, HO>(P, F, st[p], sn, cs, G.nat ? G.nat[i] : 0.0, k, cf);
      if (G.k) store_row<S>(G.k, i, k);
      if (HO && G.compl_out) G.compl_out[i] = cf;
      if (THEN == kThenNext) {
#pragma unroll
        for (int q = 0; q < S; ++q) v[q] = v[q] + G.c * k[q];
      } else if (THEN == kThenRk4) {
#pragma unroll
        for (int q = 0; q < S; ++q) v[q] += (d[0][q] + 2.0 * d[1][q] + 2.0 * d[2][q] + k[q]) * G.dt / 6.0;
      } else if (THEN == kThenEuler || THEN == kThenSrk) {
#pragma unroll
        for (int q = 0; q < S; ++q) v[q] = st[p][q];
        stochastic_update<S, THEN == kThenSrk>(G.noise, G.dt, (int)i, k, cf, v);
      }
      if (kSums) {
        store_row<S>(G.next, i, v);
        double w[COLS];
        field_terms<S, HO>(v, w);
        add_terms<COLS>(w, s, c);
      }
    }
  }
  if (kSums) block_sums<COLS>(s, c, G.out + (long)blockIdx.x * COLS * 2);
}

// ---------------------------------------------------------------------------
// Dormand-Prince trials.  Positions take no part in the field, so the stages before the last need the
// phases (and omegas) of the state and of the derivatives alone: the derivatives are kept as two planes,
// A = {dphi/dt, domega/dt} and B = {dx/dt, dy/dt} behind it, the stages run on a copy of the state's phases
// and a plane of stage phases.  k2's positions enter nothing and are not kept.  A trial moves 1,040
// bytes per particle at 5.1 TB/s (1,440 with whole rows at 6.2): 1,048,576 particles 214 us, 240 with rows.

enum GpThen {
  kGpStart,  // the derivative at a whole state
  kGpNext,   // the derivative at stage phases; the next stage's phases and their block sums
  kGpOut,    // ... ; the new state and its block sums
  kGpError   // the derivative at the new state; per block the largest relative error
};

struct GpStep {
  const double *x = nullptr;   // the stage: a plane (kGpNext, kGpOut) or whole rows
  const double *in = nullptr;  // its block sums
  int nb = 0;
  const double *nat = nullptr;
  double *k = nullptr, *kb = nullptr;  // the derivative's planes (kb may be null)
  const double *base = nullptr;        // the state: its phases (kGpNext) or rows
  DpTerms T{};                         // earlier derivatives; T.c[T.n] is the coefficient of this one
  double *next = nullptr, *out = nullptr;
  double dt = 0.0, eps_abs = 0.0, eps_rel = 0.0;
};

template <int S, int THEN, int NT, int PER>
__global__ __launch_bounds__(256) void gp_stage(DevParams P, GpStep G) {
  constexpr int NA = S - 2, kPart = 256 * PER;
  constexpr bool kRows = THEN == kGpStart || THEN == kGpError, kWhole = THEN == kGpOut || THEN == kGpError;
  Field F{};
  double s[2] = {}, c[2] = {}, worst = 0.0;
  for (long b = (long)blockIdx.x * kPart; b < P.n; b += (long)gridDim.x * kPart) {
    double st[PER][4];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= P.n) continue;
#pragma unroll
      for (int q = 0; q < NA; ++q) st[p][2 + q] = kRows ? G.x[i * S + 2 + q] : G.x[i * NA + q];
    }
    if (b == (long)blockIdx.x * kPart) field_of<false>(G.in, G.nb, (double)P.n, F);  // over the first loads
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= P.n) continue;
      double v[S], d[NT ? NT : 1][S], k[S], cf, sn, cs;
      if (THEN == kGpNext) {
#pragma unroll
        for (int q = 0; q < NA; ++q) v[2 + q] = G.base[i * NA + q];
      } else if (kWhole) {
        load_row<S>(G.base, i, v);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const double *a = G.T.k[j], *xy = a + (long)P.n * NA;
#pragma unroll
        for (int q = 0; q < NA; ++q) d[j][2 + q] = a[i * NA + q];
        if (kWhole) {
          d[j][0] = xy[2 * i];
          d[j][1] = xy[2 * i + 1];
        }
      }
      phasor_of(st[p][2], sn, cs);
      derivative<S, false>(P, F, st[p], sn, cs, G.nat ? G.nat[i] : 0.0, k, cf);
#pragma unroll
      for (int q = 0; q < NA; ++q) G.k[i * NA + q] = k[2 + q];
      if (G.kb) {
        G.kb[2 * i] = k[0];
        G.kb[2 * i + 1] = k[1];
      }
      if (THEN == kGpNext || THEN == kGpOut) {
#pragma unroll
        for (int q = THEN == kGpOut ? 0 : 2; q < S; ++q) {
#pragma unroll
          for (int j = 0; j < NT; ++j) v[q] = v[q] + G.T.c[j] * d[j][q];
          v[q] = v[q] + G.T.c[NT] * k[q];
        }
        if (THEN == kGpOut) {
          store_row<S>(G.next, i, v);
        } else {
#pragma unroll
          for (int q = 0; q < NA; ++q) G.next[i * NA + q] = v[2 + q];
        }
        double w[2];
        phasor_of(v[2], w[1], w[0]);
        add_terms<2>(w, s, c);
      } else if (THEN == kGpError) {
#pragma unroll
        for (int q = 0; q < S; ++q) {
          double err = G.T.c[0] * d[0][q];
#pragma unroll
          for (int j = 1; j < NT; ++j) err = err + G.T.c[j] * d[j][q];
          err = err + G.T.c[NT] * k[q];
          worst = fmax(worst, fabs(err) / (G.eps_abs + G.eps_rel * (1.0 * fabs(v[q]) + (1.0 * G.dt) * fabs(d[0][q]))));
        }
      }
    }
  }
  if (THEN == kGpNext || THEN == kGpOut) block_sums<2>(s, c, G.out + (long)blockIdx.x * 4);
  if (THEN == kGpError) {
    __shared__ double red[256];
    red[threadIdx.x] = worst;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + off]);
      __syncthreads();
    }
    if (threadIdx.x == 0) G.out[blockIdx.x] = red[0];
  }
}

// the first stage's phases x + c0 k (k: plane A), the state's phases beside them, the block sums
template <int S, int PER>
__global__ __launch_bounds__(256) void gp_first(int n, const double *__restrict__ x, const double *__restrict__ k,
                                                double c0, double *__restrict__ xa, double *__restrict__ out,
                                                double *__restrict__ part) {
  constexpr int NA = S - 2, kPart = 256 * PER;
  double s[2] = {}, c[2] = {};
  for (long b = (long)blockIdx.x * kPart; b < n; b += (long)gridDim.x * kPart) {
    double v[PER][NA], w[PER][NA];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= n) continue;
#pragma unroll
      for (int q = 0; q < NA; ++q) {
        v[p][q] = x[i * S + 2 + q];
        w[p][q] = k[i * NA + q];
      }
    }
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const long i = b + p * 256 + threadIdx.x;
      if (i >= n) continue;
#pragma unroll
      for (int q = 0; q < NA; ++q) {
        xa[i * NA + q] = v[p][q];
        w[p][q] = v[p][q] + c0 * w[p][q];
        out[i * NA + q] = w[p][q];
      }
      double t[2];
      phasor_of(w[p][0], t[1], t[0]);
      add_terms<2>(t, s, c);
    }
  }
  block_sums<2>(s, c, part + (long)blockIdx.x * 4);
}

// x + sum_j c_j k_j in whole rows (the dense output)
template <int S>
__global__ __launch_bounds__(256) void gp_combine(int n, const double *__restrict__ x, DpTerms T,
                                                  double *__restrict__ out) {
  constexpr int NA = S - 2;
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= n) return;
  double v[S], d[kDpMaxTerms][S];
  load_row<S>(x, i, v);
#pragma unroll
  for (int j = 0; j < kDpMaxTerms; ++j) {
    const double *a = T.k[j], *xy = a + (long)n * NA;
    d[j][0] = xy[2 * i];
    d[j][1] = xy[2 * i + 1];
#pragma unroll
    for (int q = 0; q < NA; ++q) d[j][2 + q] = a[i * NA + q];
  }
#pragma unroll
  for (int q = 0; q < S; ++q) {
#pragma unroll
    for (int j = 0; j < kDpMaxTerms; ++j) v[q] = v[q] + T.c[j] * d[j][q];
    out[i * S + q] = v[q];
  }
}

// planes back to rows
template <int S>
__global__ __launch_bounds__(256) void gp_rows(int n, const double *__restrict__ planes, double *__restrict__ rows) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int q = 0; q < S; ++q)
    rows[i * S + q] = q < 2 ? planes[(long)n * (S - 2) + 2 * i + q] : planes[i * (S - 2) + q - 2];
}

// a's upper half of the wave and b's lower half change places: a + b then holds a's half sums in the
// lower half and b's in the upper one (ROW: the same for odd and even rows of 16 lanes)
template <bool ROW>
__device__ __forceinline__ double swap_add(double a, double b) {
  union { double d; unsigned w[2]; } u, v;
  u.d = a;
  v.d = b;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const auto r = ROW ? __builtin_amdgcn_permlane16_swap(u.w[q], v.w[q], false, false)
                       : __builtin_amdgcn_permlane32_swap(u.w[q], v.w[q], false, false);
    u.w[q] = r[0];
    v.w[q] = r[1];
  }
  return u.d + v.d;
}

// the sums of a, b, c, d over a wave: in lane 15 of the rows of 16 lanes that column_of names
__device__ __forceinline__ double four_sums(double a, double b, double c, double d) {
  double x = swap_add<true>(swap_add<false>(a, b), swap_add<false>(c, d));
  x += dpp<0x111, 0xf>(x);  // row_shr:1
  x += dpp<0x112, 0xf>(x);
  x += dpp<0x114, 0xf>(x);
  x += dpp<0x118, 0xf>(x);
  return x;
}
__device__ __forceinline__ int column_of(int lane) { return ((lane >> 4) & 1) * 2 + (lane >> 5); }

// Up to 256 * PPT particles: one workgroup, the particles in registers, nsteps steps.  The chain of a
// stage is a phasor, the sums over the workgroup (register moves, one LDS exchange) and the
// derivative.  Cosines and sines are added in two parts, multiples of 2^-40, whose sums are exact in any order,
// and the rest, whose sums err by 2^-80; the omega-weighted ones, which have no such bound, carry their rounding
// errors over a thread's particles and over the waves, as the block sums of larger systems do over their blocks
// (all of them that way: n = 1,000 20 us more for 80 stages).  The four waves have a SIMD each, and one wave of independent particles issues nearly
// every cycle it is given, so the particles are split over registers before they are split over more
// waves, whose reductions would only add instructions.
enum GfStepper { kSmallRk4, kSmallEuler, kSmallSrk };

template <int S, int STEPPER, int PPT>
__global__ __launch_bounds__(256) void gf_small(DevParams P, int nsteps, double dt, double *__restrict__ state,
                                                const double *__restrict__ nat, double *__restrict__ k1,
                                                double *__restrict__ k2, double *__restrict__ k3,
                                                double *__restrict__ k4, double *__restrict__ compl_out, GfNoise Z) {
  constexpr bool HO = STEPPER == kSmallSrk;
  constexpr int COLS = HO ? 4 : 2;
  constexpr bool kOne = PPT == 1;  // a block's sums alone, plain
  __shared__ double sh[2][HO && !kOne ? 8 : 4][4];  // the waves' sums
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double y[PPT][S], st[PPT][S], w[PPT], sn[PPT], cs[PPT];
#pragma unroll
  for (int p = 0; p < PPT; ++p) {
    const int i = p * 256 + threadIdx.x;
    w[p] = i < P.n && nat ? nat[i] : 0.0;
#pragma unroll
    for (int q = 0; q < S; ++q) {
      y[p][q] = st[p][q] = i < P.n ? state[(long)i * S + q] : 0.0;
      // the first stage is the state + 0 * k1 (RungeKutta4StepperPtr.cpp:50), which a k1 that is not
      // finite turns into NaN; after the first step such a k1 is in the state itself
      if (STEPPER == kSmallRk4 && i < P.n) st[p][q] = y[p][q] + 0.0 * k1[(long)i * S + q];
    }
  }
  int flip = 0;
  const auto field = [&](Field &F) {
    bool far = false;
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      small_sincos(st[p][2], 0.0, sn[p], cs[p]);
      far = far || !(fabs(st[p][2]) <= 0x1p30);
    }
    if (far) {
#pragma unroll
      for (int p = 0; p < PPT; ++p)
        if (!(fabs(st[p][2]) <= 0x1p30)) sincos(st[p][2], &sn[p], &cs[p]);
    }
    double s[4] = {}, m[2] = {}, e[2] = {};  // the parts of the cosines and of the sines; the weighted ones
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const bool in = p * 256 + (int)threadIdx.x < P.n;
      const double c1 = in ? cs[p] : 0.0, s1 = in ? sn[p] : 0.0;
      constexpr double kSplit = 6144.0;  // 1.5 2^12: of up to 2^11 terms
      const double ch = kOne ? c1 : (c1 + kSplit) - kSplit, sh1 = kOne ? s1 : (s1 + kSplit) - kSplit;
      const double w[2] = {HO && in ? st[p][S - 1] * c1 : 0.0, HO && in ? st[p][S - 1] * s1 : 0.0};
      if (kOne) {
        s[0] = c1, s[1] = s1, s[2] = w[0], s[3] = w[1];
        continue;
      }
      s[0] += ch;
      s[1] += sh1;
      s[2] += c1 - ch;
      s[3] += s1 - sh1;
      if (HO) add_terms<2>(w, m, e);
    }
    double t = four_sums(s[0], s[1], s[2], s[3]);
    if ((lane & 15) == 15) sh[flip][column_of(lane)][wv] = t;
    if (HO && !kOne) {
      t = four_sums(m[0], m[1], e[0], e[1]);
      if ((lane & 15) == 15) sh[flip][(HO && !kOne ? 4 : 0) + column_of(lane)][wv] = t;
    }
    __syncthreads();
    const auto four = [](const double *x) { return (x[0] + x[1]) + (x[2] + x[3]); };
    double v[COLS];
#pragma unroll
    for (int q = 0; q < 2; ++q) v[q] = (kOne ? four(sh[flip][q]) : four(sh[flip][q]) + four(sh[flip][2 + q])) / (double)P.n;
    if (HO)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (kOne) {
          v[COLS - 2 + q] = four(sh[flip][2 + q]) / (double)P.n;
          continue;
        }
        const double *x = sh[flip][HO && !kOne ? 4 + q : 0];
        double r, u, z, d0, d1, d2;
        two_sum(x[0], x[1], r, d0);
        two_sum(x[2], x[3], u, d1);
        two_sum(r, u, z, d2);
        v[COLS - 2 + q] = (z + (((d0 + d1) + d2) + four(sh[flip][HO && !kOne ? 6 + q : 0]))) / (double)P.n;
      }
    flip ^= 1;  // the other half is free: every wave had read it before this barrier
    F.zx = v[0];
    F.zy = v[1];
    if (HO) {
      F.wx = v[COLS - 2];
      F.wy = v[COLS - 1];
    }
    finish_field<HO>(F);
  };
  for (int step = 0; step < nsteps; ++step) {
    const bool last = step + 1 == nsteps;
    Field F{};
    if (STEPPER == kSmallRk4) {
      double tot[PPT][S];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        field(F);
        double *kb = g == 0 ? k1 : (g == 1 ? k2 : (g == 2 ? k3 : k4));
#pragma unroll
        for (int p = 0; p < PPT; ++p) {
          const int i = p * 256 + threadIdx.x;
          double k[S], cf;
          derivative<S, false>(P, F, st[p], sn[p], cs[p], w[p], k, cf);
          if (last && i < P.n) store_row<S>(kb, i, k);
          const double kc = (g < 2 ? 0.5 : 1.0) * dt;
#pragma unroll
          for (int q = 0; q < S; ++q) {
            tot[p][q] = g == 0 ? k[q] : (g < 3 ? tot[p][q] + 2.0 * k[q] : tot[p][q] + k[q]);
            if (g < 3) st[p][q] = y[p][q] + kc * k[q];
          }
        }
      }
#pragma unroll
      for (int p = 0; p < PPT; ++p)
#pragma unroll
        for (int q = 0; q < S; ++q) st[p][q] = y[p][q] = y[p][q] + tot[p][q] * dt / 6.0;
    } else {
      field(F);
#pragma unroll
      for (int p = 0; p < PPT; ++p) {
        const int i = p * 256 + threadIdx.x;
        if (i >= P.n) continue;
        double k[S], cf;
        derivative<S, HO>(P, F, st[p], sn[p], cs[p], w[p], k, cf);
        if (HO && last) compl_out[i] = cf;
        stochastic_update<S, HO>(Z, dt, i, k, cf, st[p]);
      }
      ++Z.step;
    }
  }
#pragma unroll
  for (int p = 0; p < PPT; ++p) {
    const int i = p * 256 + threadIdx.x;
    if (i < P.n) store_row<S>(state, i, st[p]);
  }
}

// One particle per thread shortens the chain of a launch, four at a time share the field and the
// reductions.  A Runge-Kutta step (one, four): n = 4,096: 17, 24 us; 65,536: 21, 26 us; 262,144: 44, 35 us.
inline bool gf_wide(int n) { return n > 131072; }
inline int gf_blocks(int n) {
  const int part = gf_wide(n) ? 1024 : 256;
  const int nb = (n + part - 1) / part;
  return nb < kMaxBlocks ? nb : kMaxBlocks;
}

template <int S, bool HO>
void first(hipStream_t st, int n, const double *x, const double *k0, double c0, double *part) {
  const auto run = [&](auto kernel) { kernel<<<dim3(gf_blocks(n)), dim3(256), 0, st>>>(n, x, k0, c0, part); };
  gf_wide(n) ? run(gf_first<S, HO, 4>) : run(gf_first<S, HO, 1>);
}

template <int S, bool HO, int THEN>
void stage(hipStream_t st, const DevParams &P, GfStep &G) {
  G.nb = gf_blocks(P.n);
  const auto run = [&](auto kernel) { kernel<<<dim3(G.nb), dim3(256), 0, st>>>(P, G); };
  gf_wide(P.n) ? run(gf_stage<S, HO, THEN, 4>) : run(gf_stage<S, HO, THEN, 1>);
}

template <int S, bool HO>
void rhs(hipStream_t st, const DevParams &P, const double *x, const double *kprev, double kc, double *part,
         const double *nat, double *k, double *compl_out) {
  first<S, HO>(st, P.n, x, kprev, kc, part);
  GfStep G{};
  G.x = x;
  G.kprev = kprev;
  G.kc = kc;
  G.in = part;
  G.nat = nat;
  G.k = k;
  G.compl_out = compl_out;
  stage<S, HO, kThenNothing>(st, P, G);
}

template <int S, bool HO>
void rk4(hipStream_t st, const DevParams &P, long nsteps, double dt, double *state, double *tmp, double *const *k,
         double *part, const double *nat, double *compl_out) {
  double *in = part, *out = part + gf_part_doubles(P.n) / 2;
  first<S, HO>(st, P.n, state, k[0], 0.0, in);  // state + 0 * k1, RungeKutta4StepperPtr.cpp:50
  for (long s = 0; s < nsteps; ++s)
    for (int g = 0; g < 4; ++g) {
      GfStep G{};
      G.x = g == 0 ? state : tmp;
      G.kprev = s == 0 && g == 0 ? k[0] : nullptr;  // later a k1 that is not finite is in the state
      G.in = in;
      G.nat = nat;
      G.k = g < 3 || s + 1 == nsteps ? k[g] : nullptr;
      G.compl_out = compl_out;
      G.base = state;
      G.out = out;
      G.dt = dt;
      if (g < 3) {
        G.c = (g < 2 ? 0.5 : 1.0) * dt;
        G.next = tmp;
        stage<S, HO, kThenNext>(st, P, G);
      } else {
        G.k1 = k[0];
        G.k2 = k[1];
        G.k3 = k[2];
        G.next = state;
        stage<S, HO, kThenRk4>(st, P, G);
      }
      double *t = in;
      in = out;
      out = t;
    }
}

template <int S, bool SRK>
void stochastic(hipStream_t st, const DevParams &P, long nsteps, double dt, double *state, double *part,
                const double *nat, double *compl_out, GfNoise Z) {
  double *in = part, *out = part + gf_part_doubles(P.n) / 2;
  first<S, SRK>(st, P.n, state, nullptr, 0.0, in);
  for (long s = 0; s < nsteps; ++s) {
    GfStep G{};
    G.x = state;
    G.in = in;
    G.nat = nat;
    G.compl_out = s + 1 == nsteps ? compl_out : nullptr;
    G.next = state;
    G.out = out;
    G.dt = dt;
    G.noise = Z;
    stage<S, SRK, SRK ? kThenSrk : kThenEuler>(st, P, G);
    ++Z.step;
    double *t = in;
    in = out;
    out = t;
  }
}

// Largest systems of one workgroup.  A step there, in launches: Runge-Kutta n = 2,048: 10, 17 us (twice
// as many do not fit its registers); Euler n = 1,024: 3.4, 5.4 us, 2,048: 6.6, 5.4 us; stochastic
// Runge-Kutta 4.5, 6.5 and 7.8, 6.5 us.
constexpr int kSmallRk4N = 2048, kSmallStochasticN = 1024;
constexpr int kSmallSteps = 1024;  // steps of one launch

template <int S, int STEPPER>
void small(hipStream_t st, const DevParams &P, long nsteps, double dt, double *state, const double *nat,
           double *const *k, double *compl_out, GfNoise Z) {
  for (long s = 0; s < nsteps; s += kSmallSteps) {
    const int m = (int)(nsteps - s < kSmallSteps ? nsteps - s : kSmallSteps);
    const auto run = [&](auto kernel) {
      kernel<<<dim3(1), dim3(256), 0, st>>>(P, m, dt, state, nat, k[0], k[1], k[2], k[3], compl_out, Z);
    };
    if (P.n <= 256)
      run(gf_small<S, STEPPER, 1>);
    else if (P.n <= 512)
      run(gf_small<S, STEPPER, 2>);
    else if (P.n <= 1024)
      run(gf_small<S, STEPPER, 4>);
    else if constexpr (STEPPER == kSmallRk4)
      run(gf_small<S, STEPPER, 8>);
    Z.step += m;
  }
}

}  // namespace

size_t gf_part_doubles(int n) { return (size_t)2 * gf_blocks(n) * 8; }

void launch_global(hipStream_t st, const DevParams &P, const double *x, const double *kprev, double kc, double *part,
                   const double *nat, double *k_next, double *compl_out) {
  if (P.s == 3)
    rhs<3, false>(st, P, x, kprev, kc, part, nat, k_next, compl_out);
  else if (P.higher_order)
    rhs<4, true>(st, P, x, kprev, kc, part, nat, k_next, compl_out);
  else
    rhs<4, false>(st, P, x, kprev, kc, part, nat, k_next, compl_out);
}

void launch_global_rk4(hipStream_t st, const DevParams &P, long nsteps, double dt, double *state, double *tmp,
                       double *const *k, double *part, const double *nat, double *compl_out) {
  if (P.s == 3) {
    if (P.n <= kSmallRk4N)
      small<3, kSmallRk4>(st, P, nsteps, dt, state, nat, k, nullptr, GfNoise{});
    else
      rk4<3, false>(st, P, nsteps, dt, state, tmp, k, part, nat, nullptr);
  } else if (P.higher_order) {
    rk4<4, true>(st, P, nsteps, dt, state, tmp, k, part, nat, compl_out);
  } else if (P.n <= kSmallRk4N) {
    small<4, kSmallRk4>(st, P, nsteps, dt, state, nat, k, nullptr, GfNoise{});
  } else {
    rk4<4, false>(st, P, nsteps, dt, state, tmp, k, part, nat, nullptr);
  }
}

void launch_global_stochastic(hipStream_t st, const DevParams &P, bool srk, long nsteps, double dt, double *state,
                              double *part, const double *nat, double *compl_out, const GfNoise &Z) {
  double *none[4] = {nullptr, nullptr, nullptr, nullptr};
  const bool one = P.n <= kSmallStochasticN;
  if (srk) {
    if (one)
      small<4, kSmallSrk>(st, P, nsteps, dt, state, nat, none, compl_out, Z);
    else
      stochastic<4, true>(st, P, nsteps, dt, state, part, nat, compl_out, Z);
  } else if (P.s == 4) {
    if (one)
      small<4, kSmallEuler>(st, P, nsteps, dt, state, nat, none, nullptr, Z);
    else
      stochastic<4, false>(st, P, nsteps, dt, state, part, nat, nullptr, Z);
  } else {
    if (one)
      small<3, kSmallEuler>(st, P, nsteps, dt, state, nat, none, nullptr, Z);
    else
      stochastic<3, false>(st, P, nsteps, dt, state, part, nat, nullptr, Z);
  }
}

namespace {
template <int S, int THEN, int NT>
void gp(hipStream_t st, const DevParams &P, GpStep &G) {
  G.nb = gf_blocks(P.n);
  const auto run = [&](auto kernel) { kernel<<<dim3(G.nb), dim3(256), 0, st>>>(P, G); };
  gf_wide(P.n) ? run(gp_stage<S, THEN, NT, 4>) : run(gp_stage<S, THEN, NT, 1>);
}

template <int S>
void gp_start(hipStream_t st, const DevParams &P, const double *x, double *part, const double *nat, double *k) {
  first<S, false>(st, P.n, x, nullptr, 0.0, part);
  GpStep G{};
  G.x = x;
  G.in = part;
  G.nat = nat;
  G.k = k;
  G.kb = k + (long)P.n * (S - 2);
  gp<S, kGpStart, 0>(st, P, G);
}

template <int S>
int gp_trial(hipStream_t st, const DevParams &P, const DpTrial &D, const double *nat, double *part) {
  const long na = (long)P.n * (S - 2);
  double *p0 = part, *p1 = part + gf_part_doubles(P.n) / 2;
  double *tmp = D.tmp, *xa = D.tmp + na;
  const auto first = [&](auto kernel) {
    kernel<<<dim3(gf_blocks(P.n)), dim3(256), 0, st>>>(P.n, D.x, D.k[0], D.first, xa, tmp, p0);
  };
  gf_wide(P.n) ? first(gp_first<S, 4>) : first(gp_first<S, 1>);
  GpStep G{};
  G.nat = nat;
  G.dt = D.dt;
  G.eps_abs = D.eps_abs;
  G.eps_rel = D.eps_rel;
  // stage g (k2 .. k6) takes the block sums in one half and leaves the next ones in the other
  for (int g = 1; g <= 5; ++g) {
    G.x = tmp;
    G.in = g & 1 ? p0 : p1;
    G.out = g & 1 ? p1 : p0;
    G.k = D.k[g];
    G.kb = g == 1 ? nullptr : D.k[g] + na;
    G.base = g < 5 ? xa : D.x;
    G.T = D.terms[g - 1];
    G.next = g < 5 ? tmp : D.out;
    switch (g) {
      case 1: gp<S, kGpNext, 1>(st, P, G); break;
      case 2: gp<S, kGpNext, 2>(st, P, G); break;
      case 3: gp<S, kGpNext, 3>(st, P, G); break;
      case 4: gp<S, kGpNext, 4>(st, P, G); break;
      default: gp<S, kGpOut, 4>(st, P, G);
    }
  }
  G.x = D.out;
  G.in = p1;
  G.out = p0;
  G.k = D.k[6];
  G.kb = D.k[6] + na;
  G.base = D.x;
  G.T = D.terms[5];
  gp<S, kGpError, 5>(st, P, G);
  return G.nb;
}
}  // namespace

void launch_dp_global_start(hipStream_t st, const DevParams &P, const double *x, double *part, const double *nat,
                            double *k) {
  P.s == 4 ? gp_start<4>(st, P, x, part, nat, k) : gp_start<3>(st, P, x, part, nat, k);
}

int launch_dp_global_trial(hipStream_t st, const DevParams &P, const DpTrial &D, const double *nat, double *part) {
  return P.s == 4 ? gp_trial<4>(st, P, D, nat, part) : gp_trial<3>(st, P, D, nat, part);
}

void launch_dp_global_combine(hipStream_t st, int s, int n, const double *x, const DpTerms &T, double *out) {
  const dim3 nb((unsigned)((n + 255L) / 256));
  if (s == 4)
    gp_combine<4><<<nb, dim3(256), 0, st>>>(n, x, T, out);
  else
    gp_combine<3><<<nb, dim3(256), 0, st>>>(n, x, T, out);
}

void launch_dp_global_rows(hipStream_t st, int s, int n, const double *planes, double *rows) {
  const dim3 nb((unsigned)((n + 255L) / 256));
  if (s == 4)
    gp_rows<4><<<nb, dim3(256), 0, st>>>(n, planes, rows);
  else
    gp_rows<3><<<nb, dim3(256), 0, st>>>(n, planes, rows);
}

}  // namespace spss
