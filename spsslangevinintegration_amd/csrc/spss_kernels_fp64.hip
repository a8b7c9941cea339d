// spss_kernels_fp64.hip -- FP64 kernels: the cell list on general boxes and grids, Verlet lists, the steppers'
// updates and the reductions (all pairs, the cell list on the unit box and the global field have files of
// their own).
//
// The general cell list's sums are accumulated pair by pair in the order the reference visits the pairs
// (stencil order, then ascending j), so results agree with it to the last few ulps of the device
// sin/cos; the Verlet sums go through phasors (spss_pairs64.hpp).  Built with -ffp-contract=off.
#pragma clang fp contract(off)

#include "spss_device.hpp"
#include "spss_launch.hpp"
#include "spss_pairs64.hpp"
#include "spss_scan.hpp"

#include <type_traits>

namespace spss {

// ---------------------------------------------------------------------------
// stage state y + (k_coef*dt)*k_prev, ParticleSystemFirstOrderPtr.cpp:234-241
__global__ void k_stage(long m, const double *__restrict__ state, const double *__restrict__ kprev,
                        double kc_dt, double *__restrict__ stage) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) stage[k] = state[k] + kc_dt * kprev[k];
}

// the stage of an all-zero k_prev: state + 0.0 is what state + kc_dt * 0.0 gives for any finite
// kc_dt (-0.0 becomes +0.0), without reading a zero vector
__global__ void k_stage_zero(long m, const double *__restrict__ state, double *__restrict__ stage) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) stage[k] = state[k] + 0.0;
}

// ---------------------------------------------------------------------------
// Cell list by a stable device counting sort over the cell keys.
// Keys: ParticleSystemFirstOrderPtr.cpp:364-381.  Buckets in ascending particle
// index (:388-391) come from the stable rank pass below.

template <int S>
__global__ void k_cell_keys(DevParams P, const double *__restrict__ stage, int ncx, int ncy,
                            int *__restrict__ key, int *__restrict__ slot, int *__restrict__ count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  double xw, yw;
  key_wrap<S>(P, stage[(long)i * S], stage[(long)i * S + 1], xw, yw);
  int c = cell_coord(yw, ncy) * ncx + cell_coord(xw, ncx);
  key[i] = c;
  slot[i] = atomicAdd(count + c, 1);
}

__global__ void k_scatter(int n, const int *__restrict__ key, const int *__restrict__ slot,
                          const int *__restrict__ start, int *__restrict__ tmp) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) tmp[start[key[i]] + slot[i]] = i;
}

// Each cell's members in ascending particle index (the order in which the FP64 pair loop sums a
// cell's members).  Cells of at most 64 members (every cell at the densities of the workloads) are
// sorted by one wave each (wave_sort64, grid-stride over cells); the members of denser cells are
// then ranked one thread each by counting the smaller indices of their cell (grid-stride over the
// particles, so a single cell holding most particles is spread over the whole grid).
__global__ __launch_bounds__(256) void k_stable_rank(int n, int ncells, const int *__restrict__ key,
                                                     const int *__restrict__ start, const int *__restrict__ tmp,
                                                     int *__restrict__ sorted) {
  const int lane = threadIdx.x & 63;
  for (int c = blockIdx.x * 4 + (threadIdx.x >> 6); c < ncells; c += gridDim.x * 4) {
    const int b = start[c], m = start[c + 1] - b;
    if (m > 64) continue;  // the whole wave
    const int v = wave_sort64(lane < m ? tmp[b + lane] : 0x7fffffff, lane);
    if (lane < m) sorted[b + lane] = v;
  }
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int c = key[i];
    const int b = start[c], e = start[c + 1];
    if (e - b <= 64) continue;
    int r = 0;
    for (int t = b; t < e; ++t) r += tmp[t] < i ? 1 : 0;
    sorted[b + r] = i;
  }
}

// linked-list pair loop, ParticleSystemFirstOrderPtr.cpp:398-466 (x_i wrapped, x_j as stored) and
// ParticleSystemSecondOrderPtr.cpp:318-381 (model 6: both wrapped when outside the box, ClassA).
// Threads walk particles in cell order for locality; sums follow the stencil order of :83-88.
template <int S>
__global__ __launch_bounds__(kBlock) void k_linked_list(DevParams P, const double *__restrict__ stage, int ncx,
                                                        int ncy, const int *__restrict__ start,
                                                        const int *__restrict__ sorted,
                                                        const double *__restrict__ nat, double *__restrict__ k_next,
                                                        double *__restrict__ compl_out) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P.n) return;
  const int i = sorted[t];
  double st[S];
#pragma unroll
  for (int q = 0; q < S; ++q) st[q] = stage[(long)i * S + q];
  double x_i, y_i;
  key_wrap<S>(P, st[0], st[1], x_i, y_i);
  const double phi_i = st[Slots<S>::phi];
  const double omega_i = (S == 3) ? 0.0 : st[Slots<S>::omega];
  const int cx = cell_coord(x_i, ncx), cy = cell_coord(y_i, ncy);
  PairAcc a{0.0, 0.0, 0.0};
  for (int dyc = -1; dyc <= 1; ++dyc) {
    const int jy = adjust_cell(cy + dyc, ncy);
    for (int dxc = -1; dxc <= 1; ++dxc) {
      const int jx = adjust_cell(cx + dxc, ncx);
      const int c = jy * ncx + jx;
      const int e = start[c + 1];
      for (int u = start[c]; u < e; ++u) {
        const int j = sorted[u];
        if (j == i) continue;
        const double *sj = stage + (long)j * S;
        double x_j = sj[0], y_j = sj[1];
        if (S == 6) key_wrap<6>(P, x_j, y_j, x_j, y_j);  // :356-359
        pair_term<S>(P, x_i, y_i, phi_i, omega_i, x_j, y_j, sj[Slots<S>::phi],
                     (S == 3) ? 0.0 : sj[Slots<S>::omega], a);
      }
    }
  }
  write_k<S>(P, st, i, a, nat ? nat[i] : 0.0, k_next, compl_out);
}

// ---------------------------------------------------------------------------
// Verlet lists.  Build over all pairs (ParticleSystemFirstOrderPtr.cpp:497-543: x_i as stored)
// or from the cell stencil (:643-743: x_i wrapped).  Two passes: counts, then lists written in
// the reference's visiting order after a scan of the counts.
//
// Several lanes share a particle (LPP of a wave, a power of two): a list or a cell is read as
// contiguous runs and thousands of particles fill the chip, where one thread per particle left it to
// 79 workgroups at n = 20,011 (list build, both passes: 480 -> 53 us).

// position of a lane among those of its group of LPP whose flag is set, and their number
template <int LPP>
__device__ __forceinline__ int group_rank(bool flag, int &total) {
  const int lane = threadIdx.x & 63, g = lane & ~(LPP - 1);
  unsigned long long m = __ballot(flag) >> g;
  if (LPP < 64) m &= (1ull << (LPP & 63)) - 1;
  total = __popcll(m);
  return __popcll(m & ((1ull << (lane - g)) - 1));
}

// one run [b, e) of candidates of particle i (ids from `sorted`, or the run itself when null) by a
// group of LPP lanes, in order; returns how many are within the list radius.  A list holds the ids,
// and beside them the positions in `sorted`, by which the pair loop reads.  Every lane of the group
// takes part in every round.
template <int S, int LPP, bool FILL>
__device__ __forceinline__ int list_run(const DevParams &P, const double *__restrict__ stage,
                                        const int *__restrict__ sorted, double rmax2, int i, double x_i, double y_i,
                                        int b, int e, int w, int *__restrict__ vlist, int *__restrict__ vslot) {
  int found = 0;
  for (int u0 = b; u0 < e; u0 += LPP) {
    const int u = u0 + (threadIdx.x & (LPP - 1));
    const int j = u < e ? (sorted ? sorted[u] : u) : i;
    bool in = false;
    if (j != i) {
      double dx, dy;
      class_c_unsigned(P, x_i, y_i, stage[(long)j * S], stage[(long)j * S + 1], dx, dy);
      in = dx * dx + dy * dy <= rmax2;
    }
    int total;
    const int r = group_rank<LPP>(in, total);
    if (FILL && in) {
      vlist[w + found + r] = j;
      if (vslot) vslot[w + found + r] = u;
    }
    found += total;
  }
  return found;
}

constexpr int kBuildLanes = 16;

template <int S, bool FILL>
__global__ __launch_bounds__(kBlock) void k_verlet_build_all(DevParams P, const double *__restrict__ stage,
                                                             double rmax2, int *__restrict__ vcount,
                                                             const int *__restrict__ vstart, int *__restrict__ vlist,
                                                             int *__restrict__ vslot) {
  constexpr int LPP = 64;  // a wave per particle: the runs are all n particles
  const int i = (blockIdx.x * kBlock + threadIdx.x) / LPP;
  if (i >= P.n) return;
  const int c = list_run<S, LPP, FILL>(P, stage, nullptr, rmax2, i, stage[(long)i * S], stage[(long)i * S + 1], 0, P.n,
                                       FILL ? vstart[i] : 0, vlist, vslot);
  if (!FILL && (threadIdx.x & (LPP - 1)) == 0) vcount[i] = c;
}

template <int S, bool FILL>
__global__ __launch_bounds__(kBlock) void k_verlet_build_cells(DevParams P, const double *__restrict__ stage, int ncx,
                                                               int ncy, const int *__restrict__ start,
                                                               const int *__restrict__ sorted, double rmax2,
                                                               int *__restrict__ vcount,
                                                               const int *__restrict__ vstart,
                                                               int *__restrict__ vlist, int *__restrict__ vslot) {
  constexpr int LPP = kBuildLanes;
  const int t = (blockIdx.x * kBlock + threadIdx.x) / LPP;
  // the ballots of a wave need all of its lanes: groups past the end repeat the last particle
  const int i = sorted[min(t, P.n - 1)];  // cell order: neighbouring groups read the same cells
  double x_i, y_i;
  key_wrap<S>(P, stage[(long)i * S], stage[(long)i * S + 1], x_i, y_i);
  const int cx = cell_coord(x_i, ncx), cy = cell_coord(y_i, ncy);
  const int w = FILL ? vstart[i] : 0;
  int cnt = 0;
  for (int dyc = -1; dyc <= 1; ++dyc) {
    const int jy = adjust_cell(cy + dyc, ncy);
    for (int dxc = -1; dxc <= 1; ++dxc) {
      const int c = jy * ncx + adjust_cell(cx + dxc, ncx);
      cnt += list_run<S, LPP, FILL>(P, stage, sorted, rmax2, i, x_i, y_i, start[c], start[c + 1], w + cnt, vlist, vslot);
    }
  }
  if (!FILL && t < P.n && (threadIdx.x & (LPP - 1)) == 0) vcount[i] = cnt;
}

// stage state in the order of the lists' build (order null: as it is), and what the pair sums read of
// it: x, y wrapped into the box (NaN farther out than the guard band covers) and the phasor in the frame
// of the phase that particle 0's state has; om: omega
template <int S>
__device__ __forceinline__ void stage_record(const DevParams &P, const double *v, double ref, int t,
                                             const VerletStage &V) {
#pragma unroll
  for (int q = 0; q < S; ++q) V.stage[(long)t * S + q] = v[q];
  double sn, cs, xw, yw;
  frame_phasor_any(v[2], ref, sn, cs);
  apply_pbc(P, v[0], v[1], xw, yw);
  const bool near = fabs(v[0]) <= kFar64 * P.xs && fabs(v[1]) <= kFar64 * P.ys;
  reinterpret_cast<double4 *>(V.rec)[t] = make_double4(near ? xw : __builtin_nan(""), yw, sn, cs);
  if (S == 4) V.om[t] = v[S - 1];
}

// vmax: the step's displacement maxima, cleared (may be null)
template <int S>
__global__ __launch_bounds__(kBlock) void k_stage_order(DevParams P, const double *__restrict__ state,
                                                        const double *__restrict__ kprev, double kc_dt,
                                                        const int *__restrict__ order, VerletStage V,
                                                        unsigned long long *__restrict__ vmax) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (vmax && t < kVerletMax) vmax[t * kVerletMaxStep] = 0ull;
  if (t >= P.n) return;
  const long i = order ? order[t] : t;
  double v[S];
#pragma unroll
  for (int q = 0; q < S; ++q) v[q] = state[i * S + q] + (kprev ? kc_dt * kprev[i * S + q] : 0.0);
  stage_record<S>(P, v, frame_ref(state[2]), t, V);
}

// Verlet pair loop, ParticleSystemFirstOrderPtr.cpp:553-613 (x_i as stored), through the phasors
// (spss_pairs64.hpp): LPP lanes per particle take every LPP-th entry of its list, their sums are added in
// a fixed tree.  The records lie in the cell order of the lists' build, where the entries of a list are
// runs of neighbours: a group's reads are a few lines instead of one line per entry.  n = 20,011, ~600
// entries of which 140 in range: 404 us with one thread per particle and a sine per pair, 32 with 16
// lanes, records in list order and sin(d - alpha), 18.5 through the phasors (8, 32, 64 lanes: 27, 22, 24),
// bound by the 32 bytes per entry from the caches (20 TB/s).
// THEN: 0 the derivative alone; 1 the next Runge-Kutta stage base + kc k beside it, for the next launch; 2
// the step, base += (k1 + 2 k2 + 2 k3 + k) dt / 6, and its largest squared displacement.
// A step was ten launches (four stages, four sums, the combination, the maximum), now five: n = 20,011 of
// 600 entries, five steps with the state's transfers: 647 us, now 513.
template <int S, int LPP, bool HO, int THEN>
__global__ __launch_bounds__(kBlock) void k_verlet_pairs(DevParams P, double band, const double *__restrict__ vstage,
                                                         const double4 *__restrict__ rec,
                                                         const double *__restrict__ om, VerletThen N,
                                                         const int *__restrict__ order,
                                                         const int *__restrict__ vstart, const int *__restrict__ vslot,
                                                         const double *__restrict__ nat, double *__restrict__ k_next,
                                                         double *__restrict__ compl_out) {
  const int t = (int)(((long)blockIdx.x * kBlock + threadIdx.x) / LPP), l = threadIdx.x & (LPP - 1);
  const int i = t < P.n ? (order ? order[t] : t) : -1;
  PhasorSums q;
  double4 own{};
  double om_i = 0.0;
  double pre = 0.0, old = 0.0, k4[S] = {};  // THEN 2: component l of k1 + 2 k2 + 2 k3 and of the state
  if (THEN == 2 && i >= 0 && l < S) {
    const long c = (long)i * S + l;
    pre = N.k1[c] + 2.0 * N.k2[c] + 2.0 * N.k3[c];
    old = N.base[c];
  }
  if (i >= 0) {
    own = rec[t];
    if (HO) om_i = om[t];
    int u = vstart[i] + l;
    const int e = vstart[i + 1];
    if (u < e) {
      // the next entry's record and the position of the one after it are read while this one is added
      int j = vslot[u], j1 = u + LPP < e ? vslot[u + LPP] : j;
      double4 r = rec[j];
      for (; u < e; u += LPP) {
        const int j2 = u + 2 * LPP < e ? vslot[u + 2 * LPP] : j1;
        const double4 r1 = rec[j1];
        const double ax = fabs(own.x - r.x), ay = fabs(own.y - r.y);
        const double dx = fmin(ax, P.xs - ax), dy = fmin(ay, P.ys - ay);
        const double d = __builtin_fma(dx, dx, __builtin_fma(dy, dy, -P.rho2));
        bool in = d < 0.0;
        if (!(fabs(d) > band)) {  // rare: the reference's own test on the stored positions
          const long a = (long)t * S, b = (long)j * S;
          in = pair_in_range<S>(P, vstage[a], vstage[a + 1], vstage[b], vstage[b + 1]);
        }
        if (in) {
          q.S += r.z;
          q.C += r.w;
          q.card += 1.0;
          if (HO) {
            const double o = om[j] - om_i;
            q.TS += o * r.z;
            q.TC += o * r.w;
          }
        }
        j = j1;
        j1 = j2;
        r = r1;
      }
    }
  }
#pragma unroll
  for (int off = LPP / 2; off > 0; off >>= 1) {
    q.S += __shfl_down(q.S, off, LPP);
    q.C += __shfl_down(q.C, off, LPP);
    q.card += __shfl_down(q.card, off, LPP);
    if (HO) {
      q.TS += __shfl_down(q.TS, off, LPP);
      q.TC += __shfl_down(q.TC, off, LPP);
    }
  }
  if (i >= 0 && l == 0) {
    double st[S], sn, cs;
#pragma unroll
    for (int k = 0; k < S; ++k) st[k] = vstage[(long)t * S + k];
    phasor_of(st[2], sn, cs);
    write_k<S>(P, st, i, pair_acc<S>(P, q, own.z, own.w), nat ? nat[i] : 0.0, sn, cs, k_next,
               compl_out);
    const long ii = (long)i * S;
    if (THEN == 1) {
      double v[S];
#pragma unroll
      for (int k = 0; k < S; ++k) v[k] = N.base[ii + k] + N.kc * k_next[ii + k];  // what k_next holds: see write_k
      stage_record<S>(P, v, frame_ref(N.base[2]), t, N.next);
    } else if (THEN == 2) {
#pragma unroll
      for (int k = 0; k < S; ++k) k4[k] = k_next[ii + k];
    }
  }
  // CalculateMaxDisplacement's dist2; not a number counts for nothing.  One atomic per workgroup, where it would
  // raise what is there, the groups' maxima a cache line each: n = 20,011 1.6 us more than THEN 1; per wave with
  // sixteen maxima to a line 10.5, per workgroup 8.8
  if (THEN == 2) {
    __shared__ double wave[kBlock / 64];
    double k = 0.0, tot = 0.0;
#pragma unroll
    for (int c = 0; c < S; ++c) {
      const double v = __shfl(k4[c], 0, LPP);
      if (l == c) k = v;
    }
    if (i >= 0 && l < S) {
      tot = (pre + k) * N.dt / 6.0;
      N.base[(long)i * S + l] = old + tot;
    }
    const double dx = __shfl(tot, 0, LPP), dy = __shfl(tot, 1, LPP);
    double far = dx * dx + dy * dy;
    for (int off = 32; off > 0; off >>= 1) far = fmax(far, __shfl_xor(far, off, 64));
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x / 64] = far;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kBlock / 64; ++w) far = fmax(far, wave[w]);
      unsigned long long *m = N.vmax + (blockIdx.x & (kVerletMax - 1)) * kVerletMaxStep, v = __double_as_longlong(far);
      if (far > 0.0 && v > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(m, v);
    }
  }
}

// ---------------------------------------------------------------------------
// global polar order field, ParticleSystemFirstOrderPtr.cpp:177-223.
// Sums (cos, sin, w cos, w sin) per block in a fixed tree, then in block order.

__device__ __forceinline__ void two_sum(double a, double b, double &s, double &e) {
  s = a + b;
  double bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

// the final reductions: loads issued together per lane
constexpr int kFinalBatch = 16;

// the 64 compensated lane pairs (sum, correction) of a wave combined pairwise in a fixed tree
// (lane l with lane l + 32, then + 16, ...); lane 0 returns sum + correction
__device__ __forceinline__ double wave_combine(double s, double c) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double s2 = __shfl_down(s, off, 64), c2 = __shfl_down(c, off, 64);
    double t, e;
    two_sum(s, s2, t, e);
    s = t;
    c = c + c2 + e;
  }
  return s + c;
}

// ---------------------------------------------------------------------------
// steppers.  Each writes the step's total displacement only as the per-block
// max of dx^2 + dy^2 that CalculateMaxDisplacement needs (:841-850).

__device__ __forceinline__ void block_max_store(double v, double *partial) {
  __shared__ double sh[kBlock];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + off]);
    __syncthreads();
  }
  if (threadIdx.x == 0 && partial) partial[blockIdx.x] = sh[0];
}

// RungeKutta4StepperPtr.cpp:78-87
template <int S>
__global__ __launch_bounds__(kBlock) void k_rk4_combine(int n, double *__restrict__ state, const double *__restrict__ k1,
                                                        const double *__restrict__ k2, const double *__restrict__ k3,
                                                        const double *__restrict__ k4, double dt,
                                                        double *__restrict__ max_partial) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  double m2 = 0.0;
  if (i < n) {
    double tot[S];
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const long k = (long)i * S + q;
      tot[q] = (k1[k] + 2.0 * k2[k] + 2.0 * k3[k] + k4[k]) * dt / 6.0;
      state[k] += tot[q];
    }
    m2 = tot[0] * tot[0] + tot[1] * tot[1];
  }
  block_max_store(m2, max_partial);
}

__device__ __forceinline__ double draw(int mode, const double *noise, long idx, uint64_t seed, uint32_t particle,
                                       uint32_t which, uint64_t step) {
  if (mode == 1) return noise[idx];  // injected (host array already copied to the device)
  if (mode == 3) {
    double z0, z1;
    philox_normal2(seed, particle, which >> 1, step, z0, z1);
    return (which & 1) ? z1 : z0;
  }
  return 0.0;
}

// StochasticEulerStepperPtr.hpp:40-73 (model 4), StochasticEulerStepper.hpp:33-51 +
// ParticleSystemSecondOrder.cpp:439-451 (model 6, draws for slots 2, 3, 5), model 3 on phi.
template <int S>
__global__ __launch_bounds__(kBlock) void k_euler(int n, double *__restrict__ state, const double *__restrict__ f,
                                                  double dt, double sqrt_dt, double int_phi, double int_r,
                                                  int noise_mode, const double *__restrict__ noise, uint64_t seed,
                                                  uint64_t step, double *__restrict__ max_partial) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  double m2 = 0.0;
  if (i < n) {
    const long ii = (long)i * S;
    if (S == 4) {
      double dW = sqrt_dt * draw(noise_mode, noise, i, seed, i, 0, step);
      double t0 = f[ii] * dt, t1 = f[ii + 1] * dt, t2 = f[ii + 2] * dt;
      double t3 = f[ii + 3] * dt + int_phi * dW;
      state[ii] += t0;
      state[ii + 1] += t1;
      state[ii + 2] += t2;
      state[ii + 3] += t3;
      m2 = t0 * t0 + t1 * t1;
    } else if (S == 3) {
      double dW = sqrt_dt * draw(noise_mode, noise, i, seed, i, 0, step);
      double t0 = f[ii] * dt, t1 = f[ii + 1] * dt;
      double t2 = f[ii + 2] * dt + int_phi * dW;
      state[ii] += t0;
      state[ii + 1] += t1;
      state[ii + 2] += t2;
      m2 = t0 * t0 + t1 * t1;
    } else {
      double g2 = int_r * draw(noise_mode, noise, 3L * i, seed, i, 0, step);
      double g3 = int_r * draw(noise_mode, noise, 3L * i + 1, seed, i, 1, step);
      double g5 = int_phi * draw(noise_mode, noise, 3L * i + 2, seed, i, 2, step);
      const double g[6] = {0.0, 0.0, g2, g3, 0.0, g5};
#pragma unroll
      for (int q = 0; q < 6; ++q) state[ii + q] += dt * f[ii + q] + sqrt_dt * g[q];
    }
  }
  block_max_store(m2, max_partial);
}

// StochasticRungeKuttaStepperPtr.hpp:50-76 (model 4).  c15 = 0.5*pow(dt,1.5), is3 = 1/sqrt(3),
// sq2d = sqrt(2*D_phi) come from the host so they round exactly as there.
__global__ __launch_bounds__(kBlock) void k_srk(int n, double *__restrict__ state, const double *__restrict__ f,
                                                const double *__restrict__ C, double dt, double sqrt_dt,
                                                double c15, double is3, double sq2d, double friction,
                                                int noise_mode, const double *__restrict__ noise, uint64_t seed,
                                                uint64_t step, double *__restrict__ max_partial) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  double m2 = 0.0;
  if (i < n) {
    double U_1 = draw(noise_mode, noise, 2L * i, seed, i, 0, step);
    double U_2 = draw(noise_mode, noise, 2L * i + 1, seed, i, 1, step);
    double delta_W_i = U_1 * sqrt_dt;
    double delta_Z_i = c15 * (U_1 + is3 * U_2);
    const long ii = (long)i * 4;
    const double f0 = f[ii], f1 = f[ii + 1], f2 = f[ii + 2], f3 = f[ii + 3];
    double t0 = f0 * dt - 0.5 * f2 * f1 * dt * dt;
    double t1 = f1 * dt + 0.5 * f2 * f0 * dt * dt;
    double t2 = f2 * dt + 0.5 * f3 * dt * dt + sq2d * delta_Z_i;
    double t3 = f3 * dt + 0.5 * (C[i] - friction * f3) * dt * dt + sq2d * (delta_W_i - friction * delta_Z_i);
    state[ii] += t0;
    state[ii + 1] += t1;
    state[ii + 2] += t2;
    state[ii + 3] += t3;
    m2 = t0 * t0 + t1 * t1;
  }
  block_max_store(m2, max_partial);
}

// max of the block partials
__global__ void k_max_final(int nb, const double *__restrict__ partial, double *__restrict__ out) {
  __shared__ double sh[kBlock];
  double m = 0.0;
  for (int b0 = threadIdx.x; b0 < nb; b0 += kBlock * kFinalBatch) {
    double x[kFinalBatch];
#pragma unroll
    for (int k = 0; k < kFinalBatch; ++k) x[k] = b0 + kBlock * k < nb ? partial[b0 + kBlock * k] : 0.0;
#pragma unroll
    for (int k = 0; k < kFinalBatch; ++k) m = fmax(m, x[k]);
  }
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + off]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

// max of dx^2+dy^2 over a total-displacement vector (CalculateMaxDisplacement on a given vector)
__global__ __launch_bounds__(kBlock) void k_disp_max(int n, int s, const double *__restrict__ tot,
                                                     double *__restrict__ max_partial) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  double m2 = 0.0;
  if (i < n) {
    double dx = tot[(long)i * s], dy = tot[(long)i * s + 1];
    m2 = dx * dx + dy * dy;
  }
  block_max_store(m2, max_partial);
}

// ---------------------------------------------------------------------------
// observers and utilities

// order parameter sums: per-block compensated (cos, sin) sums of state[s*i + slot]
__global__ __launch_bounds__(kBlock) void k_order_partial(int n, int s, int slot, const double *__restrict__ state,
                                                          double *__restrict__ partial) {
  __shared__ double sh[2][kBlock];
  __shared__ double shc[2][kBlock];
  int i = blockIdx.x * kBlock + threadIdx.x;
  double c = 0.0, sn = 0.0;
  if (i < n) {
    double phi = state[(long)i * s + slot];
    c = cos(phi);
    sn = sin(phi);
  }
  sh[0][threadIdx.x] = c;
  sh[1][threadIdx.x] = sn;
  shc[0][threadIdx.x] = 0.0;
  shc[1][threadIdx.x] = 0.0;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        double t, e;
        two_sum(sh[q][threadIdx.x], sh[q][threadIdx.x + off], t, e);
        sh[q][threadIdx.x] = t;
        shc[q][threadIdx.x] += shc[q][threadIdx.x + off] + e;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[(long)blockIdx.x * 4 + 0] = sh[0][0];
    partial[(long)blockIdx.x * 4 + 1] = sh[1][0];
    partial[(long)blockIdx.x * 4 + 2] = shc[0][0];
    partial[(long)blockIdx.x * 4 + 3] = shc[1][0];
  }
}

// the (cos, sin) block partials summed with compensation, one wave per column: each lane takes
// every 64th block, then the wave combines its 64 compensated pairs in a fixed tree
__global__ __launch_bounds__(128) void k_order_final(int nb, const double *__restrict__ partial, double n,
                                                     double *__restrict__ out) {
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double s = 0.0, c = 0.0;
  for (int b0 = lane; b0 < nb; b0 += 64 * kFinalBatch) {
    double x[kFinalBatch], y[kFinalBatch];
#pragma unroll
    for (int k = 0; k < kFinalBatch; ++k) {
      const int b = b0 + 64 * k;
      x[k] = b < nb ? partial[(long)b * 4 + q] : 0.0;
      y[k] = b < nb ? partial[(long)b * 4 + 2 + q] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kFinalBatch; ++k) {
      if (b0 + 64 * k < nb) {
        double t, e;
        two_sum(s, x[k], t, e);
        s = t;
        c += e + y[k];
      }
    }
  }
  const double total = wave_combine(s, c);
  if (lane == 0) out[q] = total / n;
}

// ApplyPeriodicBoundaryConditions(Real*, long), PeriodicBoundaryConditions.cpp:147-155
__global__ void k_apply_pbc(int n, int s, double *__restrict__ state, double xs, double ys, double xrs, double yrs) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long ii = (long)i * s;
  state[ii] -= floor(state[ii] * xrs) * xs;
  state[ii + 1] -= floor(state[ii + 1] * yrs) * ys;
}

// AveragingObserver::operator(), AveragingObserver.cpp:29-37
__global__ void k_accumulate(long m, const double *__restrict__ state, double *__restrict__ acc) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) acc[k] = state[k] + acc[k];
}

__global__ void k_fill_double(long m, double *__restrict__ p, double v) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) p[k] = v;
}

// plain streaming copy, one 16-byte vector per thread: measures attainable HBM bandwidth and
// calibrates the FETCH_SIZE / WRITE_SIZE counters against a kernel of known traffic.  Without a
// grid-stride loop every load is issued as soon as its wave starts, which keeps more bytes in
// flight than a loop over a fixed grid (on MI355X at 1 GiB: ~6.2 TB/s against ~4.6 TB/s for 4096
// workgroups striding)
__global__ __launch_bounds__(256) void k_copy16(long n16, const uint4 *__restrict__ src, uint4 *__restrict__ dst) {
  const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n16) dst[k] = src[k];
}

__global__ void k_fill_int(long m, int *__restrict__ p, int v) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) p[k] = v;
}

__global__ void k_iota(int n, int *__restrict__ p) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = k;
}

// ---------------------------------------------------------------------------
// host-side launchers

static inline unsigned nblk(long m, int b = kBlock) { return (unsigned)((m + b - 1) / b); }

void launch_stage(hipStream_t st, long m, const double *state, const double *kprev, double kc_dt, double *stage) {
  if (kprev)
    k_stage<<<dim3(nblk(m)), dim3(kBlock), 0, st>>>(m, state, kprev, kc_dt, stage);
  else
    k_stage_zero<<<dim3(nblk(m)), dim3(kBlock), 0, st>>>(m, state, stage);
}

#define SPSS_DISPATCH_S(S, ...) \
  switch (S) {                   \
    case 3: { constexpr int SS = 3; __VA_ARGS__; } break; \
    case 4: { constexpr int SS = 4; __VA_ARGS__; } break; \
    case 6: { constexpr int SS = 6; __VA_ARGS__; } break; \
    default: break;              \
  }

void launch_cell_build(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy, CellBuffers &cb) {
  const int m = ncx * ncy;
  SPSS_DISPATCH_S(P.s, k_cell_keys<SS><<<dim3(nblk(P.n)), dim3(kBlock), 0, st>>>(P, stage, ncx, ncy, cb.key, cb.slot, cb.count));
  launch_scan(st, cb.count, cb.start, m, cb.blocksum);
  k_scatter<<<dim3(nblk(P.n)), dim3(kBlock), 0, st>>>(P.n, cb.key, cb.slot, cb.start, cb.tmp);
  k_stable_rank<<<dim3(std::max((m + 3) / 4, (int)nblk(P.n))), dim3(256), 0, st>>>(P.n, m, cb.key, cb.start, cb.tmp,
                                                                                 cb.sorted);
}

void launch_linked_list(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                        const CellBuffers &cb, const double *nat, double *k_next, double *compl_out) {
  SPSS_DISPATCH_S(P.s, k_linked_list<SS><<<dim3(nblk(P.n)), dim3(kBlock), 0, st>>>(P, stage, ncx, ncy, cb.start, cb.sorted, nat, k_next, compl_out));
}

void launch_scan(hipStream_t st, int *count, int *start, int m, int *blocksum) {
  const int nb = scan_blocks(m);
  scan_local<<<dim3(nb), dim3(256), 0, st>>>(count, nullptr, m, start, blocksum);
  scan_add<<<dim3(nb), dim3(256), 0, st>>>(count, nullptr, m, start, blocksum, nb, nullptr);
}

void launch_verlet_count_all(hipStream_t st, const DevParams &P, const double *stage, double rmax2, int *vcount) {
  SPSS_DISPATCH_S(P.s, k_verlet_build_all<SS, false><<<dim3(nblk(64L * P.n)), dim3(kBlock), 0, st>>>(P, stage, rmax2, vcount, nullptr, nullptr, nullptr));
}
void launch_verlet_fill_all(hipStream_t st, const DevParams &P, const double *stage, double rmax2,
                            const int *vstart, int *vlist, int *vslot) {
  SPSS_DISPATCH_S(P.s, k_verlet_build_all<SS, true><<<dim3(nblk(64L * P.n)), dim3(kBlock), 0, st>>>(P, stage, rmax2, nullptr, vstart, vlist, vslot));
}
void launch_verlet_count_cells(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                               const CellBuffers &cb, double rmax2, int *vcount) {
  SPSS_DISPATCH_S(P.s, k_verlet_build_cells<SS, false><<<dim3(nblk((long)kBuildLanes * P.n)), dim3(kBlock), 0, st>>>(P, stage, ncx, ncy, cb.start, cb.sorted, rmax2, vcount, nullptr, nullptr, nullptr));
}
void launch_verlet_fill_cells(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                              const CellBuffers &cb, double rmax2, const int *vstart, int *vlist, int *vslot) {
  SPSS_DISPATCH_S(P.s, k_verlet_build_cells<SS, true><<<dim3(nblk((long)kBuildLanes * P.n)), dim3(kBlock), 0, st>>>(P, stage, ncx, ncy, cb.start, cb.sorted, rmax2, nullptr, vstart, vlist, vslot));
}
void launch_stage_order(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                        const int *order, const VerletStage &V, unsigned long long *vmax) {
  if (P.s == 4)
    k_stage_order<4><<<dim3(nblk(P.n)), dim3(kBlock), 0, st>>>(P, state, kprev, kc_dt, order, V, vmax);
  else
    k_stage_order<3><<<dim3(nblk(P.n)), dim3(kBlock), 0, st>>>(P, state, kprev, kc_dt, order, V, vmax);
}

template <int S, bool HO, int THEN>
static void verlet_pairs_as(hipStream_t st, const DevParams &P, const VerletStage &V, const int *order,
                            const int *vstart, const int *vslot, const double *nat, double *k_next,
                            double *compl_out, const VerletThen &N) {
  // 16 lanes read a list in contiguous 64-byte runs; fewer than 16,384 particles need a wave each to
  // fill the chip
  const double4 *rec = reinterpret_cast<const double4 *>(V.rec);
  const double band = pair_band(P.rho2, P.xs, P.ys);
  if (P.n < 16384)
    k_verlet_pairs<S, 64, HO, THEN><<<dim3(nblk(64L * P.n)), dim3(kBlock), 0, st>>>(
        P, band, V.stage, rec, V.om, N, order, vstart, vslot, nat, k_next, compl_out);
  else
    k_verlet_pairs<S, 16, HO, THEN><<<dim3(nblk(16L * P.n)), dim3(kBlock), 0, st>>>(
        P, band, V.stage, rec, V.om, N, order, vstart, vslot, nat, k_next, compl_out);
}

void launch_verlet_pairs(hipStream_t st, const DevParams &P, const VerletStage &V, const int *order,
                         const int *vstart, const int *vslot, const double *nat, double *k_next, double *compl_out,
                         const VerletThen *then) {
  const VerletThen N = then ? *then : VerletThen{};
  const auto as = [&](auto s, auto ho) {
    constexpr int S = decltype(s)::value;
    constexpr bool HO = decltype(ho)::value;
    if (!then)
      verlet_pairs_as<S, HO, 0>(st, P, V, order, vstart, vslot, nat, k_next, compl_out, N);
    else if (N.next.stage)
      verlet_pairs_as<S, HO, 1>(st, P, V, order, vstart, vslot, nat, k_next, compl_out, N);
    else
      verlet_pairs_as<S, HO, 2>(st, P, V, order, vstart, vslot, nat, k_next, compl_out, N);
  };
  if (P.s == 3)
    as(std::integral_constant<int, 3>{}, std::false_type{});
  else if (P.higher_order)
    as(std::integral_constant<int, 4>{}, std::true_type{});
  else
    as(std::integral_constant<int, 4>{}, std::false_type{});
}

void launch_rk4_combine(hipStream_t st, int s, int n, double *state, const double *k1, const double *k2,
                        const double *k3, const double *k4, double dt, double *max_partial) {
  SPSS_DISPATCH_S(s, k_rk4_combine<SS><<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, state, k1, k2, k3, k4, dt, max_partial));
}

void launch_euler(hipStream_t st, int s, int n, double *state, const double *f, double dt, double sqrt_dt,
                  double int_phi, double int_r, int noise_mode, const double *noise, uint64_t seed, uint64_t step,
                  double *max_partial) {
  SPSS_DISPATCH_S(s, k_euler<SS><<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, state, f, dt, sqrt_dt, int_phi, int_r, noise_mode, noise, seed, step, max_partial));
}

void launch_srk(hipStream_t st, int n, double *state, const double *f, const double *C, double dt, double sqrt_dt,
                double c15, double is3, double sq2d, double friction, int noise_mode, const double *noise,
                uint64_t seed, uint64_t step, double *max_partial) {
  k_srk<<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, state, f, C, dt, sqrt_dt, c15, is3, sq2d, friction, noise_mode, noise, seed, step, max_partial);
}

void launch_max_final(hipStream_t st, int nb, const double *partial, double *out) {
  k_max_final<<<dim3(1), dim3(kBlock), 0, st>>>(nb, partial, out);
}

void launch_disp_max(hipStream_t st, int n, int s, const double *tot, double *partial) {
  k_disp_max<<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, s, tot, partial);
}

void launch_order_parameter(hipStream_t st, int n, int s, int slot, const double *state, double *partial,
                            double *out) {
  const int nb = (int)nblk(n);
  k_order_partial<<<dim3(nb), dim3(kBlock), 0, st>>>(n, s, slot, state, partial);
  k_order_final<<<dim3(1), dim3(128), 0, st>>>(nb, partial, (double)n, out);
}

void launch_apply_pbc(hipStream_t st, int n, int s, double *state, double xs, double ys, double xrs, double yrs) {
  k_apply_pbc<<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, s, state, xs, ys, xrs, yrs);
}

void launch_accumulate(hipStream_t st, long m, const double *state, double *acc) {
  k_accumulate<<<dim3(nblk(m)), dim3(kBlock), 0, st>>>(m, state, acc);
}

void launch_fill_double(hipStream_t st, long m, double *p, double v) {
  if (m > 0) k_fill_double<<<dim3(nblk(m)), dim3(kBlock), 0, st>>>(m, p, v);
}

void launch_copy16(hipStream_t st, long n16, const void *src, void *dst) {
  if (n16 > 0)
    k_copy16<<<dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st>>>(n16, (const uint4 *)src, (uint4 *)dst);
}

void launch_fill_int(hipStream_t st, long m, int *p, int v) {
  if (m > 0) k_fill_int<<<dim3(nblk(m)), dim3(kBlock), 0, st>>>(m, p, v);
}

void launch_iota(hipStream_t st, int n, int *p) {
  if (n > 0) k_iota<<<dim3(nblk(n)), dim3(kBlock), 0, st>>>(n, p);
}

}  // namespace spss
