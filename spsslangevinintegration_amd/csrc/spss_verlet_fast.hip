// spss_verlet_fast.hip -- Verlet neighbour lists in FP32C precision (exact mode): models 3 and 4,
// stochastic Euler and Runge-Kutta steps, rebuilds decided on the device.
//
// Reference: EvaluateInteractionsWithVerletNeighborList and ...WithLinkedListAndVerletNeighborList
// (ParticleSystemFirstOrderPtr.cpp:470-815) with CalculateMaxDisplacement (:836-861), in this
// library's exact mode: r_max = rho + skin, candidates from cells of side >= r_max, so every list
// holds every j within r_max and each step's neighbour set is {j : |r_ij| <= rho} whatever the
// rebuild schedule.  The schedule itself follows the exact mode of the FP64 path: after every
// step acc += sqrt(max_i |dr_i|^2), rebuild when acc + that step's value > (r_max - rho) / 2.
//
// Layout (the resident copy): particles in the cell order of the last rebuild on a grid of
// side Hv = 1/int(1/r_max); between rebuilds they keep their slots.  Per slot: FP64 state
// (double-buffered by step), id, natural frequency, cell, FP32 snapshot {x, y, cos phi, sin phi} and
// FP32 omega (double-buffered with the state).
//
// Grids of at most kRowTileCols columns have row tiles of the rebuild's cell order (spans of whole
// cells of one row, as for the cell-list pair kernel).  The step is one workgroup per tile: the 3 x (W + 2)
// cells around its W cells go into LDS and the sums over the particles within rho come from the matrix
// cores (spss_mfma_pairs.hpp).  The cells of the last rebuild hold every candidate until the next one,
// so no list is read; the tiles that overflow the stage or a workgroup walk those cells (vt_rest), and lists
// are built for vf_lists alone, from the state that the last rebuild left in the scratch arrays.  Snapshots of tiled
// grids hold positions from the centre of the particle's cell.  At N = 1M, 53 neighbours, skin
// 0.2 rho, stochastic Runge-Kutta: 113 us per step (about a third each: staging, sums, update), where walking
// 16-bit lists from LDS took 125, bound by LDS reads, and building them 190 per rebuild.
//
// Wider grids keep an ELL list of width K per slot with its length, in blocks of 256 slots and chunks of
// four entries (lslot), and walk it through global memory (vr_lists, vs_step): FP32 distances as
// x_j - x_i minus its nearest integer, sixteen entries per pass, phasor sums in four FP32 partials
// flushed into FP64.  Either way a guard band around rho^2 is decided with the reference's FP64 ClassC
// formula on the stored positions, so neighbour sets are exact.
//
// One step is a rebuild -- launches that return at once unless the device flag asks for one:
// the flag, cell keys and histogram; the scan's blocks; starts and bucket fill; stable rank and gather into
// scratch with the row tiles; back into the resident arrays with the new snapshot -- and the step,
// which ends with the Euler/SRK update of step_particle, the new snapshot and the step's largest
// squared displacement (maxima by group of workgroups), which the next step's first launch turns into its
// flag on the device.  No host synchronisation: steps replay from HIP graphs.  Seven launches (tiled
// grids): at N = 16,384 they are the step's time, 29 us, where ten took 34.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/spss_hip.h"
#include "spss_launch.hpp"
#include "spss_mfma_pairs.hpp"
#include "spss_scan.hpp"
#include "spss_step.hpp"
#include "spss_tiles.hpp"
#include "spss_verlet_fast.hpp"

namespace spss {

namespace {
thread_local std::string g_verr;
constexpr int kVB = 256;         // threads per workgroup
constexpr int kVGraphSteps = 10;  // steps of the bulk graph (even: the state buffers end where they started)
constexpr int kGateGrid = 1024;   // workgroups of the launches that run on rebuilds only
}  // namespace

// device control block
constexpr int kGroups = 64, kLineU64 = 16;  // workgroup groups of the displacement maximum, a 128-byte line each
struct VCtl {
  int flag;                     // rebuild before this step (should_update_lists_), set by vr_keys
  int force;                    // the resident copy was just entered: rebuild
  double acc[2];                // accumulated_displacement_, by the parity of the step that reads it
  unsigned long long step;      // Philox step of graph-replayed steps
  int nrest;                    // items of vt_rest since the last rebuild
  int pad;
  // the last step's largest |dr|^2 by group of workgroups (workgroup b in group b % kGroups), as the
  // bits of a non-negative double, one word per cache line so that the groups' atomics run apart
  unsigned long long gmax[kGroups * kLineU64];
};

struct VArgs {
  int n, ncv, cells, K;
  double rmax2;           // FP64 list radius squared
  double half_skin;       // (r_max - rho) / 2
  double h;               // the cells' side, 1 / ncv
  float r2c, r2h, r2k;    // guard band around rho^2: |d^2 - r2c| <= r2h is decided in FP64
  float m2c, m2h;         // guard band around r_max^2 (list build)
  float unit, rho_u, r2_u, drift;  // tiled grids: kMUnit per cell side; rho, rho^2 and 1 + half the skin in units
  VCtl *ctl;
};

__device__ __forceinline__ bool gate_off(const VArgs &A) { return A.ctl->flag == 0; }

// a row or column at most one outside the grid
__device__ __forceinline__ int wrap_row(int c, int nc) { return c < 0 ? c + nc : (c >= nc ? c - nc : c); }

// device addresses of fields of the control block, formed on the host without dereferencing it
static int *ctl_flag(VCtl *c) { return reinterpret_cast<int *>(reinterpret_cast<char *>(c) + offsetof(VCtl, flag)); }
static unsigned long long *ctl_step(VCtl *c) {
  return reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(c) + offsetof(VCtl, step));
}

// snapshot entry: wrapped position and unit phasor, each computed in FP64 and rounded once
__device__ __forceinline__ float4 vsnap_of(const DevParams &P, const double *st) {
  double xw, yw, sn, cn;
  apply_pbc(P, st[0], st[1], xw, yw);
  phasor_of(st[2], sn, cn);
  return make_float4((float)xw, (float)yw, (float)cn, (float)sn);
}

// the snapshot of a tiled grid: the position from the centre of the particle's cell of the last rebuild
// (nearest image), which FP32 holds to 2^-24 of the cell instead of the box
__device__ __forceinline__ float4 vsnap_cell(const DevParams &P, const double *st, int cx, int cy, double h) {
  double xw, yw, sn, cn;
  apply_pbc(P, st[0], st[1], xw, yw);
  xw -= ((double)cx + 0.5) * h;
  yw -= ((double)cy + 0.5) * h;
  xw -= rint(xw);
  yw -= rint(yw);
  phasor_of(st[2], sn, cn);
  return make_float4((float)xw, (float)yw, (float)cn, (float)sn);
}

// FP32 squared minimum-image distance minus c2
__device__ __forceinline__ float dd_of(float4 o, float xi, float yi, float c2) {
  float dx = o.x - xi;
  dx -= __builtin_rintf(dx);
  float dy = o.y - yi;
  dy -= __builtin_rintf(dy);
  return __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, -c2));
}

// entry t of slot p in the ELL lists of width K (a multiple of 16): blocks of 256 slots, inside a
// block chunks of 4 consecutive entries of one slot, slot-major (the chunks of entries 4c..4c+3 of
// the block's 256 slots side by side).  A builder writes a slot's entries four at a time, the loads
// of a chunk by a wave's lanes are one contiguous run, and a particle's entries lie 4 KB apart
// (with one n-long array per entry they would each sit on a page of their own).
__host__ __device__ __forceinline__ long lslot(long p, long t, int K) {
  return ((((p >> 8) * (K >> 2) + (t >> 2)) * 256 + (p & 255)) << 2) + (t & 3);
}

// ---------------------------------------------------------------------------
// rebuild (every launch returns at once when the flag is clear)

// Before the rest: CalculateMaxDisplacement's bookkeeping (ParticleSystemFirstOrderPtr.cpp:851-860) in
// the exact mode (one step of margin) from the last step's group maxima, by every wave for itself; the
// first workgroup leaves the result for the launches after this one, and advances the graph's Philox step.
template <int S>
__global__ __launch_bounds__(kVB) void vr_keys(DevParams P, VArgs A, int parity, unsigned long long *step_inc,
                                               const double *__restrict__ state, int *__restrict__ key,
                                               int *__restrict__ slotc, int *__restrict__ count) {
  {
    double m = __longlong_as_double((long long)A.ctl->gmax[(threadIdx.x & 63) * kLineU64]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    const double stepd = sqrt(m), acc = A.ctl->acc[parity] + stepd;
    const int flag = A.ctl->force || acc + stepd > A.half_skin;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      A.ctl->flag = flag;
      if (flag) A.ctl->nrest = 0;  // vr_settle adds them again
      A.ctl->acc[1 - parity] = flag ? 0.0 : acc;
      if (step_inc) *step_inc += 1ull;
    }
    if (!flag) return;
  }
  // the particles are in the last rebuild's cell order and have moved less than half the skin
  // since, so a wave holds a few runs of equal keys: one atomic per run, the run's lanes take
  // consecutive places after it (the order inside a cell is settled by vr_gather)
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int nwave = (A.n + 63) & ~63;  // every lane of a wave takes the same trips
  for (int p = blockIdx.x * kVB + threadIdx.x; p < nwave; p += gridDim.x * kVB) {
    const bool valid = p < A.n;
    int c = -1;
    if (valid) {
      double xw, yw;
      apply_pbc(P, state[(long)p * S], state[(long)p * S + 1], xw, yw);
      c = cell_coord(yw, A.ncv) * A.ncv + cell_coord(xw, A.ncv);
      key[p] = c;
    }
    const int pc = __shfl_up(c, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || pc != c);
    const int seg = 63 - __clzll((long long)(heads & (below | (1ull << lane))));  // this run's first lane
    int base = 0;
    if (valid && seg == lane) {
      const unsigned long long later = lane == 63 ? 0ull : heads >> (lane + 1);
      const int len = later ? __ffsll((long long)later) : 64 - lane;
      base = atomicAdd(count + c, len);
    }
    base = __shfl(base, seg, 64);
    if (valid) slotc[p] = base + (lane - seg);
  }
}

// the maxima cleared for this step, and the bucket fill.  local (grids of at most kScanLds scan blocks): the
// starts inside the scan blocks, completed here with the blocks' totals; the counts cleared for their
// next use
constexpr int kScanLds = 512;
__global__ __launch_bounds__(kVB) void vr_scatter(VArgs A, const int *__restrict__ key, const int *__restrict__ slotc,
                                                  const int *__restrict__ local, const int *__restrict__ blocksum,
                                                  int nsb, int *__restrict__ count, int *__restrict__ start,
                                                  int *__restrict__ tmp) {
  if (blockIdx.x == 0 && threadIdx.x < kGroups) {
    A.ctl->gmax[threadIdx.x * kLineU64] = 0ull;
    if (threadIdx.x == 0) A.ctl->force = 0;
  }
  if (gate_off(A)) return;
  if (!local) {
    for (int p = blockIdx.x * kVB + threadIdx.x; p < A.n; p += gridDim.x * kVB) tmp[start[key[p]] + slotc[p]] = p;
    return;
  }
  __shared__ int off[kScanLds];
  if (threadIdx.x < 64) {
    int run = 0;
    for (int b = threadIdx.x; b - (int)threadIdx.x < nsb; b += 64) {
      const int v = b < nsb ? blocksum[b] : 0, incl = wave_incl_scan(v, threadIdx.x);
      if (b < nsb) off[b] = run + incl - v;
      run += __shfl(incl, 63, 64);
    }
  }
  __syncthreads();
  for (int t = blockIdx.x * kVB + threadIdx.x; t < max(A.n, A.cells); t += gridDim.x * kVB) {
    if (t < A.n) {
      const int c = key[t];
      tmp[local[c] + off[c / (256 * kScanItems)] + slotc[t]] = t;
    }
    if (t < A.cells) {
      start[t] = local[t] + off[t / (256 * kScanItems)];
      count[t] = 0;
    }
    if (t == 0) start[A.cells] = A.n;
  }
}

// The row tiles of rows [4 * blockIdx.x, 4 * blockIdx.x + 4), a wave each.  A tile is no wider than its staged
// cells fit the stage, where those of a single column do: at 24 particles a cell one tile of a hundred would not
// by its particles alone, and a few tiles that walk lists hold up every step (1M particles: 8 us).
__device__ __forceinline__ void vt_tiles(const int *__restrict__ start, int nc, int wcap, int cmax,
                                         int4 *__restrict__ tiles) {
  __shared__ int R[6][kRowTileCols + 1];  // starts of the rows, and of those around them
  const int row0 = blockIdx.x * 4;
  for (int e = threadIdx.x; e < 6 * (nc + 1); e += kVB) {
    const int r = e / (nc + 1), row = row0 + r - 1;
    if (row <= nc) R[r][e - r * (nc + 1)] = start[wrap_row(row, nc) * nc + e - r * (nc + 1)];
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, row = row0 + w;
  if (row >= nc) return;
  const auto fits = [&](int a, int e) {
    int total = 0;
    for (int r = w; r < w + 3; ++r) {
      int v = R[r][min(e + 1, nc)] - R[r][max(a - 1, 0)];
      if (a == 0) v += R[r][nc] - R[r][nc - 1];
      if (e == nc) v += R[r][1] - R[r][0];
      total += (v + 15) & ~15;
    }
    return total <= kMStage;
  };
  row_tiles(R[w + 1], 0, row, nc, wcap, cmax, tiles + (long)row * cmax,
            [&](int a, int e) { return fits(a, e) || !fits(a, a + 1); });
}

// each cell's particles in ascending previous slot, gathered into the new order in scratch: cells
// of at most 64 particles one wave each (wave_sort64), then the particles of denser cells one
// thread each, ranked by counting (grid-stride over the particles: a dense cluster is spread over
// the whole grid)
template <int S>
__global__ __launch_bounds__(kVB) void vr_gather(VArgs A, const int *__restrict__ key, const int *__restrict__ start,
                                                 const int *__restrict__ tmp, const double *__restrict__ state,
                                                 const int *__restrict__ id, const double *__restrict__ nat,
                                                 double *__restrict__ sstate, int *__restrict__ sid,
                                                 double *__restrict__ snat, int *__restrict__ scell,
                                                 int4 *__restrict__ tiles, int wcap, int cmax) {
  if (gate_off(A)) return;
  // the row tiles of the new order (tiled grids), one wave per row in the first workgroups: they
  // need only the final cell starts
  if (tiles && (int)blockIdx.x * 4 < A.ncv) vt_tiles(start, A.ncv, wcap, cmax, tiles);
  const int lane = threadIdx.x & 63;
  auto move = [&](int p, int q, int c) {
#pragma unroll
    for (int k = 0; k < S; ++k) sstate[(long)q * S + k] = state[(long)p * S + k];
    sid[q] = id[p];
    if (nat) snat[q] = nat[p];
    scell[q] = c;
  };
  for (int c = blockIdx.x * (kVB / 64) + (threadIdx.x >> 6); c < A.cells; c += gridDim.x * (kVB / 64)) {
    const int b = start[c], m = start[c + 1] - b;
    if (m > 64) continue;  // the whole wave
    const int v = wave_sort64(lane < m ? tmp[b + lane] : 0x7fffffff, lane);
    if (lane < m) move(v, b + lane, c);
  }
  for (int p = blockIdx.x * kVB + threadIdx.x; p < A.n; p += gridDim.x * kVB) {
    const int c = key[p];
    const int b = start[c], e = start[c + 1];
    if (e - b <= 64) continue;
    int r = 0;
    for (int t = b; t < e; ++t) r += tmp[t] < p ? 1 : 0;
    move(p, b + r, c);
  }
}

// The lists: the candidates of the 3 x 3 cells around the particle's cell in the stencil order of
// ParticleSystemFirstOrderPtr.cpp:83-88, ascending slot inside a cell; j is listed when its
// distance from the wrapped x_i to the stored x_j is within r_max (:694-739).  FP32 test outside a
// guard band, the reference's FP64 ClassC formula inside it.
// The list of slot q read from global memory.
// EXACT: every pair by the FP64 formula (tiled grids, whose snapshots are relative to the cells).
template <int S, bool EXACT>
__device__ __forceinline__ void list_of_slot(const DevParams &P, const VArgs &A, const int *__restrict__ start,
                                             const int *__restrict__ cell, const double *__restrict__ state,
                                             const float4 *__restrict__ snap, int *__restrict__ list,
                                             int *__restrict__ len, int q) {
  const int c = cell[q];
  const int cx = c % A.ncv, cy = c / A.ncv;
  const float4 me = EXACT ? make_float4(0.f, 0.f, 0.f, 0.f) : snap[q];
  double xi, yi;
  apply_pbc(P, state[(long)q * S], state[(long)q * S + 1], xi, yi);
  int w = 0;
  for (int dyc = -1; dyc <= 1; ++dyc) {
    const int jy = adjust_cell(cy + dyc, A.ncv);
    for (int dxc = -1; dxc <= 1; ++dxc) {
      const int cj = jy * A.ncv + adjust_cell(cx + dxc, A.ncv);
      const int e = start[cj + 1];
      for (int u = start[cj]; u < e; ++u) {
        if (u == q) continue;
        const float dd = EXACT ? 0.f : dd_of(snap[u], me.x, me.y, A.m2c);
        bool in = dd < 0.f;
        if (EXACT || __builtin_fabsf(dd) <= A.m2h) {
          double dx, dy;
          class_c_unsigned(P, xi, yi, state[(long)u * S], state[(long)u * S + 1], dx, dy);
          in = dx * dx + dy * dy <= A.rmax2;
        }
        if (in) {
          if (w < A.K) list[lslot(q, w, A.K)] = u;
          ++w;
        }
      }
    }
  }
  // a list longer than the width is not stored: the step walks that particle's 3 x 3 cells instead
  len[q] = w <= A.K ? w : -1;
}

template <int S>
__global__ __launch_bounds__(kVB) void vr_lists(DevParams P, VArgs A, const int *__restrict__ start,
                                                const int *__restrict__ cell, const double *__restrict__ state,
                                                const float4 *__restrict__ snap, int *__restrict__ list,
                                                int *__restrict__ len) {
  if (gate_off(A)) return;
  const int q = blockIdx.x * kVB + threadIdx.x;
  if (q < A.n) list_of_slot<S, false>(P, A, start, cell, state, snap, list, len, q);
}

// ---------------------------------------------------------------------------
// the step

// Four candidates against particle p: weights, phasor partials (and omega-weighted for SRK).  The
// candidates are list entries t .. t+3 of slot p (CELLS = false) or the slots t .. t+3 of a cell of
// the last rebuild (CELLS = true: a particle whose list outgrew the width; p itself is skipped).
// TAIL: only those below `end` count.
template <int S, bool SRK, bool TAIL, bool CELLS>
__device__ __forceinline__ void walk4(const DevParams &P, const VArgs &A, const int *__restrict__ list,
                                      const float4 *__restrict__ snap, const float *__restrict__ omega,
                                      const double *__restrict__ state, int p, int t, int end, float xi, float yi,
                                      const double *pi, float *ax, float *ay, float &an, float *bx, float *by) {
  int j[4];
  float4 o[4];
  float dd[4], m[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool in = !TAIL || t + k < end;
    j[k] = CELLS ? (in ? t + k : p) : (in ? list[lslot(p, t + k, A.K)] : p);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    o[k] = snap[j[k]];
    dd[k] = dd_of(o[k], xi, yi, A.r2c);
    m[k] = __builtin_amdgcn_fmed3f(-A.r2k * dd[k], 0.f, 1.f);
  }
  const float dmin = __builtin_fminf(__builtin_fminf(__builtin_fabsf(dd[0]), __builtin_fabsf(dd[1])),
                                     __builtin_fminf(__builtin_fabsf(dd[2]), __builtin_fabsf(dd[3])));
  if (dmin <= A.r2h) {  // rare: the reference's FP64 test (x_i as stored, rhs_verlet's :566-581)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (__builtin_fabsf(dd[k]) <= A.r2h) {
        double dx, dy;
        class_c_unsigned(P, pi[0], pi[1], state[(long)j[k] * S], state[(long)j[k] * S + 1], dx, dy);
        m[k] = dx * dx + dy * dy <= P.rho2 ? 1.f : 0.f;
      }
  }
  if (TAIL || CELLS) {
#pragma unroll
    for (int k = 0; k < 4; ++k) m[k] = ((!TAIL || t + k < end) && (!CELLS || j[k] != p)) ? m[k] : 0.f;
  }
  an += (m[0] + m[1]) + (m[2] + m[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    ax[k] = __builtin_fmaf(m[k], o[k].z, ax[k]);
    ay[k] = __builtin_fmaf(m[k], o[k].w, ay[k]);
    if (SRK) {
      const float mo = m[k] * omega[j[k]];
      bx[k] = __builtin_fmaf(mo, o[k].z, bx[k]);
      by[k] = __builtin_fmaf(mo, o[k].w, by[k]);
    }
  }
}

// candidates [a, b) (list entries, or cell slots with CELLS) in groups of four, four FP32 partials per
// sum flushed into FP64 every 16 candidates
template <int S, bool SRK, bool CELLS>
__device__ __forceinline__ void walk_range(const DevParams &P, const VArgs &A, const int *__restrict__ list,
                                           const float4 *__restrict__ snap, const float *__restrict__ omega,
                                           const double *__restrict__ state, int p, int a, int b, float xi, float yi,
                                           const double *pi, double &sx, double &sy, double &tx, double &ty,
                                           int &nnb) {
  for (int t0 = a; t0 < b; t0 += 16) {
    float ax[4] = {0.f, 0.f, 0.f, 0.f}, ay[4] = {0.f, 0.f, 0.f, 0.f}, an = 0.f;
    float bx[4] = {0.f, 0.f, 0.f, 0.f}, by[4] = {0.f, 0.f, 0.f, 0.f};
    const int te = min(t0 + 16, b);
    int t = t0;
    for (; t + 4 <= te; t += 4)
      walk4<S, SRK, false, CELLS>(P, A, list, snap, omega, state, p, t, te, xi, yi, pi, ax, ay, an, bx, by);
    if (t < te) walk4<S, SRK, true, CELLS>(P, A, list, snap, omega, state, p, t, te, xi, yi, pi, ax, ay, an, bx, by);
    sx += ((double)ax[0] + (double)ax[1]) + ((double)ax[2] + (double)ax[3]);
    sy += ((double)ay[0] + (double)ay[1]) + ((double)ay[2] + (double)ay[3]);
    nnb += (int)an;
    if (SRK) {
      tx += ((double)bx[0] + (double)bx[1]) + ((double)bx[2] + (double)bx[3]);
      ty += ((double)by[0] + (double)by[1]) + ((double)by[2] + (double)by[3]);
    }
  }
}

// The list entries [0, L) of slot p, sixteen per pass, in the order and 4-slot grouping of
// walk_range: each half of a pass issues its eight list loads, then its eight gathers of the
// snapshot (and omega), before any arithmetic, so a wave keeps eight dependent load pairs in
// flight instead of four; entries past L are the slot itself with weight zero.
template <int S, bool SRK>
__device__ __forceinline__ void walk_list(const DevParams &P, const VArgs &A, const int *__restrict__ list,
                                          const float4 *__restrict__ snap, const float *__restrict__ omega,
                                          const double *__restrict__ state, int p, int L, float xi, float yi,
                                          const double *pi, double &sx, double &sy, double &tx, double &ty,
                                          int &nnb) {
  for (int t0 = 0; t0 < L; t0 += 16) {
    float ax[4] = {0.f, 0.f, 0.f, 0.f}, ay[4] = {0.f, 0.f, 0.f, 0.f}, an = 0.f;
    float bx[4] = {0.f, 0.f, 0.f, 0.f}, by[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 16; h += 8) {
      int j[8];
      float4 o[8];
      float om[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) j[k] = t0 + h + k < L ? list[lslot(p, t0 + h + k, A.K)] : p;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        o[k] = snap[j[k]];
        if (SRK) om[k] = omega[j[k]];
      }
#pragma unroll
      for (int g = 0; g < 8; g += 4) {
        float dd[4], m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          dd[k] = dd_of(o[g + k], xi, yi, A.r2c);
          m[k] = __builtin_amdgcn_fmed3f(-A.r2k * dd[k], 0.f, 1.f);
        }
        const float dmin = __builtin_fminf(__builtin_fminf(__builtin_fabsf(dd[0]), __builtin_fabsf(dd[1])),
                                           __builtin_fminf(__builtin_fabsf(dd[2]), __builtin_fabsf(dd[3])));
        if (dmin <= A.r2h) {  // rare: the reference's FP64 test, as in walk4
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (__builtin_fabsf(dd[k]) <= A.r2h) {
              double dx, dy;
              class_c_unsigned(P, pi[0], pi[1], state[(long)j[g + k] * S], state[(long)j[g + k] * S + 1], dx, dy);
              m[k] = dx * dx + dy * dy <= P.rho2 ? 1.f : 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) m[k] = t0 + h + g + k < L ? m[k] : 0.f;
        an += (m[0] + m[1]) + (m[2] + m[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          ax[k] = __builtin_fmaf(m[k], o[g + k].z, ax[k]);
          ay[k] = __builtin_fmaf(m[k], o[g + k].w, ay[k]);
          if (SRK) {
            const float mo = m[k] * om[g + k];
            bx[k] = __builtin_fmaf(mo, o[g + k].z, bx[k]);
            by[k] = __builtin_fmaf(mo, o[g + k].w, by[k]);
          }
        }
      }
    }
    sx += ((double)ax[0] + (double)ax[1]) + ((double)ax[2] + (double)ax[3]);
    sy += ((double)ay[0] + (double)ay[1]) + ((double)ay[2] + (double)ay[3]);
    nnb += (int)an;
    if (SRK) {
      tx += ((double)bx[0] + (double)bx[1]) + ((double)bx[2] + (double)bx[3]);
      ty += ((double)by[0] + (double)by[1]) + ((double)by[2] + (double)by[3]);
    }
  }
}

// workgroups in an XCD-aware order: the hardware deals consecutive workgroups to the 8 XCDs in
// turn, so workgroup b takes the particle block (b % 8) * per + b / 8 and every XCD walks one
// contiguous eighth of the slots (neighbours' snapshots then stay in that XCD's L2); the grid is
// a multiple of 8 and blocks past the slots only take part in the displacement maximum
__device__ __forceinline__ int xcd_block(int b, int nblocks) {
  const int per = nblocks >> 3;
  return (b & 7) * per + (b >> 3);
}

// The step's largest squared displacement, for the next step's vr_keys: wave, workgroup, then one atomic per
// workgroup on the maximum of its group (kGroups words on their own cache lines).  (A last-workgroup
// count in the step kernel needs a release fence per workgroup, which writes the XCD's L2 back:
// 0.45 ms per step at N = 1M with 7,000 workgroups.)
__device__ __forceinline__ void step_max(const VArgs &A, double d2, double *wred) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) d2 = fmax(d2, __shfl_xor(d2, o, 64));
  if ((threadIdx.x & 63) == 0) wred[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double bm = wred[0];
    for (int w = 1; w < kVB / 64; ++w) bm = fmax(bm, wred[w]);
    if (bm > 0.0)
      atomicMax(&A.ctl->gmax[(blockIdx.x & (kGroups - 1)) * kLineU64], (unsigned long long)__double_as_longlong(bm));
  }
}

template <int S, bool SRK>
__global__ __launch_bounds__(kVB) void vs_step(DevParams P, VArgs A, StepArgs U, const int *__restrict__ list,
                                               const int *__restrict__ len, const int *__restrict__ start,
                                               const int *__restrict__ cell, const double *__restrict__ state,
                                               const int *__restrict__ id, const double *__restrict__ nat,
                                               const float4 *__restrict__ snap, const float *__restrict__ omega,
                                               double *__restrict__ nstate, float4 *__restrict__ nsnap,
                                               float *__restrict__ nomega, double *__restrict__ compl_out) {
  __shared__ double wmax[kVB / 64];
  const int p = xcd_block((int)blockIdx.x, (int)gridDim.x) * kVB + threadIdx.x;
  double d2 = 0.0;
  if (p < A.n) {
    const double *pi = state + (long)p * S;
    const float4 me = snap[p];
    const int L = len[p];
    double sx = 0.0, sy = 0.0, tx = 0.0, ty = 0.0;
    int nnb = 0;
    if (L >= 0) {
      walk_list<S, SRK>(P, A, list, snap, omega, state, p, L, me.x, me.y, pi, sx, sy, tx, ty, nnb);
    } else {  // (rare) the list outgrew the width: the 3 x 3 cells of the last rebuild hold every candidate
      const int c = cell[p];
      const int cx = c % A.ncv, cy = c / A.ncv;
      for (int dyc = -1; dyc <= 1; ++dyc)
        for (int dxc = -1; dxc <= 1; ++dxc) {
          const int cj = adjust_cell(cy + dyc, A.ncv) * A.ncv + adjust_cell(cx + dxc, A.ncv);
          walk_range<S, SRK, true>(P, A, list, snap, omega, state, p, start[cj], start[cj + 1], me.x, me.y, pi, sx,
                                   sy, tx, ty, nnb);
        }
    }
    Coef K;
    K.xi = P.xi;
    K.sigma = P.sigma;
    K.int_phi = U.int_phi;
    K.sq2d = U.sq2d;
    K.seed = U.seed;
    const uint64_t step = U.step_dev ? (uint64_t)*U.step_dev : U.step;
    const int i = id[p];
    double out[S], C;
    step_particle<S, SRK>(P, K, pi, i, nat ? nat[p] : 0.0, make_double2(sx, sy), make_double2(tx, ty), nnb, U,
                          step, out, C, &d2);
#pragma unroll
    for (int k = 0; k < S; ++k) nstate[(long)p * S + k] = out[k];
    nsnap[p] = vsnap_of(P, out);
    nomega[p] = S == 4 ? (float)out[3] : 0.f;
    if (SRK && compl_out) compl_out[i] = C;
  }
  step_max(A, d2, wmax);
}

// ---------------------------------------------------------------------------
// Row tiles of the rebuild's cell order (grids of at most kRowTileCols columns).  One workgroup
// per tile -- a span of whole cells of one row, as for the cell-list pair kernel -- stages the
// snapshots (and omega) of the 3 x (W + 2) cells around its W cells, which hold every candidate until
// the next rebuild, and takes the sums over them on the matrix cores (spss_mfma_pairs.hpp): a
// superset of the lists, whose pairs beyond rho count for nothing, with no list read.  Tiles whose cells
// overflow the stage or whose particles outnumber the workgroup walk those cells through global memory.

constexpr int kVCols = 48;  // staged columns W + 2

struct VtPlan {
  int cglob[3 * kVCols];                  // first slot of staged cell (r, q), at r * (W + 2) + q
  unsigned short cpos[3 * (kVCols + 1)];  // its start in staged row r, at r * (W + 3) + q, and behind it the row's end
  int len[3];                             // particles of the staged rows (cpos: meant for rows that fit the stage)
};

// the staging plan of tile (row, ca, cb): rows row-1 .. row+1, columns ca-1 .. cb (each wrapped
// once); returns the staged total of whole units per row (the same for every thread)
__device__ __forceinline__ int vt_plan(const VArgs &A, const int *__restrict__ start, int row, int ca, int cb,
                                       VtPlan &L) {
  const int ncols = cb - ca + 2, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (w < 3) {  // a wave per row, a lane per cell (at most kVCols): exclusive prefix of the counts
    int g0 = 0, v = 0;
    if (lane < ncols) {
      const int c = wrap_row(row + w - 1, A.ncv) * A.ncv + wrap_row(ca - 1 + lane, A.ncv);
      g0 = start[c];
      v = start[c + 1] - g0;
    }
    const int incl = wave_incl_scan(v, lane);
    if (lane < ncols) L.cglob[w * ncols + lane] = g0;
    if (lane <= ncols) L.cpos[w * (ncols + 1) + lane] = (unsigned short)(incl - v);
    if (lane == 63) L.len[w] = incl;
  }
  __syncthreads();
  return ((L.len[0] + 15) & ~15) + ((L.len[1] + 15) & ~15) + ((L.len[2] + 15) & ~15);
}

// whether a workgroup of vt_step takes a tile of nt particles and that staged total; the others are cut into items
constexpr int kRestItem = 64;
__device__ __forceinline__ bool vt_takes(int total, int nt) { return total <= kMStage && nt <= kVB; }

// back into the resident arrays, with the snapshot of the new order
template <int S>
__global__ __launch_bounds__(kVB) void vr_settle(DevParams P, VArgs A, const double *__restrict__ sstate,
                                                 const int *__restrict__ sid, const double *__restrict__ snat,
                                                 const int *__restrict__ scell, double *__restrict__ state,
                                                 int *__restrict__ id, double *__restrict__ nat,
                                                 int *__restrict__ cell, float4 *__restrict__ snap,
                                                 float *__restrict__ omega, const int *__restrict__ start,
                                                 const int4 *__restrict__ tiles, int ntiles, int2 *__restrict__ rest) {
  if (gate_off(A)) return;
  for (int q = blockIdx.x * kVB + threadIdx.x; q < A.n; q += gridDim.x * kVB) {
    double st[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
      st[k] = sstate[(long)q * S + k];
      state[(long)q * S + k] = st[k];
    }
    id[q] = sid[q];
    if (nat) nat[q] = snat[q];
    const int c = scell[q];
    cell[q] = c;
    snap[q] = tiles ? vsnap_cell(P, st, c % A.ncv, c / A.ncv, A.h) : vsnap_of(P, st);
    omega[q] = S == 4 ? (float)st[3] : 0.f;
  }
  // tiled grids: the tiles that the workgroups of vt_step cannot take, in items of vt_rest
  __shared__ VtPlan L;
  __shared__ int at;
  for (int tile = tiles ? blockIdx.x : ntiles; tile < ntiles; tile += gridDim.x) {  // (the same for the whole workgroup)
    const int4 td = tiles[tile];
    const int row = td.y, ca = td.z, cb = td.w;
    if (ca >= cb) continue;  // an unused tile slot
    __syncthreads();  // the previous tile's plan is consumed
    const int total = vt_plan(A, start, row, ca, cb, L);
    const int gtb = start[row * A.ncv + ca], nt = start[row * A.ncv + cb] - gtb;
    if (vt_takes(total, nt)) continue;
    const int items = (nt + kRestItem - 1) / kRestItem;
    if (threadIdx.x == 0) at = atomicAdd(&A.ctl->nrest, items);
    __syncthreads();
    for (int u = threadIdx.x; u < items; u += kVB)
      rest[at + u] = make_int2(gtb + u * kRestItem, min(kRestItem, nt - u * kRestItem));
  }
}

template <int W>
struct VtLds {
  MStage<W> M;
  VtPlan plan;
  unsigned char col[kVB];  // staged column of the tile's particles
  float most[kVB / 64][3];  // of the waves' staged values
  double wmax[kVB / 64];
};

// The sums of the tile's particles over the staged cells.  Positions are
// taken from the tile's centre.  False: a staged value is not finite (the same for every thread).
template <int S, int W>
__device__ __forceinline__ bool vt_sums(const DevParams &P, const VArgs &A, int row, int ca, int cb, int gtb, int ntile,
                                        const int *__restrict__ cell, const double *__restrict__ state,
                                        const float4 *__restrict__ snap, const float *__restrict__ omega,
                                        VtLds<W> &Ls, MSums &sum) {
  constexpr int kPasses = 5;  // chunks of 64 entries per wave: at most kMStage / 64 and two for the rows' rests
  const VtPlan &L = Ls.plan;
  const int ncols = cb - ca + 2, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l0 = __builtin_amdgcn_readfirstlane(L.len[0]), l1 = __builtin_amdgcn_readfirstlane(L.len[1]);
  const int l2 = __builtin_amdgcn_readfirstlane(L.len[2]);
  const int b1 = (l0 + 15) & ~15, b2 = b1 + ((l1 + 15) & ~15);
  // positions from the tile's centre, the cell's side kMUnit; |x| <= xm with the particles within half the
  // skin of their cells.  A coordinate is rounded to 22 bits, so separations up to rho err by 2^-22 xm:
  // `tight` is twice what d^2 errs by.  The product's roundings are at most 96 of 2^-24 of |x|^2 on top.
  const float unit = A.unit, r2 = A.r2_u;
  const float xm = 0.5f * kMUnit * (float)(cb - ca) + A.drift, ym = 0.5f * kMUnit + A.drift;
  const float tight = 0x1p-20f * A.rho_u * (xm + ym + A.rho_u), band = tight + 96.f * 0x1p-24f * (xm * xm + ym * ym);

  // the staged particles: a row's cells are one run of slots, but for a first column left of the box
  // and a last one right of it
  const bool lw = ca == 0, rw = cb == A.ncv;
  const int s0 = __builtin_amdgcn_readfirstlane(L.cglob[0]), s1 = __builtin_amdgcn_readfirstlane(L.cglob[ncols]);
  const int s2 = __builtin_amdgcn_readfirstlane(L.cglob[2 * ncols]);
  // the number of a cell of staged column 0 (of any row's extension to the left)
  const int f0 = wrap_row(row - 1, A.ncv) * A.ncv + ca - 1, f1 = row * A.ncv + ca - 1;
  const int f2 = wrap_row(row + 1, A.ncv) * A.ncv + ca - 1;
  const int c0 = (l0 + 63) >> 6, c1 = c0 + ((l1 + 63) >> 6), c2 = c1 + ((l2 + 63) >> 6);
  float4 v[kPasses];
  float om[kPasses], most[3] = {0.f, 0.f, 0.f};  // the largest |omega|, |cos phi|, |sin phi|; infinite: not all are finite
  int at[kPasses], to[kPasses];  // first entry of the wave's chunk; entries of its row from there
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int ch = 4 * p + wave;
    const int r = ch < c0 ? 0 : (ch < c1 ? 1 : 2), t0 = 64 * (ch - (r == 0 ? 0 : (r == 1 ? c0 : c1)));
    at[p] = (r == 0 ? 0 : (r == 1 ? b1 : b2)) + t0;
    to[p] = ch < c2 ? (r == 0 ? l0 : (r == 1 ? l1 : l2)) - t0 : 0;
    v[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    om[p] = 0.f;
    if (lane < to[p]) {
      const int t = t0 + lane;
      int g = (r == 0 ? s0 : (r == 1 ? s1 : s2)) + t;
      int q;  // staged column
      if (lw || rw) {
        const int e = r * (ncols + 1);
        const bool left = lw && t < L.cpos[e + 1], right = rw && t >= L.cpos[e + ncols - 1];
        const int c = left ? 0 : (right ? ncols - 1 : (lw ? 1 : 0));
        g = L.cglob[r * ncols + c] + (t - L.cpos[e + c]);
        q = left ? 0 : (right ? ncols - 1 : cell[g] - (r == 0 ? f0 : (r == 1 ? f1 : f2)));
      } else {
        q = cell[g] - (r == 0 ? f0 : (r == 1 ? f1 : f2));
      }
      v[p] = snap[g];
      if (W == kMOmega) om[p] = omega[g];
      v[p].x = __builtin_fmaf(v[p].x, unit, kMUnit * ((float)q - 0.5f * (float)(cb - ca + 1)));
      v[p].y = __builtin_fmaf(v[p].y, unit, kMUnit * (float)(r - 1));
      const float big = __builtin_fabsf(v[p].x) + __builtin_fabsf(v[p].y) + __builtin_fabsf(v[p].z) +
                        __builtin_fabsf(v[p].w) + __builtin_fabsf(om[p]);
      most[0] = __builtin_fmaxf(most[0], big < 0x1p100f ? __builtin_fabsf(om[p]) : __builtin_inff());
      most[1] = __builtin_fmaxf(most[1], __builtin_fabsf(v[p].z));
      most[2] = __builtin_fmaxf(most[2], __builtin_fabsf(v[p].w));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) most[k] = __builtin_fmaxf(most[k], __shfl_xor(most[k], o, 64));
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 3; ++k) Ls.most[wave][k] = most[k];
  if ((int)threadIdx.x < ntile) Ls.col[threadIdx.x] = (unsigned char)(cell[gtb + threadIdx.x] - row * A.ncv - ca + 1);
  m_init(Ls.M);
  __syncthreads();
  MScale scale[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float m = __builtin_fmaxf(__builtin_fmaxf(Ls.most[0][k], Ls.most[1][k]), __builtin_fmaxf(Ls.most[2][k], Ls.most[3][k]));
    if (k == 0 && !(m < 0x1p100f)) return false;
    scale[k] = m_scale(m, k == 0 ? kMMarkOmega : kMMark);
  }
  const float uo = ldexpf(1.f, scale[0].up), uc = ldexpf(1.f, scale[1].up), us = ldexpf(1.f, scale[2].up);
#pragma unroll
  for (int p = 0; p < kPasses; ++p)
    if (lane < ((to[p] + 15) & ~15))
      m_write<W>(Ls.M, at[p] + lane, lane < to[p], v[p].x, v[p].y, v[p].z * uc, v[p].w * us, om[p] * uo, scale[1],
                 scale[2], scale[0]);
  __syncthreads();
  const int first = b1 + L.cpos[ncols + 2] + 64 * wave, count = min(max(ntile - 64 * wave, 0), 64);
  if (count == 0) return true;
  const int p = gtb + 64 * wave + lane;
  const float4 me = lane < count ? snap[p] : make_float4(0.f, 0.f, 0.f, 0.f);
  const float mo = W == kMOmega && lane < count ? omega[p] : 0.f;
  sum = m_sums<W>(
      Ls.M, first, count, 3, r2, band, me.z * uc, me.w * us, mo * uo, scale[1], scale[2], scale[0],
      [&](int i, int r, int &a, int &b) {
        const int e = r * (ncols + 1), base = r == 0 ? 0 : (r == 1 ? b1 : b2);
        a = base + L.cpos[e + Ls.col[64 * wave + i] - 1];
        b = base + L.cpos[e + Ls.col[64 * wave + min(i + 15, count - 1)] + 2];
      },
      [&](int i, int e) {
        // differences of the staged positions first: their band is narrower
        const uint2 pe = m_pos(Ls.M, e), po = m_pos(Ls.M, first + i);
        const float dx = m_value(pe.x) - m_value(po.x), dy = m_value(pe.y) - m_value(po.y);
        const float dd = __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, -r2));
        if (__builtin_fabsf(dd) > tight) return dd < 0.f;
        // the reference's FP64 test (x_i as stored, rhs_verlet's :566-581)
        const int r = e < b1 ? 0 : (e < b2 ? 1 : 2), t = e - (r == 0 ? 0 : (r == 1 ? b1 : b2));
        const unsigned short *cpos = L.cpos + r * (ncols + 1);
        int q = 0, hi = ncols - 1;  // the last cell that starts at or before t holds it
        while (q < hi) {
          const int mid = (q + hi + 1) >> 1;
          if (cpos[mid] <= t) q = mid; else hi = mid - 1;
        }
        const double *pi = state + (long)(gtb + 64 * wave + i) * S;
        const double *pj = state + (long)(L.cglob[r * ncols + q] + t - cpos[q]) * S;
        double ddx, ddy;
        class_c_unsigned(P, pi[0], pi[1], pj[0], pj[1], ddx, ddy);
        return ddx * ddx + ddy * ddy <= P.rho2;
      });
  return true;
}

// The sums of slot p of a tiled grid through global memory, over a part of each of the 3 x 3 cells of the last
// rebuild: FP32 distances between snapshots, which are relative to their cells (their errors are within the
// guard band that vs_step's have), the band decided by the reference's FP64 test (x_i as stored, rhs_verlet's
// :566-581); phasor sums in four FP32 partials flushed into FP64 every U candidates.  Neighbouring lanes are
// particles of one cell and read the same candidates, in order, where lists of a dense cell scatter.
template <int S, bool SRK, int U>
__device__ __forceinline__ MSums vt_walk(const DevParams &P, const VArgs &A, const int *__restrict__ start,
                                         const int *__restrict__ cell, const double *__restrict__ state,
                                         const float4 *__restrict__ snap, const float *__restrict__ omega, int p,
                                         int part = 0, int parts = 1) {
  static_assert(U % 4 == 0 && U <= 16, "partials of four candidates at most");
  MSums m;
  const float4 me = snap[p];
  const double *pi = state + (long)p * S;
  const int c = cell[p], cx = c % A.ncv, cy = c / A.ncv;
  const float h = (float)A.h;
  for (int k = 0; k < 9; ++k) {
    const int dxc = k % 3 - 1, dyc = k / 3 - 1;
    const int cj = adjust_cell(cy + dyc, A.ncv) * A.ncv + adjust_cell(cx + dxc, A.ncv);
    const int first = start[cj], count = start[cj + 1] - first;
    const int b = first + (int)((long)count * (part + 1) / parts);
    const float xi = me.x - (float)dxc * h, yi = me.y - (float)dyc * h;
    for (int t0 = first + (int)((long)count * part / parts); t0 < b; t0 += U) {
      float4 o[U];
      float om[U], ax[4] = {}, ay[4] = {}, bx[4] = {}, by[4] = {};
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = min(t0 + u, b - 1);
        o[u] = snap[j];
        if (SRK) om[u] = omega[j];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dx = o[u].x - xi, dy = o[u].y - yi;
        const float dd = __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, -A.r2c));
        bool in = dd < 0.f;
        if (__builtin_fabsf(dd) <= A.r2h) {  // rare
          const double *pj = state + (long)min(t0 + u, b - 1) * S;
          double ddx, ddy;
          class_c_unsigned(P, pi[0], pi[1], pj[0], pj[1], ddx, ddy);
          in = ddx * ddx + ddy * ddy <= P.rho2;
        }
        in = in && t0 + u < b && t0 + u != p;
        m.n += in ? 1 : 0;
        ax[u & 3] += in ? o[u].z : 0.f;
        ay[u & 3] += in ? o[u].w : 0.f;
        if (SRK) {
          bx[u & 3] += in ? om[u] * o[u].z : 0.f;
          by[u & 3] += in ? om[u] * o[u].w : 0.f;
        }
      }
      m.sx += ((double)ax[0] + (double)ax[1]) + ((double)ax[2] + (double)ax[3]);
      m.sy += ((double)ay[0] + (double)ay[1]) + ((double)ay[2] + (double)ay[3]);
      if (SRK) {
        m.tx += ((double)bx[0] + (double)bx[1]) + ((double)bx[2] + (double)bx[3]);
        m.ty += ((double)by[0] + (double)by[1]) + ((double)by[2] + (double)by[3]);
      }
    }
  }
  return m;
}

// The step of slot p (vs_step's per-particle work) from its sums.  Returns |dr|^2.
template <int S, bool SRK>
__device__ __forceinline__ double vt_particle(const DevParams &P, const VArgs &A, const StepArgs &U, const Coef &K,
                                              uint64_t step, const double *__restrict__ state,
                                              const int *__restrict__ id, const double *__restrict__ nat,
                                              double *__restrict__ nstate, float4 *__restrict__ nsnap,
                                              float *__restrict__ nomega, double *__restrict__ compl_out,
                                              const MSums &m, int p, int cx, int cy) {
  const int i = id[p];
  double out[S], C, dp2;
  step_particle<S, SRK>(P, K, state + (long)p * S, i, nat ? nat[p] : 0.0, make_double2(m.sx, m.sy),
                        make_double2(m.tx, m.ty), m.n, U, step, out, C, &dp2);
#pragma unroll
  for (int k = 0; k < S; ++k) nstate[(long)p * S + k] = out[k];
  nsnap[p] = vsnap_cell(P, out, cx, cy, A.h);
  nomega[p] = S == 4 ? (float)out[3] : 0.f;
  if (SRK && compl_out) compl_out[i] = C;
  return dp2;
}

__device__ __forceinline__ Coef vt_coef(const DevParams &P, const StepArgs &U) {
  Coef K;
  K.xi = P.xi;
  K.sigma = P.sigma;
  K.int_phi = U.int_phi;
  K.sq2d = U.sq2d;
  K.seed = U.seed;
  return K;
}

// The particles of the tiles that vt_step's workgroups cannot take (cells of more than a hundred particles:
// dense clusters), 64 a workgroup, a quarter of the candidates per wave; launched before vt_step; their
// displacements join the group maxima too.  30,000 particles of 940 neighbours each: 118 us an Euler
// step (580 by walking lists, 1,267 by FP64 distances along them).
// (A launch of its own: as extra workgroups of vt_step, its particle loop would raise vt_step's registers.)
template <int S, bool SRK>
__global__ __launch_bounds__(kVB) void vt_rest(DevParams P, VArgs A, StepArgs U, const int2 *__restrict__ rest,
                                               const int *__restrict__ start, const int *__restrict__ cell,
                                               const double *__restrict__ state, const int *__restrict__ id,
                                               const double *__restrict__ nat, const float4 *__restrict__ snap,
                                               const float *__restrict__ omega, double *__restrict__ nstate,
                                               float4 *__restrict__ nsnap, float *__restrict__ nomega,
                                               double *__restrict__ compl_out) {
  static_assert(kRestItem == 64, "a lane per particle, in every wave");
  constexpr int kWaves = kVB / 64;
  __shared__ double sum[kWaves][SRK ? 4 : 2][64];
  __shared__ int num[kWaves][64];
  __shared__ double wmax[kWaves];
  const int items = A.ctl->nrest;
  if (items == 0) return;  // the usual case: every tile fits its workgroup
  const Coef K = vt_coef(P, U);
  const uint64_t step = U.step_dev ? (uint64_t)*U.step_dev : U.step;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double d2 = 0.0;
  for (int t = blockIdx.x; t < items; t += gridDim.x) {
    const int2 it = rest[t];
    const int p = it.x + min(lane, it.y - 1);
    MSums m = vt_walk<S, SRK, 8>(P, A, start, cell, state, snap, omega, p, w, kWaves);
    sum[w][0][lane] = m.sx;
    sum[w][1][lane] = m.sy;
    if (SRK) {
      sum[w][SRK ? 2 : 0][lane] = m.tx;
      sum[w][SRK ? 3 : 0][lane] = m.ty;
    }
    num[w][lane] = m.n;
    __syncthreads();
    if (w == 0 && lane < it.y) {
      const auto all = [&](int q) { return ((sum[0][q][lane] + sum[1][q][lane]) + sum[2][q][lane]) + sum[3][q][lane]; };
      m.sx = all(0);
      m.sy = all(1);
      if (SRK) {
        m.tx = all(SRK ? 2 : 0);
        m.ty = all(SRK ? 3 : 0);
      }
      m.n = num[0][lane] + num[1][lane] + num[2][lane] + num[3][lane];
      const int c = cell[p];
      d2 = fmax(d2, vt_particle<S, SRK>(P, A, U, K, step, state, id, nat, nstate, nsnap, nomega, compl_out, m, p,
                                        c % A.ncv, c / A.ncv));
    }
    __syncthreads();
  }
  step_max(A, d2, wmax);
}

// The step of a tile's particles, one per lane (vt_rest has the tiles that do not fit), and the step's
// largest displacement as in vs_step.
// (three workgroups per CU: no more registers than the vector ones, so that the products' results need
// not be moved out of the accumulation registers)
template <int S, bool SRK>
__global__ __launch_bounds__(kVB, 3) void vt_step(DevParams P, VArgs A, StepArgs U, const int4 *__restrict__ tiles,
                                               int ntiles, const int *__restrict__ start,
                                               const int *__restrict__ cell, const double *__restrict__ state,
                                               const int *__restrict__ id, const double *__restrict__ nat,
                                               const float4 *__restrict__ snap, const float *__restrict__ omega,
                                               double *__restrict__ nstate, float4 *__restrict__ nsnap,
                                               float *__restrict__ nomega, double *__restrict__ compl_out) {
  constexpr int W = SRK ? kMOmega : kMPlain;
  __shared__ VtLds<W> Ls;
  const int tile = xcd_block((int)blockIdx.x, (int)gridDim.x);
  const int4 td = tile < ntiles ? tiles[tile] : make_int4(0, 0, 0, 0);
  double d2 = 0.0;
  if (td.z < td.w) {  // the same for the whole workgroup
    const int row = td.y, ca = td.z, cb = td.w;
    const int total = vt_plan(A, start, row, ca, cb, Ls.plan);
    const int gtb = Ls.plan.cglob[cb - ca + 3];
    const int ntile = start[row * A.ncv + cb] - gtb;
    if (vt_takes(total, ntile)) {
      MSums sum;
      const bool have = vt_sums<S, W>(P, A, row, ca, cb, gtb, ntile, cell, state, snap, omega, Ls, sum);
      const int u = threadIdx.x, p = gtb + u;
      if (u < ntile) {
        // (rare) staged values that are not finite, or small ones beside a large one out of range
        if (!have || sum.n == kMOpen) sum = vt_walk<S, SRK, 4>(P, A, start, cell, state, snap, omega, p);
        d2 = vt_particle<S, SRK>(P, A, U, vt_coef(P, U), U.step_dev ? (uint64_t)*U.step_dev : U.step, state, id, nat,
                                 nstate, nsnap, nomega, compl_out, sum, p, cell[p] - row * A.ncv, row);
      }
    }
  }
  step_max(A, d2, Ls.wmax);
}

// the largest particle count of any 3 x 3 block of cells (the candidates of one list)
__global__ __launch_bounds__(kVB) void vc_block_max(VArgs A, const int *__restrict__ count, int *__restrict__ out) {
  const int c = blockIdx.x * kVB + threadIdx.x;
  if (c >= A.cells) return;
  const int cx = c % A.ncv, cy = c / A.ncv;
  int s = 0;
  for (int dy = -1; dy <= 1; ++dy)
    for (int dx = -1; dx <= 1; ++dx) s += count[adjust_cell(cy + dy, A.ncv) * A.ncv + adjust_cell(cx + dx, A.ncv)];
  atomicMax(out, s);
}

__global__ void vc_enter(VCtl *c) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    c->flag = c->force = 1;  // should_update_lists_ starts true (ParticleSystemFirstOrderPtr.cpp:99)
    c->acc[0] = c->acc[1] = 0.0;
  }
  for (int g = threadIdx.x; g < kGroups; g += blockDim.x) c->gmax[g * kLineU64] = 0ull;
}

__global__ void vc_set_step(VCtl *c, unsigned long long v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) c->step = v;
}

__global__ __launch_bounds__(kVB) void vc_iota(int n, int *__restrict__ id) {
  const int p = blockIdx.x * kVB + threadIdx.x;
  if (p < n) id[p] = p;
}

// the lists of the last rebuild from the state that it left in the scratch arrays
template <int S>
__global__ __launch_bounds__(kVB) void vc_lists(DevParams P, VArgs A, const int *__restrict__ start,
                                                const int *__restrict__ cell, const double *__restrict__ state,
                                                int *__restrict__ list, int *__restrict__ len) {
  const int q = blockIdx.x * kVB + threadIdx.x;
  if (q < A.n) list_of_slot<S, true>(P, A, start, cell, state, nullptr, list, len, q);
}

template <int S>
__global__ __launch_bounds__(kVB) void vc_unpermute(int n, const double *__restrict__ vstate, const int *__restrict__ id,
                                                    double *__restrict__ state) {
  const int p = blockIdx.x * kVB + threadIdx.x;
  if (p >= n) return;
  const int i = id[p];
#pragma unroll
  for (int k = 0; k < S; ++k) state[(long)i * S + k] = vstate[(long)p * S + k];
}

// ---------------------------------------------------------------------------
// host side

struct VerletFast {
  int n = 0, s = 4, ncv = 1, cells = 1, K = 0, nsb = 1;
  double rho = 0.0, r_max = 0.0;
  VArgs A{};
  double *vstate[2] = {nullptr, nullptr};
  float4 *vsnap[2] = {nullptr, nullptr};
  float *vomega[2] = {nullptr, nullptr};
  int *vid = nullptr, *vcell = nullptr;
  double *vnat = nullptr;
  int *list = nullptr, *len = nullptr;
  // row tiles of the rebuild's cell order (grids of at most kRowTileCols columns): ncv rows of vt_cmax slots
  bool tiled = false;
  int vt_wcap = 0, vt_cmax = 0;
  int4 *vtiles = nullptr;
  int2 *rest = nullptr;  // items of vt_rest
  int *local = nullptr, *key = nullptr, *slotc = nullptr, *count = nullptr, *start = nullptr, *tmp = nullptr, *blocksum = nullptr;
  double *sstate = nullptr, *snat = nullptr;
  int *sid = nullptr, *scell = nullptr;
  VCtl *ctl = nullptr;
  int *bmax = nullptr;
  size_t list_cap = 0;    // ints allocated for the lists
  bool resident = false, resident_nat = false;
  int cur = 0;
  struct StepGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
  } sg[2][2];  // [bulk, single step][parity]
  int sg_srk = -1, sg_higher = -1;
  double sg_dt = 0.0, sg_dphi = 0.0, sg_friction = 0.0;
  uint64_t sg_seed = 0;
  const double *sg_nat = nullptr;
  double *sg_compl = nullptr;
  long captures = 0;
};

const char *vf_last_error() { return g_verr.c_str(); }

static int vfail(int code, const std::string &m) {
  g_verr = m;
  return code;
}

#define VCHK(call)                                                                                      \
  do {                                                                                                  \
    hipError_t e_ = (call);                                                                             \
    if (e_ != hipSuccess) return vfail(SPSS_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

static unsigned vblocks(long n) { return (unsigned)((n + kVB - 1) / kVB); }

static void drop_graphs(VerletFast *v) {
  for (auto &row : v->sg)
    for (auto &g : row) {
      if (g.exec) hipGraphExecDestroy(g.exec);
      if (g.graph) hipGraphDestroy(g.graph);
      g.exec = nullptr;
      g.graph = nullptr;
    }
}

void vf_destroy(VerletFast *v) {
  if (!v) return;
  drop_graphs(v);
  void *b[] = {v->vstate[0], v->vstate[1], v->vsnap[0], v->vsnap[1], v->vomega[0], v->vomega[1], v->vid,
               v->vcell,     v->vnat,      v->list,     v->len,      v->key,       v->slotc,     v->count,
               v->start,     v->tmp,       v->blocksum, v->sstate,   v->snat,      v->sid,       v->scell,
               v->ctl,       v->bmax,      v->vtiles,   v->local,  v->rest};
  for (void *p : b) hipFree(p);
  delete v;
}

int vf_create(VerletFast **out, hipStream_t st, const DevParams &P, double rho, double r_max) {
  *out = nullptr;
  if (P.s != 3 && P.s != 4) return vfail(SPSS_ERR_UNSUPPORTED, "FP32C Verlet lists are implemented for models 3 and 4");
  if (P.xs != 1.0 || P.ys != 1.0)
    return vfail(SPSS_ERR_UNSUPPORTED, "FP32C Verlet lists assume the unit box of the reference's cell grid");
  if (!(r_max > rho)) return vfail(SPSS_ERR_INVALID, "the Verlet skin must be positive");
  const int ncv = (int)(1.0 / r_max);
  if (ncv < 3)
    return vfail(SPSS_ERR_UNSUPPORTED, "FP32C Verlet lists need int(1/r_max) >= 3 (use the FP64 precision there)");
  VerletFast *v = new VerletFast();
  const int n = P.n;
  v->n = n;
  v->s = P.s;
  v->ncv = ncv;
  v->cells = ncv * ncv;
  v->nsb = scan_blocks(v->cells);
  v->rho = rho;
  v->r_max = r_max;
  hipError_t e = hipSuccess;
  auto A = [&](hipError_t r) {
    if (e == hipSuccess) e = r;
  };
  const size_t nn = (size_t)n;
  for (int b = 0; b < 2; ++b) {
    A(hipMalloc(&v->vstate[b], sizeof(double) * nn * P.s));
    A(hipMalloc(&v->vsnap[b], sizeof(float4) * nn));
    A(hipMalloc(&v->vomega[b], sizeof(float) * nn));
  }
  A(hipMalloc(&v->vid, sizeof(int) * nn));
  A(hipMalloc(&v->vcell, sizeof(int) * nn));
  A(hipMalloc(&v->vnat, sizeof(double) * nn));
  A(hipMalloc(&v->len, sizeof(int) * nn));
  A(hipMalloc(&v->key, sizeof(int) * nn));
  A(hipMalloc(&v->slotc, sizeof(int) * nn));
  A(hipMalloc(&v->count, sizeof(int) * (size_t)v->cells));
  A(hipMalloc(&v->start, sizeof(int) * ((size_t)v->cells + 1)));
  A(hipMalloc(&v->tmp, sizeof(int) * nn));
  A(hipMalloc(&v->blocksum, sizeof(int) * ((size_t)v->nsb + 1)));
  A(hipMalloc(&v->sstate, sizeof(double) * nn * P.s));
  A(hipMalloc(&v->snat, sizeof(double) * nn));
  A(hipMalloc(&v->sid, sizeof(int) * nn));
  A(hipMalloc(&v->scell, sizeof(int) * nn));
  A(hipMalloc(&v->ctl, sizeof(VCtl)));
  A(hipMalloc(&v->bmax, sizeof(int)));
  v->tiled = ncv <= kRowTileCols;
  if (v->tiled) {
    // slots per row: the greedy spans of a row 1.5x the mean at about 94% of a tile each (or 80% of what
    // the mean density leaves them of the stage, vt_tiles), plus 2, and at least enough spans of vt_wcap
    // columns to cover a row
    v->vt_wcap = kVCols - 2;
    const double row_mean = (double)n / (double)ncv, cell_mean = row_mean / (double)ncv;
    const double cols = std::max(1.0, std::floor((kMStage - 24) / (3.0 * cell_mean)) - 2.0);
    v->vt_cmax = std::max((ncv + v->vt_wcap - 1) / v->vt_wcap,
                          (int)std::min((double)ncv, std::ceil(1.5 * row_mean / std::min(0.94 * kTileCap, 0.8 * cols * cell_mean)) + 2));
    A(hipMalloc(&v->local, sizeof(int) * (size_t)v->cells));
    A(hipMalloc(&v->vtiles, sizeof(int4) * (size_t)ncv * v->vt_cmax));
    A(hipMalloc(&v->rest, sizeof(int2) * ((size_t)n / kRestItem + (size_t)ncv * v->vt_cmax)));  // a ragged item per tile
  }
  if (e != hipSuccess) {
    vf_destroy(v);
    return vfail(SPSS_ERR_DEVICE, std::string("Verlet list buffers: ") + hipGetErrorString(e));
  }
  launch_fill_int(st, v->cells, v->count, 0);
  launch_fill_int(st, (long)(sizeof(VCtl) / sizeof(int)), reinterpret_cast<int *>(v->ctl), 0);
  // guard bands: coordinates in [0, 1] rounded once to FP32 (<= 2^-25 each), the difference and
  // the nearest-integer shift exact, so |dx| errs by <= 2^-24; the squared distance then by
  // <= 2 sqrt(2) r 2^-24 plus a few ulps -- times a safety factor of 8
  const double eps = std::ldexp(1.0, -24);
  auto band = [&](double r) { return r * r * std::max(8.0 * (2.0 * std::sqrt(2.0) * eps / r + 4.0 * eps), 64.0 * eps); };
  VArgs &a = v->A;
  a.n = n;
  a.ncv = ncv;
  a.cells = v->cells;
  a.rmax2 = r_max * r_max;
  a.half_skin = 0.5 * (r_max - rho);
  a.h = 1.0 / (double)ncv;
  a.r2c = (float)(rho * rho);
  a.r2h = (float)band(rho);
  a.r2k = (float)std::ldexp(1.0, std::ilogb(4.0 / (double)a.r2h) + 1);  // power of two, r2k * r2h > 4
  a.m2c = (float)(r_max * r_max);
  a.unit = (float)(kMUnit * (double)ncv);
  a.rho_u = (float)(rho * (double)a.unit);
  a.r2_u = (float)(rho * rho * (double)a.unit * (double)a.unit);
  a.drift = (float)(kMUnit * (1.0 + a.half_skin * ncv));
  a.m2h = (float)band(r_max);
  a.ctl = v->ctl;
  *out = v;
  return SPSS_OK;
}

int vf_list_width(const VerletFast *v) { return v ? v->K : 0; }
bool vf_is_resident(const VerletFast *v) { return v && v->resident; }
void vf_drop(VerletFast *v) {
  if (v) v->resident = false;
}
long vf_graph_captures(const VerletFast *v) { return v ? v->captures : 0; }

bool vf_graph_ready(const VerletFast *v, const double *nat, int srk) {
  (void)srk;  // omega is kept for every model-4 step, so either stepper may follow the other
  return v && v->resident && (nat != nullptr) == v->resident_nat;
}

// Entry into the resident copy.  The list width K is sized here from the state entered: the
// densest 3 x 3 block of cells holds bmax candidates, i.e. a local density of bmax / (9 Hv^2), so a
// list holds about lam = bmax pi r_max^2 / (9 Hv^2); K = 1.5 lam + 6 sqrt(lam) + 32 (at most bmax
// + 16) leaves room for the density to grow.  A list that outgrows K later is not stored
// (vf_lists reports it); entering again from a fresh state sizes K anew.
int vf_enter(VerletFast *v, hipStream_t st, const DevParams &P, int srk, const double *state, const double *nat) {
  (void)srk;
  const unsigned nb = vblocks(v->n);
  VCHK(hipMemcpyAsync(v->vstate[0], state, sizeof(double) * (size_t)v->n * v->s, hipMemcpyDeviceToDevice, st));
  vc_iota<<<nb, kVB, 0, st>>>(v->n, v->vid);
  if (nat) VCHK(hipMemcpyAsync(v->vnat, nat, sizeof(double) * (size_t)v->n, hipMemcpyDeviceToDevice, st));
  vc_enter<<<1, 64, 0, st>>>(v->ctl);
  // the cell counts of the state entered (the flag is set: vr_keys runs), their densest 3 x 3
  // block, and the counts cleared again for the first rebuild
  launch_fill_int(st, 1, v->bmax, 0);
  if (v->s == 4)
    vr_keys<4><<<nb, kVB, 0, st>>>(P, v->A, 0, nullptr, v->vstate[0], v->key, v->slotc, v->count);
  else
    vr_keys<3><<<nb, kVB, 0, st>>>(P, v->A, 0, nullptr, v->vstate[0], v->key, v->slotc, v->count);
  vc_block_max<<<vblocks(v->cells), kVB, 0, st>>>(v->A, v->count, v->bmax);
  int bmax = 0;
  VCHK(hipMemcpyAsync(&bmax, v->bmax, sizeof(int), hipMemcpyDeviceToHost, st));
  launch_fill_int(st, v->cells, v->count, 0);
  VCHK(hipStreamSynchronize(st));
  const double Hv = 1.0 / (double)v->ncv;
  const double lam = (double)bmax * M_PI * v->r_max * v->r_max / (9.0 * Hv * Hv);
  int K = (int)std::ceil(1.5 * lam + 6.0 * std::sqrt(lam) + 32.0);
  K = std::max(16, std::min(K, bmax + 16));
  K = (K + 15) / 16 * 16;
  // an upper bound on the width from the environment (memory cap; lists beyond it walk their cells)
  if (const char *cap = std::getenv("SPSS_VERLET_WIDTH_CAP")) K = std::max(4, std::min(K, std::atoi(cap)));
  K = (K + 15) / 16 * 16;  // whole chunks of four entries, whole passes of sixteen
  const size_t need = ((size_t)v->n + 255) / 256 * 256 * (size_t)K;  // lslot's blocks of 256 slots
  if (need > v->list_cap) {
    drop_graphs(v);  // captured launches hold the old list pointer
    hipFree(v->list);
    v->list = nullptr;
    v->list_cap = 0;
    VCHK(hipMalloc(&v->list, sizeof(int) * need));
    v->list_cap = need;
  }
  if (K != v->K) drop_graphs(v);  // the width is a launch argument of the captured steps
  v->K = K;
  v->A.K = K;
  VCHK(hipGetLastError());
  v->cur = 0;
  v->resident = true;
  v->resident_nat = nat != nullptr;
  return SPSS_OK;
}

// the rebuild launches (gated on the device flag) and the step, from buffer v->cur
template <int S, bool SRK>
static void launch_step(VerletFast *v, hipStream_t st, const DevParams &P, const StepArgs &U, double *compl_out) {
  const int c = v->cur, o = 1 - c;
  const unsigned nb = vblocks(v->n);
  const VArgs &A = v->A;
  const double *nat = v->resident_nat ? v->vnat : nullptr;
  // the rebuild launches return at once on most steps: a fixed grid of at most kGateGrid
  // workgroups (grid-stride loops) keeps what they cost then down to a dispatch
  const unsigned gg = std::min(nb, (unsigned)kGateGrid);
  vr_keys<S><<<gg, kVB, 0, st>>>(P, A, c, U.step_inc, v->vstate[c], v->key, v->slotc, v->count);
  scan_local<<<v->nsb, 256, 0, st>>>(v->count, nullptr, v->cells, v->tiled ? v->local : v->start, v->blocksum,
                                     ctl_flag(A.ctl));
  if (!v->tiled)
    scan_add<<<v->nsb, 256, 0, st>>>(v->count, nullptr, v->cells, v->start, v->blocksum, v->nsb, nullptr,
                                     ctl_flag(A.ctl));
  vr_scatter<<<gg, kVB, 0, st>>>(A, v->key, v->slotc, v->local, v->blocksum, v->nsb, v->count, v->start, v->tmp);
  // tiled grids: the row tiles of the new order are built by vr_gather's first workgroups, so its
  // grid covers a wave per row as well
  const unsigned sg = v->tiled ? std::max(gg, (unsigned)((v->ncv + 3) / 4)) : gg;
  vr_gather<S><<<sg, kVB, 0, st>>>(A, v->key, v->start, v->tmp, v->vstate[c], v->vid, nat, v->sstate, v->sid, v->snat,
                                   v->scell, v->tiled ? v->vtiles : nullptr, v->vt_wcap, v->vt_cmax);
  const int ntiles = v->tiled ? v->ncv * v->vt_cmax : 0;
  vr_settle<S><<<gg, kVB, 0, st>>>(P, A, v->sstate, v->sid, v->snat, v->scell, v->vstate[c], v->vid,
                                   nat ? v->vnat : nullptr, v->vcell, v->vsnap[c], v->vomega[c], v->start,
                                   v->tiled ? v->vtiles : nullptr, ntiles, v->rest);
  if (v->tiled) {
    const unsigned tg = (unsigned)((ntiles + 7) / 8 * 8);  // a multiple of 8 for xcd_block
    vt_rest<S, SRK><<<kGateGrid, kVB, 0, st>>>(P, A, U, v->rest, v->start, v->vcell, v->vstate[c], v->vid, nat,
                                               v->vsnap[c], v->vomega[c], v->vstate[o], v->vsnap[o], v->vomega[o],
                                               SRK ? compl_out : nullptr);
    vt_step<S, SRK><<<tg, kVB, 0, st>>>(P, A, U, v->vtiles, ntiles, v->start, v->vcell, v->vstate[c], v->vid, nat,
                                        v->vsnap[c], v->vomega[c], v->vstate[o], v->vsnap[o], v->vomega[o],
                                        SRK ? compl_out : nullptr);
  } else {
    vr_lists<S><<<nb, kVB, 0, st>>>(P, A, v->start, v->vcell, v->vstate[c], v->vsnap[c], v->list, v->len);
    const unsigned nb8 = (nb + 7u) & ~7u;  // a multiple of 8 for xcd_block
    vs_step<S, SRK><<<nb8, kVB, 0, st>>>(P, A, U, v->list, v->len, v->start, v->vcell, v->vstate[c], v->vid, nat,
                                         v->vsnap[c], v->vomega[c], v->vstate[o], v->vsnap[o], v->vomega[o],
                                         SRK ? compl_out : nullptr);
  }
}

static StepArgs vstep_args(double dt, double D_phi, double friction, int noise_mode, const double *noise,
                           uint64_t seed, uint64_t step) {
  StepArgs U{};
  U.dt = dt;
  U.sqrt_dt = std::sqrt(dt);
  U.int_phi = std::sqrt(2.0 * D_phi);
  U.c15 = 0.5 * std::pow(dt, 1.5);
  U.is3 = 1.0 / std::sqrt(3.0);
  U.sq2d = std::sqrt(2.0 * D_phi);
  U.friction = friction;
  U.noise_mode = noise_mode;
  U.noise = noise;
  U.seed = seed;
  U.step = step;
  return U;
}

static void step_impl(VerletFast *v, hipStream_t st, const DevParams &P, bool do_srk, const StepArgs &U,
                      double *compl_out) {
  if (do_srk)
    launch_step<4, true>(v, st, P, U, compl_out);
  else if (v->s == 4)
    launch_step<4, false>(v, st, P, U, compl_out);
  else
    launch_step<3, false>(v, st, P, U, compl_out);
  v->cur = 1 - v->cur;
}

int vf_step(VerletFast *v, hipStream_t st, const DevParams &P, int srk, const double *state, const double *nat,
            double *compl_out, double dt, double D_phi, double friction, int noise_mode, const double *noise,
            uint64_t seed, uint64_t step) {
  const bool do_srk = srk && v->s == 4;
  if (!vf_graph_ready(v, nat, do_srk)) {
    const int rc = vf_enter(v, st, P, do_srk, state, nat);
    if (rc != SPSS_OK) return rc;
  }
  step_impl(v, st, P, do_srk, vstep_args(dt, D_phi, friction, noise_mode, noise, seed, step), compl_out);
  VCHK(hipGetLastError());
  return SPSS_OK;
}

static int capture(VerletFast *v, hipStream_t st, const DevParams &P, bool do_srk, const StepArgs &U,
                   double *compl_out, int steps, VerletFast::StepGraph &g) {
  const int cur0 = v->cur;
  hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed);
  if (e != hipSuccess) return vfail(SPSS_ERR_DEVICE, std::string("hipStreamBeginCapture: ") + hipGetErrorString(e));
  for (int k = 0; k < steps; ++k) step_impl(v, st, P, do_srk, U, compl_out);
  hipGraph_t graph = nullptr;
  e = hipStreamEndCapture(st, &graph);
  v->cur = cur0;  // nothing ran
  if (e != hipSuccess) {
    if (graph) hipGraphDestroy(graph);
    (void)hipGetLastError();
    return vfail(SPSS_ERR_DEVICE, std::string("capture of the Verlet step graph failed: ") + hipGetErrorString(e));
  }
  hipGraphExec_t exec = nullptr;
  e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    hipGraphDestroy(graph);
    return vfail(SPSS_ERR_DEVICE, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
  }
  g.graph = graph;
  g.exec = exec;
  ++v->captures;
  return SPSS_OK;
}

static StepArgs graph_setup(VerletFast *v, const DevParams &P, bool do_srk, const double *nat, double *compl_out,
                            double dt, double D_phi, double friction, uint64_t seed) {
  const bool same = v->sg_srk == (int)do_srk && v->sg_higher == P.higher_order && v->sg_dt == dt &&
                    v->sg_dphi == D_phi && v->sg_friction == friction && v->sg_seed == seed && v->sg_nat == nat &&
                    v->sg_compl == compl_out;
  if (!same) {
    drop_graphs(v);
    v->sg_srk = do_srk;
    v->sg_higher = P.higher_order;
    v->sg_dt = dt;
    v->sg_dphi = D_phi;
    v->sg_friction = friction;
    v->sg_seed = seed;
    v->sg_nat = nat;
    v->sg_compl = compl_out;
  }
  StepArgs U = vstep_args(dt, D_phi, friction, 3, nullptr, seed, 0);
  U.step_dev = ctl_step(v->ctl);
  U.step_inc = ctl_step(v->ctl);
  return U;
}

static int ensure_graph(VerletFast *v, hipStream_t st, const DevParams &P, bool do_srk, const StepArgs &U,
                        double *compl_out, int size) {
  VerletFast::StepGraph &g = v->sg[size == 1 ? 1 : 0][v->cur];
  if (g.exec) return SPSS_OK;
  return capture(v, st, P, do_srk, U, compl_out, size, g);
}

int vf_prepare_graphs(VerletFast *v, hipStream_t st, const DevParams &P, int srk, const double *state,
                      const double *nat, double *compl_out, double dt, double D_phi, double friction, uint64_t seed) {
  (void)state;
  const bool do_srk = srk && v->s == 4;
  if (!vf_graph_ready(v, nat, do_srk)) return vfail(SPSS_ERR_INVALID, "no resident copy to capture steps of");
  const StepArgs U = graph_setup(v, P, do_srk, nat, compl_out, dt, D_phi, friction, seed);
  for (int side = 0; side < 2; ++side) {
    for (int size : {kVGraphSteps, 1}) {
      const int rc = ensure_graph(v, st, P, do_srk, U, compl_out, size);
      if (rc != SPSS_OK) {
        if (side) v->cur = 1 - v->cur;
        return rc;
      }
    }
    v->cur = 1 - v->cur;
  }
  return SPSS_OK;
}

long vf_run_graph(VerletFast *v, hipStream_t st, const DevParams &P, int srk, const double *state, const double *nat,
                  double *compl_out, double dt, double D_phi, double friction, uint64_t seed, uint64_t step,
                  long nsteps) {
  (void)state;
  const bool do_srk = srk && v->s == 4;
  if (nsteps < 1 || !vf_graph_ready(v, nat, do_srk)) return 0;
  const StepArgs U = graph_setup(v, P, do_srk, nat, compl_out, dt, D_phi, friction, seed);
  const long reps = nsteps / kVGraphSteps, rest = nsteps % kVGraphSteps;
  int rc = SPSS_OK;
  if (reps > 0) rc = ensure_graph(v, st, P, do_srk, U, compl_out, kVGraphSteps);
  for (int side = 0; side < 2 && side < rest && rc == SPSS_OK; ++side) {
    if (side) v->cur = 1 - v->cur;
    rc = ensure_graph(v, st, P, do_srk, U, compl_out, 1);
    if (side) v->cur = 1 - v->cur;
  }
  if (rc != SPSS_OK) return -1;
  vc_set_step<<<1, 64, 0, st>>>(v->ctl, (unsigned long long)step - 1ull);  // vr_keys advances it first
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    g_verr = std::string("vc_set_step: ") + hipGetErrorString(e);
    return -1;
  }
  for (long r = 0; r < reps; ++r)
    if ((e = hipGraphLaunch(v->sg[0][v->cur].exec, st)) != hipSuccess) {
      g_verr = std::string("hipGraphLaunch: ") + hipGetErrorString(e);
      return -1;
    }
  for (long r = 0; r < rest; ++r) {
    if ((e = hipGraphLaunch(v->sg[1][v->cur].exec, st)) != hipSuccess) {
      g_verr = std::string("hipGraphLaunch: ") + hipGetErrorString(e);
      return -1;
    }
    v->cur = 1 - v->cur;
  }
  return nsteps;
}

int vf_sync(VerletFast *v, hipStream_t st, double *state) {
  if (!v->resident) return SPSS_OK;
  const unsigned nb = vblocks(v->n);
  if (v->s == 4)
    vc_unpermute<4><<<nb, kVB, 0, st>>>(v->n, v->vstate[v->cur], v->vid, state);
  else
    vc_unpermute<3><<<nb, kVB, 0, st>>>(v->n, v->vstate[v->cur], v->vid, state);
  VCHK(hipGetLastError());
  return SPSS_OK;
}

int vf_status(VerletFast *v, hipStream_t st, int *should_update, double *acc) {
  VCtl c{};
  if (v->resident) {
    VCHK(hipMemcpyAsync(&c, v->ctl, sizeof(VCtl), hipMemcpyDeviceToHost, st));
    VCHK(hipStreamSynchronize(st));
  } else {
    c.force = 1;  // the next step enters and rebuilds
  }
  // what the next vr_keys will find
  double m = 0.0;
  for (int g = 0; g < kGroups; ++g) {
    double d;
    std::memcpy(&d, &c.gmax[g * kLineU64], sizeof(d));
    m = std::max(m, d);
  }
  const double stepd = std::sqrt(m), a = c.acc[v->cur] + stepd;
  const int flag = c.force || a + stepd > v->A.half_skin;
  if (should_update) *should_update = flag;
  if (acc) *acc = flag ? 0.0 : a;
  return SPSS_OK;
}

int vf_lists(VerletFast *v, hipStream_t st, const DevParams &P, std::vector<int> *counts, std::vector<int> *flat) {
  const int n = v->n;
  counts->assign(n, 0);
  flat->clear();
  if (!v->resident) return SPSS_OK;
  int force = 0;
  VCHK(hipMemcpyAsync(&force, reinterpret_cast<char *>(v->ctl) + offsetof(VCtl, force), sizeof(int),
                      hipMemcpyDeviceToHost, st));
  VCHK(hipStreamSynchronize(st));
  if (force) return SPSS_OK;  // no rebuild since entry: the arrays of the last one are another state's, or unwritten
  if (v->tiled) {  // the tiles' steps need no lists
    const unsigned nb = vblocks(n);
    if (v->s == 4)
      vc_lists<4><<<nb, kVB, 0, st>>>(P, v->A, v->start, v->vcell, v->sstate, v->list, v->len);
    else
      vc_lists<3><<<nb, kVB, 0, st>>>(P, v->A, v->start, v->vcell, v->sstate, v->list, v->len);
    VCHK(hipGetLastError());
  }
  std::vector<int> id(n), len(n), list(((size_t)n + 255) / 256 * 256 * (size_t)v->K);
  VCHK(hipMemcpyAsync(id.data(), v->vid, sizeof(int) * n, hipMemcpyDeviceToHost, st));
  VCHK(hipMemcpyAsync(len.data(), v->len, sizeof(int) * n, hipMemcpyDeviceToHost, st));
  VCHK(hipMemcpyAsync(list.data(), v->list, sizeof(int) * list.size(), hipMemcpyDeviceToHost, st));
  VCHK(hipStreamSynchronize(st));
  for (int p = 0; p < n; ++p)
    if (len[p] < 0)
      return vfail(SPSS_ERR_CAPACITY, "some Verlet lists outgrew the width " + std::to_string(v->K) +
                                          " and are not stored (those particles walk their 3 x 3 cells)");
  std::vector<int> slot_of(n);
  for (int p = 0; p < n; ++p) slot_of[id[p]] = p;
  for (int i = 0; i < n; ++i) {
    const int p = slot_of[i];
    (*counts)[i] = len[p];
    for (int t = 0; t < len[p]; ++t) flat->push_back(id[list[lslot(p, t, v->K)]]);
  }
  return SPSS_OK;
}

}  // namespace spss
