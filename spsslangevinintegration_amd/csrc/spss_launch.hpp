// spss_launch.hpp -- host-side launchers of the HIP kernels (one per kernel family).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "spss_device.hpp"

namespace spss {

// records the message spss_last_error() returns and passes the code through
int set_error(int code, const std::string &msg);

// what the observers need of a handle: its stream and its master state, up to date
struct SystemView {
  hipStream_t stream;
  const double *state;  // device, AoS FP64, original particle order
  int n, s;
  double x_size, y_size, x_rsize, y_rsize;
};
}  // namespace spss
struct spss_system;
namespace spss {
int system_view(spss_system *h, SystemView *v);
// device scratch of at least `bytes` bytes, kept by the handle; what it holds is lost at the next call
int system_scratch(spss_system *h, size_t bytes, void **p);
class HostCopy;
HostCopy &system_copy(spss_system *h);

// two HIP events timing a stretch of one stream, destroyed with the object (also on the early
// returns of an error path)
struct EventPair {
  hipEvent_t start = nullptr, stop = nullptr;
  hipError_t create() {
    const hipError_t e = hipEventCreate(&start);
    return e == hipSuccess ? hipEventCreate(&stop) : e;
  }
  // milliseconds between the two records, after waiting for the second
  hipError_t elapsed(float *ms) {
    const hipError_t e = hipEventSynchronize(stop);
    return e == hipSuccess ? hipEventElapsedTime(ms, start, stop) : e;
  }
  EventPair() = default;
  EventPair(const EventPair &) = delete;
  EventPair &operator=(const EventPair &) = delete;
  ~EventPair() {
    if (start) (void)hipEventDestroy(start);
    if (stop) (void)hipEventDestroy(stop);
  }
};

// HIP-event timer around one kernel family, enabled on request (bench instrumentation):
// records an event pair per launch on the launching stream, sums the durations on read.
struct KernelTimer {
  bool on = false;
  int used = 0;
  hipEvent_t ev[2 * 4096];
  bool created = false;
  void begin(hipStream_t st) {
    if (!on || used >= 4096) return;
    if (!created) {
      for (auto &e : ev) hipEventCreate(&e);
      created = true;
    }
    hipEventRecord(ev[2 * used], st);
  }
  void end(hipStream_t st) {
    if (!on || used >= 4096) return;
    hipEventRecord(ev[2 * used + 1], st);
    ++used;
  }
  double total_ms() {
    double t = 0.0;
    for (int k = 0; k < used; ++k) {
      float ms = 0.f;
      hipEventSynchronize(ev[2 * k + 1]);
      hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]);
      t += ms;
    }
    return t;
  }
  ~KernelTimer() {
    if (created)
      for (auto &e : ev) hipEventDestroy(e);
  }
};

// device buffers of one cell list (stable counting sort over cell keys)
struct CellBuffers {
  int *key = nullptr;     // [n] cell key of each particle
  int *slot = nullptr;    // [n] arrival slot from the histogram atomics
  int *count = nullptr;   // [cells] histogram, left zeroed by the scan
  int *start = nullptr;   // [cells + 1] exclusive scan of count
  int *tmp = nullptr;     // [n] unstable bucket fill
  int *sorted = nullptr;  // [n] particle indices, cell-major, ascending index inside a cell
  int *blocksum = nullptr;  // [scan_blocks(cells) + 1] totals of the scan's workgroups
  int cells = 0;
};

// stage = state + kc_dt * kprev; kprev null: an all-zero k_prev
void launch_stage(hipStream_t st, long m, const double *state, const double *kprev, double kc_dt, double *stage);
// all-pairs RHS: the stage state with its records (the first call), then the pair sums with workgroups
// of kAllPairsConfigs[config][0] particles and j-tiles of kAllPairsConfigs[config][1] (identical sums
// for every config; kAllPairsDefault is {256, 256}) and the derivative
constexpr int kAllPairsConfigCount = 6;
constexpr int kAllPairsDefault = 4;
extern const int kAllPairsConfigs[kAllPairsConfigCount][2];
struct AllPairsScratch {
  double *rec = nullptr;   // [4 n] {x, y, sin psi, cos psi} per particle
  double *om = nullptr;    // [n] omega
  double *part = nullptr;  // [nseg][5][n] the segments' sums
  int nseg = 0;
};
int all_pairs_segments(int n);
void launch_all_pairs_stage(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                            double *stage, const AllPairsScratch &W);
void launch_all_pairs(hipStream_t st, const DevParams &P, const AllPairsScratch &W, const double *stage,
                      const double *nat, double *k_next, double *compl_out, int config = kAllPairsDefault);
// the same derivative of up to kAllPairsFew particles in one launch, without a workspace
constexpr int kAllPairsFew = 64;
void launch_all_pairs_few(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                          const double *nat, double *k_next, double *compl_out);
void launch_cell_build(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy, CellBuffers &cb);
void launch_linked_list(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                        const CellBuffers &cb, const double *nat, double *k_next, double *compl_out);
// the FP64 linked list on a unit box of 3 x 3 to 1448 x 1448 cells (spss_cells64.hip); other boxes,
// coarser grids, where the reference visits cells more than once, and finer ones, whose cells are
// mostly empty below a hundred million particles, take the two calls above
struct Cells64 {
  char *mem = nullptr;                 // the allocation that holds them all
  int *order[2] = {nullptr, nullptr};  // [n] particle of each sorted position: the last build's, the next one's
  int cur = 0;
  int *key = nullptr, *slot = nullptr, *count = nullptr, *blocksum = nullptr;
  int *bad = nullptr;    // [2] some particle is out of the cheap tests' range; extra chunks
  int *extra = nullptr;  // [2 (n / 128 + rows)] the extra chunks
  int *local = nullptr, *start = nullptr;      // [cells + 1] starts inside a scan block, starts
  int *tmp = nullptr;                          // [2 n]
  double *pre = nullptr, *snap = nullptr;      // [s n] stage state in the last build's and in this one's order
};
bool cells64_serves(const DevParams &P, int ncx, int ncy);
void launch_cells64_build(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                          int nc, Cells64 &B);
void launch_cells64_pairs(hipStream_t st, const DevParams &P, int nc, const Cells64 &B, const double *nat,
                          double *k_next, double *compl_out);
void launch_iota(hipStream_t st, int n, int *p);
// exclusive scan of count[0..m) into start[0..m]; count is left zeroed; blocksum: scratch of
// scan_blocks(m) + 1 ints (spss_scan.hpp)
void launch_scan(hipStream_t st, int *count, int *start, int m, int *blocksum);
// Verlet lists: counts, then for every particle the ids of its entries (vlist) and their positions
// in the candidates' order (vslot: in cb.sorted, or the ids again over all pairs; may be null)
void launch_verlet_count_all(hipStream_t st, const DevParams &P, const double *stage, double rmax2, int *vcount);
void launch_verlet_fill_all(hipStream_t st, const DevParams &P, const double *stage, double rmax2,
                            const int *vstart, int *vlist, int *vslot);
void launch_verlet_count_cells(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                               const CellBuffers &cb, double rmax2, int *vcount);
void launch_verlet_fill_cells(hipStream_t st, const DevParams &P, const double *stage, int ncx, int ncy,
                              const CellBuffers &cb, double rmax2, const int *vstart, int *vlist, int *vslot);
// the stage state in the order of the lists' build (null: over all pairs), with the records and omegas that
// the pair sums over it read
struct VerletStage {
  double *stage = nullptr;  // [s n]
  double *rec = nullptr;    // [4 n] {x, y, sin psi, cos psi}
  double *om = nullptr;     // [n]
};
// what follows a derivative of the Runge-Kutta stepper in the same launch: the next stage (next set), or
// the end of the step
constexpr int kVerletMax = 64, kVerletMaxStep = 16;  // maxima of groups of workgroups, a cache line each
struct VerletThen {
  double *base = nullptr;  // the state
  double kc = 0.0, dt = 0.0;
  VerletStage next;
  const double *k1 = nullptr, *k2 = nullptr, *k3 = nullptr;
  unsigned long long *vmax = nullptr;  // [kVerletMax kVerletMaxStep] bits of the largest squared displacements
};
void launch_stage_order(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                        const int *order, const VerletStage &V, unsigned long long *vmax = nullptr);
void launch_verlet_pairs(hipStream_t st, const DevParams &P, const VerletStage &V, const int *order,
                         const int *vstart, const int *vslot, const double *nat, double *k_next, double *compl_out,
                         const VerletThen *then = nullptr);
// the global field (spss_global64.hip).  part: gf_part_doubles(n) doubles of scratch in two halves of
// block sums; kprev may be null
size_t gf_part_doubles(int n);
void launch_global(hipStream_t st, const DevParams &P, const double *x, const double *kprev, double kc, double *part,
                   const double *nat, double *k_next, double *compl_out);
// nsteps of the Runge-Kutta stepper; k: k1..k4 (left with those of the last step), tmp: a stage state
void launch_global_rk4(hipStream_t st, const DevParams &P, long nsteps, double dt, double *state, double *tmp,
                       double *const *k, double *part, const double *nat, double *compl_out);
struct GfNoise {
  int mode = 0;  // 0 none, 1 array, 3 Philox
  const double *array = nullptr;
  uint64_t seed = 0, step = 0;
  double sqrt_dt = 0.0, amp = 0.0, c15 = 0.0, is3 = 0.0, friction = 0.0;
};
// nsteps of the stochastic Euler (not with the complementary force) or Runge-Kutta stepper
void launch_global_stochastic(hipStream_t st, const DevParams &P, bool srk, long nsteps, double dt, double *state,
                              double *part, const double *nat, double *compl_out, const GfNoise &Z);
void launch_rk4_combine(hipStream_t st, int s, int n, double *state, const double *k1, const double *k2,
                        const double *k3, const double *k4, double dt, double *max_partial);
void launch_euler(hipStream_t st, int s, int n, double *state, const double *f, double dt, double sqrt_dt,
                  double int_phi, double int_r, int noise_mode, const double *noise, uint64_t seed, uint64_t step,
                  double *max_partial);
void launch_srk(hipStream_t st, int n, double *state, const double *f, const double *C, double dt, double sqrt_dt,
                double c15, double is3, double sq2d, double friction, int noise_mode, const double *noise,
                uint64_t seed, uint64_t step, double *max_partial);
void launch_max_final(hipStream_t st, int nb, const double *partial, double *out);

// Dormand-Prince 5(4): out = 1.0 * x + c[0] * k[0] + ... + c[n-1] * k[n-1] over m values (a stage
// state, the step's output or a dense-output state), and the step's error norm
constexpr int kDpMaxTerms = 6;
struct DpTerms {
  const double *k[kDpMaxTerms];
  double c[kDpMaxTerms];
  int n;
};
void launch_dp_combine(hipStream_t st, long m, const double *x, const DpTerms &T, double *out);
// max over the m = s * n values of |sum_j c_j k_j| / (eps_abs + eps_rel * (|x_old| + dt * |dxdt_old|))
// into out[0] (partial: one double per 256 particles); returns the number of partials
int launch_dp_error(hipStream_t st, int n, int s, const double *x_old, const double *dxdt_old, const DpTerms &T,
                    double dt, double eps_abs, double eps_rel, double *partial, double *out);
// the same over the global field.  Derivatives are two planes: [(s-2) n] of phases (and omegas), then
// [2 n] of positions.
struct DpTrial {
  const double *x = nullptr;  // the state
  double *out = nullptr;      // the new state
  double *k[7] = {};          // k1 (given) .. k6, the derivative at `out`
  double *tmp = nullptr;      // [s n]
  double first = 0.0;         // the coefficient of k1 in the first stage
  DpTerms terms[6] = {};      // of the later stages, the new state and the error: n earlier derivatives, and
                              // as c[n] the coefficient of the one formed there
  double dt = 0.0, eps_abs = 0.0, eps_rel = 0.0;
};
void launch_dp_global_start(hipStream_t st, const DevParams &P, const double *x, double *part, const double *nat,
                            double *k);
// the error norm's block maxima go to the front of part; their number is returned
int launch_dp_global_trial(hipStream_t st, const DevParams &P, const DpTrial &D, const double *nat, double *part);
void launch_dp_global_combine(hipStream_t st, int s, int n, const double *x, const DpTerms &T, double *out);
void launch_dp_global_rows(hipStream_t st, int s, int n, const double *planes, double *rows);
void launch_disp_max(hipStream_t st, int n, int s, const double *tot, double *partial);
void launch_order_parameter(hipStream_t st, int n, int s, int slot, const double *state, double *partial,
                            double *out);
void launch_apply_pbc(hipStream_t st, int n, int s, double *state, double xs, double ys, double xrs, double yrs);
void launch_accumulate(hipStream_t st, long m, const double *state, double *acc);
void launch_fill_double(hipStream_t st, long m, double *p, double v);
void launch_fill_int(hipStream_t st, long m, int *p, int v);
void launch_copy16(hipStream_t st, long n16, const void *src, void *dst);

}  // namespace spss
