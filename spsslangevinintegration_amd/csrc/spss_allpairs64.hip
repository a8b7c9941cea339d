// spss_allpairs64.hip -- the FP64 all-pairs right-hand side,
// ParticleSystemFirstOrderPtr.cpp:225-316 / ParticleSystemSecondOrderPtr.cpp:155-230.
//
//   ap_stage   the stage state, and per particle a 32-byte record {x, y, sin psi, cos psi} (wrapped
//              position, phasor in the frame of particle 0's phase) and omega
//   ap_pairs   grid (groups of BLOCK particles) x (segments of the j's): the phasor sums of every
//              particle over one segment, j ascending
//   ap_finish  the segments' sums added in ascending order, the derivative
//   ap_few     all of it, for up to 64 particles
//
// What bounds it: VALU issue, 14 instructions per pair (the test, the weight, three sums).  One
// thread per particle over all j leaves most of the chip idle below some 10^5 particles (17
// workgroups at n = 4,099), hence the segments: their number depends on n alone, so every
// workgroup shape gives the same sums bit for bit.  n = 4,099, rho = 0.6: 2,023 us per evaluation
// with sin and cos per pair and one workgroup per 256 particles, 29 us with the three kernels
// (pairs 20, finish 5, stage 4; the pair loop's share of the issue rate is ~30%, its two waves per
// SIMD do not cover the LDS latency at this size).
#pragma clang fp contract(off)

#include "spss_launch.hpp"
#include "spss_pairs64.hpp"

namespace spss {

namespace {

// a record whose x is this sends its tile to the exact loop: position far outside the box (model 6:
// outside it at all, ClassA is no minimum image there), or a phase without a finite phasor
constexpr double kExactMark = __builtin_huge_val();

// the record of a particle whose stage state is st
template <int S>
__device__ __forceinline__ double4 record(const DevParams &P, const double (&st)[S], double ref) {
  double x, y, sn, cs;
  apply_pbc(P, st[0], st[1], x, y);
  frame_phasor_any(st[Slots<S>::phi], ref, sn, cs);
  bool fine = fabs(sn) <= 1.5 && fabs(st[0]) <= kFar64 * P.xs && fabs(st[1]) <= kFar64 * P.ys;
  if (S == 6) fine = fine && st[0] >= 0.0 && st[0] < P.xs && st[1] >= 0.0 && st[1] < P.ys;
  if (S == 4 && P.higher_order) fine = fine && fabs(st[Slots<S>::omega]) < 1e300;
  return make_double4(fine ? x : kExactMark, y, sn, cs);
}

template <int S>
__global__ __launch_bounds__(256) void ap_stage(DevParams P, const double *__restrict__ state,
                                                const double *__restrict__ kprev,
                                                double kc_dt, double *__restrict__ stage, double4 *__restrict__ rec,
                                                double *__restrict__ om) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.n) return;
  constexpr int kPhi = Slots<S>::phi;
  const double ref = frame_ref(state[kPhi] + (kprev ? kc_dt * kprev[kPhi] : 0.0));
  double st[S];
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const long e = (long)i * S + q;
    st[q] = state[e] + (kprev ? kc_dt * kprev[e] : 0.0);
    stage[e] = st[q];
  }
  if (S == 4 && P.higher_order) om[i] = st[Slots<S>::omega];
  rec[i] = record<S>(P, st, ref);
}

__device__ __forceinline__ void add_pair(PhasorSums &a, double w, double s, double c) {
  a.S = __builtin_fma(w, s, a.S);
  a.C = __builtin_fma(w, c, a.C);
  a.card += w;
}

// four entries from t0 on of a staged tile of cnt j's against the PPL particles of a lane by the
// cheap test; MASKED: fewer than four are left, or some may be the lane's own particles
template <int S, bool HO, int PPL, int T, bool MASKED>
__device__ __forceinline__ void four_j(const DevParams &P, double band, double neg_slope,
                                       const double *__restrict__ stage, const double4 *tile, const double *tom, int i0,
                                       int j0, int t0, int cnt, const double (&x_i)[PPL], const double (&y_i)[PPL],
                                       const double (&om_i)[PPL], PhasorSums (&a)[PPL]) {
  double w[PPL][4], near = 1e300;
  double4 r[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) r[u] = tile[MASKED ? min(t0 + u, cnt - 1) : t0 + u];
#pragma unroll
  for (int p = 0; p < PPL; ++p)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      double dx = fabs(r[u].x - x_i[p]), dy = fabs(r[u].y - y_i[p]);
      dx = fmin(dx, P.xs - dx);
      dy = fmin(dy, P.ys - dy);
      const double t = __builtin_fma(dx, dx, __builtin_fma(dy, dy, -P.rho2));
      near = fmin(near, fabs(t));
      w[p][u] = pair_weight(t, neg_slope);
      if (MASKED && (t0 + u >= cnt || j0 + t0 + u == i0 + p * T + (int)threadIdx.x)) w[p][u] = 0.0;
    }
  if (near <= band) {  // rare: the reference's own test decides these pairs
#pragma unroll
    for (int p = 0; p < PPL; ++p)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = j0 + t0 + u;
        const bool there = !MASKED || (t0 + u < cnt && j != i0 + p * T + (int)threadIdx.x);
        w[p][u] = there && pair_in_range<S>(P, x_i[p], y_i[p], stage[(long)j * S], stage[(long)j * S + 1]) ? 1.0 : 0.0;
      }
  }
#pragma unroll
  for (int p = 0; p < PPL; ++p)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      add_pair(a[p], w[p][u], r[u].z, r[u].w);
      if (HO) {
        const double wo = w[p][u] * (tom[MASKED ? min(t0 + u, cnt - 1) : t0 + u] - om_i[p]);
        a[p].TS = __builtin_fma(wo, r[u].z, a[p].TS);
        a[p].TC = __builtin_fma(wo, r[u].w, a[p].TC);
      }
    }
}

// particle j, its record r and omega om_j, by the reference's own test
template <int S, bool HO, int PPL, int T>
__device__ __forceinline__ void exact_j(const DevParams &P, const double *__restrict__ stage, const double4 &r,
                                        double om_j, int i0, int j, const double (&x_i)[PPL], const double (&y_i)[PPL],
                                        const double (&om_i)[PPL], PhasorSums (&a)[PPL]) {
  const double x_j = stage[(long)j * S], y_j = stage[(long)j * S + 1];
#pragma unroll
  for (int p = 0; p < PPL; ++p) {
    const int i = i0 + p * T + threadIdx.x;
    if (i != j && pair_in_range<S>(P, x_i[p], y_i[p], x_j, y_j)) {
      add_pair(a[p], 1.0, r.z, r.w);
      if (HO) {
        a[p].TS = __builtin_fma(om_j - om_i[p], r.z, a[p].TS);
        a[p].TC = __builtin_fma(om_j - om_i[p], r.w, a[p].TC);
      }
    }
  }
}

// PPL particles per lane (BLOCK / PPL threads): a tile entry read from LDS serves PPL pairs, which
// halves the LDS reads per pair (at one particle per lane they take as long as the arithmetic)
template <int S, bool HO, int BLOCK, int JT, int PPL>
__global__ __launch_bounds__(BLOCK / PPL) void ap_pairs(DevParams P, double band, double neg_slope, int seglen,
                                                        const double *__restrict__ stage,
                                                        const double4 *__restrict__ rec, const double *__restrict__ om,
                                                        double *__restrict__ part) {
  constexpr int T = BLOCK / PPL;
  __shared__ double4 tile[JT];
  __shared__ double tom[HO ? JT : 1];
  const int n = P.n;
  const int i0 = blockIdx.x * BLOCK;
  const int jb = blockIdx.y * seglen, je = min(n, jb + seglen);
  double x_i[PPL], y_i[PPL], om_i[PPL];
  bool mine_ok = true;
#pragma unroll
  for (int p = 0; p < PPL; ++p) {
    const int i = i0 + p * T + threadIdx.x;
    x_i[p] = y_i[p] = om_i[p] = 0.0;
    if (i < n) {
      if (HO) {
        om_i[p] = stage[(long)i * S + Slots<S>::omega];
        mine_ok = mine_ok && fabs(om_i[p]) < 1e300;
      }
      x_i[p] = stage[(long)i * S];
      y_i[p] = stage[(long)i * S + 1];
      if (S == 6)  // model 6 wraps nothing (ParticleSystemSecondOrderPtr.cpp:188-193)
        mine_ok = mine_ok && x_i[p] >= 0.0 && x_i[p] < P.xs && y_i[p] >= 0.0 && y_i[p] < P.ys;
      else
        apply_pbc(P, x_i[p], y_i[p], x_i[p], y_i[p]);  // ParticleSystemFirstOrderPtr.cpp:270
    }
  }
  PhasorSums a[PPL];
  for (int j0 = jb; j0 < je; j0 += JT) {
    const int cnt = min(JT, je - j0);
    __syncthreads();
    bool ok = mine_ok;
    for (int q = threadIdx.x; q < cnt; q += T) {
      const double4 r = rec[j0 + q];
      ok = ok && r.x != kExactMark;
      tile[q] = r;
      if (HO) tom[q] = om[j0 + q];
    }
    if (__syncthreads_and(ok)) {
      // only tiles that hold some of the workgroup's own particles compare i with j
      const bool own = j0 < i0 + BLOCK && j0 + cnt > i0;
      int t0 = 0;
      if (!own)
        for (; t0 + 4 <= cnt; t0 += 4)
          four_j<S, HO, PPL, T, false>(P, band, neg_slope, stage, tile, tom, i0, j0, t0, cnt, x_i, y_i, om_i, a);
      for (; t0 < cnt; t0 += 4)
        four_j<S, HO, PPL, T, true>(P, band, neg_slope, stage, tile, tom, i0, j0, t0, cnt, x_i, y_i, om_i, a);
    } else {
      for (int t = 0; t < cnt; ++t)
        exact_j<S, HO, PPL, T>(P, stage, tile[t], HO ? tom[t] : 0.0, i0, j0 + t, x_i, y_i, om_i, a);
    }
  }
  double *out = part + (long)blockIdx.y * (HO ? 5 : 3) * n;
#pragma unroll
  for (int p = 0; p < PPL; ++p) {
    const int i = i0 + p * T + threadIdx.x;
    if (i >= n) continue;
    out[i] = a[p].S;
    out[(long)n + i] = a[p].C;
    out[2L * n + i] = a[p].card;
    if (HO) {
      out[3L * n + i] = a[p].TS;
      out[4L * n + i] = a[p].TC;
    }
  }
}

// 64 particles per workgroup, a quarter of the segments per wave (one thread per particle over all
// segments leaves most of the chip idle at a few thousand particles: 10.7 against 6 us at n = 4,099)
template <int S, bool HO>
__global__ __launch_bounds__(256) void ap_finish(DevParams P, int nseg, const double *__restrict__ stage,
                                                 const double *__restrict__ part, const double *__restrict__ nat,
                                                 double *__restrict__ k_next, double *__restrict__ compl_out) {
  constexpr int Q = HO ? 5 : 3;
  __shared__ double sh[3][Q][64];
  const int n = P.n, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  const int gb = wv * nseg / 4, ge = (wv + 1) * nseg / 4;
  double v[Q] = {};
  for (int g0 = gb; i < n && g0 < ge; g0 += 8) {  // the loads of eight segments in flight, then their sums in order
    double x[8][Q];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < Q; ++q) x[u][q] = g0 + u < ge ? part[((long)(g0 + u) * Q + q) * n + i] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < Q; ++q) v[q] += x[u][q];
  }
  if (wv > 0)
#pragma unroll
    for (int q = 0; q < Q; ++q) sh[wv - 1][q][lane] = v[q];
  __syncthreads();
  if (wv > 0 || i >= n) return;
#pragma unroll
  for (int q = 0; q < Q; ++q) v[q] = ((v[q] + sh[0][q][lane]) + sh[1][q][lane]) + sh[2][q][lane];
  PhasorSums a;
  a.S = v[0];
  a.C = v[1];
  a.card = v[2];
  if (HO) {
    a.TS = v[3];
    a.TC = v[4];
  }
  double st[S];
#pragma unroll
  for (int q = 0; q < S; ++q) st[q] = stage[(long)i * S + q];
  double s_i, c_i;
  frame_phasor_any(st[Slots<S>::phi], frame_ref(stage[Slots<S>::phi]), s_i, c_i);
  const PairAcc pa = pair_acc<S>(P, a, s_i, c_i);
  write_k<S>(P, st, i, pa, nat ? nat[i] : 0.0, k_next, compl_out);
}

// Up to 64 particles: stage, pair sums and derivative in one launch of one wave, the stage and its records in LDS.
// The same sums as by the kernels above (one segment); a Runge-Kutta step of 2 particles in 14 to 18 us for 51, of 64
// in 28 for 58.  (One wave is the line: 65 particles take 52 by the three launches.)
// (kprev and k_next may be the same array: every lane has read kprev before the wave writes.)
constexpr int kFew = kAllPairsFew;

template <int S, bool HO>
__global__ __launch_bounds__(kFew) void ap_few(DevParams P, double band, double neg_slope,
                                               const double *__restrict__ state, const double *kprev, double kc_dt,
                                               const double *__restrict__ nat, double *k_next, double *compl_out) {
  __shared__ double4 tile[kFew];
  __shared__ double tom[kFew], stage[kFew * S];
  const int n = P.n, i = threadIdx.x;
  constexpr int kPhi = Slots<S>::phi;
  const double ref = frame_ref(state[kPhi] + (kprev ? kc_dt * kprev[kPhi] : 0.0));
  double st[S] = {}, x_i[1] = {0.0}, y_i[1] = {0.0}, om_i[1] = {0.0};
  bool ok = true;
  double4 mine{};
  if (i < n) {
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const int e = i * S + q;
      st[q] = state[e] + (kprev ? kc_dt * kprev[e] : 0.0);
      stage[e] = st[q];
    }
    mine = record<S>(P, st, ref);
    ok = mine.x != kExactMark;
    tile[i] = mine;
    if (S == 6) {
      x_i[0] = st[0];
      y_i[0] = st[1];
    } else {
      apply_pbc(P, st[0], st[1], x_i[0], y_i[0]);
    }
    if (HO) tom[i] = om_i[0] = st[Slots<S>::omega];
  }
  PhasorSums a[1];
  if (__syncthreads_and(ok)) {
    for (int t0 = 0; t0 < n; t0 += 4)
      four_j<S, HO, 1, kFew, true>(P, band, neg_slope, stage, tile, tom, 0, 0, t0, n, x_i, y_i, om_i, a);
  } else {
    for (int j = 0; j < n; ++j)
      exact_j<S, HO, 1, kFew>(P, stage, tile[j], tom[j], 0, j, x_i, y_i, om_i, a);
  }
  if (i >= n) return;
  const PairAcc pa = pair_acc<S>(P, a[0], mine.z, mine.w);
  write_k<S>(P, st, i, pa, nat ? nat[i] : 0.0, k_next, compl_out);
}

template <int S, bool HO, int BLOCK, int JT>
void pairs_as(hipStream_t st, const DevParams &P, const AllPairsScratch &W, const double *stage) {
  constexpr int PPL = BLOCK >= 128 ? 2 : 1;
  const dim3 grid((unsigned)((P.n + BLOCK - 1) / BLOCK), (unsigned)W.nseg);
  const double band = pair_band(P.rho2, P.xs, P.ys);
  ap_pairs<S, HO, BLOCK, JT, PPL><<<grid, dim3(BLOCK / PPL), 0, st>>>(
      P, band, pair_neg_slope(band), (P.n + W.nseg - 1) / W.nseg, stage, (const double4 *)W.rec, W.om, W.part);
}

template <int S, bool HO>
void rhs_as(hipStream_t st, const DevParams &P, const AllPairsScratch &W, const double *stage, const double *nat,
            double *k_next, double *compl_out, int config) {
  switch (config) {
    case 0: pairs_as<S, HO, 64, 64>(st, P, W, stage); break;
    case 1: pairs_as<S, HO, 64, 256>(st, P, W, stage); break;
    case 2: pairs_as<S, HO, 128, 128>(st, P, W, stage); break;
    case 3: pairs_as<S, HO, 128, 512>(st, P, W, stage); break;
    case 5: pairs_as<S, HO, 256, 512>(st, P, W, stage); break;
    default: pairs_as<S, HO, 256, 256>(st, P, W, stage); break;
  }
  ap_finish<S, HO><<<dim3((P.n + 63) / 64), dim3(256), 0, st>>>(P, W.nseg, stage, W.part, nat, k_next, compl_out);
}

}  // namespace

const int kAllPairsConfigs[kAllPairsConfigCount][2] = {{64, 64}, {64, 256}, {128, 128}, {128, 512},
                                                        {256, 256}, {256, 512}};

// segments of the j's: 64 fill the chip from some thousand particles on (17 groups x 64 segments x 2
// waves at n = 4,099); more particles bring their own groups, and 2^19 / n of them keep the
// partial sums within 2^19 particles' worth (21 MB)
int all_pairs_segments(int n) {
  const long by_work = (n + 63) / 64, by_size = (1L << 19) / n;
  long g = by_work < 64 ? by_work : 64;
  if (g > by_size) g = by_size;
  return g < 1 ? 1 : (int)g;
}

void launch_all_pairs_stage(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                            double *stage, const AllPairsScratch &W) {
  const dim3 nb((P.n + 255) / 256);
  double4 *rec = (double4 *)W.rec;
  switch (P.s) {
    case 3: ap_stage<3><<<nb, dim3(256), 0, st>>>(P, state, kprev, kc_dt, stage, rec, W.om); break;
    case 4: ap_stage<4><<<nb, dim3(256), 0, st>>>(P, state, kprev, kc_dt, stage, rec, W.om); break;
    case 6: ap_stage<6><<<nb, dim3(256), 0, st>>>(P, state, kprev, kc_dt, stage, rec, W.om); break;
    default: break;
  }
}

void launch_all_pairs_few(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                          const double *nat, double *k_next, double *compl_out) {
  const double band = pair_band(P.rho2, P.xs, P.ys), slope = pair_neg_slope(band);
  const dim3 wg(kFew);
  switch (P.s) {
    case 3: ap_few<3, false><<<1, wg, 0, st>>>(P, band, slope, state, kprev, kc_dt, nat, k_next, compl_out); break;
    case 4:
      if (P.higher_order)
        ap_few<4, true><<<1, wg, 0, st>>>(P, band, slope, state, kprev, kc_dt, nat, k_next, compl_out);
      else
        ap_few<4, false><<<1, wg, 0, st>>>(P, band, slope, state, kprev, kc_dt, nat, k_next, compl_out);
      break;
    case 6: ap_few<6, false><<<1, wg, 0, st>>>(P, band, slope, state, kprev, kc_dt, nat, k_next, compl_out); break;
    default: break;
  }
}

void launch_all_pairs(hipStream_t st, const DevParams &P, const AllPairsScratch &W, const double *stage,
                      const double *nat, double *k_next, double *compl_out, int config) {
  switch (P.s) {
    case 3: rhs_as<3, false>(st, P, W, stage, nat, k_next, compl_out, config); break;
    case 4:
      if (P.higher_order)
        rhs_as<4, true>(st, P, W, stage, nat, k_next, compl_out, config);
      else
        rhs_as<4, false>(st, P, W, stage, nat, k_next, compl_out, config);
      break;
    case 6: rhs_as<6, false>(st, P, W, stage, nat, k_next, compl_out, config); break;
    default: break;
  }
}

}  // namespace spss
