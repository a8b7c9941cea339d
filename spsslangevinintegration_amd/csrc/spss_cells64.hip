// spss_cells64.hip -- the FP64 linked-list right-hand side on a unit box with at least 3 x 3 cells,
// ParticleSystemFirstOrderPtr.cpp:318-468 / ParticleSystemSecondOrderPtr.cpp:232-385.
//
//   c64_keys    the stage state in the order of the previous build, cell keys, histogram
//   scan_local  cell starts inside blocks of cells
//   c64_place   cell starts, bucket fill
//   c64_rank    ascending particle index inside every cell; the stage state in the new cell order
//   c64_pairs   the phasor sums over the 3 x 3 cells (spss_pairs64.hpp) and the derivative
//
// The previous build's order is only a hint (any permutation is right): particles move by a small
// part of a cell between evaluations, so in that order the histogram needs one atomic per run of
// equal keys in a wave and the gathers of c64_rank are nearly contiguous.  The states reach cell
// order once, in c64_keys; everything behind it reads neighbouring lines.
#pragma clang fp contract(off)

#include <algorithm>

#include "spss_launch.hpp"
#include "spss_pairs64.hpp"
#include "spss_scan.hpp"

namespace spss {

namespace {

template <int S>
__global__ __launch_bounds__(256) void c64_keys(DevParams P, const double *__restrict__ state,
                                                const double *__restrict__ kprev,
                                                double kc_dt, const int *__restrict__ order, int nc,
                                                double *__restrict__ pre, int *__restrict__ key,
                                                int *__restrict__ slot, int *__restrict__ count, int *__restrict__ bad) {
  const int t = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
  if (t < 2) bad[t] = 0;  // and the number of extra chunks
  int c = -1;
  if (t < P.n) {
    const long i = order[t];
    double st[S];
#pragma unroll
    for (int q = 0; q < S; ++q) st[q] = state[i * S + q] + (kprev ? kc_dt * kprev[i * S + q] : 0.0);
#pragma unroll
    for (int q = 0; q < S; ++q) pre[(long)t * S + q] = st[q];
    double xw, yw;
    key_wrap<S>(P, st[0], st[1], xw, yw);
    c = cell_coord(yw, nc) * nc + cell_coord(xw, nc);
  }
  // one atomic per run of equal keys
  const int before = __shfl_up(c, 1, 64);
  const unsigned long long heads = __ballot(lane == 0 || c != before);
  const int head = 63 - __clzll(heads & (~0ull >> (63 - lane)));
  const unsigned long long later = head == 63 ? 0ull : heads >> (head + 1);
  int base = 0;
  if (lane == head && c >= 0) base = atomicAdd(count + c, later ? __ffsll((long long)later) : 64 - head);
  base = __shfl(base, head, 64);
  if (t < P.n) {
    key[t] = c;
    slot[t] = base + lane - head;
  }
}

// Bucket fill, and the second half of the scan beside it: `local` holds the starts inside blocks of
// 256 * kScanItems cells, the blocks' offsets come from their totals (every workgroup sums them
// itself: one launch less than a kernel that adds them first).  The final starts go to `start`, the
// histogram is cleared.  Rows of more than `cap` particles, what their own workgroups of c64_pairs take, leave the
// rest in extra chunks of tb particles for all of its workgroups: {row, first position}.
constexpr int kPlaceBlocks = 1024;  // scan blocks at most (2 million cells)
__global__ __launch_bounds__(256) void c64_place(int n, int m, int nc, int nblk, int cap, int tb,
                                                 const int *__restrict__ key,
                                                 const int *__restrict__ slot, const int *__restrict__ local,
                                                 const int *__restrict__ total, const int *__restrict__ order,
                                                 int *__restrict__ start, int *__restrict__ count,
                                                 int2 *__restrict__ tmp, int *__restrict__ extras,
                                                 int2 *__restrict__ extra) {
  __shared__ int off[kPlaceBlocks + 1];
  if (threadIdx.x < 64) {
    int run = 0;
    for (int b0 = 0; b0 < nblk; b0 += 64) {
      const int lane = threadIdx.x, own = b0 + lane < nblk ? total[b0 + lane] : 0;
      int v = own;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
      }
      if (b0 + lane < nblk) off[b0 + lane] = run + v - own;
      run += __shfl(v, 63, 64);
    }
    if (threadIdx.x == 0) off[nblk] = run;
  }
  __syncthreads();
  for (int t = blockIdx.x * 256 + threadIdx.x; t < max(n, m + 1); t += gridDim.x * 256) {
    if (t < n) {
      const int c = key[t];
      tmp[local[c] + off[c / (256 * kScanItems)] + slot[t]] = make_int2(order[t], t);
    }
    if (t < m) {
      start[t] = local[t] + off[t / (256 * kScanItems)];
      count[t] = 0;
    }
    if (t == m) start[m] = off[nblk];
    if (t < nc) {
      const int a = t * nc, b = a + nc;
      const int r0 = local[a] + off[a / (256 * kScanItems)], r1 = b < m ? local[b] + off[b / (256 * kScanItems)] : off[nblk];
      const int chunks = (r1 - r0 - cap + tb - 1) / tb;
      if (r1 - r0 > cap) {
        int2 *to = extra + atomicAdd(extras, chunks);
        for (int k = 0; k < chunks; ++k) to[k] = make_int2(t, r0 + cap + k * tb);
      }
    }
  }
}

// Position p of the bucket fill goes to the slot of its rank among its cell's particle indices.
// `bad` is set by a particle that the cheap test or the phasors cannot serve: far outside the box, a
// phase beyond kPhase64 (NaN and infinity too), model 6 wrapped to exactly 1 (ClassA takes |dx| = 1 as a distance).
template <int S>
__global__ __launch_bounds__(256) void c64_rank(DevParams P, int nc, const int *__restrict__ key,
                                                const int *__restrict__ start, const int2 *__restrict__ tmp,
                                                const double *__restrict__ pre, int *__restrict__ order,
                                                double *__restrict__ snap, int *__restrict__ bad) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= P.n) return;
  const int2 me = tmp[p];
  const int c = key[me.y], b = start[c], e = start[c + 1];
  int r = 0;
  for (int u = b; u < e; ++u) r += tmp[u].x < me.x ? 1 : 0;
  double st[S];
#pragma unroll
  for (int q = 0; q < S; ++q) st[q] = pre[(long)me.y * S + q];
  order[b + r] = me.x;
#pragma unroll
  for (int q = 0; q < S; ++q) snap[(long)(b + r) * S + q] = st[q];
  bool fine = fabs(st[0]) <= kFar64 && fabs(st[1]) <= kFar64 && fabs(st[Slots<S>::phi]) <= kPhase64;
  if (S == 4 && P.higher_order) fine = fine && fabs(st[Slots<S>::omega]) < 1e300;
  if (S == 6) {
    double xw, yw;
    key_wrap<S>(P, st[0], st[1], xw, yw);
    fine = fine && xw < 1.0 && yw < 1.0;
  }
  if (!fine) *bad = 1;
}

constexpr int kCols = 64;   // staged columns of a tile at most

template <bool HO, int CAP, int TB>
struct Stage64 {
  double4 rec[CAP];  // x, y (the periodic image next to the tile), sin psi, cos psi
  double om[HO ? CAP : 1];
  int offs[3][kCols + 1];  // staged entries before each staged column of a row of cells
  int first[3][kCols];     // its first sorted position
  int col[TB];             // cell column of each particle of the workgroup
  int cut;                 // particles of the tile (past it: beyond kCols columns)
};

// the sums over the candidates [u, u + 4) (MASKED: only those before e) of a staged window
template <int S, bool HO, bool MASKED, class LDS, class EXACT>
__device__ __forceinline__ void four_pairs(const DevParams &P, double band, double neg_slope, const LDS &L, int u, int e,
                                           double x_i, double y_i, double om_i, PhasorSums &a, const EXACT &exact) {
  double w[4], near = 1e300;
  double4 r[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = L.rec[MASKED ? min(u + q, e - 1) : u + q];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double dx = r[q].x - x_i, dy = r[q].y - y_i;
    const double t = __builtin_fma(dx, dx, __builtin_fma(dy, dy, -P.rho2));
    near = fmin(near, fabs(t));
    w[q] = pair_weight(t, neg_slope);
    if (MASKED && u + q >= e) w[q] = 0.0;
  }
  if (near <= band) {  // rare: the reference's own test decides
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = (!MASKED || u + q < e) && exact(u + q) ? 1.0 : 0.0;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    a.S = __builtin_fma(w[q], r[q].z, a.S);
    a.C = __builtin_fma(w[q], r[q].w, a.C);
    a.card += w[q];
    if (HO) {
      const double wo = w[q] * (L.om[MASKED ? min(u + q, e - 1) : u + q] - om_i);
      a.TS = __builtin_fma(wo, r[q].z, a.TS);
      a.TC = __builtin_fma(wo, r[q].w, a.TC);
    }
  }
}

// One workgroup per TB particles of a row of cells (chunk k of row r; then the extra chunks of longer rows, shared
// out over all workgroups: 30,000 particles in one row of 33 in 0.38 ms, 3.8 with a row left to its own), one per
// lane in cell order: the three rows of cells around them are staged into LDS, positions as the periodic image next
// to the tile, so that a separation is a plain difference; dense cells pass through the stage in windows of CAP
// entries.  A lane walks the three column ranges of its particle, contiguous in the stage, in the reference's
// stencil order
// (ParticleSystemFirstOrderPtr.cpp:83-88).
template <int S, bool HO, int TB, int CAP>
__global__ __launch_bounds__(TB, HO ? 3 : 4) void c64_pairs(DevParams P, double band, double neg_slope, int nc, int rows8,
                                                const int *__restrict__ start, const int *__restrict__ order,
                                                const double *__restrict__ snap, const int *__restrict__ bad,
                                                const int2 *__restrict__ extra, const double *__restrict__ nat,
                                                double *__restrict__ k_next, double *__restrict__ compl_out) {
  constexpr int kPhi = Slots<S>::phi, kOm = S == 3 ? 2 : Slots<S>::omega;
  __shared__ Stage64<HO, CAP, TB> L;
  // workgroups go round the eight XCDs: each takes an eighth of the rows, so that neighbouring rows
  // share an L2
  int row = (blockIdx.x & 7) * rows8 + (blockIdx.x >> 3);
  const int extras = bad[1];
  int next = blockIdx.y * gridDim.x + blockIdx.x;  // of the extra chunks
  int base = row < nc ? start[row * nc] + (int)blockIdx.y * TB : 0, r1 = row < nc ? start[(row + 1) * nc] : 0;
  bool own = base < r1;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (;; own = false) {
    if (!own) {
      if (next >= extras) break;
      const int2 it = extra[next];
      next += gridDim.x * gridDim.y;
      row = it.x;
      base = it.y;
      r1 = start[(row + 1) * nc];
    }
    const int last = min(r1, base + TB);
    if (*bad) {  // pair by pair, the reference's expressions
      for (int g = base + threadIdx.x; g < last; g += TB) {
        double st[S], x_i, y_i;
#pragma unroll
        for (int q = 0; q < S; ++q) st[q] = snap[(long)g * S + q];
        key_wrap<S>(P, st[0], st[1], x_i, y_i);
        const int cx = cell_coord(x_i, nc);
        PairAcc a{0.0, 0.0, 0.0};
        for (int k = -1; k <= 1; ++k)
          for (int dc = -1; dc <= 1; ++dc) {
            const int c = adjust_cell(row + k, nc) * nc + adjust_cell(cx + dc, nc);
            for (int u = start[c]; u < start[c + 1]; ++u) {
              if (u == g) continue;
              const double *sj = snap + (long)u * S;
              double x_j = sj[0], y_j = sj[1];
              if (S == 6) key_wrap<6>(P, x_j, y_j, x_j, y_j);  // ParticleSystemSecondOrderPtr.cpp:356-359
              pair_term<S>(P, x_i, y_i, st[kPhi], S == 3 ? 0.0 : st[kOm], x_j, y_j, sj[kPhi], S == 3 ? 0.0 : sj[kOm], a);
            }
          }
        const int i = order[g];
        write_k<S>(P, st, i, a, nat ? nat[i] : 0.0, k_next, compl_out);
      }
      continue;
    }
    const int g = base + threadIdx.x, gi = min(g, last - 1);  // a lane past the end repeats the last particle
    double x_i, y_i;
    key_wrap<S>(P, snap[(long)gi * S], snap[(long)gi * S + 1], x_i, y_i);
    const double phi_i = snap[(long)gi * S + kPhi];
    const int cx = cell_coord(x_i, nc);
    const double ref = frame_ref(snap[(long)base * S + kPhi]);
    if (g < last) L.col[threadIdx.x] = cx;
    if (threadIdx.x == 0) L.cut = last;
    int done = base;  // particles before it are finished
    while (done < last) {
      __syncthreads();
      // the tile: particles [done, cut) whose cells span at most kCols - 2 columns
      const int ca = L.col[done - base];
      int cut = last;
      if (L.col[last - 1 - base] > ca + kCols - 3) {  // a sparse row (the same for all threads)
        if (g >= done && g < last && cx > ca + kCols - 3) atomicMin(&L.cut, g);
        __syncthreads();
        cut = L.cut;
        __syncthreads();
        if (threadIdx.x == 0) L.cut = last;
      }
      const int cb = L.col[cut - 1 - base];
      const int ncols = cb - ca + 3;
      // staging plan: counts of the staged columns of each row and their prefix sums
      for (int k = wv; k < 3; k += TB / 64) {
        const int cbase = adjust_cell(row + k - 1, nc) * nc;
        int s0 = 0, cnt = 0;
        if (lane < ncols) {
          const int c = cbase + adjust_cell(ca - 1 + lane, nc);
          s0 = start[c];
          cnt = start[c + 1] - s0;
        }
        int incl = cnt;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int v = __shfl_up(incl, off, 64);
          if (lane >= off) incl += v;
        }
        if (lane < ncols) {
          L.offs[k][lane] = incl - cnt;
          L.first[k][lane] = s0;
        }
        if (lane == ncols - 1) L.offs[k][ncols] = incl;
      }
      __syncthreads();
      const int n0 = L.offs[0][ncols], n1 = n0 + L.offs[1][ncols], total = n1 + L.offs[2][ncols];
      const auto rowbase = [n0, n1](int k) { return k == 0 ? 0 : (k == 1 ? n0 : n1); };
      const bool mine = g >= done && g < cut;  // a lane takes part if its particle lies in the tile
      const int ql = cx - ca;                  // its first staged column
      PhasorSums a;
      double s_i = 0.0, c_i = 0.0, om_i = 0.0;
      if (mine) {
        // a particle meets itself among its candidates: its own term is taken off beforehand (those with omegas are
        // zeros)
        frame_phasor(phi_i, ref, s_i, c_i);
        a.S = -s_i;
        a.C = -c_i;
        a.card = -1.0;
        if (HO) om_i = snap[(long)gi * S + kOm];
      }
      for (int w0 = 0; w0 < total; w0 += CAP) {
        const int w1 = min(total, w0 + CAP);
        if (w0 > 0) __syncthreads();
        // a row's staged columns are one run of the cell order, but for those across the box's edge;
        // positions and phases first, so that a thread's loads are in flight together
        constexpr int IT = (CAP + TB - 1) / TB;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
          const int v = it * TB + (int)threadIdx.x, vv = w0 + v;
          if (vv >= w1) continue;
          const int k = vv < n0 ? 0 : (vv < n1 ? 1 : 2), o = vv - rowbase(k);
          const bool left = ca == 0 && o < L.offs[k][1], right = cb == nc - 1 && o >= L.offs[k][ncols - 1];
          const int q = left ? 0 : (right ? ncols - 1 : (ca == 0 ? 1 : 0));
          const double *sj = snap + ((long)L.first[k][q] + o - L.offs[k][q]) * S;
          double xw, yw;
          key_wrap<S>(P, sj[0], sj[1], xw, yw);
          const int jrow = row + k - 1;
          L.rec[v] = make_double4(xw + (left ? -1.0 : (right ? 1.0 : 0.0)),
                                  yw + (jrow < 0 ? -1.0 : (jrow >= nc ? 1.0 : 0.0)), sj[kPhi], 0.0);
          if (HO) L.om[v] = sj[kOm];
        }
        for (int v = threadIdx.x; v < w1 - w0; v += TB) {  // a thread's own entries
          double sn, cs;
          frame_phasor(L.rec[v].z, ref, sn, cs);
          L.rec[v].z = sn;
          L.rec[v].w = cs;
        }
        __syncthreads();
        if (mine) {
          // the reference's test of the staged entry u: its sorted position from the staging plan
          const auto exact = [&](int u) {
            const int v = w0 + u, k = v < n0 ? 0 : (v < n1 ? 1 : 2);
            int q = 0;
            while (rowbase(k) + L.offs[k][q + 1] <= v) ++q;
            const double *sj = snap + ((long)L.first[k][q] + v - rowbase(k) - L.offs[k][q]) * S;
            double x_j = sj[0], y_j = sj[1];
            if (S == 6) key_wrap<6>(P, x_j, y_j, x_j, y_j);
            return pair_in_range<S>(P, x_i, y_i, x_j, y_j);
          };
#pragma unroll 1
          for (int k = 0; k < 3; ++k) {
            int u = max(rowbase(k) + L.offs[k][ql], w0) - w0;
            const int e = min(rowbase(k) + L.offs[k][ql + 3], w1) - w0;
            PhasorSums r;  // a sum per row of cells: shorter chains of roundings
            for (; u + 4 <= e; u += 4) four_pairs<S, HO, false>(P, band, neg_slope, L, u, e, x_i, y_i, om_i, r, exact);
            if (u < e) four_pairs<S, HO, true>(P, band, neg_slope, L, u, e, x_i, y_i, om_i, r, exact);
            a.S += r.S;
            a.C += r.C;
            a.card += r.card;
            if (HO) {
              a.TS += r.TS;
              a.TC += r.TC;
            }
          }
        }
      }
      if (mine) {
        const int i = order[g];
        double st[S];
#pragma unroll
        for (int q = 0; q < S; ++q) st[q] = snap[(long)g * S + q];
        const PairAcc acc = pair_acc<S>(P, a, s_i, c_i);
        double sn, cs;
        small_sincos(st[kPhi], 0.0, sn, cs);
        write_k<S>(P, st, i, acc, nat ? nat[i] : 0.0, sn, cs, k_next, compl_out);
      }
      done = cut;
    }
  }
}

// 256 particles a workgroup of c64_pairs stage the fewest entries per particle; below some ten thousand
// particles 128 a workgroup fill the chip better (per evaluation of model 6: 39.6 -> 36 us at
// n = 20,000 against 42.2 -> 43.6 us at n = 50,000)
int chunk(int n) { return n >= 40960 ? 256 : 128; }
// chunks of a row of mean length, one more for the spread
int row_chunks(int n, int nc) {
  const long per_row = (n + nc - 1) / nc;
  return (int)std::min<long>((per_row + per_row / 8) / chunk(n) + 1, 65535);
}

template <int S>
void build(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt, int nc,
           Cells64 &B) {
  const dim3 nb((unsigned)((P.n + 255) / 256)), tb(256);
  const int m = nc * nc, next = B.cur ^ 1;
  c64_keys<S><<<nb, tb, 0, st>>>(P, state, kprev, kc_dt, B.order[B.cur], nc, B.pre, B.key, B.slot, B.count, B.bad);
  const int nblk = scan_blocks(m);
  scan_local<><<<dim3(nblk), tb, 0, st>>>(B.count, nullptr, m, B.local, B.blocksum);
  // by the cells too, of which few particles may have many (200 on 2 million: 2,674 us an evaluation by the
  // particles alone, now 46)
  const dim3 np(std::max(nb.x, std::min((unsigned)(m / 256 + 1), 2048u)));
  c64_place<<<np, tb, 0, st>>>(P.n, m, nc, nblk, row_chunks(P.n, nc) * chunk(P.n), chunk(P.n), B.key, B.slot, B.local,
                               B.blocksum, B.order[B.cur], B.start, B.count, (int2 *)B.tmp, B.bad + 1, (int2 *)B.extra);
  c64_rank<S><<<nb, tb, 0, st>>>(P, nc, B.key, B.start, (const int2 *)B.tmp, B.pre, B.order[next], B.snap, B.bad);
  B.cur = next;
}

template <int S, bool HO, int TB, int CAP>
void pairs_as(hipStream_t st, const DevParams &P, int nc, const Cells64 &B, const double *nat, double *k_next,
              double *compl_out) {
  const int rows8 = (nc + 7) / 8;
  const double band = pair_band(P.rho2, 1.0, 1.0);
  c64_pairs<S, HO, TB, CAP><<<dim3((unsigned)rows8 * 8, (unsigned)row_chunks(P.n, nc)), dim3(TB), 0, st>>>(
      P, band, pair_neg_slope(band), nc, rows8, B.start, B.order[B.cur], B.snap, B.bad, (const int2 *)B.extra, nat,
      k_next, compl_out);
}

template <int S, bool HO>
void pairs(hipStream_t st, const DevParams &P, int nc, const Cells64 &B, const double *nat, double *k_next,
           double *compl_out) {
  if (chunk(P.n) == 256)
    pairs_as<S, HO, 256, 1152>(st, P, nc, B, nat, k_next, compl_out);
  else
    pairs_as<S, HO, 128, 640>(st, P, nc, B, nat, k_next, compl_out);
}

}  // namespace

bool cells64_serves(const DevParams &P, int ncx, int ncy) {
  return P.xs == 1.0 && P.ys == 1.0 && ncx == ncy && ncx >= 3 && ncx <= 1448 &&
         scan_blocks((long)ncx * ncy) <= kPlaceBlocks;
}

void launch_cells64_build(hipStream_t st, const DevParams &P, const double *state, const double *kprev, double kc_dt,
                          int nc, Cells64 &B) {
  switch (P.s) {
    case 3: build<3>(st, P, state, kprev, kc_dt, nc, B); break;
    case 4: build<4>(st, P, state, kprev, kc_dt, nc, B); break;
    case 6: build<6>(st, P, state, kprev, kc_dt, nc, B); break;
    default: break;
  }
}

void launch_cells64_pairs(hipStream_t st, const DevParams &P, int nc, const Cells64 &B, const double *nat,
                          double *k_next, double *compl_out) {
  switch (P.s) {
    case 3: pairs<3, false>(st, P, nc, B, nat, k_next, compl_out); break;
    case 4:
      if (P.higher_order)
        pairs<4, true>(st, P, nc, B, nat, k_next, compl_out);
      else
        pairs<4, false>(st, P, nc, B, nat, k_next, compl_out);
      break;
    case 6: pairs<6, false>(st, P, nc, B, nat, k_next, compl_out); break;
    default: break;
  }
}

}  // namespace spss
