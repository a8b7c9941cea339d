// spss_observer.hip -- the reference's trajectory and summary outputs and its restart from the
// last saved frame (the spss_frame*, spss_summary*, spss_*_last_frame part of the C ABI).
//
// Frame (BinaryObserverFirstOrderPtr.cpp:108-121, BinaryObserverFirstOrder.cpp:101-122): a float
// time, then the s*n state values as floats.  Models 3 and 4 wrap the float copy: x and y by the
// float overload of PeriodicBoundaryConditions::ApplyPeriodicBoundaryConditions
// (PeriodicBoundaryConditions.cpp:137-145), phi by phi -= floor(phi / 2 pi) * 2 pi; each of these
// runs in double on the float value and is rounded back to float, as the float -= double of the
// reference does.  Model 6 writes the raw float copy (BinaryObserverSecondOrderPtr.cpp:108-113).
//
// Summary (BinaryObserverFirstOrderPtr.cpp:126-146, BinaryObserverSecondOrderPtr.cpp:175-193):
// Z = (1/n) sum_i ((float) cos phi_i + i (float) sin phi_i), accumulated in complex<float> in
// particle order; the line "t \t |Z| \t arg Z" with the default stream formatting.  The phasors
// are computed in parallel and summed with the rounding of every addition in particle order
// (spss_seqsum.hpp), so the float sums are the reference's; |Z| and arg Z are taken on the host with
// std::abs / std::arg of complex<float>.
//
// Restart (SimulationEngineFirstOrderPtr.cpp:70-94): the last complete frame of a file, found
// from the file size, its floats widened to double.
#include <hip/hip_runtime.h>

#include <cmath>
#include <complex>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/spss_hip.h"
#include "spss_hostcopy.hpp"
#include "spss_launch.hpp"
#include "spss_seqsum.hpp"

using namespace spss;

namespace {

constexpr double kTwoPi = 6.283185307179586476925286766559;

__global__ void ob_frame(const double *__restrict__ state, long m, int s, int wrap, double xs, double ys, double xrs,
                         double yrs, float *__restrict__ out) {
  const long k = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (k >= m) return;
  float v = (float)state[k];
  if (wrap) {
    const int q = (int)(k % s);
    if (q == 0)
      v = (float)((double)v - floor((double)v * xrs) * xs);
    else if (q == 1)
      v = (float)((double)v - floor((double)v * yrs) * ys);
    else if (q == 2)
      v = (float)((double)v - floor((double)v / kTwoPi) * kTwoPi);
  }
  out[k] = v;
}

// cosines into ph, sines into ph + npad; zeros from n to npad
__global__ void ob_phasors(const double *__restrict__ state, int n, long npad, int s, int slot,
                           float *__restrict__ ph) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= npad) return;
  float re = 0.f, im = 0.f;
  if (i < n) {
    const double phi = state[i * s + slot];
    re = (float)cos(phi);
    im = (float)sin(phi);
  }
  ph[i] = re;
  ph[npad + i] = im;
}

// The complex<float> accumulation of the reference, in particle order (spss_seqsum.hpp).  One lane
// adding term by term waited out a load per addition: 58.9 ms at n = 1,048,576.  Here ob_runs maps
// runs of L terms for 64 exponents (a wave per run and component, an exponent per lane), ob_long_runs
// composes 16 of them, and ob_walk goes through the long runs, into their runs where a long one
// leaves its binade, and term by term where a run does (n = 1,048,576, random phases: about half of
// the long runs, a tenth to a third of the runs).  121 + 11 us for the maps, 1.1-1.7 ms for the walk:
// 4.5 cycles per addition left (370,000 at most of the million), 340 per map looked up.
__global__ __launch_bounds__(256) void ob_runs(const float *__restrict__ ph, long npad, int L, int nruns,
                                               SeqMap *__restrict__ runs) {
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int run = w >> 1, comp = w & 1;
  if (run >= nruns) return;
  const float scale = ldexpf(1.f, 23 - (lane + kSeqExp0));
  const float limit = fminf(4194304.f, (float)(1 << 30) / (float)L);
  const float *c = ph + comp * npad + (long)run * L;
  SeqMap m = seq_identity();
  for (int i0 = 0; i0 < L; i0 += 64) {
    const float v = c[i0 + lane];
    for (int k = 0; k < 64; ++k) {
      const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
      seq_term(m, t * scale, limit);
    }
  }
  runs[((long)run * 2 + comp) * 64 + lane] = m;
}

__global__ __launch_bounds__(256) void ob_long_runs(const SeqMap *__restrict__ runs, int nruns, int nlong, int limit,
                                                    SeqMap *__restrict__ longs) {
  const long t = blockIdx.x * 256L + threadIdx.x;  // (long run, component, exponent)
  if (t >= nlong * 128L) return;
  const int q = (int)(t >> 7), rest = (int)(t & 127);
  SeqMap m = seq_identity();
  for (int r = q * kSeqLevel; r < min(nruns, (q + 1) * kSeqLevel); ++r) m = seq_compose(m, runs[r * 128L + rest], limit);
  longs[t] = m;
}

// s through the map in lane k of m: true if it stayed in its binade
__device__ __forceinline__ bool seq_pass(const SeqMap &m, int k, float &s) {
  if (s == 0.f) return seq_zeros(__builtin_amdgcn_readlane(m.reach, k));
  const int S = seq_units(s), p = S & 1;
  const int inc = __builtin_amdgcn_readlane(p ? m.inc[1] : m.inc[0], k);
  const int lo = __builtin_amdgcn_readlane(p ? m.lo[1] : m.lo[0], k);
  const int hi = __builtin_amdgcn_readlane(p ? m.hi[1] : m.hi[0], k);
  const int reach = __builtin_amdgcn_readlane(m.reach, k);
  if (!seq_stays(S, lo, hi, reach)) return false;
  s = seq_value(S + inc, s);
  return true;
}

__device__ __forceinline__ float wave_uniform(float s) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s)));
}

// s + the 256 terms at v, one by one: a quarter is read while the one before it is added
__device__ __forceinline__ void add_terms(const float4 *v, float &s) {
  float4 a[16], b[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) a[t] = v[t];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    if (h < 3)
#pragma unroll
      for (int t = 0; t < 16; ++t) b[t] = v[16 * (h + 1) + t];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      s = s + a[t].x;
      s = s + a[t].y;
      s = s + a[t].z;
      s = s + a[t].w;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) a[t] = b[t];
  }
}

// what the walk needs of one long run: its maps (an exponent per lane), its 16 runs' maps for the
// exponents k0, k0 + 1, k0 - 1, k0 - 2 (lane = run + 16 * exponent), and its terms if L == 256
struct SeqGroup {
  SeqMap lm, rm;
  int k0;
  float4 t[kSeqLevel];
};

// WHOLE: runs of 256 terms, whose long run fits the LDS
template <bool WHOLE>
struct SeqWalk {
  const float4 *c;
  const SeqMap *runs, *longs;
  int L, nlong, comp, lane;

  __device__ __forceinline__ void run_maps(SeqGroup &g, int q, int k0) const {
    const int e = lane >> 4, k = k0 + (e == 0 ? 0 : (e == 1 ? 1 : 1 - e));
    g.k0 = k0;
    g.rm = runs[(q * kSeqLevel + (lane & 15)) * 128L + comp * 64 + max(0, min(63, k))];
  }

  // (past the end: the last one again)
  __device__ __forceinline__ void load(SeqGroup &g, int q, float s) const {
    q = min(q, nlong - 1);
    g.lm = longs[q * 128L + comp * 64 + lane];
    run_maps(g, q, max(0, seq_lookup(wave_uniform(s))));
    if (WHOLE)
#pragma unroll
      for (int t = 0; t < kSeqLevel; ++t) g.t[t] = c[((long)q * kSeqLevel + t) * 64 + lane];
  }

  __device__ __forceinline__ void walk(SeqGroup &g, int q, float4 *terms, float &s) const {
    if (q >= nlong) return;
    s = wave_uniform(s);
    const int kl = seq_lookup(s);
    if (kl >= 0 && seq_pass(g.lm, kl, s)) return;
    if (WHOLE) {
#pragma unroll
      for (int t = 0; t < kSeqLevel; ++t) terms[64 * t + lane] = g.t[t];
      __syncthreads();
    }
    for (int r = 0; r < kSeqLevel; ++r) {
      s = wave_uniform(s);
      const int k = seq_lookup(s);
      if (k >= 0) {
        if (k - g.k0 > 1 || k - g.k0 < -2) run_maps(g, q, k);
        const int d = k - g.k0;
        if (seq_pass(g.rm, r + 16 * (d >= 0 ? d : 1 - d), s)) continue;
      }
      if (WHOLE) {
        add_terms(terms + r * 64, s);
        continue;
      }
      for (int i0 = 0; i0 < L; i0 += 256) {
        __syncthreads();
        terms[lane] = c[(((long)q * kSeqLevel + r) * L + i0) / 4 + lane];
        __syncthreads();
        add_terms(terms, s);
      }
    }
    if (WHOLE) __syncthreads();
  }
};

// One wave per component (blockIdx.x); the next long run is on its way while one is walked,
// and the chain of additions is what is left to wait for.
template <bool WHOLE>
__global__ __launch_bounds__(64) void ob_walk(const float *__restrict__ ph, long npad, int L, int nlong,
                                              const SeqMap *__restrict__ runs, const SeqMap *__restrict__ longs,
                                              float *__restrict__ out) {
  __shared__ float4 terms[WHOLE ? kSeqLevel * 64 : 64];
  const int comp = blockIdx.x;
  const SeqWalk<WHOLE> W{(const float4 *)(ph + comp * npad), runs, longs, L, nlong, comp, (int)threadIdx.x};
  float s = 0.f;
  SeqGroup a, b;
  W.load(a, 0, s);
  for (int q = 0; q < nlong; q += 2) {
    W.load(b, q + 1, s);
    W.walk(a, q, terms, s);
    W.load(a, q + 2, s);
    W.walk(b, q + 1, terms, s);
  }
  if (threadIdx.x == 0) out[comp] = s;
}

// Up to 16,384 terms (64 KB of LDS): phasors and their sum in one launch, a workgroup per component and its first
// wave adding term by term, 4.5 cycles each.  The maps' launches alone take longer: 22 us a call against 63 at
// n = 10, 34 against 73 at 4,096, 73 against 100 at 16,384.
constexpr int kSeqFew = 16384;

__global__ __launch_bounds__(512) void ob_few(const double *__restrict__ state, int n, int s, int slot,
                                               float *__restrict__ out) {
  __shared__ float4 terms[kSeqFew / 4];
  const int comp = blockIdx.x, npad = (n + 255) & ~255;
  for (int i = threadIdx.x; i < npad; i += 512) {
    float v = 0.f;
    if (i < n) {
      const double phi = state[(long)i * s + slot];
      v = (float)(comp ? sin(phi) : cos(phi));
    }
    ((float *)terms)[i] = v;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  float sum = 0.f;
  for (int i = 0; i < npad; i += 256) add_terms(terms + i / 4, sum);
  if (threadIdx.x == 0) out[comp] = sum;
}

int check(hipError_t e, const char *what) {
  return e == hipSuccess ? SPSS_OK : set_error(SPSS_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

#define OCHK(call)                                \
  do {                                            \
    int r_ = check((call), #call);                \
    if (r_ != SPSS_OK) return r_;                 \
  } while (0)

// the 1 + s*n floats of a frame into host memory
int frame_to_host(spss_system *sys, double t, float *host) {
  SystemView v{};
  int rc = system_view(sys, &v);
  if (rc != SPSS_OK) return rc;
  const long m = (long)v.s * v.n;
  float *d = nullptr;
  if ((rc = system_scratch(sys, sizeof(float) * m, (void **)&d)) != SPSS_OK) return rc;
  const unsigned nb = (unsigned)((m + 255) / 256);
  if (m > 0)
    hipLaunchKernelGGL(ob_frame, dim3(nb), dim3(256), 0, v.stream, v.state, m, v.s, v.s == 6 ? 0 : 1, v.x_size,
                       v.y_size, v.x_rsize, v.y_rsize, d);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = system_copy(sys).to_host(host + 1, d, sizeof(float) * m, v.stream);
  OCHK(e);
  host[0] = (float)t;
  return SPSS_OK;
}

int summary_sums(spss_system *sys, float *re, float *im, int *n_out) {
  SystemView v{};
  int rc = system_view(sys, &v);
  if (rc != SPSS_OK) return rc;
  if (v.n < 1) return set_error(SPSS_ERR_INVALID, "no particles");
  const int slot = v.s == 6 ? 4 : 2;
  float *out = nullptr;
  if (v.n <= kSeqFew) {
    if ((rc = system_scratch(sys, 2 * sizeof(float), (void **)&out)) != SPSS_OK) return rc;
    hipLaunchKernelGGL(ob_few, dim3(2), dim3(512), 0, v.stream, v.state, v.n, v.s, slot, out);
  } else {
    // runs of 256 terms, longer ones beyond 2^22 particles; whole long runs, filled up with zeros
    int L = 256;
    while (v.n / L >= 16384) L *= 2;
    const int nlong = (int)((v.n + (long)L * kSeqLevel - 1) / ((long)L * kSeqLevel)), nruns = nlong * kSeqLevel;
    const long npad = (long)nruns * L;
    SeqMap *runs = nullptr;
    const size_t maps = ((size_t)nruns + nlong) * 128;
    if ((rc = system_scratch(sys, maps * sizeof(SeqMap) + sizeof(float) * (2 * npad + 2), (void **)&runs)) != SPSS_OK)
      return rc;
    SeqMap *longs = runs + (size_t)nruns * 128;
    float *ph = (float *)(runs + maps);
    out = ph + 2 * npad;
    hipLaunchKernelGGL(ob_phasors, dim3((unsigned)(npad / 256)), dim3(256), 0, v.stream, v.state, v.n, npad, v.s, slot, ph);
    hipLaunchKernelGGL(ob_runs, dim3(nruns / 2), dim3(256), 0, v.stream, ph, npad, L, nruns, runs);
    hipLaunchKernelGGL(ob_long_runs, dim3((nlong * 128 + 255) / 256), dim3(256), 0, v.stream, runs, nruns, nlong,
                       (1 << 30) / (L * kSeqLevel), longs);
    if (L == 256)
      hipLaunchKernelGGL(ob_walk<true>, dim3(2), dim3(64), 0, v.stream, ph, npad, L, nlong, runs, longs, out);
    else
      hipLaunchKernelGGL(ob_walk<false>, dim3(2), dim3(64), 0, v.stream, ph, npad, L, nlong, runs, longs, out);
  }
  hipError_t e = hipGetLastError();
  float h[2] = {0.f, 0.f};
  if (e == hipSuccess) e = hipMemcpyAsync(h, out, sizeof(h), hipMemcpyDeviceToHost, v.stream);
  if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
  OCHK(e);
  *re = h[0];
  *im = h[1];
  *n_out = v.n;
  return SPSS_OK;
}

}  // namespace

extern "C" {

int spss_frame(spss_system *sys, double t, float *host_frame) {
  if (!sys || !host_frame) return set_error(SPSS_ERR_INVALID, "NULL argument");
  return frame_to_host(sys, t, host_frame);
}

int spss_frame_append(spss_system *sys, const char *path, double t) {
  if (!sys || !path) return set_error(SPSS_ERR_INVALID, "NULL argument");
  SystemView v{};
  int rc = system_view(sys, &v);
  if (rc != SPSS_OK) return rc;
  std::vector<float> buf(1 + (size_t)v.s * v.n);
  if ((rc = frame_to_host(sys, t, buf.data())) != SPSS_OK) return rc;
  FILE *f = std::fopen(path, "ab");
  if (!f) return set_error(SPSS_ERR_INVALID, std::string("cannot open ") + path);
  const size_t w = std::fwrite(buf.data(), sizeof(float), buf.size(), f);
  const int closed = std::fclose(f);
  if (w != buf.size() || closed != 0) return set_error(SPSS_ERR_INVALID, std::string("cannot write ") + path);
  return SPSS_OK;
}

int spss_summary(spss_system *sys, float *abs_z, float *arg_z) {
  if (!sys || !abs_z || !arg_z) return set_error(SPSS_ERR_INVALID, "NULL argument");
  float re = 0.f, im = 0.f;
  int n = 0;
  int rc = summary_sums(sys, &re, &im, &n);
  if (rc != SPSS_OK) return rc;
  std::complex<float> z(re, im);
  z /= (float)n;
  *abs_z = std::abs(z);
  *arg_z = std::arg(z);
  return SPSS_OK;
}

int spss_summary_append(spss_system *sys, const char *path, double t) {
  if (!sys || !path) return set_error(SPSS_ERR_INVALID, "NULL argument");
  float a = 0.f, g = 0.f;
  int rc = spss_summary(sys, &a, &g);
  if (rc != SPSS_OK) return rc;
  FILE *f = std::fopen(path, "a");
  if (!f) return set_error(SPSS_ERR_INVALID, std::string("cannot open ") + path);
  // operator<< of a float with the default stream settings prints it as %g of its double value
  const int w = std::fprintf(f, "%g\t%g\t%g\n", (double)(float)t, (double)a, (double)g);
  const int closed = std::fclose(f);
  if (w < 0 || closed != 0) return set_error(SPSS_ERR_INVALID, std::string("cannot write ") + path);
  return SPSS_OK;
}

int spss_read_last_frame(const char *path, int s, int n, float *t, double *state) {
  if (!path || !t || !state) return set_error(SPSS_ERR_INVALID, "NULL argument");
  if (s < 1 || n < 1) return set_error(SPSS_ERR_INVALID, "s and n must be >= 1");
  FILE *f = std::fopen(path, "rb");
  if (!f) return set_error(SPSS_ERR_INVALID, std::string("cannot open ") + path);
  const long frame = (1L + (long)s * n) * (long)sizeof(float);
  long size = -1;
  if (std::fseek(f, 0, SEEK_END) == 0) size = std::ftell(f);
  const long t_max = size > 0 ? size / frame : 0;
  if (t_max < 1) {
    std::fclose(f);
    return set_error(SPSS_ERR_INVALID, std::string("no complete frame in ") + path);
  }
  std::vector<float> buf((size_t)s * n);
  bool ok = std::fseek(f, frame * (t_max - 1), SEEK_SET) == 0;
  ok = ok && std::fread(t, sizeof(float), 1, f) == 1;
  ok = ok && std::fread(buf.data(), sizeof(float), buf.size(), f) == buf.size();
  std::fclose(f);
  if (!ok) return set_error(SPSS_ERR_INVALID, std::string("cannot read ") + path);
  for (size_t k = 0; k < buf.size(); ++k) state[k] = (double)buf[k];
  return SPSS_OK;
}

int spss_load_last_frame(spss_system *sys, const char *path, double *t) {
  if (!sys || !path) return set_error(SPSS_ERR_INVALID, "NULL argument");
  SystemView v{};
  int rc = system_view(sys, &v);
  if (rc != SPSS_OK) return rc;
  std::vector<double> st((size_t)v.s * v.n);
  float tf = 0.f;
  if ((rc = spss_read_last_frame(path, v.s, v.n, &tf, st.data())) != SPSS_OK) return rc;
  if ((rc = spss_set_state(sys, st.data())) != SPSS_OK) return rc;
  if (t) *t = (double)tf;
  return SPSS_OK;
}

}  // extern "C"
