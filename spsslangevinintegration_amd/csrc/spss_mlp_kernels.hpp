// spss_mlp_kernels.hpp -- device code of the sweep-screen network (included by spss_mlp.hip).
//
// Networks of any width: one launch per layer and direction, 256 threads, 32 x 32 output tiles; reductions are staged
// through LDS in chunks of 64 and summed in ascending index order with FMAs, without atomics,
// so that every result is reproducible bit for bit.  Matrices are row-major FP32.
#pragma once

#include <hip/hip_runtime.h>

namespace spss {
namespace mlp {

constexpr int kT = 32;    // edge of an output tile
constexpr int kK = 64;    // reduction chunk staged in LDS
constexpr int kTB = 256;  // threads per block: 32 columns x 8 row groups, 4 rows each

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }

// d/dz [z Phi(z)] = Phi(z) + z phi(z)
__device__ __forceinline__ float gelu_grad(float z) {
  const float cdf = 0.5f * (1.f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return __builtin_fmaf(z, pdf, cdf);
}

// Z[b, o] = sum_i A[row(b), i] W[o, i] + bias[o]; H[b, o] = gelu(Z[b, o]) when H is given.
// row(b) = (a_off + b) mod a_mod: a ring over the resident training set for the input layer.
__global__ __launch_bounds__(kTB) void ml_fwd(const float *A, long a_off, long a_mod, int B, int in, int out,
                                              const float *W, const float *bias, float *Z, float *H) {
  __shared__ float sa[kT][kK + 1];
  __shared__ float sw[kT][kK + 1];
  const int b0 = blockIdx.x * kT, o0 = blockIdx.y * kT;
  const int tx = threadIdx.x % kT, ty = threadIdx.x / kT;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < in; i0 += kK) {
    const int kk = min(kK, in - i0);
    for (int e = threadIdx.x; e < kT * kK; e += kTB) {
      const int r = e / kK, c = e % kK;
      float va = 0.f, vw = 0.f;
      if (c < kk) {
        if (b0 + r < B) va = A[((a_off + b0 + r) % a_mod) * in + i0 + c];
        if (o0 + r < out) vw = W[(long)(o0 + r) * in + i0 + c];
      }
      sa[r][c] = va;
      sw[r][c] = vw;
    }
    __syncthreads();
    for (int c = 0; c < kk; ++c) {
      const float w = sw[tx][c];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = __builtin_fmaf(sa[ty + 8 * q][c], w, acc[q]);
    }
    __syncthreads();
  }
  const int o = o0 + tx;
  if (o >= out) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int b = b0 + ty + 8 * q;
    if (b < B) {
      const float z = acc[q] + bias[o];
      Z[(long)b * out + o] = z;
      if (H) H[(long)b * out + o] = gelu(z);
    }
  }
}

// mean squared error over the B x m outputs: D = 2 (Y - T) / (B m), loss = sum (Y - T)^2 / (B m)
// (FP64 partial sums in a fixed tree); targets of row b at T[(t_off + b) mod t_mod]
__global__ __launch_bounds__(kTB) void ml_mse(const float *Y, const float *T, long t_off, long t_mod, int B, int m,
                                              float *D, float *loss) {
  __shared__ double red[kTB];
  const float scale = 2.f / (float)(B * m);
  double s = 0.0;
  for (int e = threadIdx.x; e < B * m; e += kTB) {
    const int b = e / m, j = e % m;
    const float d = Y[e] - T[((t_off + b) % t_mod) * m + j];
    D[e] = scale * d;
    s += (double)d * (double)d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = kTB / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = (float)(red[0] / (double)(B * m));
}

// dW[o, i] = sum_b D[b, o] A[row(b), i], b ascending; column i == in is the bias (A = 1)
__global__ __launch_bounds__(kTB) void ml_bwd_weight(const float *D, int B, int out, const float *A, long a_off,
                                                     long a_mod, int in, float *dW, float *db) {
  __shared__ float sd[kK][kT + 1];
  __shared__ float sa[kK][kT + 1];
  const int o0 = blockIdx.x * kT, i0 = blockIdx.y * kT;
  const int tx = threadIdx.x % kT, ty = threadIdx.x / kT;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int bb = 0; bb < B; bb += kK) {
    const int kk = min(kK, B - bb);
    for (int e = threadIdx.x; e < kK * kT; e += kTB) {
      const int r = e / kT, c = e % kT;
      float vd = 0.f, va = 0.f;
      if (r < kk) {
        if (o0 + c < out) vd = D[(long)(bb + r) * out + o0 + c];
        const int i = i0 + c;
        if (i < in) va = A[((a_off + bb + r) % a_mod) * in + i];
        else if (i == in) va = 1.f;
      }
      sd[r][c] = vd;
      sa[r][c] = va;
    }
    __syncthreads();
    for (int r = 0; r < kk; ++r) {
      const float a = sa[r][tx];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = __builtin_fmaf(sd[r][ty + 8 * q], a, acc[q]);
    }
    __syncthreads();
  }
  const int i = i0 + tx;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int o = o0 + ty + 8 * q;
    if (o >= out) continue;
    if (i < in) dW[(long)o * in + i] = acc[q];
    else if (i == in) db[o] = acc[q];
  }
}

// G[b, i] = (sum_o D[b, o] W[o, i]) gelu'(Zp[b, i]), o ascending
__global__ __launch_bounds__(kTB) void ml_bwd_data(const float *D, int B, int out, int in, const float *W,
                                                   const float *Zp, float *G) {
  __shared__ float sd[kT][kK + 1];
  __shared__ float sw[kK][kT + 1];
  const int b0 = blockIdx.x * kT, i0 = blockIdx.y * kT;
  const int tx = threadIdx.x % kT, ty = threadIdx.x / kT;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int o0 = 0; o0 < out; o0 += kK) {
    const int kk = min(kK, out - o0);
    for (int e = threadIdx.x; e < kT * kK; e += kTB) {
      const int r = e / kK, c = e % kK;
      sd[r][c] = (c < kk && b0 + r < B) ? D[(long)(b0 + r) * out + o0 + c] : 0.f;
      const int rr = e / kT, cc = e % kT;
      sw[rr][cc] = (rr < kk && i0 + cc < in) ? W[(long)(o0 + rr) * in + i0 + cc] : 0.f;
    }
    __syncthreads();
    for (int c = 0; c < kk; ++c) {
      const float w = sw[c][tx];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = __builtin_fmaf(sd[ty + 8 * q][c], w, acc[q]);
    }
    __syncthreads();
  }
  const int i = i0 + tx;
  if (i >= in) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int b = b0 + ty + 8 * q;
    if (b < B) G[(long)b * in + i] = acc[q] * gelu_grad(Zp[(long)b * in + i]);
  }
}

// Adam (Kingma & Ba 2015) in the form of torch.optim.Adam without weight decay:
//   m = b1 m + (1 - b1) g,  v = b2 v + (1 - b2) g^2,
//   p -= (lr / (1 - b1^t)) m / (sqrt(v) / sqrt(1 - b2^t) + eps)
__global__ __launch_bounds__(kTB) void ml_adam(float *p, const float *g, float *m, float *v, long n, float b1,
                                               float b2, float step_size, float inv_sqrt_bc2, float eps) {
  for (long e = blockIdx.x * (long)kTB + threadIdx.x; e < n; e += (long)gridDim.x * kTB) {
    const float gr = g[e];
    const float mm = __builtin_fmaf(b1, m[e], (1.f - b1) * gr);
    const float vv = __builtin_fmaf(b2, v[e], (1.f - b2) * gr * gr);
    m[e] = mm;
    v[e] = vv;
    p[e] -= step_size * mm / (sqrtf(vv) * inv_sqrt_bc2 + eps);
  }
}

// ---------------------------------------------------------------------------
// Narrow networks (every width at most kNarrow, parameters within kNarrowParams): the whole
// network stays in LDS, a launch covers all layers.  Every sum runs over the same terms in the
// same order as in the kernels above, so the results are the same bits.

constexpr int kNarrow = 128;
constexpr int kMaxNet = 8;               // layers
constexpr int kNarrowParams = 35840;     // floats of padded weights and biases in LDS (140 KB)

struct Net {
  int L;
  int dims[kMaxNet + 1];
  long woff[kMaxNet], boff[kMaxNet];
  float *act[kMaxNet + 1];  // act[l], l >= 1: gelu(Z_{l-1}), batch x dims[l]
  float *dz[kMaxNet];       // dL/dZ_l, batch x dims[l + 1]
  float *y;                 // network output, batch x dims[L]
};

// LDS pitch of a row of W_l: 16-byte aligned, and a 16-byte read of 16 neighbouring rows falls into
// all 64 banks where in is a multiple of 64
__host__ __device__ inline int narrow_pitch(int in) { return ((in + 3) & ~3) + 4; }
__host__ __device__ inline int narrow_floats(const int *dims, int L) {
  int f = 0;
  for (int l = 0; l < L; ++l) f += dims[l + 1] * narrow_pitch(dims[l]);
  return f;
}

constexpr int kTrainRows = 2;  // rows per workgroup
constexpr int kRowsTB = 512;   // its threads: as many for the load of the weights as for the rows

// ring index of batch row b (off, b < mod)
__device__ __forceinline__ long ring(long off, long b, long mod) {
  const long r = off + b;
  return r < mod ? r : r - mod;
}

// a barrier for what the workgroup exchanges through LDS: unlike __syncthreads it does not wait for
// stores to memory to arrive (1-2 us after every layer)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// sum over k < n of a[k] w[k], k ascending; a and w 16-byte aligned in LDS.  The reads of 64 terms are
// issued before the first of them is added.
__device__ __forceinline__ float dot_row(const float *a, const float *w, int n) {
  float acc = 0.f;
  int k = 0;
  for (; k + 64 <= n; k += 64) {
    float4 x[16], y[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) x[q] = ((const float4 *)(a + k))[q], y[q] = ((const float4 *)(w + k))[q];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      acc = __builtin_fmaf(x[q].x, y[q].x, acc);
      acc = __builtin_fmaf(x[q].y, y[q].y, acc);
      acc = __builtin_fmaf(x[q].z, y[q].z, acc);
      acc = __builtin_fmaf(x[q].w, y[q].w, acc);
    }
  }
#pragma unroll 4
  for (; k < n; ++k) acc = __builtin_fmaf(a[k], w[k], acc);
  return acc;
}

// the same down a column of w (pitch step)
__device__ __forceinline__ float dot_column(const float *a, const float *w, int step, int n) {
  float acc = 0.f;
  int k = 0;
  for (; k + 32 <= n; k += 32) {
    float4 x[8];
    float y[32];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = ((const float4 *)(a + k))[q];
#pragma unroll
    for (int q = 0; q < 32; ++q) y[q] = w[(k + q) * step];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      acc = __builtin_fmaf(x[q].x, y[4 * q], acc);
      acc = __builtin_fmaf(x[q].y, y[4 * q + 1], acc);
      acc = __builtin_fmaf(x[q].z, y[4 * q + 2], acc);
      acc = __builtin_fmaf(x[q].w, y[4 * q + 3], acc);
    }
  }
#pragma unroll 4
  for (; k < n; ++k) acc = __builtin_fmaf(a[k], w[k * step], acc);
  return acc;
}

// One pass of two rows through the network and back, a thread per row and unit: activations, output
// and the gradients with respect to every Z.  A batch of 256 rows is 128 workgroups; at this size
// nothing but the chains of FMAs (128 per layer), the load of the weights (137 KB per workgroup from
// L2) and the launch is left.  Batch 256, 3 x 128 hidden: 14.4 us for what took eight launches
// (forward 4 x 10.7, backward 3 x 8.4, loss 3.9 us).  What counted on the way: no wait for stores at
// the barriers, 16-byte LDS reads, a thread per row and unit (a thread for both rows' unit, or loads
// straight into LDS a word at a time: 24 us).
__global__ __launch_bounds__(kRowsTB) void ml_rows(Net N, const float *__restrict__ p, const float *__restrict__ X,
                                                   const float *__restrict__ T, long off, long mod, int B) {
  extern __shared__ __align__(16) float sh[];
  __shared__ float zs[kMaxNet][kTrainRows][kNarrow];         // Z of every layer
  __shared__ __align__(16) float h[2][kTrainRows][kNarrow];  // the layer's input, then gradients
  const int tid = threadIdx.x, b0 = blockIdx.x * kTrainRows;
  const int L = N.L, d0 = N.dims[0], m = N.dims[L];
  const int r = tid / kNarrow, u = tid % kNarrow;  // this thread's row and unit
  const bool row = r < kTrainRows, there = row && b0 + r < B;
  float bias[kMaxNet], t = 0.f, x = 0.f;
#pragma unroll
  for (int l = 0; l < kMaxNet; ++l) bias[l] = row && l < L && u < N.dims[l + 1] ? p[N.boff[l] + u] : 0.f;
  if (there && u < d0) x = X[ring(off, b0 + r, mod) * d0 + u];
  if (there && u < m) t = T[ring(off, b0 + r, mod) * m + u];
  int at = 0;
  for (int l = 0; l < L; ++l) {
    const int in = N.dims[l], out = N.dims[l + 1], pitch = narrow_pitch(in);
    const float *w = p + N.woff[l];
    if (in % 4 == 0 && N.woff[l] % 4 == 0) {
      const int q = in / 4, n4 = out * q;
#pragma unroll 8
      for (int e = tid; e < n4; e += kRowsTB) {
        const int o = e / q;
        *(float4 *)(sh + at + o * pitch + 4 * (e - o * q)) = ((const float4 *)w)[e];
      }
    } else {
      for (int e = tid; e < out * in; e += kRowsTB) sh[at + (e / in) * pitch + e % in] = w[e];
    }
    at += out * pitch;
  }
  if (row && u < d0) h[0][r][u] = x;
  lds_barrier();
  at = 0;
  int cur = 0;
  for (int l = 0; l < L; ++l) {
    const int in = N.dims[l], out = N.dims[l + 1], pitch = narrow_pitch(in);
    if (row && u < out) {
      float bl = 0.f;
#pragma unroll
      for (int k = 0; k < kMaxNet; ++k) bl = k == l ? bias[k] : bl;
      const float z = dot_row(h[cur][r], sh + at + u * pitch, in) + bl;
      zs[l][r][u] = z;
      const float g = gelu(z);
      h[cur ^ 1][r][u] = g;
      if (there) {
        if (l + 1 < L)
          N.act[l + 1][(long)(b0 + r) * out + u] = g;
        else
          N.y[(long)(b0 + r) * out + u] = z;
      }
    }
    lds_barrier();
    at += out * pitch;
    cur ^= 1;
  }
  // dL/dY of the mean squared error, then back through the layers
  const float scale = 2.f / (float)(B * m);
  if (row && u < m) {
    const float g = scale * (zs[L - 1][r][u] - t);
    h[0][r][u] = g;
    if (there) N.dz[L - 1][(long)(b0 + r) * m + u] = g;
  }
  lds_barrier();
  cur = 0;
  for (int l = L - 1; l > 0; --l) {
    const int in = N.dims[l], out = N.dims[l + 1], pitch = narrow_pitch(in);
    at -= out * pitch;
    if (row && u < in) {
      const float g = dot_column(h[cur][r], sh + at + u, pitch, out) * gelu_grad(zs[l - 1][r][u]);
      h[cur ^ 1][r][u] = g;
      if (there) N.dz[l - 1][(long)(b0 + r) * in + u] = g;
    }
    lds_barrier();
    cur ^= 1;
  }
}

struct AdamArgs {
  float b1, b2, step_size, inv_sqrt_bc2, eps;
};

constexpr int kGT = 16;    // edge of a gradient tile: one output per thread
constexpr int kGB = 256;   // batch rows in LDS at a time

__host__ __device__ inline int narrow_tiles(int in, int out) {
  return ((out + kGT - 1) / kGT) * ((in + kGT) / kGT);  // in + 1 columns: the bias is the last
}

// dW_l = D_l^T A_l with the bias as an extra column, b ascending, for all layers in one launch (a
// 16 x 16 tile per workgroup: ~160 of them for 3 x 128 hidden, where a layer's 16 tiles of 32 x 32
// left most of the chip idle: 4 x 20.3 -> 6.6 us at batch 256), then the Adam update of the tile's
// parameters (g: the gradients alone, no update).  The last workgroup takes the loss.
__global__ __launch_bounds__(kTB) void ml_grad(Net N, float *__restrict__ p, float *__restrict__ m1,
                                               float *__restrict__ m2, float *__restrict__ g,
                                               const float *__restrict__ X, const float *__restrict__ T, long off,
                                               long mod, int B, AdamArgs A, float *__restrict__ loss) {
  __shared__ __align__(16) float sd[kGT][kGB + 4], sa[kGT][kGB + 4];
  const int tid = threadIdx.x, tx = tid % kGT, ty = tid / kGT;
  int t = blockIdx.x, l = 0;
  while (l < N.L && t >= narrow_tiles(N.dims[l], N.dims[l + 1])) t -= narrow_tiles(N.dims[l], N.dims[l + 1]), ++l;
  if (l == N.L) {  // the loss, in the order of ml_mse
    __shared__ double red[kTB];
    const int m = N.dims[N.L];
    double s = 0.0;
    for (int e = tid; e < B * m; e += kTB) {
      const float d = N.y[e] - T[ring(off, e / m, mod) * m + e % m];
      s += (double)d * (double)d;
    }
    red[tid] = s;
    __syncthreads();
    for (int k = kTB / 2; k > 0; k >>= 1) {
      if (tid < k) red[tid] += red[tid + k];
      __syncthreads();
    }
    if (tid == 0) *loss = (float)(red[0] / (double)(B * m));
    return;
  }
  const int in = N.dims[l], out = N.dims[l + 1], across = (in + kGT) / kGT;
  const int o0 = (t / across) * kGT, i0 = (t % across) * kGT;
  const float *D = N.dz[l], *Al = l == 0 ? X : N.act[l];
  const int o = o0 + ty, i = i0 + tx;
  const bool mine = o < out && i <= in;
  const long e = mine ? (i < in ? N.woff[l] + (long)o * in + i : N.boff[l] + o) : 0;
  float pe = 0.f, m1e = 0.f, m2e = 0.f;  // on their way while the sums run
  if (mine && !g) {
    pe = p[e];
    m1e = m1[e];
    m2e = m2[e];
  }
  float acc = 0.f;
  for (int bb = 0; bb < B; bb += kGB) {
    const int kk = min(kGB, B - bb);
    if (bb > 0) __syncthreads();
    const int c = tid % kGT;
    const bool dc = o0 + c < out, ac = i0 + c < in;
    float vd[kGB / kGT], va[kGB / kGT];
#pragma unroll
    for (int q = 0; q < kGB / kGT; ++q) {
      const int r = tid / kGT + q * kGT;
      vd[q] = 0.f;
      va[q] = i0 + c == in ? 1.f : 0.f;
      if (r < kk && dc) vd[q] = D[(long)(bb + r) * out + o0 + c];
      if (r < kk && ac) va[q] = Al[(l == 0 ? ring(off, bb + r, mod) : (long)(bb + r)) * in + i0 + c];
    }
#pragma unroll
    for (int q = 0; q < kGB / kGT; ++q) {
      sd[c][tid / kGT + q * kGT] = vd[q];
      sa[c][tid / kGT + q * kGT] = va[q];
    }
    __syncthreads();
    const float4 *d4 = (const float4 *)sd[ty], *a4 = (const float4 *)sa[tx];
    int r = 0;
#pragma unroll 4
    for (; r + 4 <= kk; r += 4) {
      const float4 d = d4[r / 4], a = a4[r / 4];
      acc = __builtin_fmaf(d.x, a.x, acc);
      acc = __builtin_fmaf(d.y, a.y, acc);
      acc = __builtin_fmaf(d.z, a.z, acc);
      acc = __builtin_fmaf(d.w, a.w, acc);
    }
    for (; r < kk; ++r) acc = __builtin_fmaf(sd[ty][r], sa[tx][r], acc);
  }
  if (!mine) return;
  if (g) {
    g[e] = acc;
    return;
  }
  const float mm = __builtin_fmaf(A.b1, m1e, (1.f - A.b1) * acc);
  const float vv = __builtin_fmaf(A.b2, m2e, (1.f - A.b2) * acc * acc);
  m1[e] = mm;
  m2[e] = vv;
  p[e] = pe - A.step_size * mm / (sqrtf(vv) * A.inv_sqrt_bc2 + A.eps);
}

// Forward pass of 16 Q rows per workgroup through all layers, on the matrix cores (v_mfma_f32_16x16x4_f32: an
// FP32 multiply-add per term, k ascending, so the sums are those of the kernels above bit for bit): the rows'
// activations in LDS, a wave's up to 32 outputs of all rows in its registers, the weights straight from
// the caches with the next sixteen inputs' on their way.  A layer's outputs replace its inputs once
// every wave has its sums.  100,000 rows of 3 x 128 hidden: 201 us (34 TFLOP/s; the products 60, the error
// functions of the GELUs 75, neither beside the other), 219 for FMAs of the vector units with the weights
// through LDS.  The call is bound by the rows' way up: 32,768 of them take 54 us.  64 rows a workgroup (Q = 4) read the
// weights least often; where they leave units idle, 16 (Q = 1): one row of 3 x 128 hidden 50 us a call instead of 62.
constexpr int kPP = kNarrow + 4;  // pitch of a row's activations: a product's 16 rows x 4 inputs in 64 banks

typedef float mlp4 __attribute__((ext_vector_type(4)));

template <int Q>  // 16 Q rows
__global__ __launch_bounds__(kTB, 4) void ml_predict(Net N, const float *__restrict__ p, const float *__restrict__ X,
                                                     int n, float *__restrict__ Y) {
  constexpr int kPR = 16 * Q;
  __shared__ __align__(16) float a[kPR * kPP];
  const int tid = threadIdx.x, b0 = blockIdx.x * kPR, R = min(kPR, n - b0);
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int d0 = N.dims[0], d4 = (d0 + 3) & ~3;
  for (int e = tid; e < kPR * d4; e += kTB) {
    const int r = e / d4, i = e - r * d4;
    a[r * kPP + i] = r < R && i < d0 ? X[(long)(b0 + r) * d0 + i] : 0.f;
  }
  __syncthreads();
  for (int l = 0; l < N.L; ++l) {
    const int in = N.dims[l], out = N.dims[l + 1], tiles = (out + 15) / 16;
    const float *wl = p + N.woff[l], *bias = p + N.boff[l];
    const bool last = l + 1 == N.L, two = wave + 4 < tiles;
    mlp4 acc[2][Q] = {};  // outputs 16 (wave + 4 t) + c of rows 16 q + 4 g ..
    float bo[2] = {};
    if (wave < tiles) {
      const int o0 = 16 * wave + c, o1 = o0 + 64;
      bo[0] = o0 < out ? bias[o0] : 0.f;
      bo[1] = o1 < out ? bias[o1] : 0.f;
      float w[2][4], v[2][4];
      const auto load = [&](int k0, float (&to)[2][4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = k0 + 4 * s + g;
          to[0][s] = k < in && o0 < out ? wl[o0 * in + k] : 0.f;
          to[1][s] = two && k < in && o1 < out ? wl[o1 * in + k] : 0.f;
        }
      };
      load(0, w);
      for (int k0 = 0; k0 < in; k0 += 16) {
        load(k0 + 16, v);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (k0 + 4 * s >= in) break;
          float x[Q];
#pragma unroll
          for (int q = 0; q < Q; ++q) x[q] = a[(16 * q + c) * kPP + k0 + 4 * s + g];
#pragma unroll
          for (int q = 0; q < Q; ++q) acc[0][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q], w[0][s], acc[0][q], 0, 0, 0);
          if (two)
#pragma unroll
            for (int q = 0; q < Q; ++q)
              acc[1][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q], w[1][s], acc[1][q], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int s = 0; s < 4; ++s) w[t][s] = v[t][s];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (wave + 4 * t >= tiles) continue;
      const int o = 16 * (wave + 4 * t) + c;
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * q + 4 * g + r;
          const float z = acc[t][q][r] + bo[t];
          if (!last)
            a[row * kPP + o] = o < out ? gelu(z) : 0.f;  // zeros past the last output: the next layer's padding (an
                                                         // infinite input times its zero weights is none)
          else if (row < R && o < out)
            Y[(long)(b0 + row) * out + o] = z;
        }
    }
    __syncthreads();
  }
}

}  // namespace mlp
}  // namespace spss
