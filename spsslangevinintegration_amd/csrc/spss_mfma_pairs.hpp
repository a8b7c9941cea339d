// spss_mfma_pairs.hpp -- neighbour phasor sums of FP32C precision on the matrix cores: one wave takes
// sixteen particles of a row of cells at a time against the union of their stencils, staged in LDS.
//
// With positions from the tile's centre, |x_i - x_j|^2 - r^2 = -2 x_i . x_j + |x_j|^2 + (|x_i|^2 - r^2) is a
// short product: v_mfma_f32_16x16x16_f16 gives it for sixteen candidates by sixteen particles, with the
// last term as the accumulator's start.  A coordinate is the sum of two halves of eleven bits, whose four
// products take four of the sixteen places, |x_j|^2 two.  The sign is the range test (v_perm spreads a
// sign over a byte: -1 within, 0 beyond); the few pairs that rounding could decide are decided one
// by one.
//
// The phasors are staged as 38-bit fixed-point numbers, their five signed bytes in planes, cosines and sines
// each on the scale of the tile's largest; the omega-weighted ones as 46-bit numbers on the scale of the
// tile's largest |omega| beside.  The sums over the neighbours are then products of 0/-1 bytes and digit bytes,
// sixteen particles by sixteen planes by 64 candidates in a v_mfma_i32_16x16x64_i8: whole numbers, exact in
// any order and grouping.  An FP32 phasor is kept whole from 2^-13 of the scale on, and beside one of 2^-9
// in range what smaller ones lose (2^-38) is below that one's own rounding to FP32 (2^-34): these sums
// are closer to the exact ones than FP32 partial sums are; so for the weighted ones beside one of 2^-18 (the
// bulk of a Lorentzian clipped at 200 of its widths is at 2^-8).  Planes of marks tell, by the same
// product, whether there is one in range; where there is none (beside a particle far off its neighbours in the
// same tile) the caller takes the sums itself.
//
// Bound: the vector units, 42 operations per 1,024 pairs where a walk over candidates takes 180, and
// what comes before and after.  Cycles of a SIMD per 1,024 pairs, measured alone: this product 71 (by
// v_mfma_f32_16x16x4_f32 139, and nothing else issues meanwhile), signs to bytes and the band's minimum
// 85 (by v_cvt_pk_u8_f32, which takes eight cycles, 180), the digit products 34; the loop 244.
#pragma once

#include <hip/hip_runtime.h>

#include "spss_tiles.hpp"

namespace spss {

typedef int mint4 __attribute__((ext_vector_type(4)));
typedef float mfloat4 __attribute__((ext_vector_type(4)));
typedef _Float16 mhalf2 __attribute__((ext_vector_type(2)));
typedef _Float16 mhalf4 __attribute__((ext_vector_type(4)));

constexpr int kMStage = 1040;         // staged entries: particles, and padding to whole units of 16 per row (what
                                      // leaves four workgroups to a CU; three: 16 of 115 us at 1M particles)
constexpr int kMPlane = kMStage + 16; // and one unit out of every range
constexpr int kMDigits = kMPlane / 4 + 4;  // words of a digit plane: sixteen planes, 12 banks apart, in 64 banks
constexpr int kMUnits = kMStage / 16 + 16; // units of one group's candidates, and sixteen out of every range
constexpr float kMUnit = 1024.f;      // positions: cells to |x| < 25 in halves, their second halves not denormal
constexpr float kMSquare = 0x1p-14f;  // squares in halves
constexpr float kMFar = 3e4f;         // "|x|^2" of padding at x = 0, in squares: beyond every range

// W: words of digits per entry: the first four digits of cos and of sin, the last one of both and the two marks;
// the first digits of omega cos and omega sin, their last two in one word
constexpr int kMPlain = 3, kMOmega = 6;
template <int W>
struct MStage {
  // entry 4c + j: x1 x2 y1 y2 at pos[j >> 1][2c + (j & 1)]; the squares' halves of entries 4c, 4c + 2, 4c + 1,
  // 4c + 3 at sq[4c ..]
  alignas(16) uint2 pos[2][kMPlane / 2];
  unsigned sq[kMPlane];
  unsigned limb[4 * W][kMDigits];
  unsigned ones[4];
  unsigned char units[4][4][kMUnits];      // per wave and group: its units
};

__device__ __forceinline__ unsigned m_pack(_Float16 lo, _Float16 hi) {
  return __builtin_bit_cast(unsigned, mhalf2{lo, hi});
}
__device__ __forceinline__ unsigned m_halves(float x) {  // x as a sum of two halves
  const _Float16 a = (_Float16)x, b = (_Float16)(x - (float)a);
  return m_pack(a, b);
}
__device__ __forceinline__ float m_value(unsigned w) {
  const mhalf2 h = __builtin_bit_cast(mhalf2, w);
  return (float)h[0] + (float)h[1];
}
__device__ __forceinline__ int m_square(int e) { return (e & ~3) | ((e & 1) << 1) | ((e >> 1) & 1); }

template <int W>
__device__ __forceinline__ void m_place(MStage<W> &L, int e, uint2 xy, float square) {
  L.pos[(e >> 1) & 1][(e >> 2) * 2 + (e & 1)] = xy;
  L.sq[m_square(e)] = m_halves(square);
}
template <int W>
__device__ __forceinline__ uint2 m_pos(const MStage<W> &L, int e) {
  return L.pos[(e >> 1) & 1][(e >> 2) * 2 + (e & 1)];
}

template <int W>
__device__ __forceinline__ void m_init(MStage<W> &L) {
  if (threadIdx.x < 16) m_place(L, kMStage + threadIdx.x, make_uint2(0u, 0u), kMFar);
  if (threadIdx.x < 4) L.ones[threadIdx.x] = 0x01010101u;
}

// lanes 4q..4q+3 hold a word of digits each: lane 4q + b returns digit b of the four (exchanges with
// lane ^ 1, then with lane ^ 2)
__device__ __forceinline__ unsigned quad_transpose(unsigned w, unsigned s1, unsigned s2) {
  const unsigned t = __builtin_amdgcn_perm((unsigned)__builtin_amdgcn_mov_dpp((int)w, 0xb1, 0xf, 0xf, true), w, s1);
  return __builtin_amdgcn_perm((unsigned)__builtin_amdgcn_mov_dpp((int)t, 0x4e, 0xf, 0xf, true), t, s2);
}

// a component's scale: its values in the tile times 2^up are below 2^30
struct MScale {
  int up;
  float mark;  // values from there on are marked
};
// most: the tile's largest value (< 2^100)
__device__ __forceinline__ MScale m_scale(float most, float mark) {
  const bool none = !(most > 0x1p-90f);  // such values may as well be zeros: they lose 2^-127 at most
  return {none ? 119 : 29 - ilogbf(most), none ? 0.f : mark};
}
constexpr float kMMark = 0x1p21f, kMMarkOmega = 0x1p12f;

// v = hi + 2^-LOW lo for |v| <= 2^30
template <int LOW>
__device__ __forceinline__ int m_fixed(float v, int &lo) {
  const float h = __builtin_rintf(v);
  lo = (int)__builtin_rintf((v - h) * (float)(1 << LOW));
  return (int)h;
}
// whether both components of an entry are marked
__device__ __forceinline__ unsigned m_marked(float x, MScale kx, float y, MScale ky) {
  return __builtin_fabsf(x) >= kx.mark && __builtin_fabsf(y) >= ky.mark ? 1u : 0u;
}
// signed digits of a 32-bit number, and of a smaller one's two
__device__ __forceinline__ unsigned m_digits(int q) { return ((unsigned)q + 0x80808080u) ^ 0x80808080u; }
__device__ __forceinline__ unsigned m_digits16(int q) { return (((unsigned)q + 0x8080u) ^ 0x8080u) & 0xffffu; }

// entry e of the stage (not valid: padding, its values zero); the lanes of a quad have consecutive entries
// of one unit and come here together; x, y in cells / kMUnit; c, s, om: scaled
template <int W>
__device__ __forceinline__ void m_write(MStage<W> &L, int e, bool valid, float x, float y, float c, float s,
                                        float om, MScale kc, MScale ks, MScale ko) {
  const int lane = threadIdx.x & 63;
  const unsigned s1 = lane & 1 ? 0x03070105u : 0x06020400u, s2 = lane & 2 ? 0x03020706u : 0x05040100u;
  const uint2 xy = make_uint2(m_halves(x), m_halves(y));
  const float xr = m_value(xy.x), yr = m_value(xy.y);
  m_place(L, e, xy, valid ? kMSquare * __builtin_fmaf(xr, xr, yr * yr) : kMFar);
  unsigned *const d = L.limb[lane & 3] + (e >> 2);
  constexpr int kNext = 4 * kMDigits;  // the same digit of the next word
  int lc, ls;
  const int hc = m_fixed<7>(c, lc), hs = m_fixed<7>(s, ls);
  d[0] = quad_transpose(m_digits(hc), s1, s2);
  d[kNext] = quad_transpose(m_digits(hs), s1, s2);
  unsigned low = (lc & 0xff) | (ls & 0xff) << 8 | m_marked(c, kc, s, ks) << 16;
  if (W == kMOmega) {
    const float vx = om * (c * 0x1p-30f), vy = om * (s * 0x1p-30f);
    low |= m_marked(vx, ko, vy, ko) << 24;
    const int hx = m_fixed<15>(vx, lc), hy = m_fixed<15>(vy, ls);
    d[3 * kNext] = quad_transpose(m_digits(hx), s1, s2);
    d[4 * kNext] = quad_transpose(m_digits(hy), s1, s2);
    d[5 * kNext] = quad_transpose(m_digits16(lc) | m_digits16(ls) << 16, s1, s2);
  }
  d[2 * kNext] = quad_transpose(low, s1, s2);
}

struct MSums {
  double sx = 0.0, sy = 0.0, tx = 0.0, ty = 0.0;  // without the particle itself
  int n = 0;                                      // kMOpen: nothing marked in range
};
constexpr int kMOpen = -1;

// The sums of the wave's `count` particles (one per lane, entries first .. first + count - 1 of the stage
// in cell order); r2: the squared radius in staged units, band: what rounding may move a squared
// distance by; range(lane, r, a, b): the entries [a, b) of row r of the stencils of particles [lane,
// lane + 16); in(lane, e): the exact range test of particle `lane` and entry e.  c, s, om: the lane's own
// phasor and omega, scaled, which its sums are rid of.  (Its own mark counts too: with the other component
// its value weighs by that much in what is made of the sums.)
template <int W, class RANGE, class IN>
__device__ __forceinline__ MSums m_sums(MStage<W> &L, int first, int count, int nrows, float r2, float band, float c,
                                        float s, float om, MScale kc, MScale ks, MScale ko, RANGE range, IN in) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
  MSums out;
  int sx[2] = {0, 0}, sy[2] = {0, 0}, kx = 0, ky = 0, tx[2] = {0, 0}, ty[2] = {0, 0}, lx = 0, ly = 0;
  int mp = 0, mo = 0;  // marked phasors, weighted ones in range
  // the units of each group's candidates, four groups at once, one row per lane
  int total = 0;
  {
    int a = 0, b = 0;
    if (i < nrows && 16 * g < count) range(16 * g, i, a, b);
    const int u0 = a >> 4, m = b > a ? ((b + 15) >> 4) - u0 : 0;
    total = m;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const int t = __shfl_up(total, o, 16);
      if (i >= o) total += t;
    }
    unsigned char *list = L.units[wave][g];
    for (int t = 0; t < m; ++t) list[total - m + t] = (unsigned char)(u0 + t);
    total = __shfl(total, 15, 16);
    list[total + i] = (unsigned char)(kMStage / 16);  // the last pass's rest, and what is read ahead
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
  // the lane's part of the product: halves of its unit's entries 4 (i & 3) .. + 3
  const char *fb = (g < 2 ? reinterpret_cast<const char *>(L.pos[0]) : reinterpret_cast<const char *>(L.sq)) + 16 * (i & 3);
  constexpr int kSecond = sizeof(L.pos[0]);
  const int second = g < 2 ? kSecond : 0;
  // the planes: the phasors' ten digits, the marks, ones; the weighted ones' twelve digits
  const char *l1 = i < 12 ? reinterpret_cast<const char *>(L.limb[i]) : reinterpret_cast<const char *>(L.ones);
  const int m1 = i < 12 ? -1 : 0;
  const char *l2 = reinterpret_cast<const char *>(L.limb[W == kMOmega && i < 12 ? 12 + i : 0]);
  for (int gr = 0; 16 * gr < count; ++gr) {
    const bool real = 16 * gr + i < count;
    const uint2 own = m_pos(L, real ? first + 16 * gr + i : kMStage);
    const float xi = m_value(own.x), yi = m_value(own.y);
    // particles that are not: beyond every range
    const float ai = real ? __builtin_fmaf(xi, xi, yi * yi) - r2 : 2.f * kMFar / kMSquare;
    const mfloat4 a4 = {ai, ai, ai, ai};
    const unsigned pick = g == 0 ? 0x05040504u : 0x07060706u;  // a coordinate's first or second half, twice
    const mhalf2 two = {(_Float16)-2.f, (_Float16)-2.f}, sq = {(_Float16)(1.f / kMSquare), (_Float16)(1.f / kMSquare)};
    const mhalf2 none = {(_Float16)0.f, (_Float16)0.f};
    const mhalf2 hx = __builtin_bit_cast(mhalf2, __builtin_amdgcn_perm(own.x, own.x, pick)) * two;
    const mhalf2 hy = __builtin_bit_cast(mhalf2, __builtin_amdgcn_perm(own.y, own.y, pick)) * two;
    // the product's other side for entries 0, 1 and 2, 3 of four (of the squares, see MStage)
    const mhalf2 b0 = g < 2 ? hx : (g == 2 ? sq : none), b1 = g < 2 ? hy : none;
    const mhalf2 b2 = g < 2 ? hx : none, b3 = g < 2 ? hy : (g == 2 ? sq : none);
    const mhalf4 v0 = {b0[0], b0[1], b1[0], b1[1]}, v1 = {b2[0], b2[1], b3[0], b3[1]};
    mint4 s1 = {0, 0, 0, 0}, s2 = {0, 0, 0, 0};
    const unsigned char *uf = L.units[wave][gr] + (i >> 2), *ul = L.units[wave][gr] + g;
    const int n = __builtin_amdgcn_readlane(total, 16 * gr);
    struct Entries {
      mint4 a, b;
    };
    const auto features = [&](int e) {
      const char *f = fb + 4 * e;
      return Entries{*reinterpret_cast<const mint4 *>(f), *reinterpret_cast<const mint4 *>(f + second)};
    };
    struct Products {
      mfloat4 t[4];
    };
    const auto half4 = [](int lo, int hi) { return __builtin_bit_cast(mhalf4, make_uint2((unsigned)lo, (unsigned)hi)); };
    const auto products = [&](const Entries &f) {
      Products r;
      r.t[0] = __builtin_amdgcn_mfma_f32_16x16x16f16(half4(f.a[0], f.a[1]), v0, a4, 0, 0, 0);
      r.t[1] = __builtin_amdgcn_mfma_f32_16x16x16f16(half4(f.a[2], f.a[3]), v0, a4, 0, 0, 0);
      r.t[2] = __builtin_amdgcn_mfma_f32_16x16x16f16(half4(f.b[0], f.b[1]), v1, a4, 0, 0, 0);
      r.t[3] = __builtin_amdgcn_mfma_f32_16x16x16f16(half4(f.b[2], f.b[3]), v1, a4, 0, 0, 0);
      return r;  // t[q][r]: entry 4r + q of the lane's unit
    };
    const auto bits = [](float t) { return __builtin_bit_cast(unsigned, t); };
    int el = 16 * ul[0], ef = 16 * uf[0];
    for (int u = 0; u < n; u += 4) {
      const Products c = products(features(ef));
      const mint4 d1 = *reinterpret_cast<const mint4 *>(l1 + (el & m1));
      const int el0 = el;
      el = 16 * ul[u + 4];
      ef = 16 * uf[u + 4];
      mint4 w;
      float least = __builtin_fabsf(c.t[0][0]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // selector 9, 11: the second, the first operand's sign over a byte; 12: 0
        w[r] = (int)(__builtin_amdgcn_perm(bits(c.t[1][r]), bits(c.t[0][r]), 0x0c0c0b09u) |
                     __builtin_amdgcn_perm(bits(c.t[3][r]), bits(c.t[2][r]), 0x0b090c0cu));
        if (r) least = __builtin_fminf(least, __builtin_fabsf(c.t[0][r]));
        least = __builtin_fminf(least, __builtin_fabsf(c.t[1][r]));
        least = __builtin_fminf(__builtin_fminf(least, __builtin_fabsf(c.t[2][r])), __builtin_fabsf(c.t[3][r]));
      }
      if (least <= band) {  // rare
        unsigned open = 0;  // entries to decide
#pragma unroll
        for (int e = 0; e < 16; ++e) open |= __builtin_fabsf(c.t[e & 3][e >> 2]) <= band ? 1u << e : 0u;
        for (; open; open &= open - 1) {
          const int e = __builtin_ctz(open);
          const unsigned mask = 0xffu << (8 * (e & 3)), byte = in(16 * gr + i, el0 + e) ? mask : 0u;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (e >> 2 == r) w[r] = (int)(((unsigned)w[r] & ~mask) | byte);
        }
      }
      s1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d1, w, s1, 0, 0, 0);
      if (W == kMOmega) s2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const mint4 *>(l2 + el0), w, s2, 0, 0, 0);
    }
    // lanes i and 16 + i hold the first digits of the cosines' and the sines' sums, lane 32 + i the last ones and
    // the marks, lane 48 + i the count; lane 16 gr + i takes them, in pairs
    const int p0 = s1[0] + (s1[1] << 8), p1 = s1[2] + (s1[3] << 8);
    const int x0 = __shfl(p0, i), x1 = __shfl(p1, i), y0 = __shfl(p0, 16 + i), y1 = __shfl(p1, 16 + i);
    const int z0 = __shfl(s1[0], 32 + i), z1 = __shfl(s1[1], 32 + i), cn = __shfl(s1[0], 48 + i);
    const int c0 = __shfl(s1[2], 32 + i), c1 = W == kMOmega ? __shfl(s1[3], 32 + i) : 0;
    if (g == gr) {
      sx[0] = x0, sx[1] = x1, sy[0] = y0, sy[1] = y1, kx = z0, ky = z1;
      out.n = -cn;
      mp = c0;
      mo = c1;
    }
    if (W == kMOmega) {
      const int q0 = s2[0] + (s2[1] << 8), q1 = s2[2] + (s2[3] << 8);
      const int u0 = __shfl(q0, i), u1 = __shfl(q1, i), v0 = __shfl(q0, 16 + i), v1 = __shfl(q1, 16 + i);
      const int a = __shfl(q0, 32 + i), b = __shfl(q1, 32 + i);
      if (g == gr) {
        tx[0] = u0, tx[1] = u1, ty[0] = v0, ty[1] = v1;
        lx = a;
        ly = b;
      }
    }
  }
  const auto whole = [](const int *q) { return fma((double)q[1], 65536.0, (double)q[0]); };
  int lc, ls;
  const int hc = m_fixed<7>(c, lc), hs = m_fixed<7>(s, ls);
  out.sx = ldexp(-(whole(sx) + (double)hc + 0x1p-7 * (double)(kx + lc)), -kc.up);
  out.sy = ldexp(-(whole(sy) + (double)hs + 0x1p-7 * (double)(ky + ls)), -ks.up);
  if (W == kMOmega) {
    const int hx = m_fixed<15>(om * (c * 0x1p-30f), lc), hy = m_fixed<15>(om * (s * 0x1p-30f), ls);
    out.tx = ldexp(-(whole(tx) + (double)hx + 0x1p-15 * (double)(lx + lc)), 30 - ko.up - kc.up);
    out.ty = ldexp(-(whole(ty) + (double)hy + 0x1p-15 * (double)(ly + ls)), 30 - ko.up - ks.up);
  }
  if (out.n > 1 && (mp == 0 || (W == kMOmega && mo == 0))) {
    out.n = kMOpen;
    return out;
  }
  --out.n;
  return out;
}

}  // namespace spss
