// spss_seqsum.hpp -- the float sum s = ((c_0 + c_1) + c_2) + ... with the rounding of every addition,
// as a loop over the terms gives it, computed in parallel.
//
// While |s| stays in one binade [2^e, 2^(e+1)), s is a whole multiple S of u = 2^(e-23) and adding c
// adds a whole number to S: c / u rounded to the nearest, ties to the even sum, so that the number
// depends on S through its parity alone.  A run of terms is then a map from the parity of S to the
// increment of S, maps compose, and with the least and the largest value that S takes on the way one
// can see whether it left the binade.  Every run of terms is therefore summed ahead for every
// exponent e and both parities, by all of the chip; a walk over the runs picks the map of its own
// exponent and parity, and adds the terms one by one only where a run crosses into another binade.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace spss {

constexpr int kSeqExp0 = -33;  // exponents covered: kSeqExp0 + [0, 64)
constexpr int kSeqLevel = 16;  // runs composed into a long run

struct SeqMap {
  int inc[2];       // increment of S by its parity at the start
  int lo[2], hi[2]; // least and largest increment on the way (the start's 0 among them)
  int reach;        // a bound of |c / u| + 1 of every term, 1 for zeros alone; kSeqNever: no statement
  int pad;
};
constexpr int kSeqNever = 0x7fffffff;

__host__ __device__ __forceinline__ SeqMap seq_identity() { return SeqMap{{0, 0}, {0, 0}, {0, 0}, 1, 0}; }

// one more term: v = c / u (exact); terms beyond `limit` could overflow the run's sums
__host__ __device__ __forceinline__ void seq_term(SeqMap &m, float v, float limit) {
  const float a = v < 0.f ? -v : v;
  if (!(a <= limit)) {  // NaN too
    m.reach = kSeqNever;
    return;
  }
  if (m.reach == kSeqNever) return;
  // d is exact (of v's last place and at most half), which v less its floor is not: -(0.5 - 2^-25) leaves 0.5 there
  const float w = rintf(v), d = v - w;
  const int k = (int)w, other = d == 0.5f ? 1 : (d == -0.5f ? -1 : 0);  // a tie's other whole number, from k
  const int need = a > 0.f ? (int)a + 2 : 1;
  m.reach = need > m.reach ? need : m.reach;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    m.inc[p] += k + (((p + m.inc[p] + k) & 1) ? other : 0);
    m.lo[p] = m.inc[p] < m.lo[p] ? m.inc[p] : m.lo[p];
    m.hi[p] = m.inc[p] > m.hi[p] ? m.inc[p] : m.hi[p];
  }
}

// first a, then b
__host__ __device__ __forceinline__ SeqMap seq_compose(const SeqMap &a, const SeqMap &b, int limit) {
  SeqMap m;
  m.pad = 0;
  m.reach = a.reach > b.reach ? a.reach : b.reach;
  if (m.reach > limit) m.reach = kSeqNever;
  if (m.reach == kSeqNever) {
    m.inc[0] = m.inc[1] = m.lo[0] = m.lo[1] = m.hi[0] = m.hi[1] = 0;
    return m;
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int t = a.inc[p], q = (p + t) & 1;
    m.inc[p] = t + (q ? b.inc[1] : b.inc[0]);
    const int l = t + (q ? b.lo[1] : b.lo[0]), h = t + (q ? b.hi[1] : b.hi[0]);
    m.lo[p] = l < a.lo[p] ? l : a.lo[p];
    m.hi[p] = h > a.hi[p] ? h : a.hi[p];
  }
  return m;
}

// exponent slot of s (0..63), or -1
__host__ __device__ __forceinline__ int seq_slot(float s) {
  union { float f; uint32_t u; } b;
  b.f = s;
  const int e = (int)((b.u >> 23) & 0xff) - 127 - kSeqExp0;
  return e >= 0 && e < 64 ? e : -1;
}

// the slot to look s up in (zero: the smallest), or -1
__host__ __device__ __forceinline__ int seq_lookup(float s) { return s == 0.f ? 0 : seq_slot(s); }

// whether a run whose map has this reach leaves a zero sum at zero: its terms are all zeros (increments of
// zero do not tell: every exponent's unit has terms too small for it)
__host__ __device__ __forceinline__ bool seq_zeros(int reach) { return reach == 1; }

// s as a multiple of its ulp
__host__ __device__ __forceinline__ int seq_units(float s) {
  union { float f; uint32_t u; } b;
  b.f = s;
  const int m = (int)((b.u & 0x7fffff) | 0x800000);
  return (b.u >> 31) ? -m : m;
}

// whether a run with these bounds keeps S inside its binade.  An exact sum S + c / u is within 1/2 of
// the whole number it was rounded to, so whole numbers strictly inside the binade prove that every
// sum lay in it and was rounded to multiples of u.
__host__ __device__ __forceinline__ bool seq_stays(int S, int lo, int hi, int reach) {
  if (reach == kSeqNever) return false;
  const int a = S > 0 ? S + lo : -(S + hi), b = S > 0 ? S + hi : -(S + lo);
  return a > 1 << 23 && b < 1 << 24;
}

// the float of S units at the exponent of `like` (|S| in [2^23, 2^24))
__host__ __device__ __forceinline__ float seq_value(int S, float like) {
  union { float f; uint32_t u; } b;
  b.f = like;
  const uint32_t m = (uint32_t)(S < 0 ? -S : S) & 0x7fffff;
  b.u = (S < 0 ? 0x80000000u : 0u) | (b.u & 0x7f800000u) | m;
  return b.f;
}

}  // namespace spss
