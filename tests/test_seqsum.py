"""The maps of spss_seqsum.hpp, compiled for the host and walked as the summary's kernels walk them, against
the plain loop of float additions: equal bit for bit.  The terms are those whose rounding can go wrong:
next to multiples of a quarter of a unit of the sum's last place, ties of both parities, sign changes,
partial sums across binades, subnormals."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spsslangevinintegration_amd", "csrc")

SOURCE = r"""
#include <algorithm>
#include <cmath>
#include <vector>
using std::max;
using std::min;
#include "spss_seqsum.hpp"
using namespace spss;

extern "C" float loop_sum(const float *c, long n, float s) {
  for (long i = 0; i < n; ++i) s = s + c[i];
  return s;
}

// the terms behind s, in runs of L and long runs of kSeqLevel of them; *by_map: terms taken through maps
extern "C" float map_sum(const float *c, long n, int L, float s, long *by_map) {
  const long nlong = (n + (long)L * kSeqLevel - 1) / ((long)L * kSeqLevel), nruns = nlong * kSeqLevel;
  const auto term = [&](long i) { return i < n ? c[i] : 0.f; };
  std::vector<SeqMap> runs(nruns * 64), longs(nlong * 64);
  for (int e = 0; e < 64; ++e) {
    const float scale = ldexpf(1.f, 23 - (e + kSeqExp0)), limit = fminf(4194304.f, (float)(1 << 30) / (float)L);
    for (long r = 0; r < nruns; ++r) {
      SeqMap m = seq_identity();
      for (int i = 0; i < L; ++i) seq_term(m, term(r * L + i) * scale, limit);
      runs[r * 64 + e] = m;
    }
    for (long q = 0; q < nlong; ++q) {
      SeqMap m = seq_identity();
      for (long r = q * kSeqLevel; r < (q + 1) * kSeqLevel; ++r)
        m = seq_compose(m, runs[r * 64 + e], (1 << 30) / (L * kSeqLevel));
      longs[q * 64 + e] = m;
    }
  }
  const auto pass = [&](const std::vector<SeqMap> &maps, long r) {
    const int k = seq_lookup(s);
    if (k < 0) return false;
    const SeqMap &m = maps[r * 64 + k];
    if (s == 0.f) return seq_zeros(m.reach);
    const int S = seq_units(s), p = S & 1;
    if (!seq_stays(S, m.lo[p], m.hi[p], m.reach)) return false;
    s = seq_value(S + m.inc[p], s);
    return true;
  };
  *by_map = 0;
  for (long q = 0; q < nlong; ++q) {
    if (pass(longs, q)) {
      *by_map += (long)L * kSeqLevel;
      continue;
    }
    for (long r = q * kSeqLevel; r < (q + 1) * kSeqLevel; ++r) {
      if (pass(runs, r))
        *by_map += L;
      else
        for (int i = 0; i < L; ++i) s = s + term(r * L + i);
    }
  }
  return s;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("seqsum")
    (d / "check.cpp").write_text(SOURCE)
    out = str(d / "check.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(rocm, "include"), "-I" + CSRC, str(d / "check.cpp"), "-o", out], check=True)
    h = ctypes.CDLL(out)
    h.loop_sum.restype = h.map_sum.restype = ctypes.c_float
    return h


def sums(lib, c, L=256, s=0.0):
    c = np.ascontiguousarray(c, dtype=np.float32)
    p, n = c.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(c.size)
    by_map = ctypes.c_long()
    a = lib.loop_sum(p, n, ctypes.c_float(s))
    b = lib.map_sum(p, n, ctypes.c_int(L), ctypes.c_float(s), ctypes.byref(by_map))
    return np.float32(a), np.float32(b), by_map.value


# in units of the sum's last place: multiples of a quarter and their neighbours
NEAR = sorted({float(np.nextafter(np.float32(v), np.float32(w))) for q in range(-9, 10) for v in [0.25 * q]
               for w in (v, -10.0, 10.0)} | {2.0 ** -30, -2.0 ** -30})


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("start", [8388608 + 12345, 8388608 + 12346])
@pytest.mark.parametrize("exponent", [0, -20, 5])
def test_one_term_of_every_kind(lib, start, sign, exponent):
    for v in NEAR:
        a, b, by_map = sums(lib, [v * 2.0 ** exponent], 16, sign * start * 2.0 ** exponent)
        assert a == b and by_map > 0, (v, a, b)


@pytest.mark.parametrize("exponent", [0, -20, 5])
def test_runs_of_near_ties(lib, exponent):
    rng = np.random.default_rng(5)
    for L in (16, 256):
        for s0 in (8388608 + 5000, -(8388608 + 5001), 16777216 - 4000):
            c = rng.choice(NEAR, 20000) * 2.0 ** exponent
            a, b, by_map = sums(lib, c, L, s0 * 2.0 ** exponent)
            assert a == b and by_map > 0, (L, s0, a, b)


def test_a_sum_that_near_ties_drag(lib):
    # 140,000 phasors near 0.95, then pairs whose second term is just short of half a unit
    c = np.concatenate([np.full(140000, 0.95), np.tile([0.95, np.cos(1.5786089058042636)], 2000)])
    a, b, by_map = sums(lib, c)
    assert a == b and by_map > 70000, (a, b, by_map)


@pytest.mark.parametrize("seed", range(6))
def test_sums_across_binades(lib, seed):
    rng = np.random.default_rng(seed)
    n = int(rng.integers(1, 60000))
    c = np.cos(rng.uniform(0, 2 * np.pi, n) if seed % 2 else rng.normal(0.0, 0.3 * seed, n)).astype(np.float32)
    c[rng.random(n) < 0.01] *= np.float32(2.0 ** -140)  # subnormals among them
    a, b, _ = sums(lib, c)
    assert a == b


@pytest.mark.parametrize("term", [1e-18, -1e-18, 2.0 ** -57, 2.0 ** -58, 1e-30, 1e-42])
def test_tiny_terms_at_a_zero_sum(lib, term):
    for n in (1, 256, 1000, 5000):
        for c in (np.full(n, term), np.concatenate([np.zeros(4096), np.full(n, term)]),
                  np.tile([0.0, term, -term], n)):
            a, b, _ = sums(lib, c)
            assert a == b, (n, a, b)


def test_zeros_pass_by_map(lib):
    a, b, by_map = sums(lib, np.concatenate([np.zeros(4096), -np.zeros(4096), [1.0]]))
    assert a == b == 1.0 and by_map >= 8192
