"""The pieces and threads of spss_hostcopy.hpp on the host, over a stand-in for the HIP runtime that copies at once
and counts what it is asked for: which copies are staged, when the pinned buffer comes and goes, what is copied
where it ends, and that a runtime without pinned memory is as good."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spsslangevinintegration_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstdlib>
#include <cstring>
using hipError_t = int;
using hipEvent_t = int *;
using hipStream_t = void *;
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t { int type; };
constexpr int hipSuccess = 0, hipErrorInvalidValue = 1;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
inline long pinned = 0, pinned_calls = 0, direct = 0, pieces = 0;
inline bool no_pinned = false;
inline char *pin_begin = nullptr, *pin_end = nullptr;
inline const void *registered = nullptr;
inline int hipHostMalloc(void **p, size_t n, unsigned) {
  if (no_pinned) return 2;
  *p = malloc(n);
  pin_begin = (char *)*p;
  pin_end = pin_begin + n;
  pinned = (long)n;
  ++pinned_calls;
  return 0;
}
inline int hipHostFree(void *p) { free(p); pinned = 0; return 0; }
inline int hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new int(0); return 0; }
inline int hipEventDestroy(hipEvent_t e) { delete e; return 0; }
inline int hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline int hipEventSynchronize(hipEvent_t) { return 0; }
inline int hipStreamSynchronize(hipStream_t) { return 0; }
inline int hipGetLastError() { return 0; }
inline int hipGetDevice(int *d) { *d = 0; return 0; }
inline int hipSetDevice(int) { return 0; }
inline int hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  a->type = p == registered ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return p == registered ? 0 : hipErrorInvalidValue;
}
inline int hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  ++((char *)d >= pin_begin && (char *)d < pin_end ? pieces : direct);
  return 0;
}
"""

CHECK = r"""
#include <cstdint>
#include <cstdio>
#include <vector>
#include "spss_hostcopy.hpp"
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  using namespace spss;
  std::vector<char> src(70u << 20), dst(70u << 20);
  uint32_t r = 1;
  for (char &c : src) c = (char)((r = r * 1664525u + 1013904223u) >> 24);
  const auto copy = [&](HostCopy &h, size_t n) {
    std::fill(dst.begin(), dst.end(), 0);
    direct = pieces = 0;
    if (h.to_host(dst.data(), src.data(), n, nullptr) != hipSuccess) return false;
    return memcmp(dst.data(), src.data(), n) == 0 && (n == dst.size() || dst[n] == 0);
  };
  {
    HostCopy h;
    for (int k = 0; k < 3; ++k) {
      CHECK(copy(h, kCopyMin - 1));
      CHECK(direct == 1 && pinned_calls == 0);
    }
    // a handle's first large copy takes no pinned memory: many read theirs once
    CHECK(copy(h, kCopyMin) && direct == 1 && pieces == 0 && pinned_calls == 0);
    CHECK(copy(h, kCopyMin) && direct == 0 && pieces > 1 && pinned_calls == 1);
    CHECK(copy(h, kCopyMin + 4097) && direct == 0);
    const long calls = pinned_calls;
    for (size_t n : {kCopyBuffer - 1, kCopyBuffer, kCopyBuffer + 1, (size_t)(70u << 20)}) CHECK(copy(h, n) && direct == 0);
    CHECK(pinned_calls == calls + 1 && pinned <= (long)kCopyBuffer);
    registered = dst.data();
    CHECK(copy(h, kCopyBuffer) && direct == 1 && pieces == 0);
    registered = nullptr;
    CHECK(copy(h, 0));
  }
  CHECK(pinned == 0);  // given back with the handle
  no_pinned = true;
  {
    HostCopy h;
    for (int k = 0; k < 3; ++k) CHECK(copy(h, kCopyMin + 5) && direct == 1 && pieces == 0);
  }
  return 0;
}
"""


def test_staging(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "check.cpp").write_text(CHECK)
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-I" + str(tmp_path), "-I" + CSRC, str(tmp_path / "check.cpp"), "-o",
                    exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
