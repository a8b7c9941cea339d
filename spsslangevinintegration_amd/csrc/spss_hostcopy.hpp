// spss_hostcopy.hpp -- copies from device memory to a caller's ordinary (pageable) memory.
//
// The runtime stages such a copy through its own pinned memory with one thread: 20 MB take 1.16 ms, of
// which the transfer is 0.4, and 4.8 ms into memory that has no pages yet.  Here the transfer goes to a
// pinned buffer of the handle in pieces, and up to kCopyThreads threads move them on as they arrive: 0.73
// and 1.24 ms (two threads 0.68 and 3.0 at 21 MB).  Into memory that has its pages both take as long at 8 MB (0.47;
// 4 MB 0.24 and 0.37, 12 MB 0.70 and 0.55, 16 MB 0.93 and 0.62): the runtime copies less than that.  It
// also makes a handle's first copy, for which the pinned pages (1 ms) would come on top and which for
// many handles is the only one; and it copies to memory that is pinned already, and to the device, where this is
// no faster.
// Every call returns with the copy done, as before.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <system_error>
#include <thread>

namespace spss {

constexpr size_t kCopyMin = 8u << 20, kCopyBuffer = 32u << 20;  // bytes
constexpr int kCopyPieces = 16, kCopyThreads = 8;

// the pinned buffer (at most kCopyBuffer bytes) and the pieces' events, kept by a handle and given back
// with it
class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;
  ~HostCopy() { drop(); }

  hipError_t to_host(void *dst, const void *src, size_t bytes, hipStream_t st) {
    if (!staged(dst, bytes)) return direct(dst, src, bytes, hipMemcpyDeviceToHost, st);
    char *d = static_cast<char *>(dst);
    const char *s = static_cast<const char *>(src);
    for (size_t at = 0; at < bytes; at += cap_) {
      const size_t m = std::min(cap_, bytes - at), piece = piece_of(m);
      hipError_t e = hipSuccess;
      int n = 0;
      for (size_t o = 0; o < m && e == hipSuccess; o += piece, ++n) {
        e = hipMemcpyAsync(pin_ + o, s + at + o, std::min(piece, m - o), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev_[n], st);
      }
      if (e == hipSuccess)
        e = each(n, [&](int k) {
          const hipError_t r = hipEventSynchronize(ev_[k]);
          if (r == hipSuccess) std::memcpy(d + at + k * piece, pin_ + k * piece, std::min(piece, m - k * piece));
          return r;
        });
      const hipError_t drained = hipStreamSynchronize(st);  // on errors too: the buffer is free again
      if (e == hipSuccess) e = drained;
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }

 private:
  char *pin_ = nullptr;
  size_t cap_ = 0;
  bool again_ = false;  // there has been a copy of kCopyMin bytes or more
  hipEvent_t ev_[kCopyPieces] = {};

  static size_t piece_of(size_t m) { return ((m + kCopyPieces - 1) / kCopyPieces + 4095) / 4096 * 4096; }

  static hipError_t direct(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t st) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  }

  void drop() {
    for (hipEvent_t &e : ev_) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
    cap_ = 0;
  }

  // the buffer for copies of that much; false if there is none (they go to the runtime then)
  bool reserve(size_t bytes) {
    const size_t want = std::min(kCopyBuffer, piece_of(bytes) * kCopyPieces);
    if (cap_ >= want) return true;
    drop();
    bool ok = hipHostMalloc(reinterpret_cast<void **>(&pin_), want, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t &e : ev_) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
      (void)hipGetLastError();
      drop();
      return false;
    }
    cap_ = want;
    return true;
  }

  // whether a copy of that much to `host` is staged here; allocates the buffer
  bool staged(const void *host, size_t bytes) {
    if (bytes < kCopyMin) return false;
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) == hipSuccess) {
      if (a.type != hipMemoryTypeUnregistered) return false;
    } else {
      (void)hipGetLastError();  // memory that the runtime does not know
    }
    if (!again_) {
      again_ = true;
      return false;
    }
    return reserve(bytes);
  }

  // work(0) .. work(n - 1) on this thread and up to kCopyThreads - 1 others
  template <class F>
  static hipError_t each(int n, F work) {
    std::atomic<int> next{0}, error{(int)hipSuccess};
    int device = 0;
    const hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const auto run = [&] {
      for (int k; (k = next.fetch_add(1)) < n;) {
        const hipError_t r = work(k);
        if (r != hipSuccess) error = (int)r;
      }
    };
    std::thread team[kCopyThreads - 1];
    const int most = std::min({n, kCopyThreads, (int)std::max(1u, std::thread::hardware_concurrency())}) - 1;
    for (int k = 0; k < most; ++k) {
      try {
        team[k] = std::thread([&] {
          const hipError_t r = hipSetDevice(device);
          if (r == hipSuccess)
            run();
          else
            error = (int)r;
        });
      } catch (const std::system_error &) {
        break;  // the threads there are do it
      }
    }
    run();
    for (std::thread &t : team)
      if (t.joinable()) t.join();
    return (hipError_t)error.load();
  }
};

}  // namespace spss
