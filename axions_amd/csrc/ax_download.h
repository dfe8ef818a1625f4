/*
 * ax_download.h - device to host copies of states, winding maps and crossings
 * (host code only: it uses the HIP runtime, no kernel).
 */
#ifndef AXIONS_AX_DOWNLOAD_H
#define AXIONS_AX_DOWNLOAD_H

#include <hip/hip_runtime_api.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <new>
#include <thread>

namespace ax {

/* One run of a download: n values at dev, as they are (bytes) or floats
 * widened to doubles, to host. */
struct Run {
  const char *dev;
  char *host;
  size_t n;
  bool widen;
};

/* The calling thread's current device while this lives; the one it had after. */
class DeviceScope {
 public:
  explicit DeviceScope(int device) {
    error = hipGetDevice(&before_);
    if (error == hipSuccess && before_ != device) {
      error = hipSetDevice(device);
      changed_ = error == hipSuccess;
    }
  }
  ~DeviceScope() {
    if (changed_) (void)hipSetDevice(before_);
  }
  DeviceScope(const DeviceScope &) = delete;
  DeviceScope &operator=(const DeviceScope &) = delete;
  hipError_t error;

 private:
  int before_ = 0;
  bool changed_ = false;
};

/* Device to host on stream (of device), waiting for it.  The runtime takes
 * pageable memory through its own staging with one thread (17 GB/s here); runs
 * of kDirect bytes or more in all go through pinned memory (stage, allocated
 * on first use) in pieces instead, kCopiers threads each with two pieces, one
 * arriving while the other is copied out and, for FP32 lattices, widened.
 * State of 64^3 FP64 (21 MB) 1.33 -> 0.78 ms, of 64^3 FP32 1.03 -> 0.42, of
 * 160^3 FP64 (328 MB) 32 -> 11.  Throws nothing. */
constexpr size_t kDirect = (size_t)4 << 20;
constexpr size_t kPiece = (size_t)1 << 20;
constexpr int kCopiers = 4;

inline hipError_t download(int device, hipStream_t stream, char *&stage, const Run *runs, int nruns) {
  struct Piece {
    const char *dev;
    char *host;
    size_t n;   /* device bytes */
    bool widen;
  };
  auto bytes = [](const Run &r) { return r.widen ? 4 * r.n : r.n; };
  size_t total = 0, count = 0, widest = 0;
  for (int r = 0; r < nruns; ++r) {
    total += bytes(runs[r]);
    count += (bytes(runs[r]) + kPiece - 1) / kPiece;
    if (runs[r].widen) widest = std::max(widest, std::min(kPiece, bytes(runs[r])));
  }
  auto piece = [&](size_t i) -> Piece {
    int r = 0;
    for (size_t n; i >= (n = (bytes(runs[r]) + kPiece - 1) / kPiece); ++r) i -= n;
    const size_t o = i * kPiece;
    const Run &q = runs[r];
    return {q.dev + o, q.host + (q.widen ? 2 * o : o), std::min(kPiece, bytes(q) - o), q.widen};
  };
  auto out = [](const Piece &p, const char *from) {
    if (!p.widen) {
      memcpy(p.host, from, p.n);
      return;
    }
    const float *f = (const float *)from;
    double *d = (double *)p.host;
    for (size_t i = 0; i < p.n / 4; ++i) d[i] = f[i];
  };
  if (total >= kDirect && !stage) {
    const DeviceScope scope(device);
    if (scope.error != hipSuccess ||
        hipHostMalloc((void **)&stage, 2 * kCopiers * kPiece, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();   /* clear the sticky error of the failed call */
      stage = nullptr;
    }
  }
  if (total < kDirect || !stage) {
    std::unique_ptr<char[]> tmp(widest ? new (std::nothrow) char[widest] : nullptr);
    hipError_t e = widest && !tmp ? hipErrorOutOfMemory : hipSuccess;
    for (size_t i = 0; i < count && e == hipSuccess; ++i) {
      const Piece p = piece(i);
      e = hipMemcpyAsync(p.widen ? tmp.get() : p.host, p.dev, p.n, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess && p.widen) {
        e = hipStreamSynchronize(stream);
        if (e == hipSuccess) out(p, tmp.get());
      }
    }
    const hipError_t w = hipStreamSynchronize(stream);
    return e == hipSuccess ? w : e;
  }
  std::atomic<int> failed{(int)hipSuccess};
  auto copier = [&](int t) {
    const DeviceScope scope(device);   /* the events' device */
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = scope.error;
    for (int q = 0; q < 2 && e == hipSuccess; ++q) e = hipEventCreateWithFlags(&ev[q], hipEventDisableTiming);
    auto fetch = [&](size_t i, int q) {
      const Piece p = piece(i);
      if (e == hipSuccess)
        e = hipMemcpyAsync(stage + (size_t)(2 * t + q) * kPiece, p.dev, p.n, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(ev[q], stream);
    };
    if ((size_t)t < count) fetch(t, 0);
    int q = 0;
    for (size_t i = t; i < count && e == hipSuccess; i += kCopiers, q ^= 1) {
      if (i + kCopiers < count) fetch(i + kCopiers, q ^ 1);
      if (e == hipSuccess) e = hipEventSynchronize(ev[q]);
      if (e == hipSuccess) out(piece(i), stage + (size_t)(2 * t + q) * kPiece);
    }
    if (e != hipSuccess) failed = (int)e;
    for (hipEvent_t x : ev)
      if (x) (void)hipEventDestroy(x);
  };
  std::thread th[kCopiers];
  int started = 1;   /* the calling thread is the first copier */
  try {
    for (; started < kCopiers; ++started) th[started] = std::thread(copier, started);
  } catch (...) {   /* no more threads: their pieces are taken below */
  }
  copier(0);
  for (int t = started; t < kCopiers; ++t) copier(t);
  for (int t = 1; t < started; ++t) th[t].join();
  const hipError_t w = hipStreamSynchronize(stream);
  return failed != (int)hipSuccess ? (hipError_t)failed.load() : w;
}

}  // namespace ax

#endif
