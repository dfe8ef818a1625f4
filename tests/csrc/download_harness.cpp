// Test harness: the staged download (axions_amd/csrc/ax_download.h) over a
// stand-in for the HIP runtime calls it makes, in which "device" memory is
// host memory and every thread has a current device; built by
// tests/test_download_host.py with g++.
#include "../../axions_amd/csrc/ax_download.h"

#include <vector>

namespace {
thread_local int current = 0;
std::atomic<int> copies{0};
int fail_copy = -1;         // the copy that fails (-1: none)
bool fail_pinned = false;
struct Event { int device; };
constexpr int kStreamDevice = 1;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return d < 0 || d > 1 ? hipErrorInvalidDevice : hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (fail_pinned) return hipErrorOutOfMemory;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
  if (copies++ == fail_copy) return hipErrorInvalidValue;
  memcpy(to, from, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t) new Event{current}; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event *)e; return hipSuccess; }
// an event is recorded on streams of its own device
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  return ((Event *)e)->device == kStreamDevice ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

// nruns runs of n values from a device-1 lattice, called by a thread whose
// device is `device`; returns the HIP error, the thread's device afterwards in
// *after
int run_download(int device, const char *dev, char *host, size_t n, int nruns, int widen, int copy_that_fails,
                 int no_pinned, int *after) {
  copies = 0;
  fail_copy = copy_that_fails;
  fail_pinned = no_pinned != 0;
  current = device;
  std::vector<ax::Run> runs;
  const size_t from = widen ? 4 * n : n, to = widen ? 8 * n : n;
  for (int r = 0; r < nruns; ++r) runs.push_back({dev + r * from, host + r * to, n, widen != 0});
  char *stage = nullptr;
  const hipError_t e = ax::download(kStreamDevice, nullptr, stage, runs.data(), nruns);
  free(stage);
  *after = current;
  return (int)e;
}
}
