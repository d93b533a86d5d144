// The few HIP calls of transfer.hip on the host alone, for tests without a
// GPU: "device" memory is host memory, and a stream is a list of operations
// that run when someone waits for them, not before the stream's queue is
// said to have drained (busy_until).
#pragma once

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct HostStream {
  std::vector<std::function<void()>> ops;
  size_t ran = 0;
  std::chrono::steady_clock::time_point busy_until{};
  void run_to(size_t n) {
    if (ran >= n) return;
    std::this_thread::sleep_until(busy_until);
    for (; ran < n; ++ran) ops[ran]();
  }
};
struct HostEvent {
  HostStream* stream = nullptr;
  size_t at = 0;
};
using hipStream_t = HostStream*;
using hipEvent_t = HostEvent*;

// errors as HIP keeps them: a failure stays until it is fetched, a later
// success does not take it back
struct HostHip {
  hipError_t last = hipSuccess;
  bool refuse_pinned = false;
  hipError_t fail(hipError_t e) {
    last = e;
    return e;
  }
};
inline HostHip g_hip;

inline hipError_t hipGetLastError() {
  const hipError_t e = g_hip.last;
  g_hip.last = hipSuccess;
  return e;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_hip.refuse_pinned) return g_hip.fail(hipErrorOutOfMemory);
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new HostEvent;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->stream = s;
  e->at = s->ops.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->stream) e->stream->run_to(e->at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  s->run_to(s->ops.size());
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
  s->ops.push_back([=] { std::memcpy(dst, src, n); });
  return hipSuccess;
}
