// The runtime calls that rhy_transfer.hip makes, on host memory, with counts
// and switches, so that its routes can be tested without a device.
#pragma once

#include <cstdlib>
#include <cstring>
#include <mutex>

typedef int hipError_t;
typedef int hipDevice_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2,
                     hipErrorInvalidHandle = 400;
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;

struct FakeStream {
  int device;
};
struct FakeEvent {
  int device;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

namespace hostrt {
inline std::mutex lock;
inline int copies = 0, waits = 0, pinned_calls = 0, events = 0;
inline size_t pinned_bytes = 0;  // pinned and not given back
inline bool refuse_pinned = false;
inline const void *pinned_lo = nullptr, *pinned_hi = nullptr;  // pinned caller memory
inline thread_local int device = 0;
}  // namespace hostrt

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) {
  *d = hostrt::device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  hostrt::device = d;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s->device;
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = p >= hostrt::pinned_lo && p < hostrt::pinned_hi ? hipMemoryTypeHost
                                                            : hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  ++hostrt::pinned_calls;
  if (hostrt::refuse_pinned) return hipErrorOutOfMemory;
  hostrt::pinned_bytes += n;
  size_t* q = static_cast<size_t*>(std::malloc(n + 64));
  *q = n;
  *p = q + 8;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  size_t* q = static_cast<size_t*>(p) - 8;
  hostrt::pinned_bytes -= *q;
  std::free(q);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind,
                                 hipStream_t) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  ++hostrt::copies;
  std::memcpy(to, from, n);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  ++hostrt::waits;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  ++hostrt::events;
  *e = static_cast<FakeEvent*>(std::malloc(sizeof(FakeEvent)));
  (*e)->device = hostrt::device;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> hold(hostrt::lock);
  --hostrt::events;
  std::free(e);
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
