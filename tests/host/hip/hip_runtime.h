// The few runtime calls sbp_xfer.hpp makes, on the host: devices are numbers,
// device memory is host memory and a copy is done when the call returns.  A
// stream and an event belong to a device; an event is only recorded on a stream
// of its own device, and created on the thread's current one, as in HIP.
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
struct FakeStream {
  int device;
};
struct FakeEvent {
  int device;
};
using hipStream_t = FakeStream *;
using hipEvent_t = FakeEvent *;
using hipDevice_t = int;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

inline thread_local int t_device = 0;                      // a thread starts on device 0
inline thread_local hipError_t t_last = hipSuccess;        // sticky until it is read
inline std::atomic<int> g_pinned{0}, g_pinned_most{1000};  // chunks handed out, and how many may be
inline hipError_t done(hipError_t e) { return e == hipSuccess ? e : (t_last = e); }

inline hipError_t hipGetLastError()
{
  const hipError_t e = t_last;
  t_last = hipSuccess;
  return e;
}
inline hipError_t hipGetDevice(int *d) { return *d = t_device, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return t_device = d, hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = s->device, hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
  *e = static_cast<hipEvent_t>(std::malloc(sizeof(FakeEvent)));
  (*e)->device = t_device;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  return done(e->device == s->device ? hipSuccess : hipErrorInvalidHandle);
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
  if (g_pinned >= g_pinned_most) return done(hipErrorOutOfMemory);
  g_pinned++;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { return g_pinned--, std::free(p), hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
  return std::memcpy(d, s, n), hipSuccess;
}
