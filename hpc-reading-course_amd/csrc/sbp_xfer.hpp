// sbp_xfer.hpp -- moving vectors between the caller's memory and the device.
//
// The caller's memory is pageable, and a fresh result array is not even mapped
// yet.  A copy call then takes 25 us or more to set up, and a large one out of
// device memory runs at one thread's page faults and copies: 37 ms for the 403
// MB of a 4097^2 state, 22 ms into mapped pages.  So
//   - vectors of at most kZeroCopyBytes lie in pinned host memory, which the
//     kernels that convert them read or write themselves (a right-hand side
//     at 65^2, 101 KB in and out, 46 us with copy calls, 29 without; 1.05 MB in
//     53 / 72, out 56 / 360).  Beyond, the processor's copy into it is as slow
//     as the call's (1.27 MB in 66 / 69 us, 1.59 MB 80 / 74);
//   - results of kThreadedBytes and more leave through pinned chunks that a
//     few threads drain, each copying one out while the others' transfers run:
//     403 MB 10.6 ms (38), 101 MB 3.0 (9.4).  Chunks of 4 MB: 1 MB ones take 13
//     ms, a transfer's set-up each; four threads: two 20 ms, eight 9.3.  Smaller
//     results are left to one copy call: beside a caller's own threads that
//     spin for work, waiting for a processor costs more than it saves (48
//     results of 9 MB, interleaved with such work: 28 ms, with four threads 75).
// Uploads stay one copy call (13.6 ms for 403 MB).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

namespace sbp {
namespace host {

constexpr size_t kZeroCopyBytes = 5 << 18;
constexpr size_t kThreadedBytes = 64 << 20;

// Pinned chunks of one context's or ensemble's transfers, allocated by the
// first that needs them (16 MB) and freed with their owner.
class Staging {
  static constexpr int kSlots = 4;
  static constexpr size_t kChunk = 4 << 20;
  char *pin_[kSlots] = {};
  hipEvent_t ev_[kSlots] = {};

 public:
  Staging() = default;
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;
  ~Staging() { release(); }
  void release()
  {
    for (int k = 0; k < kSlots; k++) {
      if (pin_[k]) (void)hipHostFree(pin_[k]);
      if (ev_[k]) (void)hipEventDestroy(ev_[k]);
      pin_[k] = nullptr;
      ev_[k] = nullptr;
    }
  }

  // bytes of device memory src, as the stream's earlier work leaves them, to
  // dst; done when it returns
  hipError_t to_host(void *dst, const void *src, size_t bytes, hipStream_t s)
  {
    const long chunks = (long)((bytes + kChunk - 1) / kChunk);
    // the stream's device, which need not be the calling thread's
    int device = 0, callers = 0;
    hipError_t e = hipStreamGetDevice(s, &device);
    if (e == hipSuccess) e = hipGetDevice(&callers);
    if (e == hipSuccess) e = hipSetDevice(device);
    if (e != hipSuccess) return e;
    int slots = 0;
    for (; slots < kSlots && e == hipSuccess; slots += e == hipSuccess) {
      if (!ev_[slots]) e = hipEventCreateWithFlags(&ev_[slots], hipEventDisableTiming);
      if (e == hipSuccess && !pin_[slots])
        e = hipHostMalloc(reinterpret_cast<void **>(&pin_[slots]), kChunk, hipHostMallocDefault);
    }
    if (slots < kSlots) (void)hipGetLastError();  // fewer chunks, or none: a copy call
    if (slots == 0) {
      e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      const hipError_t back = hipSetDevice(callers);
      return e == hipSuccess ? back : e;
    }
    std::atomic<long> next{0};
    std::atomic<int> failed{hipSuccess};
    auto drain = [&](int k) {
      hipError_t r = hipSetDevice(device);
      for (long i; r == hipSuccess && (i = next.fetch_add(1)) < chunks;) {
        const size_t o = (size_t)i * kChunk, m = std::min(kChunk, bytes - o);
        r = hipMemcpyAsync(pin_[k], static_cast<const char *>(src) + o, m, hipMemcpyDeviceToHost, s);
        if (r == hipSuccess) r = hipEventRecord(ev_[k], s);
        if (r == hipSuccess) r = hipEventSynchronize(ev_[k]);
        if (r == hipSuccess) std::memcpy(static_cast<char *>(dst) + o, pin_[k], m);
      }
      if (r != hipSuccess) failed = r;
    };
    std::thread th[kSlots];
    int started = 1;
    try {
      for (; started < slots; started++) th[started] = std::thread(drain, started);
    } catch (const std::exception &) {  // no more threads, or no memory for one: those there are take the rest
    }
    drain(0);
    for (int k = 1; k < started; k++) th[k].join();
    const hipError_t back = hipSetDevice(callers);
    if (failed == hipSuccess) failed = back;
    return static_cast<hipError_t>(failed.load());
  }
};

// v into the buffer the kernels read: pinned host memory, once nothing in
// flight uses it, or device memory
inline hipError_t put(void *buf, bool pinned, const void *v, size_t bytes, hipStream_t s)
{
  if (!pinned) return hipMemcpyAsync(buf, v, bytes, hipMemcpyHostToDevice, s);
  const hipError_t e = hipStreamSynchronize(s);
  if (e == hipSuccess) std::memcpy(buf, v, bytes);
  return e;
}

// what the stream's kernels leave in the buffer to v; done when it returns
inline hipError_t get(Staging &st, void *v, const void *buf, bool pinned, size_t bytes, hipStream_t s)
{
  if (bytes >= kThreadedBytes) return st.to_host(v, buf, bytes, s);
  if (!pinned) {
    const hipError_t c = hipMemcpyAsync(v, buf, bytes, hipMemcpyDeviceToHost, s);
    if (c != hipSuccess) return c;
  }
  const hipError_t e = hipStreamSynchronize(s);
  if (e == hipSuccess && pinned) std::memcpy(v, buf, bytes);
  return e;
}

}  // namespace host
}  // namespace sbp
