// drain CASE: a result of several chunks through sbp::host::get on the host
// stand-in of the runtime (hip/hip_runtime.h here); prints ok, exits 0.
//   plain         as it is
//   other-device  the calling thread's device is not the stream's (and stays the thread's)
//   no-pinned     no pinned chunk to be had; one-pinned: a single one
//   no-memory     the second thread's own allocation throws std::bad_alloc
#include <hip/hip_runtime.h>

#include <cstdio>
#include <new>
#include <string>
#include <vector>

static thread_local int t_throw_at = 0;  // the calling thread's n-th allocation from here throws
void *operator new(size_t n)
{
  if (t_throw_at > 0 && --t_throw_at == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

#include "sbp_xfer.hpp"

int main(int, char **argv)
{
  const std::string how = argv[1];
  const size_t n = sbp::host::kThreadedBytes + (5 << 20) + 12345;
  std::vector<char> src(n), dst(n);
  for (size_t k = 0; k < n; k++) src[k] = (char)(k * 2654435761u >> 13);
  FakeStream stream{how == "other-device" ? 3 : 0};
  if (how == "no-pinned") g_pinned_most = 0;
  if (how == "one-pinned") g_pinned_most = 1;
  sbp::host::Staging staging;
  for (int pass = 0; pass < 2; pass++) {
    std::memset(dst.data(), 0, n);
    if (how == "no-memory") t_throw_at = 2;
    const hipError_t e = sbp::host::get(staging, dst.data(), src.data(), false, n, &stream);
    t_throw_at = 0;
    if (e != hipSuccess) return std::printf("error %d\n", (int)e), 1;
    if (dst != src) return std::printf("wrong bytes\n"), 1;
    if (t_device != 0) return std::printf("the thread's device changed\n"), 1;
    if (hipGetLastError() != hipSuccess) return std::printf("an error is left behind\n"), 1;
  }
  std::printf("ok\n");
  return 0;
}
