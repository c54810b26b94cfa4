// host_copy.cpp — see host_copy.h.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace cfx {

HostCopy::~HostCopy() {
  for (int t = 0; t < kThreads; ++t) {
    if (done_[t]) (void)hipEventDestroy(done_[t]);
    if (piece_[t]) (void)hipHostFree(piece_[t]);
  }
}

bool HostCopy::ready() {
  if (n_ > 0) return true;
  const int want = std::min<int>(kThreads, std::max(1u, std::thread::hardware_concurrency()));
  for (int t = 0; t < want; ++t) {
    if (!piece_[t] && hipHostMalloc(&piece_[t], kPiece, hipHostMallocDefault) != hipSuccess) {
      piece_[t] = nullptr;
      (void)hipGetLastError();  // no pinned memory left: go on with what there is
      break;
    }
    if (!done_[t] && hipEventCreateWithFlags(&done_[t], hipEventDisableTiming) != hipSuccess) {
      done_[t] = nullptr;
      (void)hipGetLastError();
      break;
    }
    n_ = t + 1;
  }
  return n_ > 0;
}

// Whether p is ordinary host memory.  The runtime itself copies at the link's rate
// into pinned memory, and the processor need not reach device memory at all.
static bool pageable(const void *p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

int HostCopy::to_host(void *dst, const void *src, size_t n, hipStream_t st) {
  if (hipError_t e = hipStreamSynchronize(st)) return (int)e;
  std::unique_lock<std::mutex> lock(busy_, std::defer_lock);
  if (n < kLeast || !pageable(dst) || !lock.try_lock()) return (int)hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
  if (n_ == 0) {
    asked_ += n;
    if (asked_ < kWorth) {
      lock.unlock();
      return (int)hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
    }
  }
  // events and transfers belong to the stream's device, which need not be the
  // caller's current one
  int device = 0, current = 0;
  if (hipStreamGetDevice(st, &device) != hipSuccess || hipGetDevice(&current) != hipSuccess ||
      hipSetDevice(device) != hipSuccess) {
    (void)hipGetLastError();
    return (int)hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
  }
  if (!ready()) {
    (void)hipSetDevice(current);
    return (int)hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
  }
  // about two pieces per thread at least, of 512 KiB or more
  const size_t piece = std::min(kPiece, std::max<size_t>(n / (2 * kThreads) / 4096 * 4096, 512u << 10));
  std::atomic<size_t> next{0};
  std::atomic<int> error{0};
  auto work = [&](int t) {
    int e = (int)hipSetDevice(device);
    while (e == 0 && error.load(std::memory_order_relaxed) == 0) {
      const size_t at = next.fetch_add(piece);
      if (at >= n) break;
      const size_t len = std::min(piece, n - at);
      e = (int)hipMemcpyAsync(piece_[t], (const char *)src + at, len, hipMemcpyDeviceToHost, st);
      if (e == 0) e = (int)hipEventRecord(done_[t], st);
      if (e == 0) e = (int)hipEventSynchronize(done_[t]);
      if (e == 0) std::memcpy((char *)dst + at, piece_[t], len);
    }
    if (e) error.store(e, std::memory_order_relaxed);
  };
  std::thread more[kThreads];
  const int want = (int)std::min<size_t>((size_t)n_, (n + piece - 1) / piece);
  for (int t = 1; t < want; ++t) {
    try {
      more[t] = std::thread(work, t);
    } catch (const std::system_error &) {
      break;  // the threads there are share the pieces
    }
  }
  work(0);
  for (std::thread &m : more)
    if (m.joinable()) m.join();
  (void)hipSetDevice(current);
  return error.load();
}

}  // namespace cfx
