// host_copy.h — large copies from device memory to ordinary host memory.
//
// hipMemcpy to pageable memory stages through the runtime's own pinned buffer
// on one thread; into a freshly allocated array that thread also takes the
// page faults (507 MB, the conserved state of 256x128x128 cells with 9
// species: 48 ms).  Here kThreads threads, the caller among them, each with a
// pinned piece, take pieces of the copy in turn, so that transfers, copies and
// page faults overlap: 11.5 ms, near the rate of the link.  All transfers go through
// one stream, the owner's: new streams would cost 0.2 to 4 ms each on first use.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace cfx {

class HostCopy {
 public:
  static constexpr int kThreads = 8;
  static constexpr size_t kPiece = 4u << 20;  // pinned bytes per thread
  // smaller copies go through hipMemcpy: 3.4 MB 0.22 ms there; with the threads
  // 5 MB 0.34, 9 MB 0.52, 17 MB 0.70, 68 MB 2.0 ms (hipMemcpy 6.5)
  static constexpr size_t kLeast = 8u << 20;
  // The pinned pieces and their events take 1 to 3 ms to set up, 7 for the first
  // context of a process, and what they save adds up to that over about this many
  // bytes (a process's first copy, hipMemcpy and new pieces: 17 MB 2.2 and 7.9 ms,
  // 56 MB 5.7 and 9.5, 86 MB 9.0 and 10.0, 112 MB 11.0 and 10.5).  So they are set
  // up for a copy of this size, or once the copies so far add up to it: a program
  // that fetches a field or two does not pay for them.
  static constexpr size_t kWorth = 96u << 20;
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;
  ~HostCopy();
  // n bytes of device memory src to dst, after the work on stream st; returns a
  // hipError_t.  Callers that find the pieces in use by another thread, or no
  // pinned memory, or whose dst is pinned or device memory, copy with hipMemcpy.
  int to_host(void *dst, const void *src, size_t n, hipStream_t st);

 private:
  bool ready();
  std::mutex busy_;
  size_t asked_ = 0;  // bytes asked for before the pieces were set up
  int n_ = 0;         // threads that have a piece
  void *piece_[kThreads] = {};
  hipEvent_t done_[kThreads] = {};
};

}  // namespace cfx
