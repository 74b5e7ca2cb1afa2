// Large copies from the device to the caller's pageable arrays, through pinned slots emptied by a few host
// threads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace adga_host {

// One per context: its pinned slots are allocated at the first large copy and freed with it.  A copy occupies
// the calling thread until it is complete, like a copy of pageable memory, so calls on one object do not overlap
// (a context is used by one host thread at a time).
//
// A pageable device-to-host copy of the runtime moves at the rate of one thread that copies and takes the page
// faults of a fresh array (9.8 GB/s: 27 ms for the 264 MB self-energy of the 5-orbital 16^3 workload, 9.1 ms
// here; 8 chunks of 1 MB in flight 10.6 ms, of 4 MB 8.2 ms but twice the pinned memory to set up).  Here
// each thread queues the DMA of its next chunk while it copies the last one.
class HostCopy {
 public:
  // smaller copies are left to the runtime
  static constexpr size_t MIN_BYTES = (size_t)16 << 20;
  ~HostCopy() { release(); }
  // dst (host) <- src (device) after the work queued on `s` so far; complete on return
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
  void release();

 private:
  static constexpr int THREADS = 8, SLOTS = 2;              // slots per thread
  static constexpr size_t CHUNK = (size_t)2 << 20;
  bool ensure();
  char* pinned_ = nullptr;
  hipEvent_t ev_[THREADS * SLOTS] = {};
};

}  // namespace adga_host
