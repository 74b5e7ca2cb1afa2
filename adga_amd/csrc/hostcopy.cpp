#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

namespace adga_host {

void HostCopy::release() {
  for (hipEvent_t& e : ev_) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (pinned_) (void)hipHostFree(pinned_);
  pinned_ = nullptr;
}

bool HostCopy::ensure() {
  if (pinned_) return true;
  bool ok = hipHostMalloc((void**)&pinned_, THREADS * SLOTS * CHUNK, hipHostMallocDefault) == hipSuccess;
  for (hipEvent_t& e : ev_) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    release();
    (void)hipGetLastError();  // the runtime's own copy takes over
  }
  return ok;
}

hipError_t HostCopy::to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes < MIN_BYTES || !ensure()) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  int device = 0;
  if (hipError_t e = hipGetDevice(&device)) return e;
  std::atomic<int> err{hipSuccess};
  const size_t nchunk = (bytes + CHUNK - 1) / CHUNK;
  char* const d = static_cast<char*>(dst);
  const char* const r = static_cast<const char*>(src);
  auto len = [&](size_t c) { return std::min(CHUNK, bytes - c * CHUNK); };
  // thread t takes the chunks t, t + THREADS, ..., alternating between its two slots
  auto work = [&](int t) {
    auto check = [&](hipError_t e) {
      if (e != hipSuccess) err.store(e);
      return e == hipSuccess && err.load() == hipSuccess;
    };
    if (!check(hipSetDevice(device))) return;
    auto slot = [&](size_t i) { return pinned_ + (size_t)(t * SLOTS + (int)(i % SLOTS)) * CHUNK; };
    auto event = [&](size_t i) { return ev_[t * SLOTS + (int)(i % SLOTS)]; };
    const size_t n = (size_t)t < nchunk ? (nchunk - t - 1) / THREADS + 1 : 0;  // this thread's chunks
    auto chunk = [&](size_t i) { return t + i * THREADS; };
    auto fetch = [&](size_t i) {
      return check(hipMemcpyAsync(slot(i), r + chunk(i) * CHUNK, len(chunk(i)), hipMemcpyDeviceToHost, s)) &&
             check(hipEventRecord(event(i), s));
    };
    if (n > 0 && !fetch(0)) return;
    for (size_t i = 0; i < n; ++i) {
      if (i + 1 < n && !fetch(i + 1)) return;  // its slot was emptied in the last round
      if (!check(hipEventSynchronize(event(i)))) return;
      std::memcpy(d + chunk(i) * CHUNK, slot(i), len(chunk(i)));
    }
  };
  std::thread pool[THREADS];
  int started = 0;
  try {
    for (; started < THREADS; ++started) pool[started] = std::thread(work, started);
  } catch (const std::exception&) {
    // no more threads (std::system_error) or no memory for one (std::bad_alloc; past here it would end the process,
    // with threads not joined): this one does the rest of the shares
  }
  for (int t = started; t < THREADS; ++t) work(t);
  for (int t = 0; t < started; ++t) pool[t].join();
  hipError_t e = (hipError_t)err.load();
  // after an error a slot may still be written: the stream is drained before the slots are used again
  const hipError_t es = hipStreamSynchronize(s);
  return e != hipSuccess ? e : es;
}

}  // namespace adga_host
