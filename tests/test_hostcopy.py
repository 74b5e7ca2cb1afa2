"""The threaded device-to-host copy (csrc/hostcopy.cpp) on the CPU, with a stand-in for the runtime whose copies are
memcpy: every size around its chunks arrives whole, and threads that cannot be had, whether the system or the
allocator refuses them, leave the copy to the calling thread."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

STUB = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
inline hipError_t hipHostMalloc(void** p, size_t n, int) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = (void*)1; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
"""

MAIN = r"""
#include <cstdio>
#include <new>
#include <vector>
#include "hostcopy.h"
// the allocation of this thread that fails, counted down; 0: none
static thread_local int fail_at = 0;
void* operator new(size_t n) {
  if (fail_at > 0 && --fail_at == 0) throw std::bad_alloc();
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main() {
  const size_t MB = 1 << 20;
  adga_host::HostCopy h;
  std::vector<unsigned char> src(70 * MB), dst(70 * MB);
  for (size_t i = 0; i < src.size(); ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
  for (size_t bytes : {(size_t)1, 16 * MB - 1, 16 * MB, 16 * MB + 1, 18 * MB, 31 * MB + 12345, 32 * MB, 33 * MB + 7,
                       64 * MB - 16, 69 * MB + 16})
    for (int fail = 0; fail <= (bytes >= 16 * MB ? 8 : 0); ++fail) {
      std::fill(dst.begin(), dst.end(), (unsigned char)0xee);
      fail_at = fail;
      const hipError_t e = h.to_host(dst.data(), src.data(), bytes, nullptr);
      fail_at = 0;
      bool ok = e == hipSuccess && memcmp(dst.data(), src.data(), bytes) == 0;
      for (size_t i = bytes; i < dst.size(); ++i) ok = ok && dst[i] == 0xee;
      if (!ok) { printf("bytes %zu fail %d wrong\n", bytes, fail); return 1; }
    }
  printf("ok\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_hostcopy_sizes_and_refused_threads(tmp_path):
    csrc = os.path.join(ROOT, "adga_amd", "csrc")
    os.makedirs(tmp_path / "hip")
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", str(tmp_path), "-I", csrc, str(tmp_path / "main.cpp"),
                    os.path.join(csrc, "hostcopy.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
