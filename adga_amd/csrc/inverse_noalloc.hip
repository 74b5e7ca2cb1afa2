// adga_inverse_matrix_z_noalloc: the inverse of adga_inverse_matrix_z (the same kernels, gj.hip) with every
// device buffer it needs carved from one file-scope device array, so that a call makes no device allocation.
// Each GPU the library runs on holds its own copy of the array (about 51.1 MB at the largest n) until the
// process ends; every call on a GPU shares it, so calls that overlap on one GPU race.
#include <hip/hip_runtime.h>

#include <mutex>

#include "adga_amd.h"
#include "adga_kernels.h"

namespace {

using adga::z64;

constexpr int NA_MAX_N = ADGA_INVERSE_NOALLOC_MAX_N;
constexpr long NA_MAT = (long)NA_MAX_N * NA_MAX_N;  // complex elements of a matrix buffer, three of them
constexpr long NA_G = 3L * NA_MAX_N * 16 + 1;       // the panels (gj_scratch at NA_MAX_N)
constexpr long NA_INTS = 2 * NA_MAX_N + 1;          // pivots, row states, status
constexpr long NA_ELEMS = 3 * NA_MAT + NA_G + (NA_INTS * (long)sizeof(int) + sizeof(z64) - 1) / sizeof(z64);
constexpr int NA_MAX_DEV = 64;

}  // namespace

static __device__ __align__(256) z64 scratch[NA_ELEMS];

namespace {

std::mutex na_mu;
void* na_ptr[NA_MAX_DEV] = {};

// Device address of `scratch` on the current device, looked up once per device.
hipError_t scratch_address(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= NA_MAX_DEV) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(na_mu);
  if (!na_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    na_ptr[dev] = p;
  }
  *out = na_ptr[dev];
  return hipSuccess;
}

}  // namespace

extern "C" int adga_inverse_matrix_z_noalloc(int n, double* m, int* ierr) {
  if (n < 1 || !m || !ierr) return ADGA_E_ARG;
  *ierr = 0;
  if (n > NA_MAX_N) return ADGA_E_ARG;
  if (n > adga::gj_max_n() || adga::gj_scratch(n) > (size_t)NA_G) return ADGA_E_ARG;
  void* base = nullptr;
  if (scratch_address(&base) != hipSuccess) return ADGA_E_HIP;
  z64* a = static_cast<z64*>(base);
  z64 *b = a + NA_MAT, *c = b + NA_MAT, *g = c + NA_MAT;
  int* piv = reinterpret_cast<int*>(g + NA_G);
  int *pos = piv + NA_MAX_N, *info = pos + NA_MAX_N;
  const size_t bytes = sizeof(z64) * (size_t)n * n;
  // the Fortran matrix read row-major is its transpose, and so is the inverse
  if (hipMemcpyAsync(a, m, bytes, hipMemcpyHostToDevice, nullptr) != hipSuccess) return ADGA_E_HIP;
  const z64* x = adga::launch_gj_inverse(n, a, b, c, g, piv, pos, info, nullptr);
  if (hipGetLastError() != hipSuccess) return ADGA_E_HIP;
  if (hipMemcpy(ierr, info, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess) return ADGA_E_HIP;
  if (*ierr != 0) return ADGA_E_SINGULAR;
  if (hipMemcpy(m, x, bytes, hipMemcpyDeviceToHost) != hipSuccess) return ADGA_E_HIP;
  return ADGA_OK;
}
