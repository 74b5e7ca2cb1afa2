// Sums of the lambda correction in FP64 on the device.  The physical susceptibility of a point is the sum of
// the reduced susceptibility's entries, chi_phys = sum_{i,j} chi[(i,i), (j,j)] (the entries the reference's
// reduced output keeps, hdf5_module.f90:1479-1495); the corrected one is chi^lambda = chi / (1 + lambda chi)
// = 1/(1/chi + lambda), and the sums over all points are S(lambda) = sum chi^lambda and
// S'(lambda) = -sum (chi^lambda)^2.  The reductions are two-stage with a fixed grid (a partial per block, then
// one block per lambda in a fixed order), so repeated sums are bit-identical.
#include "adga_kernels.h"

namespace adga {

namespace {
constexpr int LAM_THREADS = 256;
}

// out[p] = sum_{i,j} chi[(i*n + i) + (j*n + j)*n2 + p*n4]
__global__ void k_chi_phys(int n, long npts, const z64* __restrict__ chi, z64* __restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const int n2 = n * n;
  const z64* c = chi + p * (long)n2 * n2;
  z64 acc = mk(0.0, 0.0);
  for (int j = 0; j < n; ++j)
    for (int i = 0; i < n; ++i) acc = cadd(acc, c[(i * n + i) + (long)(j * n + j) * n2]);
  out[p] = acc;
}

void launch_chi_phys(int n, long npts, const z64* chi, z64* out, hipStream_t s) {
  hipLaunchKernelGGL(k_chi_phys, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, s, n, npts, chi, out);
}

__device__ __forceinline__ void block_reduce2(z64& a, z64& b, z64* red) {
  red[threadIdx.x] = a;
  red[LAM_THREADS + threadIdx.x] = b;
  __syncthreads();
  for (int h = LAM_THREADS / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + h]);
      red[LAM_THREADS + threadIdx.x] = cadd(red[LAM_THREADS + threadIdx.x], red[LAM_THREADS + threadIdx.x + h]);
    }
    __syncthreads();
  }
  a = red[0];
  b = red[LAM_THREADS];
}

// part[(l * nblk + blk) * 2 + {0, 1}] = block blk's sums of chi^lambda_l and (chi^lambda_l)^2; grid (nblk, nl)
__global__ void __launch_bounds__(LAM_THREADS) k_lambda_partial(long npts, const double* __restrict__ lams,
                                                                const z64* __restrict__ chi, z64* __restrict__ part) {
  __shared__ z64 red[2 * LAM_THREADS];
  const int l = blockIdx.y;
  const double lam = lams[l];
  z64 s1 = mk(0.0, 0.0), s2 = mk(0.0, 0.0);
  for (long p = (long)blockIdx.x * LAM_THREADS + threadIdx.x; p < npts; p += (long)gridDim.x * LAM_THREADS) {
    const z64 c = chi[p];
    const z64 cl = cdiv(c, mk(1.0 + lam * c.re, lam * c.im));
    s1 = cadd(s1, cl);
    s2 = cadd(s2, cmul(cl, cl));
  }
  block_reduce2(s1, s2, red);
  if (threadIdx.x == 0) {
    part[((long)l * gridDim.x + blockIdx.x) * 2] = s1;
    part[((long)l * gridDim.x + blockIdx.x) * 2 + 1] = s2;
  }
}

// out[l * 2] = scale * sum, out[l * 2 + 1] = -scale * sum of squares; one block per lambda
__global__ void __launch_bounds__(LAM_THREADS) k_lambda_final(int nblk, double scale, const z64* __restrict__ part,
                                                              z64* __restrict__ out) {
  __shared__ z64 red[2 * LAM_THREADS];
  const int l = blockIdx.x;
  z64 s1 = mk(0.0, 0.0), s2 = mk(0.0, 0.0);
  for (int b = threadIdx.x; b < nblk; b += LAM_THREADS) {
    s1 = cadd(s1, part[((long)l * nblk + b) * 2]);
    s2 = cadd(s2, part[((long)l * nblk + b) * 2 + 1]);
  }
  block_reduce2(s1, s2, red);
  if (threadIdx.x == 0) {
    out[l * 2] = cscale(s1, scale);
    out[l * 2 + 1] = cscale(s2, -scale);
  }
}

void launch_lambda_sums(long npts, int nl, int nblk, double scale, const double* lams, const z64* chi, z64* part,
                        z64* out, hipStream_t s) {
  hipLaunchKernelGGL(k_lambda_partial, dim3(nblk, nl), dim3(LAM_THREADS), 0, s, npts, lams, chi, part);
  hipLaunchKernelGGL(k_lambda_final, dim3(nl), dim3(LAM_THREADS), 0, s, nblk, scale, part, out);
}

// The safeguarded Newton iteration of a solve, one state machine per solve in device memory: an evaluation is a
// k_lambda_eval (partial sums at st->lam) and a k_lambda_step (their sum, then the host rule's next lambda or the
// end), so the host queues several and waits once instead of once per evaluation (11 evaluations of 36288 points:
// 0.55 ms with a copy to and from the host for each, 0.22 so).  Evaluations queued beyond the end return at once.
__global__ void k_lambda_init(LambdaState init, LambdaState* __restrict__ st) { *st = init; }

__global__ void __launch_bounds__(LAM_THREADS) k_lambda_eval(long npts, const LambdaState* __restrict__ st,
                                                             const z64* __restrict__ chi, z64* __restrict__ part) {
  __shared__ z64 red[2 * LAM_THREADS];
  if (st->status != LAMBDA_RUNNING) return;
  const double lam = st->lam;
  z64 s1 = mk(0.0, 0.0), s2 = mk(0.0, 0.0);
  for (long p = (long)blockIdx.x * LAM_THREADS + threadIdx.x; p < npts; p += (long)gridDim.x * LAM_THREADS) {
    const z64 c = chi[p];
    const z64 cl = cdiv(c, mk(1.0 + lam * c.re, lam * c.im));
    s1 = cadd(s1, cl);
    s2 = cadd(s2, cmul(cl, cl));
  }
  block_reduce2(s1, s2, red);
  if (threadIdx.x == 0) {
    part[blockIdx.x * 2] = s1;
    part[blockIdx.x * 2 + 1] = s2;
  }
}

__global__ void __launch_bounds__(LAM_THREADS) k_lambda_step(int nblk, double scale, const z64* __restrict__ part,
                                                             LambdaState* __restrict__ state) {
  __shared__ z64 red[2 * LAM_THREADS];
  LambdaState st = *state;
  if (st.status != LAMBDA_RUNNING) return;
  z64 s1 = mk(0.0, 0.0), s2 = mk(0.0, 0.0);
  for (int b = threadIdx.x; b < nblk; b += LAM_THREADS) {
    s1 = cadd(s1, part[b * 2]);
    s2 = cadd(s2, part[b * 2 + 1]);
  }
  block_reduce2(s1, s2, red);
  if (threadIdx.x != 0) return;
  const double sum = scale * s1.re, fx = sum - st.target, dfx = -scale * s2.re;
  auto next = [&] {  // the top of Newton's loop: the end, or the next x
    st.iters = st.k < st.maxit ? st.k : st.maxit;
    if (st.k >= st.maxit) {
      st.status = LAMBDA_MAXIT;
    } else if (fabs(fx) <= st.ftol) {
      st.status = LAMBDA_DONE;
    } else {
      double xn = dfx < 0 ? st.lam - fx / dfx : 0.5 * (st.a + st.b);
      if (!(xn > st.a && xn < st.b)) xn = 0.5 * (st.a + st.b);  // Newton left the bracket: bisect
      st.lam = xn;
    }
  };
  if (!isfinite(sum) || !isfinite(dfx)) {
    st.status = LAMBDA_NONFINITE;
  } else if (st.bracket) {  // lam = b of the bracket: f(b) < 0 is looked for
    if (fx > 0) {
      if (++st.tries > 200) {
        st.status = LAMBDA_NO_BRACKET;
      } else {
        st.a = st.b;
        st.b = st.b > 0 ? 4.0 * st.b : 1.0;
        st.lam = st.b;
      }
    } else {
      st.bracket = 0;
      next();
    }
  } else {
    (fx > 0 ? st.a : st.b) = st.lam;
    if (st.b - st.a <= 4e-16 * fmax(1.0, fabs(st.lam))) {
      st.iters = st.k + 1;
      st.status = LAMBDA_DONE;
    } else {
      ++st.k;
      next();
    }
  }
  *state = st;
}

void launch_lambda_init(const LambdaState& init, LambdaState* st, hipStream_t s) {
  hipLaunchKernelGGL(k_lambda_init, dim3(1), dim3(1), 0, s, init, st);
}

void launch_lambda_newton(long npts, int nblk, double scale, LambdaState* st, const z64* chi, z64* part, hipStream_t s) {
  hipLaunchKernelGGL(k_lambda_eval, dim3(nblk), dim3(LAM_THREADS), 0, s, npts, st, chi, part);
  hipLaunchKernelGGL(k_lambda_step, dim3(1), dim3(LAM_THREADS), 0, s, nblk, scale, part, st);
}

__global__ void k_lambda_apply(long npts, double lam, const z64* __restrict__ chi, z64* __restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const z64 c = chi[p];
  out[p] = cdiv(c, mk(1.0 + lam * c.re, lam * c.im));
}

void launch_lambda_apply(long npts, double lam, const z64* chi, z64* out, hipStream_t s) {
  hipLaunchKernelGGL(k_lambda_apply, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, s, npts, lam, chi, out);
}

}  // namespace adga
