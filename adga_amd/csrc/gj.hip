// The inverse of one complex128 matrix (adga_inverse_matrix_z) by Gauss-Jordan elimination in place with
// partial pivoting, on gfx950.
//
// One matrix gives an LU and n triangular solves too little to do at once: 463 launches of one to a few
// workgroups, most of their time a chain of 32-column panels and 32-row triangular products.  The elimination
// in place needs two launches per GJ_W columns and no right-hand sides:
//   k_gj_panel   the columns [c0, c0 + w) of all rows, in the registers of one workgroup: w pivot steps, each
//                eliminating the pivot's column in every other row, which leaves in the panel its columns G of
//                the result, and in F each step's multipliers;
//   k_gj_update  the same w steps for all other columns: what each pivot row holds when its step comes (a triangular
//                recursion of w values per column), and A' = E A - F X of these rows X (E: the identity without the
//                pivot rows), a product of inner size w on the FP64 matrix cores over the whole chip, from one
//                buffer into another (a workgroup's input rows are another's output rows).
// The product of the steps, G, would update the other columns without the recursion (A' = E A + G A[pivot rows, :]),
// but it holds the inverse of the w x w pivot block, whose condition then multiplies the error: |1 - X A| at
// n = 65 and condition 1e8 5e-8, at 1e14 1.5, where the steps one by one, like an LU, leave 3e-9 and 2e-3.
// Rows are not interchanged: the pivot of column j is the largest |re| + |im| among the rows not used yet, the
// smallest row on ties - the pivots of LAPACK's interchanged elimination as long as no tie decides between rows
// it has moved - and k_gj_unscramble puts row p_j and column i in the places j and p_i.
//
// The elimination above the pivots costs it some accuracy against an LU (relative error 2.8e-15 against 1.2e-15 at
// n = 1080); one Newton step X + (1 - X A) X, two products on the matrix cores, leaves 9e-16.  It is taken where
// the matrix is well conditioned only (k_gj_newton).
//
// n = 1080: 8.1 ms with the two host copies (the LU with n right-hand sides 24.3; 7.7 with G in the place of F and X).
#include <algorithm>

#include "adga_kernels.h"
#include "mfma_gemm.h"
#include "wave_ops.h"

namespace adga {

namespace {
constexpr int GJ_W = 16;
constexpr int GJ_SMALL = 64;  // one launch up to this size

// A candidate pivot's rank: |re| + |im| as an integer, 0 for none (a NaN, a row already used)
__device__ __forceinline__ unsigned long long pivot_key(z64 x, bool open) {
  const double v = cabs1(x);
  return open && v == v ? (unsigned long long)__double_as_longlong(v) + 1 : 0ull;
}

// the smallest of `row` over the lanes of a mask
__device__ __forceinline__ int min_row(unsigned long long mask, int row) {
  int best = 0x7fffffff;
  while (mask) {  // ties: a few lanes
    best = min(best, __builtin_amdgcn_readlane(row, __ffsll((long long)mask) - 1));
    mask &= mask - 1;
  }
  return best;
}

// The w <= GJ_W columns from c0 on, given as the columns of Pn and left as the columns of G, and the multipliers of
// step j as column j of F (n values each, so that consecutive lanes take consecutive rows), in the registers of one
// workgroup, thread t holding rows t + i NT.  One
// barrier per column: each wave publishes its best candidate with the row's values.  The column of step j is always
// register 0: each step writes the updated column c to register c - 1 and the finished one to the last, so that
// GJ_W steps leave them in order and one loop body serves all (unrolled, the body's 16 copies ran at the rate of
// instruction misses: 126 us per panel at n = 1080).  pos[r]: the column row r was the pivot of, -1 before.
//
// Bound by FP64 issue on one CU and the latency of barrier, search and reciprocal: 49 us per panel at n = 1080, 3 of
// them for F (62 us with A and G row-major and the pivot row read from LDS by every thread).
template <int RPT, int NT>
__global__ void __launch_bounds__(NT) k_gj_panel(int n, int c0, int w, const z64* __restrict__ Pn,
                                                 z64* __restrict__ G, z64* __restrict__ F, int* __restrict__ piv,
                                                 int* __restrict__ pos, int* __restrict__ info) {
  constexpr int NW = NT / 64, W = GJ_W;
  __shared__ z64 cv[2][NW][W];
  __shared__ unsigned long long ckey[2][NW];
  __shared__ int crow[2][NW];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  z64 reg[RPT][W];
  unsigned open = 0;  // bit i: the row of slot i exists and is not a pivot yet
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = t + i * NT;
    if (r < n && (c0 == 0 || pos[r] < 0)) open |= 1u << i;
#pragma unroll
    for (int c = 0; c < W; ++c) reg[i][c] = r < n && c < w ? Pn[c * n + r] : mk(0.0, 0.0);
  }
  int bad = 0;
  // the wave's candidate in the column in register 0, with its row's values
  auto search = [&](int q) __attribute__((always_inline)) {
    unsigned long long key = 0;
    int slot = 0;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const unsigned long long k = pivot_key(reg[i][0], open >> i & 1);
      const bool take = k > key;
      key = take ? k : key;
      slot = take ? i : slot;
    }
    unsigned long long who = wave_argmax(key);
    int wl = __ffsll((long long)who) - 1;
    const int row = t + slot * NT;
    if (__popcll(who) > 1 && __ballot(key != 0)) {
      const int best = min_row(who, row);
      wl = __ffsll((long long)(who & __ballot(row == best))) - 1;
    }
    if (lane == wl) {
      ckey[q][wave] = key;
      crow[q][wave] = row;
#pragma unroll
      for (int i = 0; i < RPT; ++i)
        if (slot == i) {
#pragma unroll
          for (int c = 0; c < W; ++c) cv[q][wave][c] = reg[i][c];
          // keeps the branches apart: merged, they become one store from an address into reg, i.e. scratch memory
          asm volatile("; slot %0" ::"n"(i));
        }
    }
  };
  search(0);
#pragma unroll 1
  for (int j = 0; j < W; ++j) {
    const int q = j & 1;
    if (j >= w) {  // a narrow last panel: only the registers move on
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const z64 first = reg[i][0];
#pragma unroll
        for (int c = 1; c < W; ++c) reg[i][c - 1] = reg[i][c];
        reg[i][W - 1] = first;
        if (t + i * NT < n) F[j * n + t + i * NT] = mk(0.0, 0.0);
      }
      continue;
    }
    __syncthreads();
    // the workgroup's pivot: the largest key, the smallest row on ties
    const unsigned long long k = lane < NW ? ckey[q][lane] : 0ull;
    const int krow = lane < NW ? crow[q][lane] : 0;
    const unsigned long long m = wave_argmax(k) & ((1ull << NW) - 1);
    const bool any = __ballot(k != 0) != 0;
    int bw = __ffsll((long long)m) - 1;
    if (any && __popcll(m) > 1) bw = __ffsll((long long)(m & __ballot(krow == min_row(m, krow)))) - 1;
    const int p = any ? __builtin_amdgcn_readlane(krow, bw) : -1;
    // the pivot row: lane c holds its column c, every lane takes it as a scalar
    const z64 pl = cv[q][bw][lane & (W - 1)];
    auto pr = [&](int c) { return mk(lane_value(pl.re, c), lane_value(pl.im, c)); };
    const z64 pv = pr(0);
    const bool nz = any && !(pv.re == 0.0 && pv.im == 0.0);
    if (t == 0) piv[c0 + j] = any ? p : 0;
    if (!nz && bad == 0) bad = c0 + j + 1;  // no pivot in this column: no elimination
    const z64 rp = crecip(pv);
    z64 f[RPT], last[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const z64 l = cmul(reg[i][0], rp);
      f[i] = csel(nz, l, mk(0.0, 0.0));
      last[i] = csel(nz, mk(-l.re, -l.im), reg[i][0]);
      const int wr = wave * 64 + i * NT;  // the wave's rows of slot i
      if (p >= wr && p < wr + 64) {  // uniform: the pivot is one of them; its row is pr / pivot = 0 - (-1 / pivot) pr
        const bool own = t + i * NT == p;
        if (own) pos[p] = c0 + j;
        open = own ? open & ~(1u << i) : open;
        if (nz) {
          f[i] = csel(own, mk(-rp.re, -rp.im), f[i]);
          last[i] = csel(own, rp, last[i]);
#pragma unroll
          for (int c = 1; c < W; ++c) reg[i][c] = csel(own, mk(0.0, 0.0), reg[i][c]);
        }
      }
    }
#pragma unroll
    for (int c = 1; c < W; ++c) {
      const z64 x = pr(c);
#pragma unroll
      for (int i = 0; i < RPT; ++i) reg[i][c - 1] = cfms(f[i], x, reg[i][c]);
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      reg[i][W - 1] = last[i];
      if (t + i * NT < n) F[j * n + t + i * NT] = f[i];
    }
    if (j + 1 < w) search(q ^ 1);
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = t + i * NT;
    if (r < n) {
#pragma unroll
      for (int c = 0; c < W; ++c) G[c * n + r] = c < w ? reg[i][c] : mk(0.0, 0.0);
      if (c0 == 0 && (open >> i & 1)) pos[r] = -1;
    }
  }
  if (t == 0 && (c0 == 0 || (bad != 0 && *info == 0))) *info = bad;
}

// Pn[c][r] = A(r, c) for the first w columns; rmax cleared
__global__ void __launch_bounds__(256) k_gj_first(int n, int w, const z64* __restrict__ A, z64* __restrict__ Pn,
                                                  unsigned long long* __restrict__ rmax) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e == 0) *rmax = 0;
  if (e < n * GJ_W && e % GJ_W < w) Pn[(e % GJ_W) * n + e / GJ_W] = A[(long)(e / GJ_W) * n + e % GJ_W];
}

// out(r, c) = (r a pivot of this panel ? 0 : in(r, c)) - sum_k F(r, k) x_k(c), out(r, c0 + j) = G(r, j), and the
// next panel's columns [c1, c1 + GJ_W) once more into Pn.  x_k(c) is what the pivot row p_k of step k holds then:
// x_j = in(p_j, c) - sum_{k<j} F(p_j, k) x_k, and p_j itself enters the sum from its own step on.  One wave per
// workgroup and 32 x 32 tile, the recursion of its 32 columns on as many lanes (both halves of the wave alike), the
// products' operands from L2 and LDS (inner size 16: four k of each MFMA, four MFMAs).  Bound by latency: every tile
// is in flight at once (n = 1080: 25 us, 21 with the product by G, whose error grows with the pivot block).
__global__ void __launch_bounds__(64) k_gj_update(int n, int c0, int w, const z64* __restrict__ in,
                                                  const z64* __restrict__ G, const z64* __restrict__ F,
                                                  const int* __restrict__ piv, const int* __restrict__ pos,
                                                  z64* __restrict__ out, z64* __restrict__ Pn) {
  constexpr int W = GJ_W;
  __shared__ z64 lo[W][W];   // F(p_j, k) at [k][j], k < j
  __shared__ z64 xs[W][33];  // x_k of the tile's columns
  const int lane = threadIdx.x, li = lane & 15, lg = lane >> 4, c1 = c0 + GJ_W;
  const int rt = blockIdx.y * 32, ct = blockIdx.x * 32;
  z64 x[W];
  const int xc = ct + (lane & 31);
#pragma unroll
  for (int k = 0; k < W; ++k) x[k] = k < w && xc < n ? in[(long)piv[c0 + k] * n + xc] : mk(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < W * W / 64; ++i) {
    const int k = (lane + 64 * i) / W, j = (lane + 64 * i) % W;
    lo[k][j] = k < j && j < w ? F[k * n + piv[c0 + j]] : mk(0.0, 0.0);
  }
  z64 g[2][4], a[2][4];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int r = rt + b * 16 + li, own = r < n ? pos[r] - c0 : 0;  // the step this row is the pivot of, or below 0
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = 4 * s + lg;
      const z64 f = r < n && k >= own ? F[k * n + r] : mk(0.0, 0.0);
      g[b][s] = mk(-f.re, -f.im);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < W - 1; ++k)
#pragma unroll
    for (int j = k + 1; j < W; ++j) x[j] = cfms(lo[k][j], x[k], x[j]);
#pragma unroll
  for (int k = 0; k < W; ++k)
    if (lane < 32) xs[k][lane] = x[k];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int b = 0; b < 2; ++b) a[b][s] = xs[4 * s + lg][b * 16 + li];
  f64x4 re[2][2], im[2][2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = rt + rb * 16 + Mfma<double>::row(lg, v);
      const bool keep = r < n && !(pos[r] >= c0);  // pos >= c0: a pivot of this panel (later ones are not set yet)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const int c = ct + cb * 16 + li;
        const z64 x = keep && c < n ? in[(long)r * n + c] : mk(0.0, 0.0);
        re[rb][cb][v] = x.re;
        im[rb][cb][v] = x.im;
      }
    }
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        re[rb][cb] = Mfma<double>::op(g[rb][s].re, a[cb][s].re, re[rb][cb]);
        im[rb][cb] = Mfma<double>::op(g[rb][s].re, a[cb][s].im, im[rb][cb]);
        re[rb][cb] = Mfma<double>::op(-g[rb][s].im, a[cb][s].im, re[rb][cb]);
        im[rb][cb] = Mfma<double>::op(g[rb][s].im, a[cb][s].re, im[rb][cb]);
      }
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = rt + rb * 16 + Mfma<double>::row(lg, v), c = ct + cb * 16 + li;
        if (r < n && c < n) {
          const z64 x = mk(re[rb][cb][v], im[rb][cb][v]);
          out[(long)r * n + c] = c >= c0 && c < c0 + w ? G[(c - c0) * n + r] : x;
          if (c >= c1 && c < c1 + GJ_W) Pn[(c - c1) * n + r] = x;
        }
      }
}

// out(j, p_i) = A(p_j, i)
__global__ void __launch_bounds__(256) k_gj_unscramble(int n, const z64* __restrict__ A, const int* __restrict__ piv,
                                                       z64* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y;
  if (i < n) out[(long)j * n + piv[i]] = A[(long)piv[j] * n + i];
}

// The whole elimination of n <= GJ_SMALL in one workgroup of NW waves, wave v holding the columns [16 v, 16 v + 16)
// of all rows, one row per lane.  Per column one barrier: its wave finds the pivot among its lanes and publishes
// the column; every wave takes its part of the pivot row from the pivot's lane.
template <int NW>
__global__ void __launch_bounds__(NW * 64) k_gj_small(int n, const z64* __restrict__ A, z64* __restrict__ out,
                                                      int* __restrict__ info) {
  constexpr int W = GJ_W;
  __shared__ z64 col[2][64];
  __shared__ int prow[2];
  __shared__ int order[64];  // the pivot row of each column
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave * W;
  z64 reg[W];
#pragma unroll
  for (int c = 0; c < W; ++c) reg[c] = lane < n && cw + c < n ? A[lane * n + cw + c] : mk(0.0, 0.0);
  bool open = lane < n;
  int bad = 0;
  // register 0 is the wave's column cw + j % 16, as in k_gj_panel
#pragma unroll 1
  for (int j = 0; j < NW * W; ++j) {
    const int q = j & 1;
    const bool mine = wave == j / W;
    if (mine && j < n) {
      const unsigned long long key = pivot_key(reg[0], open);
      const int p = __ballot(key != 0) ? __ffsll((long long)wave_argmax(key)) - 1 : -1;
      col[q][lane] = reg[0];
      if (lane == 0) prow[q] = p;
    }
    __syncthreads();
    const int p = j < n ? __builtin_amdgcn_readfirstlane(prow[q]) : -1;
    const z64 pv = col[q][p < 0 ? 0 : p];
    const bool nz = p >= 0 && !(pv.re == 0.0 && pv.im == 0.0);
    if (j < n) {
      if (!nz && bad == 0) bad = j + 1;  // no pivot in this column: no elimination
      if (threadIdx.x == 0) order[j] = p < 0 ? 0 : p;
    }
    const bool own = lane == p;
    open = open && !own;
    z64 first = reg[0];
    if (nz) {
      const z64 rp = crecip(pv);
      const z64 l = cmul(col[q][lane], rp);
      // the pivot's row: x / pivot = 0 - (-1 / pivot) x
      const z64 f = csel(own, mk(-rp.re, -rp.im), l);
      auto update = [&](z64 v) {
        const z64 x = mk(lane_value(v.re, p), lane_value(v.im, p));
        return cfms(f, x, csel(own, mk(0.0, 0.0), v));
      };
      first = mine ? csel(own, rp, mk(-l.re, -l.im)) : update(first);
#pragma unroll
      for (int c = 1; c < W; ++c) reg[c - 1] = update(reg[c]);
    } else {
#pragma unroll
      for (int c = 1; c < W; ++c) reg[c - 1] = reg[c];
    }
    reg[W - 1] = first;
  }
  __syncthreads();
  if (threadIdx.x == 0) *info = bad;
  // out(j, p_i) = row p_j, column i: lane r is row p_j = r
  int j = 0;
  for (int k = 0; k < n; ++k)
    if (order[k] == lane) j = k;
  if (lane < n && !bad) {
#pragma unroll
    for (int c = 0; c < W; ++c)
      if (cw + c < n) out[j * n + order[cw + c]] = reg[c];
  }
}

// C = 1 - X A and its largest element into rmax (step 0), or X + R X (step 1), n x n, R and A in the place of P and
// Q: 32 x 32 tiles, four waves.  The sums are formed in slices of 128 products, so that rounding grows with the slice
// and not with n (one sum over all of n = 1080 left 2.2e-15).  0.21 ms each at n = 1080, half the FP64 matrix rate:
// three passes over the chip.
//
// The step makes X A = 1 more accurate but not A X = 1: R's own rounding, about eps |X| |A|, enters the latter as
// A R X, eps times the square of the condition (n = 65, condition 1e8: |1 - A X| 2e-3 with the step, 3e-9 without).
// So X stays as it is (and is copied to C) where |R| is above 4 eps sqrt(n), which matrices of a condition below
// about 100 leave: there the step makes both residuals smaller (n = 1080, condition 100: 2e-14 -> 7e-15 and 1e-15).
__global__ void __launch_bounds__(256) k_gj_newton(int n, int step, const z64* __restrict__ P, const z64* __restrict__ Q,
                                                   z64* __restrict__ C, unsigned long long* __restrict__ rmax) {
  using Cfg = G3Cfg<double, 32, 32, 2, 2, 16>;
  constexpr int KS = 128;  // an even number of the tile's chunks: a slice starts in the buffer the last one has left
  __shared__ __align__(16) unsigned char lds[Cfg::LDS];
  const int rt = blockIdx.y * 32, ct = blockIdx.x * 32;
  if (step == 1 && !(__longlong_as_double((long long)*rmax) <= 4 * 2.220446049250313e-16 * sqrt((double)n))) {
    for (int e = threadIdx.x; e < 32 * 32; e += 256) {
      const int r = rt + e / 32, c = ct + e % 32;
      if (r < n && c < n) C[r * n + c] = Q[r * n + c];
    }
    return;
  }
  unsigned long long top = 0;
  for (int k = 0; k < n; k += KS)
    gemm3m_tile<double, 32, 32, 2, 2, 16>(
        P + k, n, Q + (long)k * n, n,
        [=](int r, int c) {
          return k ? C[r * n + c] : step ? Q[r * n + c] : mk(r == c ? 1.0 : 0.0, 0.0);
        },
        [=, &top](int r, int c, z64 v) {
          C[r * n + c] = v;
          const unsigned long long b = (unsigned long long)__double_as_longlong(cabs1(v)) & 0x7fffffffffffffffull;
          if (k + KS >= n && b > top) top = b;  // a NaN is above every number
        },
        n, n, min(KS, n - k), false, step == 0, rt, ct, lds);
  if (step == 1) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long v = __shfl_xor(top, o);
    top = v > top ? v : top;
  }
  if ((threadIdx.x & 63) == 0) atomicMax(rmax, top);
}

}  // namespace

// the largest panel in registers: 3 rows of each of 512 threads (n = 1536: 15 ms; the LU above: 49 ms at n = 1600)
int gj_max_n() { return 1536; }

// G, the next panel, F and one word for the Newton step's residual
size_t gj_scratch(int n) { return (size_t)3 * n * GJ_W + 1; }

z64* launch_gj_inverse(int n, z64* A, z64* B, z64* C, z64* G, int* piv, int* pos, int* info, hipStream_t s) {
  if (n <= GJ_SMALL) {
    switch ((n + GJ_W - 1) / GJ_W) {
      case 1: hipLaunchKernelGGL(k_gj_small<1>, dim3(1), dim3(64), 0, s, n, A, B, info); break;
      case 2: hipLaunchKernelGGL(k_gj_small<2>, dim3(1), dim3(128), 0, s, n, A, B, info); break;
      case 3: hipLaunchKernelGGL(k_gj_small<3>, dim3(1), dim3(192), 0, s, n, A, B, info); break;
      default: hipLaunchKernelGGL(k_gj_small<4>, dim3(1), dim3(256), 0, s, n, A, B, info); break;
    }
    return B;
  }
  z64 *Pn = G + (size_t)n * GJ_W, *F = Pn + (size_t)n * GJ_W, *src = A;
  auto* rmax = reinterpret_cast<unsigned long long*>(F + (size_t)n * GJ_W);
  const int nt = (n + 31) / 32;
  hipLaunchKernelGGL(k_gj_first, dim3((n * GJ_W + 255) / 256), dim3(256), 0, s, n, std::min(GJ_W, n), A, Pn, rmax);
  for (int c0 = 0; c0 < n; c0 += GJ_W) {
    const int w = std::min(GJ_W, n - c0);
#define ADGA_GJ(RPT, NT) \
  hipLaunchKernelGGL((k_gj_panel<RPT, NT>), dim3(1), dim3(NT), 0, s, n, c0, w, Pn, G, F, piv, pos, info)
    if (n <= 128) ADGA_GJ(1, 128);
    else if (n <= 256) ADGA_GJ(1, 256);
    else if (n <= 512) ADGA_GJ(1, 512);
    else if (n <= 1024) ADGA_GJ(2, 512);
    else ADGA_GJ(3, 512);
#undef ADGA_GJ
    hipLaunchKernelGGL(k_gj_update, dim3(nt, nt), dim3(64), 0, s, n, c0, w, src, G, F, piv, pos,
                       B, Pn);
    src = B;
    std::swap(B, C);
  }
  hipLaunchKernelGGL(k_gj_unscramble, dim3((n + 255) / 256, n), dim3(256), 0, s, n, src, piv, B);
  hipLaunchKernelGGL(k_gj_newton, dim3(nt, nt), dim3(256), 0, s, n, 0, B, A, C, rmax);
  hipLaunchKernelGGL(k_gj_newton, dim3(nt, nt), dim3(256), 0, s, n, 1, C, B, A, rmax);
  return A;
}

}  // namespace adga
