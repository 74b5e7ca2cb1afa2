// A3 (bubble), A6 (BSE build) and the FP64 right-hand side / residuals of the A7/A8 solves
// (the LU itself is in lu.hip) on gfx950.
//
// Formulation (main.F90:673-757): for each channel r the reference forms
// A = 1 - blockdiag(S_nu) C with S_nu = chi0^q(nu) diag(chi0^w(nu))^-1 - 1 and
// C = chi0^w F_r, inverts it, and forms eta = (1+gamma^w)(A^-1 - 1).  Here the
// same eta is obtained without an explicit inverse and without the cancellation
// in A^-1 - 1: eta A = (1+gamma^w)(1 - A) = (1+gamma^w) blockdiag(S) C is solved
// as M Y = B with M = A^T, Y = eta^T: by fixed-point iteration on the residual
// products below where 1 - M contracts (M is then never formed), else by LU with
// partial pivoting of M, stored row-major per matrix (row r, column c at
// r*ldm + c); the n^2 right-hand sides are extra columns of M where they do not
// fit the solve's LDS at once, so that their forward elimination happens inside
// the factorisation.  B and every residual are formed in FP64 from the unrounded
// S and C, so the residual is on the scale of eta itself.
#include <type_traits>

#include "adga_kernels.h"
#include "mfma_gemm.h"

namespace adga {

// ---------------------------------------------------------------- A3: bubble
// chi0q[b][d](i1 = i*n + j, i2 = l*n + k') = -beta/nkp sum_K G(K, nu_d)_il G(K - q_b, nu_d - omega)_k'j
// (accumulate_chi0, one_particle_quant_module.f90:274-288; k-sum main.F90:647-657).
// n <= 2: one block per (nu, point); thread = ((i,l), k-slice); n^2 accumulators per thread.
// gt2 is the table of the second factor G(K - q, nu - omega) (gt itself, or a derivative table when the
// tangent of the bubble is formed by the product rule); accumulate adds into chi0q.
template <int NN>
__global__ void __launch_bounds__(256) k_bubble(Geom g, int iwb, const int* __restrict__ qidx,
                                                const z64* __restrict__ gt, const z64* __restrict__ gt2,
                                                z64* __restrict__ chi0q, int accumulate) {
  constexpr int N2 = NN * NN;
  constexpr int NKS = 256 / N2;
  __shared__ z64 red[256];
  const int d = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const int og = t % N2, ks = t / N2;
  const int i = og / NN, l = og % NN;
  const int q = qidx[b];
  const int iwf = d - g.iwf;
  const z64* g1 = gt + (long)(iwf - g.glo) * g.nkp * N2;
  const z64* g2 = gt2 + (long)(iwf - iwb - g.glo) * g.nkp * N2;
  z64 acc[N2];
#pragma unroll
  for (int e = 0; e < N2; ++e) acc[e] = mk(0.0, 0.0);
  if (ks < NKS) {
    for (int K = ks; K < g.nkp; K += NKS) {
      z64 a = g1[(long)K * N2 + i * NN + l];
      int kq = k_minus_q(K, q, g.nkx, g.nky, g.nkz);
      const z64* row = g2 + (long)kq * N2;
#pragma unroll
      for (int e = 0; e < N2; ++e) acc[e] = cfma(a, row[e], acc[e]);  // e = k'*n + j
    }
  }
  const double f = -g.beta / g.nkp;
  z64* out = chi0q + ((long)b * g.nf + d) * g.n4;
#pragma unroll
  for (int e = 0; e < N2; ++e) {
    red[t] = acc[e];
    __syncthreads();
    if (t < N2) {
      z64 s = mk(0.0, 0.0);
      for (int kk = 0; kk < NKS; ++kk) s = cadd(s, red[kk * N2 + t]);
      // thread t = og = (i, l); e = (k', j): chi0(i1 = i*n + j, i2 = l*n + k')
      int ii = t / NN, ll = t % NN, kp = e / NN, jj = e % NN;
      z64* o = out + (ii * NN + jj) + (ll * NN + kp) * N2;
      *o = accumulate ? cadd(*o, cscale(s, f)) : cscale(s, f);
    }
    __syncthreads();
  }
}

// The same on the FP64 matrix cores for n >= 3: at one nu and q a product of inner size nkp, the rows (i, l) and
// columns (k', j) of the tables G(K, nu) and G(K - q, nu - omega) being the n^2 contiguous values of one K, in the
// 16 lanes of an MFMA's operand as they lie in memory (n = 3, 4: one 16 x 16 tile, 5: 2 x 2).  A workgroup of
// BUB_NW waves takes QB points at one nu, the points sharing the loads of the first factor and the indices of K;
// wave w takes K = 4 w .. 4 w + 3 of every 4 BUB_NW and the waves' sums meet in LDS.  Workgroups of one nu follow
// one another on one XCD, whose L2 then holds the two tables.
// Bound by the matrix rate on padded tiles (n = 3: 9 of 16 rows and columns; 45 .. 53 TFLOP/s of padded products).
// 5 orbitals, 16^3 k, 160 frequencies, 48 points: 10.2 ms with one thread per (i, l) and slice of k -> 4.97;
// 4 orbitals, 12^3, 40 frequencies, 48 points: 0.61 -> 0.33; 3 orbitals, 20^3, 60 frequencies, 41 points: 1.03 ->
// 0.93, one point 0.24 -> 0.17.
constexpr int BUB_NW = 8;
template <int NN, int QB>
__global__ void __launch_bounds__(BUB_NW * 64) k_bubble_mm(Geom g, int iwb, int npts, int nqg,
                                                           const int* __restrict__ qidx, const z64* __restrict__ gt,
                                                           const z64* __restrict__ gt2, z64* __restrict__ chi0q,
                                                           int accumulate) {
  using M = Mfma<double>;
  constexpr int N2 = NN * NN, T = (N2 + 15) / 16, STEP = 4 * BUB_NW;
  __shared__ double red[BUB_NW][8][64];
  const int per = (g.nf * nqg + 7) / 8;
  const int work = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (work >= g.nf * nqg || (int)(blockIdx.x / 8) >= per) return;
  const int d = work / nqg, b0 = (work % nqg) * QB;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = g.nkx, ny = g.nky, nz = g.nkz;
  const z64* g1 = gt + (long)(d - g.iwf - g.glo) * g.nkp * N2;
  const z64* g2 = gt2 + (long)(d - g.iwf - iwb - g.glo) * g.nkp * N2;
  int qx[QB], qy[QB], qz[QB];
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    const int q = qidx[min(b0 + u, npts - 1)];  // a partial group repeats its last point
    qz[u] = q % nz;
    qy[u] = q / nz % ny;
    qx[u] = q / (nz * ny);
  }
  int el[T];  // a lane beyond the n^2 values repeats the last: its row or column of the tile is not used
#pragma unroll
  for (int i = 0; i < T; ++i) el[i] = min(i * 16 + li, N2 - 1);
  f64x4 re[QB][T][T], im[QB][T][T];
#pragma unroll
  for (int u = 0; u < QB; ++u)
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int c = 0; c < T; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) re[u][r][c][v] = im[u][r][c][v] = 0.0;
  // the lane's K and its coordinates, advanced by STEP without divisions
  int K = 4 * wave + lg, kz = K % nz, ky = K / nz % ny, kx = K / (nz * ny) % nx;
  const int sz = STEP % nz, sy = STEP / nz % ny, sx = STEP / (nz * ny) % nx;
  struct Operands {
    z64 a[T], x[QB][T];
  };
  auto fetch = [&](Operands& o) __attribute__((always_inline)) {
    const int k = min(K, g.nkp - 1);
#pragma unroll
    for (int i = 0; i < T; ++i) o.a[i] = g1[k * N2 + el[i]];
#pragma unroll
    for (int u = 0; u < QB; ++u) {
      const int z = kz - qz[u], y = ky - qy[u], w = kx - qx[u];
      const int kq = (z < 0 ? z + nz : z) + ((y < 0 ? y + ny : y) + (w < 0 ? w + nx : w) * ny) * nz;
#pragma unroll
      for (int i = 0; i < T; ++i) o.x[u][i] = g2[kq * N2 + el[i]];
    }
    K += STEP;
    kz += sz;
    ky += sy;
    kx += sx;
    if (kz >= nz) kz -= nz, ++ky;
    if (ky >= ny) ky -= ny, ++kx;
    if (kx >= nx) kx -= nx;  // beyond nkp: only kept in range
  };
  const int full = g.nkp / STEP, steps = (g.nkp + STEP - 1) / STEP;
  auto multiply = [&](Operands& o, int step) __attribute__((always_inline)) {
    if (step >= full && step * STEP + 4 * wave + lg >= g.nkp) {  // no K of this lane's in the last step
#pragma unroll
      for (int i = 0; i < T; ++i) o.a[i] = mk(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < QB; ++u)
#pragma unroll
      for (int r = 0; r < T; ++r)
#pragma unroll
        for (int c = 0; c < T; ++c) {
          re[u][r][c] = M::op(o.a[r].re, o.x[u][c].re, re[u][r][c]);
          im[u][r][c] = M::op(o.a[r].re, o.x[u][c].im, im[u][r][c]);
          re[u][r][c] = M::op(-o.a[r].im, o.x[u][c].im, re[u][r][c]);
          im[u][r][c] = M::op(o.a[r].im, o.x[u][c].re, im[u][r][c]);
        }
  };
  Operands even, odd;  // the loads of a step are in flight during the products of the one before
  fetch(even);
  for (int k = 0; k < steps; k += 2) {
    fetch(odd);
    multiply(even, k);
    if (k + 1 == steps) break;
    fetch(even);
    multiply(odd, k + 1);
  }
  const double f = -g.beta / g.nkp;
#pragma unroll
  for (int u = 0; u < QB; ++u)
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int c = 0; c < T; ++c) {
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          red[wave][v][lane] = re[u][r][c][v];
          red[wave][4 + v][lane] = im[u][r][c][v];
        }
        __syncthreads();
        // wave v < 4: register v of every lane, D[row(lg, v)][li]
        if (wave < 4 && b0 + u < npts) {
          z64 s = mk(0.0, 0.0);
          for (int w = 0; w < BUB_NW; ++w) s = cadd(s, mk(red[w][wave][lane], red[w][4 + wave][lane]));
          const int il = r * 16 + M::row(lg, wave), kj = c * 16 + li;
          if (il < N2 && kj < N2) {
            z64* o = chi0q + ((long)(b0 + u) * g.nf + d) * g.n4 + (il / NN * NN + kj % NN) +
                     (il % NN * NN + kj / NN) * N2;
            *o = accumulate ? cadd(*o, cscale(s, f)) : cscale(s, f);
          }
        }
      }
}

void launch_bubble(const Geom& g, int iwb, int npts, const int* qidx, const z64* gt, z64* chi0q, hipStream_t s,
                   const z64* gt2, bool accumulate) {
  const z64* g2 = gt2 ? gt2 : gt;
  const int acc = accumulate ? 1 : 0;
  if (g.n >= 3) {
    // two points per workgroup once that still leaves one for every CU (five orbitals: one point fills the
    // registers; four points of fewer orbitals: 1.14 ms where two take 0.97)
    const int QB = g.n == 5 ? 1 : 2;
    const bool wide = QB > 1 && (long)g.nf * ((npts + QB - 1) / QB) >= 256;
    const int nqg = wide ? (npts + QB - 1) / QB : npts;
    const dim3 grid((unsigned)((g.nf * nqg + 7) / 8 * 8)), block(BUB_NW * 64);
#define ADGA_BUB(NN, QB) \
  hipLaunchKernelGGL((k_bubble_mm<NN, QB>), grid, block, 0, s, g, iwb, npts, nqg, qidx, gt, g2, chi0q, acc)
    if (g.n == 3) {
      if (wide) ADGA_BUB(3, 2);
      else ADGA_BUB(3, 1);
    } else if (g.n == 4) {
      if (wide) ADGA_BUB(4, 2);
      else ADGA_BUB(4, 1);
    } else {
      ADGA_BUB(5, 1);
    }
#undef ADGA_BUB
    return;
  }
  const dim3 grid(g.nf, npts);
  if (g.n == 1) hipLaunchKernelGGL(k_bubble<1>, grid, dim3(256), 0, s, g, iwb, qidx, gt, g2, chi0q, acc);
  else hipLaunchKernelGGL(k_bubble<2>, grid, dim3(256), 0, s, g, iwb, qidx, gt, g2, chi0q, acc);
}

// ---------------------------------------------------------------- S_nu
// S[b][d][a][c] = chi0q(a, c, d) winv(c, d) - delta_ac  (main.F90:685-688)
__global__ void k_smat(Geom g, int npts, const z64* __restrict__ chi0q, const z64* __restrict__ winv,
                       z64* __restrict__ S) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long tot = (long)npts * g.nf * g.n4;
  if (idx >= tot) return;
  int e = (int)(idx % g.n4);
  long bd = idx / g.n4;
  int d = (int)(bd % g.nf);
  int a = e / g.n2, c = e % g.n2;  // S row a, column c (row-major)
  z64 v = cmul(chi0q[bd * g.n4 + a + (long)c * g.n2], winv[c + d * g.n2]);
  if (a == c) v.re -= 1.0;
  S[idx] = v;
}

void launch_smat(const Geom& g, int npts, const z64* chi0q, const z64* winv, z64* S, hipStream_t s) {
  long tot = (long)npts * g.nf * g.n4;
  hipLaunchKernelGGL(k_smat, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, g, npts, chi0q, winv, S);
}

// ---------------------------------------------------------------- A6: BSE build
// M_{b,ch}(r, d*n2 + s) = delta - R_d(s, r),  R_d(s, r) = sum_i' S_b[d][s][i'] C_ch(d*n2 + i', r)
// (main.F90:693-700, transposed: M = A^T).  A workgroup owns DB frequency blocks d of one channel
// for PB points and all rows: their S_d sit in LDS, and each thread reads the n2 contiguous values
// C(d*n2 + ., r) (a row slice of C^T) once and turns them into n2 outputs per point.  Padding
// columns [N, ldm) are not written (never read).  The complex64 build (the refined path's LU
// input, whose residuals are formed in FP64 from S and C themselves) computes in FP32: its entries
// then differ from the rounded FP64 ones by a few FP32 ulps.  The complex128 build computes in FP64.
// Frequency blocks per workgroup (DB) and points per workgroup (PB, sharing each C row read).  For
// n <= 3 a workgroup's row segment is DB * n2 elements: complex64 takes 16 blocks, so that at n = 3 each
// segment is 1152 bytes and starts on a 128-byte line (8 blocks gave 576-byte segments, every other one
// starting mid-line; 21.2 -> 20.3 ms per build of 8000 matrices at N = 1080), with 2 points per
// workgroup to keep four workgroups per CU; complex128 segments of 8 blocks are already whole lines.
template <int NN, int ES>
struct BuildShape {
  static constexpr int N2 = NN * NN, N4 = N2 * N2;
  static constexpr int DB = NN <= 3 ? (ES == 8 ? 16 : 8) : 2;
  static constexpr int PB0 = 40960 / (DB * N4 * ES);
  static constexpr int PB1 = PB0 < 1 ? 1 : PB0 > 4 ? 4 : PB0;
  static constexpr int PB = NN <= 3 ? ((ES == 8 && PB1 > 2) ? 2 : PB1) : (PB1 < (ES == 8 ? 2 : 1) ? PB1 : (ES == 8 ? 2 : 1));
};

template <typename T, int NN>
__global__ void __launch_bounds__(256) k_build(Geom g, int npts, int ldm, const z64* __restrict__ S,
                                               const z64* __restrict__ c_d, const z64* __restrict__ c_m,
                                               cplx<T>* __restrict__ M) {
  using CA = cplx<T>;  // arithmetic type
  using Sh = BuildShape<NN, (int)sizeof(CA)>;
  constexpr int N2 = Sh::N2, N4 = Sh::N4, DB = Sh::DB, PB = Sh::PB;
  __shared__ CA sS[PB][DB * N4];
  // grid (point groups, channels, frequency blocks): the point group runs fastest, so the workgroups
  // resident at one time read the same column block of C, which stays in their XCDs' L2
  const int ch = blockIdx.y, b0 = blockIdx.x * PB, t = threadIdx.x;
  const int N = g.N;
  const int d0 = blockIdx.z * DB;
  const int nd = min(DB, g.nf - d0);
  const int np = min(PB, npts - b0);
  for (int pb = 0; pb < np; ++pb) {
    const z64* Sb = S + ((long)(b0 + pb) * g.nf + d0) * N4;
    for (int e = t; e < nd * N4; e += 256) sS[pb][e] = ccast<T>(Sb[e]);
  }
  __syncthreads();
  const z64* C = ch == 0 ? c_d : c_m;
  // outputs go through an LDS tile so that each row segment (nd*n2 complex) is written by consecutive
  // lanes.  QT threads share a (row, frequency block) and split its n2 outputs: one for n <= 3, four
  // for n = 4, 5 (16 or 25 outputs per row and block), whose tile would otherwise span 128 rows
  // (52 KB of complex64 at n = 5) and leave few workgroups per CU
  constexpr int QT = NN <= 3 ? 1 : 4, QS = (N2 + QT - 1) / QT;
  constexpr int RS = 256 / (DB * QT), W = DB * N2;
  const int q = t % QT, dl = (t / QT) % DB, rl = t / (QT * DB);
  const int d = d0 + dl, sq0 = q * QS, sq1 = min(N2, sq0 + QS);
  __shared__ cplx<T> tile[RS][W + 1];
  for (int r0 = 0; r0 < N; r0 += RS) {
    const int r = r0 + rl;
    const bool act = dl < nd && r < N;
    CA cc[N2];
    const z64* crow = C + (long)(act ? r : 0) * N + (act ? d : 0) * N2;
#pragma unroll
    for (int i = 0; i < N2; ++i) cc[i] = ccast<T>(crow[i]);
    for (int pb = 0; pb < np; ++pb) {
      if (act) {
        const CA* sd = sS[pb] + dl * N4;
        // not unrolled: S_d stays in LDS (hoisting its n2^2 values into registers costs occupancy)
#pragma unroll 1
        for (int sq = sq0; sq < sq1; ++sq) {
          CA acc = mk<T>(0, 0);
#pragma unroll
          for (int i = 0; i < N2; ++i) acc = cfma(sd[sq * N2 + i], cc[i], acc);
          tile[rl][dl * N2 + sq] = mk<T>((d * N2 + sq == r ? (T)1 : (T)0) - acc.re, -acc.im);
        }
      }
      __syncthreads();
      // 16-byte stores: ldm is a multiple of 16 and d0 * n2 is even, so every row segment starts
      // 16-byte aligned; non-temporal, as M is read again only by the factorisation after the whole
      // build (20.6 -> 19.2 ms per complex64 build of 8000 matrices at N = 1080, 34.8 -> 33.1 complex128)
      cplx<T>* mb = M + ((long)(2 * (b0 + pb) + ch) * N + r0) * ldm + d0 * N2;
      constexpr int VW = 16 / (int)sizeof(cplx<T>), WV = W / VW;
      static_assert(W % VW == 0, "row segment of whole 16-byte vectors");
      struct alignas(16) Vec { cplx<T> v[VW]; };
      const int lim = nd * N2;
      for (int e = t; e < RS * WV; e += 256) {
        const int row = e / WV, col = (e % WV) * VW;
        if (r0 + row >= N) continue;
        cplx<T>* dst = mb + (long)row * ldm + col;
        if (col + VW <= lim) {
          Vec x;
#pragma unroll
          for (int j = 0; j < VW; ++j) x.v[j] = tile[row][col + j];
          if constexpr (sizeof(T) == 4) {
            typedef float f4 __attribute__((ext_vector_type(4)));
            const f4 vv = {x.v[0].re, x.v[0].im, x.v[1].re, x.v[1].im};
            __builtin_nontemporal_store(vv, reinterpret_cast<f4*>(dst));
          } else {
            typedef double d2 __attribute__((ext_vector_type(2)));
            const d2 vv = {x.v[0].re, x.v[0].im};
            __builtin_nontemporal_store(vv, reinterpret_cast<d2*>(dst));
          }
        } else {
          for (int j = 0; j < VW; ++j)
            if (col + j < lim) dst[j] = tile[row][col + j];
        }
      }
      __syncthreads();
    }
  }
}

template <typename T>
void launch_build(const Geom& g, int npts, int ldm, const z64* S, const z64* cd, const z64* cm, cplx<T>* M,
                  hipStream_t s) {
#define ADGA_BUILD_CASE(NN)                                                                            \
  case NN: {                                                                                           \
    using Sh = BuildShape<NN, (int)sizeof(cplx<T>)>;                                                   \
    constexpr int DB = Sh::DB, PB = Sh::PB;                                                           \
    dim3 grid((npts + PB - 1) / PB, 2, (g.nf + DB - 1) / DB);                                         \
    hipLaunchKernelGGL((k_build<T, NN>), grid, dim3(256), 0, s, g, npts, ldm, S, cd, cm, M);          \
    break;                                                                                             \
  }
  switch (g.n) {
    ADGA_BUILD_CASE(1)
    ADGA_BUILD_CASE(2)
    ADGA_BUILD_CASE(3)
    ADGA_BUILD_CASE(4)
    ADGA_BUILD_CASE(5)
    default: break;
  }
#undef ADGA_BUILD_CASE
}
template void launch_build<float>(const Geom&, int, int, const z64*, const z64*, const z64*, c32*, hipStream_t);
template void launch_build<double>(const Geom&, int, int, const z64*, const z64*, const z64*, z64*, hipStream_t);

// ---------------------------------------------------------------- A7/A8 refinement residuals
// The residual products take their right operand row-major, one N x (npts n2) plane per channel:
// Z_ch[x][b*n2 + s] = sum_c' S_b[d][c'][i'] V[2b + ch][d*n2 + c'][s]  (x = d*n2 + i'), i.e.
// Z = blockdiag(S)^T V with the points side by side, V = Y (a solution) or, when Y is null,
// V = (1 + gamma^w_ch)^T (k_resid_zt).
// |re| + |im| as an order-preserving integer: a NaN is above every number, so a maximum keeps it
__device__ __forceinline__ unsigned long long abs_bits(z64 v) {
  return (unsigned long long)__double_as_longlong(cabs1(v)) & 0x7fffffffffffffffull;
}
__device__ __forceinline__ unsigned long long umax64(unsigned long long a, unsigned long long b) {
  return a > b ? a : b;
}

// Out[(2b + ch) N + r][s] = sum_x C_ch(x, r) Z_ch[x][b*n2 + s], plus (B - Y) at the same position
// when B is given (the residual), for the rows r >= r0: complex FP64 products by the 3M method (X = Ar Br, Y = Ai Bi,
// Z = (Ar + Ai)(Br + Bi), as gemm3m_tile), C read row-major as A(r, x) = C[r N + x], the output in the
// point-major layout of Y.  With `update` what is stored is Y plus that result (Out may be Y).  With rmax, each
// matrix's max |result| goes there from the output registers (abs_bits, combined per column in LDS), instead of
// a second pass over it.
//
// Bound by the FP64 matrix cores: four waves per workgroup, K staged through two LDS buffers in chunks of
// RG_KC, one barrier per chunk, the next k's fragments loaded ahead of each k's MFMAs, and two (64 x 64 tile,
// 32 x 32 per wave) to four (32 x 32 tile, 16 x 16 per wave) workgroups per CU, so that one's barriers run under
// another's MFMAs.  Two workgroups of a CU tend to run in step, though, and what a wave does between its last MFMA
// of a chunk and the barrier then stands still: the staging and the next loads are issued between MFMAs instead,
// from offsets computed once.  N = 1080, 13500 columns: 3.85 -> 3.43 ms, the matrix cores busy for 73 -> 80% of it
// (6% are the last round of workgroups); N = 4000, 1200 columns 4.36 -> 3.87; N = 2000, 1600 columns (32 x 32)
// 1.30 -> 1.16.  An eight-wave 128 x 64 tile, alone on its CU, is a fifth slower than four waves.
// Workgroup b runs on XCD b % 8; each XCD takes a contiguous eighth of the tiles in an order of RG_GC columns
// by all rows, so that the 64 or 128 resident workgroups of an XCD share their C and Z panels through its L2
// and no XCD holds more than one tile more than another (whole columns per XCD: N = 4000, 1200 columns 5.25
// against 4.26 ms, N = 540, 369 columns 64 against 50 us).
constexpr int RG_KC = 16, RG_GC = 8;
template <int TM, int TN>
__global__ void __launch_bounds__(256, TM == 64 ? 2 : 4)
k_resid_gemm(Geom g, int npts, int ch0, int nch, const z64* __restrict__ cd, const z64* __restrict__ cm,
             const z64* __restrict__ Zall, z64* Out, const z64* __restrict__ B, const z64* Y, int accumulate,
             int update, unsigned long long* __restrict__ rmax, int r0) {
  using V = f64x4;
  constexpr int KC = RG_KC, WR = 2, WC = 2, RB = TM / WR / 16, CB = TN / WC / 16;
  constexpr int LDA = KC + 1, LDB = TN + 8, BUF = TM * LDA + KC * LDB;  // strides without bank conflicts
  constexpr int PA = TM * KC / 256, PB = KC * TN / 256;
  __shared__ __attribute__((aligned(16))) z64 lds[2 * BUF];
  const int N = g.N, n2 = g.n2, ncol = npts * n2;
  const int ntr = (N - r0 + TM - 1) / TM, ntc = (ncol + TN - 1) / TN, per = ntr * ntc, tot = nch * per;
  const int share = (tot + 7) / 8, slot = (int)blockIdx.x >> 3, id = ((int)blockIdx.x & 7) * share + slot;
  if (slot >= share || id >= tot) return;
  const int ch = ch0 + id / per, e0 = id % per, full = ntc / RG_GC * RG_GC;
  const int gw = e0 < full * ntr ? RG_GC : ntc - full;  // columns of this tile's group
  const int gc = e0 < full * ntr ? e0 / (RG_GC * ntr) * RG_GC : full, ge = e0 - gc * ntr;
  const int rt = r0 + ge / gw * TM, ct = (gc + ge % gw) * TN;
  const z64* A = ch == 0 ? cd : cm;
  const z64* Z = Zall + (long)ch * N * ncol;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wr = (wave / WC) * (TM / WR), wc = (wave % WC) * (TN / WC), li = lane & 15, lg = lane >> 4;
  V x[RB][CB], y[RB][CB], z[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) x[rb][cb] = y[rb][cb] = z[rb][cb] = V{0, 0, 0, 0};
  // This thread's elements of a chunk: A(row + 16 i, k = kb + t % KC), Z(k = kb + SB i + t / TN, col), as
  // offsets from a base that all threads share.  Rows and columns beyond the edge are read at the last one:
  // they only enter outputs that are not stored.
  static_assert(PA == PB && PA % 2 == 0 && KC == 16, "two halves of a chunk in two of its four k steps");
  constexpr int SA = 256 / KC, SB = 256 / TN;
  const z64* At = A + (long)rt * N;
  const z64* Zt = Z + ct;
  unsigned oa[PA];  // bytes
#pragma unroll
  for (int i = 0; i < PA; ++i)
    oa[i] = (unsigned)sizeof(z64) * ((unsigned)min(i * SA + t / KC, N - 1 - rt) * (unsigned)N + (unsigned)(t % KC));
  const unsigned ob =
      (unsigned)sizeof(z64) * ((unsigned)(t / TN) * (unsigned)ncol + (unsigned)min(t % TN, ncol - 1 - ct));
  auto ld = [](const z64* base, unsigned off) {
    return *reinterpret_cast<const z64*>(reinterpret_cast<const char*>(base) + off);
  };
  z64 pa[PA], pb[PB];
  auto fetch1 = [&](int kb, int i) {  // elements i of a whole chunk
    pa[i] = ld(At + kb, oa[i]);
    pb[i] = ld(Zt + (long)(kb + i * SB) * ncol, ob);
  };
  auto fetch = [&](int kb) {
    if (kb + KC <= N) {
#pragma unroll
      for (int i = 0; i < PA; ++i) fetch1(kb, i);
      return;
    }
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      pa[i] = kb + t % KC < N ? ld(At + kb, oa[i]) : mk(0.0, 0.0);
      pb[i] = kb + i * SB + t / TN < N ? ld(Zt + (long)(kb + i * SB) * ncol, ob) : mk(0.0, 0.0);
    }
  };
  auto stage1 = [&](int b, int i) {
    z64* As = lds + b * BUF;
    z64* Bs = As + TM * LDA;
    As[(t / KC + i * SA) * LDA + t % KC] = pa[i];
    Bs[(t / TN + i * SB) * LDB + t % TN] = pb[i];
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < PA; ++i) stage1(b, i);
  };
  // the chunk in buffer b; k in [kend, KC) of a last, partial chunk are staged zeros.  With `next` >= 0 the
  // second and third of its four k steps each also write half of the staged chunk to the other buffer and
  // start the loads of the chunk at `next`, between MFMAs.
  auto compute = [&](int b, int kend, auto feed, int next) {
    const z64* Ap = lds + b * BUF + (wr + li) * LDA + lg;
    const z64* Bp = lds + b * BUF + TM * LDA + lg * LDB + wc + li;
    z64 a[2][RB], v[2][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) a[0][rb] = Ap[rb * 16 * LDA];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) v[0][cb] = Bp[cb * 16];
#pragma unroll
    for (int kk = 0; kk < KC; kk += 4) {
      const int p = (kk >> 2) & 1;
      if (kk + 4 < KC) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) a[p ^ 1][rb] = Ap[rb * 16 * LDA + kk + 4];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) v[p ^ 1][cb] = Bp[(kk + 4) * LDB + cb * 16];
      }
      if (kk >= kend) continue;
      double as[RB], vs[CB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) as[rb] = a[p][rb].re + a[p][rb].im;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) vs[cb] = v[p][cb].re + v[p][cb].im;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          x[rb][cb] = Mfma<double>::op(a[p][rb].re, v[p][cb].re, x[rb][cb]);
          y[rb][cb] = Mfma<double>::op(a[p][rb].im, v[p][cb].im, y[rb][cb]);
          z[rb][cb] = Mfma<double>::op(as[rb], vs[cb], z[rb][cb]);
          if constexpr (decltype(feed)::value) {
            constexpr int HALF = PA / 2, PER = RB * CB;
            const int j = rb * CB + cb;
            if (kk == 4 || kk == 8)
#pragma unroll
              for (int i = 0; i < HALF; ++i)
                if (i * PER / HALF == j) {
                  stage1(b ^ 1, (kk / 4 - 1) * HALF + i);
                  fetch1(next, (kk / 4 - 1) * HALF + i);
                }
          }
        }
      if constexpr (decltype(feed)::value) __builtin_amdgcn_sched_barrier(0);
    }
  };
  using Feed = std::integral_constant<bool, true>;
  using Plain = std::integral_constant<bool, false>;
  fetch(0);
  stage(0);
  if (KC < N) fetch(KC);
  __syncthreads();
  int b = 0, kb = 0;
  for (; kb + 3 * KC <= N; kb += KC) {  // a buffer is written after the barrier that ended its reading
    compute(b, KC, Feed{}, kb + 2 * KC);
    __syncthreads();
    b ^= 1;
  }
  for (; kb + KC < N; kb += KC) {
    compute(b, KC, Plain{}, 0);
    stage(b ^ 1);
    if (kb + 2 * KC < N) fetch(kb + 2 * KC);
    __syncthreads();
    b ^= 1;
  }
  auto at = [&](int r, int col) {
    const int pt = col / n2;
    return ((long)(2 * pt + ch) * N + r) * n2 + (col - pt * n2);
  };
  // what is added to the product is loaded beside the last chunk's MFMAs
  const bool add = B != nullptr || accumulate;
  z64 cin[RB][CB][4];
  if (add) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = rt + wr + rb * 16 + Mfma<double>::row(lg, v), col = ct + wc + cb * 16 + li;
          z64 c = mk(0.0, 0.0);
          if (row < N && col < ncol) {
            const long i = at(row, col);
            c = B ? csub(B[i], Y[i]) : Out[i];
          }
          cin[rb][cb][v] = c;
        }
  }
  compute(b, N - kb, Plain{}, 0);
  unsigned long long mx[CB] = {};
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    z64 yv[CB][4];  // Y again, all of a block row's loads before its stores (Out may be Y itself)
    if (update) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = rt + wr + rb * 16 + Mfma<double>::row(lg, v), col = ct + wc + cb * 16 + li;
          yv[cb][v] = row < N && col < ncol ? Y[at(row, col)] : mk(0.0, 0.0);
        }
    }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = rt + wr + rb * 16 + Mfma<double>::row(lg, v), col = ct + wc + cb * 16 + li;
        if (row < N && col < ncol) {
          z64 o = mk(x[rb][cb][v] - y[rb][cb][v], (z[rb][cb][v] - x[rb][cb][v]) - y[rb][cb][v]);
          if (add) o = cadd(cin[rb][cb][v], o);
          mx[cb] = umax64(mx[cb], abs_bits(o));
          Out[at(row, col)] = update ? cadd(yv[cb][v], o) : o;
        }
      }
  }
  if (rmax) {
    __syncthreads();  // the tile's LDS reads are done
    unsigned long long* sm = reinterpret_cast<unsigned long long*>(lds);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      unsigned long long v = mx[cb];
      v = umax64(v, __shfl_xor(v, 16));
      v = umax64(v, __shfl_xor(v, 32));
      if (lane < 16) sm[(wave / WC) * TN + wc + cb * 16 + lane] = v;
    }
    __syncthreads();
    if (t < TN && ct + t < ncol) atomicMax(&rmax[2 * ((ct + t) / n2) + ch], umax64(sm[t], sm[TN + t]));
  }
}

// Out = C_ch^T Z_ch (+ B - Y when B is given, + Out itself when accumulate), rows r0 .. N - 1.  64 x 64 tiles from
// four rounds of the chip's 512 such workgroups on; below, 32 x 32 tiles lose less to the last round and to few
// workgroups.  64 x 64 against 32 x 32, us, columns of both channels: N = 400, 1024 columns (112 tiles of 64 x 64)
// 61 / 35; N = 136, 2408 (114) 34 / 20; N = 540, 9000 (1278) 353 / 312; N = 720, 9000 (1704) 591 / 549; N = 2000, 4500
// (2304) 1899 / 1917; N = 4000, 2400 (2394) 3713 / 4227; N = 960, 12800 (3000) 1166 / 1289.  Between 1200 and 2048
// tiles either wins with how full the last round is: N = 960, 6400 (1500) 589 / 649; N = 2000, 3200 (1600) 1396 / 1355;
// N = 1080, 7200 (1938) 869 / 930.
void resid_gemm(const Geom& g, int npts, int ch0, int nch, const z64* cd, const z64* cm, const z64* Z, z64* Out,
                const z64* B, const z64* Y, hipStream_t s, bool accumulate, unsigned long long* rmax, int r0,
                bool update) {
  auto tiles = [&](int tile) {
    return nch * ((long)(g.N - r0 + tile - 1) / tile) * (((long)npts * g.n2 + tile - 1) / tile);
  };
  auto grid = [](long n) { return dim3((unsigned)((n + 7) / 8 * 8)); };
  if (tiles(64) >= 2048)
    hipLaunchKernelGGL((k_resid_gemm<64, 64>), grid(tiles(64)), dim3(256), 0, s, g, npts, ch0, nch, cd, cm, Z, Out, B,
                       Y, accumulate ? 1 : 0, update ? 1 : 0, rmax, r0);
  else
    hipLaunchKernelGGL((k_resid_gemm<32, 32>), grid(tiles(32)), dim3(256), 0, s, g, npts, ch0, nch, cd, cm, Z, Out, B,
                       Y, accumulate ? 1 : 0, update ? 1 : 0, rmax, r0);
}

// Per-matrix max |A| (|.| = |re|+|im|, abs_bits), one workgroup per matrix; `clear` (may be null) is zeroed.
__global__ void __launch_bounds__(256) k_absmax(long tot, const z64* __restrict__ A,
                                                unsigned long long* __restrict__ out,
                                                unsigned long long* __restrict__ clear) {
  __shared__ unsigned long long sr[4];
  const int m = blockIdx.x, t = threadIdx.x;
  unsigned long long v = 0;
  for (long e = t; e < tot; e += 256) v = umax64(v, abs_bits(A[(long)m * tot + e]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = umax64(v, __shfl_xor(v, o));
  if ((t & 63) == 0) sr[t >> 6] = v;
  __syncthreads();
  if (t == 0) {
    out[m] = umax64(umax64(sr[0], sr[1]), umax64(sr[2], sr[3]));
    if (clear) clear[m] = 0;
  }
}

// rel[m] = max|R| / max|B|, and rmax cleared for the next residual; a zero right-hand side counts as
// converged when the residual is zero too, a NaN in the residual gives NaN.
__global__ void k_resid_rel(int nmat, const unsigned long long* __restrict__ bmax,
                            unsigned long long* __restrict__ rmax, double* __restrict__ rel) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nmat) return;
  const double r = __longlong_as_double((long long)rmax[m]), b = __longlong_as_double((long long)bmax[m]);
  rel[m] = b > 0.0 ? r / b : (r == 0.0 ? 0.0 : INFINITY);
  rmax[m] = 0;
}

// Z = blockdiag(S)^T V with one thread per (channel, d, point b, column s) forming the n2 rows
// x = d*n2 + i' of its column: each thread reads its values of V once, and for each i' the wave writes a
// contiguous run of Z's row x (consecutive lanes hold consecutive columns b*n2 + s).  V by `mode`: Z_OPG
// (1 + gamma^w)^T, Z_Y the solution, Z_ADD Y + R with the sum stored to Y (a step of the fixed-point
// iteration: every element of Y belongs to one thread), Z_RHS B (its start; stored to Y unless that is null).
enum { Z_OPG = 0, Z_Y = 1, Z_ADD = 2, Z_RHS = 3 };
template <int N2>
__global__ void __launch_bounds__(256) k_resid_zt(Geom g, int npts, int mode, const z64* __restrict__ S,
                                                  z64* __restrict__ Y, const z64* __restrict__ R,
                                                  const z64* __restrict__ opg_d, const z64* __restrict__ opg_m,
                                                  z64* __restrict__ Z) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ncol = (long)npts * N2;
  if (idx >= 2L * g.nf * ncol) return;
  const int col = (int)(idx % ncol);
  const int r = (int)(idx / ncol), d = r % g.nf, ch = r / g.nf;
  const int b = col / N2, s = col - b * N2;
  const z64* Sd = S + ((long)b * g.nf + d) * (N2 * N2);
  z64 v[N2];
  if (mode == Z_OPG) {
    const z64* opg = ch == 0 ? opg_d : opg_m;
#pragma unroll
    for (int cp = 0; cp < N2; ++cp) v[cp] = opg[s + (long)(d * N2 + cp) * N2];
  } else {
    const long o = (long)(2 * b + ch) * g.N * N2 + (long)d * N2 * N2 + s;
    const z64* src = mode == Z_RHS ? R : Y;
#pragma unroll
    for (int cp = 0; cp < N2; ++cp) v[cp] = src[o + cp * N2];
    if (mode == Z_ADD) {
#pragma unroll
      for (int cp = 0; cp < N2; ++cp) v[cp] = cadd(v[cp], R[o + cp * N2]);
    }
    if (mode == Z_ADD || (mode == Z_RHS && Y)) {
#pragma unroll
      for (int cp = 0; cp < N2; ++cp) Y[o + cp * N2] = v[cp];
    }
  }
  z64* Zc = Z + ((long)ch * g.N + (long)d * N2) * ncol + col;
#pragma unroll
  for (int ip = 0; ip < N2; ++ip) {
    z64 acc = mk(0.0, 0.0);
#pragma unroll
    for (int cp = 0; cp < N2; ++cp) acc = cfma(Sd[cp * N2 + ip], v[cp], acc);
    Zc[(long)ip * ncol] = acc;
  }
}

// Zg[d*n2 + i'][b*n2 + s] = S_b[d][s][i'] (the channel-0 plane of the residual product's right
// operand), so that C^T Zg (k_resid_gemm) is
// gamma^q_d(s, r) = sum_d sum_i' S_b[d][s][i'] C_d(d*n2 + i', r) = sum_nu chi0^{nl,q} F^w_d
// (main.F90:693-700, the accumulation of rectanglework over nu); threads as in k_resid_zt.
template <int N2>
__global__ void __launch_bounds__(256) k_gamq_zt(Geom g, int npts, const z64* __restrict__ S, z64* __restrict__ Z) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ncol = (long)npts * N2;
  if (idx >= (long)g.nf * ncol) return;
  const int col = (int)(idx % ncol), d = (int)(idx / ncol);
  const int b = col / N2, s = col - b * N2;
  const z64* Sd = S + ((long)b * g.nf + d) * (N2 * N2) + s * N2;
  z64* Zc = Z + (long)d * N2 * ncol + col;
#pragma unroll
  for (int ip = 0; ip < N2; ++ip) Zc[(long)ip * ncol] = Sd[ip];
}

static void resid_z(const Geom& g, int npts, int mode, const z64* S, z64* Y, const z64* R, const z64* opgd,
                    const z64* opgm, z64* Z, hipStream_t s) {
  const long tz = 2L * g.nf * npts * g.n2;
#define ADGA_RZ(NN)                                                                                                 \
  case NN:                                                                                                         \
    hipLaunchKernelGGL(k_resid_zt<NN * NN>, dim3((unsigned)((tz + 255) / 256)), dim3(256), 0, s, g, npts, mode, S, \
                       Y, R, opgd, opgm, Z);                                                                       \
    break;
  switch (g.n) {
    ADGA_RZ(1) ADGA_RZ(2) ADGA_RZ(3) ADGA_RZ(4) ADGA_RZ(5)
    default: break;
  }
#undef ADGA_RZ
}

void launch_gamq_z(const Geom& g, int npts, const z64* S, z64* Z, hipStream_t s) {
  const long tz = (long)g.nf * npts * g.n2;
#define ADGA_GZ(NN)                                                                                                 \
  case NN:                                                                                                         \
    hipLaunchKernelGGL(k_gamq_zt<NN * NN>, dim3((unsigned)((tz + 255) / 256)), dim3(256), 0, s, g, npts, S, Z);     \
    break;
  switch (g.n) {
    ADGA_GZ(1) ADGA_GZ(2) ADGA_GZ(3) ADGA_GZ(4) ADGA_GZ(5)
    default: break;
  }
#undef ADGA_GZ
}

// gamma^q_d for every point of the batch, into G2 with the residual layout (point b at 2*b).  The EOM, which
// alone reads it, sums over nu >= 0 (eom_row0): half the rows, half the product.
void launch_gamq(const Geom& g, int npts, const z64* S, const z64* cd, z64* Z, z64* G2, hipStream_t s) {
  launch_gamq_z(g, npts, S, Z, s);
  resid_gemm(g, npts, 0, 1, cd, cd, Z, G2, nullptr, nullptr, s, false, nullptr, eom_row0(g));
}

// Right-hand side of the eta system: eta A = (1+gamma^w)(1 - A) = (1+gamma^w) blockdiag(S) C, i.e.
// B = M eta^T with B = C^T (blockdiag(S)^T (1+gamma^w)^T), in FP64; with V(q) the density channel adds
// (1+gamma^w_d)^T (W^T (1+gamma^w_d)^T).
void launch_rhs(const Geom& g, int npts, const z64* S, const z64* cd, const z64* cm, const z64* opgd,
                const z64* opgm, z64* Z, z64* B, hipStream_t s, const VqTerm* vq) {
  resid_z(g, npts, Z_OPG, S, nullptr, nullptr, opgd, opgm, Z, s);
  resid_gemm(g, npts, 0, 2, cd, cm, Z, B, nullptr, nullptr, s);
  if (vq) launch_vq_add(g, npts, *vq, nullptr, B, s);
}

void launch_absmax_rhs(const Geom& g, int npts, const z64* B, const ResidNorm& nrm, hipStream_t s) {
  hipLaunchKernelGGL(k_absmax, dim3(2 * npts), dim3(256), 0, s, (long)g.N * g.n2, B, nrm.bmax, nrm.rmax);
}

__global__ void k_add(long n, const z64* __restrict__ R, z64* __restrict__ Y) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) Y[i] = cadd(Y[i], R[i]);
}

void launch_add(long n, const z64* R, z64* Y, hipStream_t s) {
  hipLaunchKernelGGL(k_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, R, Y);
}

// R = B - M Y with M Y = Y - C^T (blockdiag(S)^T Y), in FP64 from the unrounded factors S and C (with V(q):
// minus (1 + gamma^w_d)^T (W^T Y) in the density channel), and with `norm` its norms.  M = 1 - T with
// T Y = C^T (blockdiag(S)^T Y), so steps Y += R from Y = B sum the series (1 + T + T^2 + ...) B.
//   RESID_OF     of Y as given, stored to R
//   RESID_START  of Y = B, RESID_STEP of the last call's Y + R, for the fixed-point iteration: without V(q) the
//                product stores Y + R over Y at once and R nowhere, five passes over a solution's array a step
//                (B, Y, Y + R, and Y, Z of the next operand) where R stored, added as the next operand is
//                formed and by a kernel of its own at the end took eight and three more; with V(q), whose term
//                is added to R by kernels after the product, the next call adds R (resid_step_pending).
bool resid_step_pending(const VqTerm* vq) { return vq != nullptr; }

void launch_residual(const Geom& g, int npts, const z64* S, const z64* cd, const z64* cm, const z64* B, z64* Y,
                     z64* Z, z64* R, const ResidNorm& nrm, hipStream_t s, const VqTerm* vq, ResidMode mode,
                     LuTimer* timer, bool norm) {
  const int nmat = 2 * npts;
  const bool start = mode == RESID_START, update = mode != RESID_OF && !resid_step_pending(vq);
  if (start)
    resid_z(g, npts, Z_RHS, S, update ? nullptr : Y, B, nullptr, nullptr, Z, s);
  else
    resid_z(g, npts, mode == RESID_STEP && !update ? Z_ADD : Z_Y, S, Y, R, nullptr, nullptr, Z, s);
  if (timer) {
    timer->mark(s);
    timer->flops += 8.0 * g.N * (double)g.N * g.n2 * nmat;
  }
  resid_gemm(g, npts, 0, 2, cd, cm, Z, update ? Y : R, B, update && start ? B : Y, s, false,
             norm && !vq ? nrm.rmax : nullptr, 0, update);
  if (timer) timer->mark(s);
  if (vq) {
    launch_vq_add(g, npts, *vq, Y, R, s);
    if (norm) hipLaunchKernelGGL(k_absmax, dim3(nmat), dim3(256), 0, s, (long)g.N * g.n2, R, nrm.rmax, nullptr);
  }
  if (norm)
    hipLaunchKernelGGL(k_resid_rel, dim3((nmat + 255) / 256), dim3(256), 0, s, nmat, nrm.bmax, nrm.rmax, nrm.rel);
}

}  // namespace adga
