// A8 (eta), A9 (chi contraction), A10 (dynamic EOM), A11 (local/static EOM) on gfx950.
#include <algorithm>

#include "adga_kernels.h"
#include "mfma_gemm.h"

namespace adga {

// eta_m(s, x) = Y[m][x][s]: Y = eta^T solves A^T eta^T = B (main.F90:740-757), and the solutions' layout
// (one N x n2 row-major block per matrix) is eta's Fortran (n2, N) layout, so the kernels below read
// eta from Y itself.

// chi_ch(q) (non-local part) = beta^-2 gamma^w_ch . (chi0^q - chi0^w) + beta^-2 eta_ch . chi0^q, where
// (X . Y)(s, s2) = sum_{d, i3} X(s, d*n2 + i3) Y(i3, s2, d)  (susc_module.f90:34-56, main.F90:666-769);
// bubble_nl(q) = sum_d chi0^q / beta^2 - sum_d chi0^w / beta^2  (main.F90:654-663).
//
// A form g . (c - w) + e . c is that with c = chi0^q of each point, w = chi0^w, g per channel and e per channel
// and point; the derivative of chi is the sum of two (product rule): (dg, de, c, w) and (g, e, dc, dw).
//
// One workgroup per point and slice of frequencies, for n >= 3: both factors of each product are loaded as they
// lie, every element into one lane of a matrix fragment, where threads that each form outputs load them n2 times
// over and are bound by the L1 cache (a thread per row and slice: three orbitals, 120 frequencies, 1500 points
// 0.69 ms, 0.33 here; a thread per output: five orbitals, 160 frequencies, 48 points 2.15 ms, 0.15 here; the
// derivative with three, 80 frequencies, 500 points 0.70 ms, 0.16 here).  Now bound by the loads of c and e
// (0.70 GB in the first, 2.1 TB/s).  Four waves take every fourth step of four x = d n2 + i3, are added in
// LDS in a fixed order, and the slices' sums by k_chi_sum.
struct ChiForm {
  const z64 *c, *w, *gd, *gm, *e;
};
template <int NT>
struct ChiForms {
  ChiForm f[NT];
};
template <int N2, int NT>
__global__ void __launch_bounds__(256) k_chi_mm(Geom g, int slices, ChiForms<NT> fs, z64* __restrict__ part) {
  constexpr int N4 = N2 * N2, T = (N2 + 15) / 16;
  __shared__ z64 sum[4][2 * N4];
  const int b = blockIdx.x, sl = blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int d0 = (int)((long)g.nf * sl / slices), d1 = (int)((long)g.nf * (sl + 1) / slices);
  const int x0 = d0 * N2, x1 = d1 * N2;
  f64x4 re[2][T][T], im[2][T][T];
#pragma unroll
  for (int ch = 0; ch < 2; ++ch)
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int q = 0; q < T; ++q) re[ch][r][q] = im[ch][r][q] = f64x4{0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    const ChiForm f = fs.f[k];
    const z64* cq = f.c + (long)b * g.nf * N4;
    const z64* eb = f.e + (long)(2 * b) * g.N * N2;
    for (int xs = x0 + 4 * wave; xs < x1; xs += 16) {
      const int x = xs + lg, d = x / N2, i3 = x - d * N2;
      const bool in = x < x1;
      z64 c[T], n[T], a[2][2][T];  // c, c - w; g and e of the two channels
#pragma unroll
      for (int q = 0; q < T; ++q) {
        const int s2 = q * 16 + li;
        const bool ok = in && s2 < N2;
        c[q] = ok ? cq[(long)d * N4 + i3 + s2 * N2] : mk(0.0, 0.0);
        n[q] = ok && s2 == i3 ? csub(c[q], f.w[x]) : c[q];
      }
#pragma unroll
      for (int r = 0; r < T; ++r) {
        const int s = r * 16 + li;
        const bool ok = in && s < N2;
        const long o = (long)x * N2 + s;
        a[0][0][r] = ok ? f.gd[o] : mk(0.0, 0.0);
        a[0][1][r] = ok ? eb[o] : mk(0.0, 0.0);
        a[1][0][r] = ok ? f.gm[o] : mk(0.0, 0.0);
        a[1][1][r] = ok ? eb[(long)g.N * N2 + o] : mk(0.0, 0.0);
      }
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int r = 0; r < T; ++r)
#pragma unroll
            for (int q = 0; q < T; ++q) {
              const z64 u = a[ch][p][r], v = p == 0 ? n[q] : c[q];
              re[ch][r][q] = Mfma<double>::op(u.re, v.re, re[ch][r][q]);
              im[ch][r][q] = Mfma<double>::op(u.re, v.im, im[ch][r][q]);
              re[ch][r][q] = Mfma<double>::op(-u.im, v.im, re[ch][r][q]);
              im[ch][r][q] = Mfma<double>::op(u.im, v.re, im[ch][r][q]);
            }
    }
  }
#pragma unroll
  for (int ch = 0; ch < 2; ++ch)
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int q = 0; q < T; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int s = r * 16 + Mfma<double>::row(lg, v), s2 = q * 16 + li;
          if (s < N2 && s2 < N2) sum[wave][ch * N4 + s + s2 * N2] = mk(re[ch][r][q][v], im[ch][r][q][v]);
        }
  __syncthreads();
  z64* out = part + ((long)b * slices + sl) * (3 * N4);
  for (int e = t; e < 2 * N4; e += 256)
    out[e] = cadd(cadd(sum[0][e], sum[1][e]), cadd(sum[2][e], sum[3][e]));
  const ChiForm f = fs.f[NT - 1];  // its c summed over the frequencies; of a derivative, minus its w
  const z64* cq = f.c + (long)b * g.nf * N4;
  for (int e = t; e < N4; e += 256) {
    z64 bs = mk(0.0, 0.0);
#pragma unroll 4
    for (int d = d0; d < d1; ++d) {
      z64 v = cq[(long)d * N4 + e];
      if (NT == 2 && e / N2 == e % N2) v = csub(v, f.w[d * N2 + e % N2]);
      bs = cadd(bs, v);
    }
    out[2 * N4 + e] = bs;
  }
}

// The slices' sums in order, over beta^2: chi_out (channel, n4) per point, and bub_out, less bubloc if given.
__global__ void __launch_bounds__(256) k_chi_sum(Geom g, int npts, int slices, const z64* __restrict__ part,
                                                 const z64* __restrict__ bubloc, z64* __restrict__ chi_out,
                                                 z64* __restrict__ bub_out) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int per = 3 * g.n4;
  if (idx >= (long)npts * per) return;
  const int b = (int)(idx / per), e = (int)(idx - (long)b * per);
  const z64* p = part + (long)b * slices * per + e;
  z64 v = p[0];
  for (int k = 1; k < slices; ++k) v = cadd(v, p[(long)k * per]);
  v = cscale(v, 1.0 / (g.beta * g.beta));
  if (e < 2 * g.n4) {
    chi_out[(long)b * 2 * g.n4 + e] = v;
  } else {
    const int f = e - 2 * g.n4;
    bub_out[(long)b * g.n4 + f] = bubloc ? csub(v, bubloc[f]) : v;
  }
}

// Slices until 2048 workgroups are in flight, of eight frequencies or more; `part` (3 n4 values per point and
// slice) fits a solution's array of 2 n4 per point and frequency.
template <int NT>
static bool chi_mm(const Geom& g, int npts, const ChiForms<NT>& fs, z64* part, const z64* bubloc, z64* chi_out,
                   z64* bub_out, hipStream_t s) {
  const int slices = std::max(1, std::min((2047 + npts) / npts, g.nf / 8));
  const dim3 grid((unsigned)npts, (unsigned)slices);
  switch (g.n) {
    case 3: hipLaunchKernelGGL((k_chi_mm<9, NT>), grid, dim3(256), 0, s, g, slices, fs, part); break;
    case 4: hipLaunchKernelGGL((k_chi_mm<16, NT>), grid, dim3(256), 0, s, g, slices, fs, part); break;
    case 5: hipLaunchKernelGGL((k_chi_mm<25, NT>), grid, dim3(256), 0, s, g, slices, fs, part); break;
    default: return false;
  }
  const long tot = (long)npts * 3 * g.n4;
  hipLaunchKernelGGL(k_chi_sum, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, g, npts, slices, part, bubloc,
                     chi_out, bub_out);
  return true;
}

bool launch_dchi_mm(const Geom& g, int npts, const z64* chi0q, const z64* dchi0q, const z64* chi0w, const z64* dchi0w,
                    const z64* gamd, const z64* gamm, const z64* dgamd, const z64* dgamm, const z64* Y, const z64* dY,
                    z64* part, z64* dchi_out, z64* dbub_out, hipStream_t s) {
  return chi_mm<2>(g, npts, {{{chi0q, chi0w, dgamd, dgamm, dY}, {dchi0q, dchi0w, gamd, gamm, Y}}}, part, nullptr,
                   dchi_out, dbub_out, s);
}

// The same for n <= 2, whose n2 values fill little of a matrix fragment, with one workgroup per point: thread (k
// slice, channel, row s) accumulates row s of chi_ch over its slice of x = d*n2 + i3 (the n2 values of chi0^q at one
// x are read by every thread of the slice), the slices are summed through LDS, and threads 0 .. n4-1 form bubble_nl (summed over d in order).
template <int N2>
__global__ void __launch_bounds__(256) k_chi_wg(Geom g, const z64* __restrict__ chi0q, const z64* __restrict__ chi0w,
                                                const z64* __restrict__ gam_d, const z64* __restrict__ gam_m,
                                                const z64* __restrict__ eta, const z64* __restrict__ bubloc,
                                                z64* __restrict__ chi_out, z64* __restrict__ bub_out) {
  constexpr int N4 = N2 * N2, KS = 256 / (2 * N2);
  __shared__ z64 part[KS][2][N4];
  const int b = blockIdx.x, t = threadIdx.x;
  const int ks = t / (2 * N2), ch = (t % (2 * N2)) / N2, s = t % N2;
  const int N = g.N;
  const z64* cq = chi0q + (long)b * g.nf * N4;
  if (ks < KS) {
    const z64* gam = ch == 0 ? gam_d : gam_m;
    const z64* et = eta + (long)(2 * b + ch) * N2 * N;
    z64 acc[N2];
#pragma unroll
    for (int s2 = 0; s2 < N2; ++s2) acc[s2] = mk(0.0, 0.0);
    const int x0 = (int)((long)N * ks / KS), x1 = (int)((long)N * (ks + 1) / KS);
#pragma unroll 2
    for (int x = x0; x < x1; ++x) {
      const int d = x / N2, i3 = x % N2;
      const z64 gv = gam[s + (long)x * N2], ev = et[s + (long)x * N2];
      const z64 w = chi0w[i3 + d * N2];  // chi0^w enters chi0^q - chi0^w where s2 == i3
      const z64* cx = cq + (long)d * N4 + i3;
#pragma unroll
      for (int s2 = 0; s2 < N2; ++s2) {
        const z64 c = cx[s2 * N2];
        acc[s2] = cfma(gv, s2 == i3 ? csub(c, w) : c, acc[s2]);
        acc[s2] = cfma(ev, c, acc[s2]);
      }
    }
#pragma unroll
    for (int s2 = 0; s2 < N2; ++s2) part[ks][ch][s + s2 * N2] = acc[s2];
  }
  __syncthreads();
  const double ib2 = 1.0 / (g.beta * g.beta);
  for (int e = t; e < 2 * N4; e += 256) {
    const int c2 = e / N4, f = e % N4;
    z64 v = mk(0.0, 0.0);
    for (int k = 0; k < KS; ++k) v = cadd(v, part[k][c2][f]);
    chi_out[((long)b * 2 + c2) * N4 + f] = cscale(v, ib2);
  }
  for (int e = t; e < N4; e += 256) {
    z64 bs = mk(0.0, 0.0);
#pragma unroll 8
    for (int d = 0; d < g.nf; ++d) bs = cadd(bs, cq[(long)d * N4 + e]);
    bub_out[(long)b * N4 + e] = csub(cscale(bs, ib2), bubloc[e]);
  }
}

// m_tot = -(U + V - U~/2) eta_d /(beta nqp) + 1.5 U~ eta_m /(beta nqp) + U gamma^q_d /(beta nqp)
//        - V gamma^w_d /(beta nqp)   (eom_module.f90:183-207; the V terms only with V(q): vq non-null).
// Output (n2, N) Fortran per point, the half nu >= 0 that the EOM sums over.
__global__ void k_mtot(Geom g, int npts, const z64* __restrict__ u, const z64* __restrict__ ut,
                       const z64* __restrict__ eta, const z64* __restrict__ gamq, z64* __restrict__ mt,
                       const int* __restrict__ qpos, const z64* __restrict__ vq, const z64* __restrict__ gamd,
                       int accumulate) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)g.n2 * g.N, half = per / 2;
  if (idx >= half * npts) return;
  int b = (int)(idx / half);
  long e = half + idx % half;
  int s = (int)(e % g.n2);
  long x = e / g.n2;
  const z64* ed = eta + (long)(2 * b) * per;
  const z64* em = eta + (long)(2 * b + 1) * per;
  const z64* gq = gamq + (long)(2 * b) * per;  // residual layout: point b at slot 2b
  const z64* v = vq ? vq + (long)qpos[b] * g.n4 : nullptr;
  z64 t1 = mk(0.0, 0.0), t2 = mk(0.0, 0.0), t3 = mk(0.0, 0.0), t4 = mk(0.0, 0.0);
  for (int a = 0; a < g.n2; ++a) {
    z64 uu = u[s + a * g.n2], uw = ut[s + a * g.n2];
    z64 uwork = mk(uu.re - 0.5 * uw.re, uu.im - 0.5 * uw.im);
    if (v) {
      const z64 va = v[s + a * g.n2];
      uwork = cadd(va, uwork);
      t4 = cfma(va, gamd[a + x * g.n2], t4);
    }
    t1 = cfma(uwork, ed[a + x * g.n2], t1);
    t2 = cfma(uw, em[a + x * g.n2], t2);
    t3 = cfma(uu, gq[a + x * g.n2], t3);
  }
  double a1 = -1.0 / g.beta / g.nqp, a2 = 1.5 / g.beta / g.nqp, a3 = 1.0 / g.beta / g.nqp;
  z64 m = cscale(t1, a1);
  m = cadd(cscale(t2, a2), m);
  m = cadd(cscale(t3, a3), m);
  if (v) m = cadd(cscale(t4, a1), m);
  z64* out = mt + b * per + e;
  *out = accumulate ? cadd(*out, m) : m;
}

// Sigma_nl(i, l, nu, k) += sum_b sum_{j,k'} m_b(i*n + j, n2*(iwf + nu) + l*n + k') G(k - q_b, nu - omega)_{jk'}
// for nu = 0 .. iwf-1 (eom_module.f90:211-227).  One thread per (i, l, nu, k); the batch is summed
// in a fixed order, so the accumulation is deterministic.
__global__ void __launch_bounds__(256) k_eom(Geom g, int iwb, int npts, const int* __restrict__ qidx,
                                             const int* __restrict__ keom, const z64* __restrict__ mt,
                                             const z64* __restrict__ gt, z64* __restrict__ sigma) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int half = g.iwf;
  if (idx >= (long)g.n2 * half * g.nkp_eom) return;
  int il = (int)(idx % g.n2);
  int nu = (int)((idx / g.n2) % half);
  int kk = (int)(idx / ((long)g.n2 * half));
  int i = il % g.n, l = il / g.n;
  int k = keom[kk] - 1;
  const z64* gw = gt + (long)(nu - iwb - g.glo) * g.nkp * g.n2;
  long col0 = (long)g.n2 * (g.iwf + nu) + l * g.n;
  long per = (long)g.n2 * g.N;
  z64 acc = mk(0.0, 0.0);
  for (int b = 0; b < npts; ++b) {
    int kq = k_minus_q(k, qidx[b], g.nkx, g.nky, g.nkz);
    const z64* gr = gw + (long)kq * g.n2;
    const z64* m = mt + (long)b * per;
    for (int j = 0; j < g.n; ++j)
      for (int kp = 0; kp < g.n; ++kp) acc = cfma(m[(i * g.n + j) + (col0 + kp) * g.n2], gr[j * g.n + kp], acc);
  }
  long o = i + (long)l * g.n + (long)(g.iws + nu) * g.n2 + (long)kk * g.n2 * (2 * g.iws);
  sigma[o] = cadd(sigma[o], acc);
}

// Sigma(i, l, -nu-1) = conj(Sigma(l, i, nu)) for nu >= 0 (eom_module.f90:157, 228); nk slices.
__global__ void k_fill_neg(Geom g, int nk, z64* __restrict__ sigma) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)g.n2 * g.iws * nk) return;
  int il = (int)(idx % g.n2);
  int nu = (int)((idx / g.n2) % g.iws);
  long kk = idx / ((long)g.n2 * g.iws);
  int i = il % g.n, l = il / g.n;
  long base = kk * g.n2 * (2 * g.iws);
  z64 v = sigma[base + l + (long)i * g.n + (long)(g.iws + nu) * g.n2];
  sigma[base + i + (long)l * g.n + (long)(g.iws - nu - 1) * g.n2] = cconj(v);
}

// Local EOM with the DMFT g: Sigma_dmft(i, l, nu) += sum_k m(i*n + k, n2*(iwf+nu) + l*n + k) g_k(nu - omega),
// m = -(1/beta) U gamma^w_d (eom_module.f90:137-158, default branch).
__global__ void k_eom_dmft(Geom g, int iwb, const z64* __restrict__ u, const z64* __restrict__ gam_d,
                           const z64* __restrict__ giw, z64* __restrict__ sdmft) {
  int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= g.n2 * g.iwf) return;
  int il = idx % g.n2, nu = idx / g.n2;
  int i = il % g.n, l = il / g.n;
  long col0 = (long)g.n2 * (g.iwf + nu) + l * g.n;
  z64 acc = mk(0.0, 0.0);
  for (int k = 0; k < g.n; ++k) {
    int a = i * g.n + k;
    z64 t = mk(0.0, 0.0);
    for (int ap = 0; ap < g.n2; ++ap) t = cfma(u[a + ap * g.n2], gam_d[ap + (col0 + k) * g.n2], t);
    z64 m = cscale(t, -1.0 / g.beta);
    z64 gl = giw[(nu - iwb + g.iwmax) + (long)k * 2 * g.iwmax];
    acc = cfma(m, gl, acc);
  }
  long o = i + (long)l * g.n + (long)(g.iws + nu) * g.n2;
  sdmft[o] = cadd(sdmft[o], acc);
}

// Local Hartree term sum_j (2 u({ii},{jj}) - u({ji},{ji})) n_j added to every frequency
// (eom_module.f90:58-70).
__global__ void k_eom_static(Geom g, const z64* __restrict__ u, const z64* __restrict__ ndmft,
                             z64* __restrict__ sdmft) {
  int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= g.n * 2 * g.iws) return;
  int i = idx % g.n, nu = idx / g.n;
  z64 acc = mk(0.0, 0.0);
  for (int j = 0; j < g.n; ++j) {
    z64 a = u[(i * g.n + i) + (long)(j * g.n + j) * g.n2];
    z64 b = u[(i * g.n + j) + (long)(i * g.n + j) * g.n2];
    acc = cfma(mk(2.0 * a.re - b.re, 2.0 * a.im - b.im), ndmft[j], acc);
  }
  long o = i + (long)i * g.n + (long)nu * g.n2;
  sdmft[o] = cadd(sdmft[o], acc);
}

void launch_chi(const Geom& g, int npts, const z64* eta, const z64* chi0q, const z64* chi0w, const z64* gamd,
                const z64* gamm, const z64* bubloc, z64* part, z64* chi_out, z64* bub_out, hipStream_t s) {
#define ADGA_CHI_WG(NN)                                                                                          \
  if (g.n == NN) {                                                                                              \
    hipLaunchKernelGGL(k_chi_wg<NN * NN>, dim3((unsigned)npts), dim3(256), 0, s, g, chi0q, chi0w, gamd, gamm, eta, \
                       bubloc, chi_out, bub_out);                                                               \
    return;                                                                                                     \
  }
  ADGA_CHI_WG(1) ADGA_CHI_WG(2)
#undef ADGA_CHI_WG
  chi_mm<1>(g, npts, {{{chi0q, chi0w, gamd, gamm, eta}}}, part, bubloc, chi_out, bub_out, s);
}

// k_mtot for n <= 3 with one thread per (point b, x) forming the n2 values s of its row: eta_d, eta_m and
// gamma^q_d at x (and gamma^w_d with V(q)) are read once per thread instead of once per output; the same
// sums in the same order as k_mtot.
template <int N2, bool VQ>
__global__ void __launch_bounds__(256) k_mtot_t(Geom g, int npts, const z64* __restrict__ u,
                                                const z64* __restrict__ ut, const z64* __restrict__ eta,
                                                const z64* __restrict__ gamq, z64* __restrict__ mt,
                                                const int* __restrict__ qpos, const z64* __restrict__ vq,
                                                const z64* __restrict__ gamd, int accumulate) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int half = g.N / 2;
  if (idx >= (long)npts * half) return;
  const int b = (int)(idx / half), x = half + (int)(idx - (long)b * half);
  const long per = (long)N2 * g.N;
  const z64* ed = eta + (long)(2 * b) * per + (long)x * N2;
  const z64* em = eta + (long)(2 * b + 1) * per + (long)x * N2;
  const z64* gq = gamq + (long)(2 * b) * per + (long)x * N2;  // residual layout: point b at slot 2b
  z64 e_d[N2], e_m[N2], g_q[N2], g_d[VQ ? N2 : 1];
#pragma unroll
  for (int a = 0; a < N2; ++a) {
    e_d[a] = ed[a];
    e_m[a] = em[a];
    g_q[a] = gq[a];
    if constexpr (VQ) g_d[a] = gamd[a + (long)x * N2];
  }
  const z64* v = VQ ? vq + (long)qpos[b] * (N2 * N2) : nullptr;
  const double a1 = -1.0 / g.beta / g.nqp, a2 = 1.5 / g.beta / g.nqp, a3 = 1.0 / g.beta / g.nqp;
  z64* out = mt + (long)b * per + (long)x * N2;
#pragma unroll
  for (int s = 0; s < N2; ++s) {
    z64 t1 = mk(0.0, 0.0), t2 = mk(0.0, 0.0), t3 = mk(0.0, 0.0), t4 = mk(0.0, 0.0);
#pragma unroll
    for (int a = 0; a < N2; ++a) {
      const z64 uu = u[s + a * N2], uw = ut[s + a * N2];
      z64 uwork = mk(uu.re - 0.5 * uw.re, uu.im - 0.5 * uw.im);
      if constexpr (VQ) {
        const z64 va = v[s + a * N2];
        uwork = cadd(va, uwork);
        t4 = cfma(va, g_d[a], t4);
      }
      t1 = cfma(uwork, e_d[a], t1);
      t2 = cfma(uw, e_m[a], t2);
      t3 = cfma(uu, g_q[a], t3);
    }
    z64 m = cscale(t1, a1);
    m = cadd(cscale(t2, a2), m);
    m = cadd(cscale(t3, a3), m);
    if constexpr (VQ) m = cadd(cscale(t4, a1), m);
    out[s] = accumulate ? cadd(out[s], m) : m;
  }
}

void launch_mtot(const Geom& g, int npts, const z64* u, const z64* ut, const z64* eta, const z64* gamq, z64* mt,
                 hipStream_t s, const int* qpos, const z64* vq, const z64* gamd, bool accumulate) {
  const long tx = (long)npts * (g.N / 2);
#define ADGA_MT(NN)                                                                                                 \
  if (g.n == NN) {                                                                                                 \
    if (vq)                                                                                                        \
      hipLaunchKernelGGL((k_mtot_t<NN * NN, true>), dim3((unsigned)((tx + 255) / 256)), dim3(256), 0, s, g, npts,  \
                         u, ut, eta, gamq, mt, qpos, vq, gamd, accumulate ? 1 : 0);                                 \
    else                                                                                                           \
      hipLaunchKernelGGL((k_mtot_t<NN * NN, false>), dim3((unsigned)((tx + 255) / 256)), dim3(256), 0, s, g, npts, \
                         u, ut, eta, gamq, mt, qpos, vq, gamd, accumulate ? 1 : 0);                                 \
    return;                                                                                                        \
  }
  ADGA_MT(1) ADGA_MT(2) ADGA_MT(3)
#undef ADGA_MT
  long tot = (long)npts * g.n2 * (g.N / 2);
  hipLaunchKernelGGL(k_mtot, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, g, npts, u, ut, eta, gamq, mt,
                     qpos, vq, gamd, accumulate ? 1 : 0);
}

void launch_eom_direct(const Geom& g, int iwb, int npts, const int* qidx, const int* keom, const z64* mt,
                       const z64* gt, z64* sigma, hipStream_t s) {
  long te = (long)g.n2 * g.iwf * g.nkp_eom;
  hipLaunchKernelGGL(k_eom, dim3((unsigned)((te + 255) / 256)), dim3(256), 0, s, g, iwb, npts, qidx, keom, mt, gt,
                     sigma);
}

void launch_eom_static_local(const Geom& g, const z64* u, const z64* ndmft, z64* sdmft, hipStream_t s) {
  hipLaunchKernelGGL(k_eom_static, dim3((g.n * 2 * g.iws + 63) / 64), dim3(64), 0, s, g, u, ndmft, sdmft);
}

void launch_eom_local(const Geom& g, int iwb, bool do_static, const z64* u, const z64* gamd, const z64* giw,
                      const z64* ndmft, z64* sdmft, hipStream_t s) {
  if (do_static)
    hipLaunchKernelGGL(k_eom_static, dim3((g.n * 2 * g.iws + 63) / 64), dim3(64), 0, s, g, u, ndmft, sdmft);
  hipLaunchKernelGGL(k_eom_dmft, dim3((g.n2 * g.iwf + 63) / 64), dim3(64), 0, s, g, iwb, u, gamd, giw, sdmft);
  hipLaunchKernelGGL(k_fill_neg, dim3((g.n2 * g.iws + 63) / 64), dim3(64), 0, s, g, 1, sdmft);
}

__global__ void k_zero_points(int npts, long len, const int* __restrict__ keep, z64* __restrict__ a) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)npts * len) return;
  if (!keep[idx / len]) a[idx] = mk(0.0, 0.0);
}

void launch_zero_points(int npts, long len, const int* keep, z64* a, hipStream_t s) {
  const long tot = (long)npts * len;
  if (tot > 0)
    hipLaunchKernelGGL(k_zero_points, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, npts, len, keep, a);
}

__global__ void k_gather(int k, long len, const int* __restrict__ sel, const z64* __restrict__ src,
                         z64* __restrict__ dst, int scatter) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)k * len) return;
  const long i = idx / len, e = idx % len;
  const long far = (long)sel[i] * len + e;
  if (scatter) dst[far] = src[idx];
  else dst[idx] = src[far];
}

void launch_gather(int k, long len, const int* sel, const z64* src, z64* dst, bool scatter, hipStream_t s) {
  const long tot = (long)k * len;
  if (tot > 0)
    hipLaunchKernelGGL(k_gather, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, k, len, sel, src, dst,
                       scatter ? 1 : 0);
}

void launch_fill_neg(const Geom& g, int nk, z64* sigma, hipStream_t s) {
  long tot = (long)g.n2 * g.iws * nk;
  hipLaunchKernelGGL(k_fill_neg, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, g, nk, sigma);
}

}  // namespace adga
