// One-particle routines around the per-(q,omega) loop (one_particle_quant_module.f90) on gfx950:
// get_giw (40-79), get_nfock (337-361), get_sigma_g_loc (124-180) and get_ndga (363-393).  Each is
// a sum of small inverses G(k, nu) = [(i nu + mu) - H(k) - dc - Sigma(k, nu)]^-1 over the k grid or
// over the frequencies nu_0 .. nu_{iwmax-1}: one thread per (k, nu) inverts in registers, one
// workgroup per fixed index reduces (wave shuffles, then the four waves through LDS).
//
// Layouts are the reference's Fortran arrays (first index fastest): hk(n,n,nkp),
// siw(-iwmax:iwmax-1, n), dc(2, n), sigma_sum(n, n, -iwfmax_small:iwfmax_small-1, nk),
// giw(-iwmax:iwmax-1, n), gloc(-iwmax:iwmax-1, n, n), n_fock / n_dga_k(nk, n, n), n_dga(n).
#include <algorithm>

#include "adga_kernels.h"
#include "small_inv.h"

namespace adga {

namespace {

constexpr int OP_NT = 256;

// G^-1(k, nu): -H(k) - Sigma off the diagonal, (i nu + mu) - H(k)_ii - dc(1,i) - Sigma_ii on it.
// Sigma is the DMFT siw (diagonal, frequency iw) when sfull is null, else the full matrix
// sfull(a, b) = sfull[a + b*n] (get_gkiw 81-104, get_gkiw_dga 107-121, get_sigma_g_loc 153-160), with the DMFT siw
// still to be added to its diagonal when `own`.
template <int NN>
__device__ __forceinline__ void ginv(const Geom& g, const z64* __restrict__ hk, int k, int iw,
                                     const z64* __restrict__ siw, const z64* __restrict__ dc,
                                     const z64* __restrict__ sfull, bool own, z64 (&a)[NN][NN]) {
  const double nu = M_PI * (2 * iw + 1) / g.beta;
#pragma unroll
  for (int i = 0; i < NN; ++i)
#pragma unroll
    for (int j = 0; j < NN; ++j) {
      const z64 h = hk[(long)k * NN * NN + i + j * NN];
      z64 v = mk(-h.re, -h.im);
      if (sfull) v = csub(v, sfull[i + j * NN]);
      a[i][j] = v;
    }
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    const z64 h = hk[(long)k * NN * NN + i + i * NN];
    z64 s = mk(0.0, 0.0);
    if (sfull) s = sfull[i + i * NN];
    if (!sfull || own) s = cadd(s, siw[(iw + g.iwmax) + (long)i * 2 * g.iwmax]);
    const z64 d = dc[2 * i];
    a[i][i] = mk(g.mu - h.re - d.re - s.re, nu - h.im - d.im - s.im);
  }
}

// Sum of v over the workgroup, returned in thread 0 (red: one slot per wave).
__device__ __forceinline__ z64 wg_sum(z64 v, z64* red) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v.re += __shfl_xor(v.re, off);
    v.im += __shfl_xor(v.im, off);
  }
  __syncthreads();  // red is free (the previous sum has been read)
  if (lane == 0) red[wave] = v;
  __syncthreads();
  z64 s = mk(0.0, 0.0);
  if (t == 0)
    for (int w = 0; w < OP_NT / 64; ++w) s = cadd(s, red[w]);
  return s;
}

// k sums at fixed nu_iw (iw = iw0 + NF blockIdx.x + 0 .. NF - 1 in [0, iwmax)) with Sigma = siw, threads over k.
//   FULL = false: giw(iw, i) = (1/nkp) sum_k G_ii, giw(-iw-1, i) = conj (get_giw).
//   FULL = true:  gloc(iw, a, b) = (1/nkp) sum_k G_ab, gloc(-iw-1) = gloc(iw)^H (get_sigma_g_loc outside the box).
// H(k) is read once for the NF frequencies: with one, 2000 frequencies at 20^3 k, three orbitals, read 2.3 GB out of
// L2 in 128 us (get_giw); with four 87 us.
template <int NN, bool FULL, int NF>
__global__ void __launch_bounds__(OP_NT) k_op_ksum(Geom g, int iw0, const z64* __restrict__ hk,
                                                   const z64* __restrict__ siw, const z64* __restrict__ dc,
                                                   z64* __restrict__ out) {
  __shared__ z64 red[OP_NT / 64];
  const int iw = iw0 + NF * blockIdx.x, t = threadIdx.x;
  constexpr int NE = FULL ? NN * NN : NN;
  z64 acc[NF][NE], x[NF][NN];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[f][e] = mk(0.0, 0.0);
    // a partial group repeats the last frequency
    const int w = min(iw + f, g.iwmax - 1);
#pragma unroll
    for (int i = 0; i < NN; ++i) x[f][i] = siw[(w + g.iwmax) + (long)i * 2 * g.iwmax];
  }
  for (int k = t; k < g.nkp; k += OP_NT) {
    z64 h[NN][NN];
#pragma unroll
    for (int i = 0; i < NN; ++i)
#pragma unroll
      for (int j = 0; j < NN; ++j) h[i][j] = hk[(long)k * NN * NN + i + j * NN];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double nu = M_PI * (2 * min(iw + f, g.iwmax - 1) + 1) / g.beta;
      z64 a[NN][NN];
#pragma unroll
      for (int i = 0; i < NN; ++i) {
#pragma unroll
        for (int j = 0; j < NN; ++j) a[i][j] = mk(-h[i][j].re, -h[i][j].im);
        const z64 d = dc[2 * i], v = h[i][i], s = x[f][i];
        a[i][i] = mk(g.mu - v.re - d.re - s.re, nu - v.im - d.im - s.im);
      }
      inv_small<NN>(a);
      if constexpr (FULL) {
#pragma unroll
        for (int i = 0; i < NN; ++i)
#pragma unroll
          for (int j = 0; j < NN; ++j) acc[f][i + j * NN] = cadd(acc[f][i + j * NN], a[i][j]);
      } else {
#pragma unroll
        for (int i = 0; i < NN; ++i) acc[f][i] = cadd(acc[f][i], a[i][i]);
      }
    }
  }
  const long w2 = 2L * g.iwmax;
  const double nk = (double)g.nkp;
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const z64 s = wg_sum(acc[f][e], red);
      const int w = iw + f;
      if (t == 0 && w < g.iwmax) {
        const z64 v = mk(s.re / nk, s.im / nk);
        if constexpr (FULL) {
          const int i = e % NN, j = e / NN;
          out[(w + g.iwmax) + i * w2 + j * w2 * NN] = v;
          out[(-w - 1 + g.iwmax) + j * w2 + i * w2 * NN] = mk(v.re, -v.im);
        } else {
          out[(w + g.iwmax) + e * w2] = v;
          out[(-w - 1 + g.iwmax) + e * w2] = mk(v.re, -v.im);
        }
      }
    }
}

// NF frequencies to a workgroup where the registers hold them (three orbitals at most) and every CU still gets a
// workgroup
template <int NN, bool FULL>
void op_ksum(const Geom& g, int iw0, const z64* hk, const z64* siw, const z64* dc, z64* out, hipStream_t s) {
  constexpr int NF = NN > 3 ? 1 : FULL ? 2 : 4;
  const int nw = g.iwmax - iw0;
  if (nw >= 256 * NF)
    hipLaunchKernelGGL((k_op_ksum<NN, FULL, NF>), dim3((nw + NF - 1) / NF), dim3(OP_NT), 0, s, g, iw0, hk, siw, dc, out);
  else if (nw > 0)
    hipLaunchKernelGGL((k_op_ksum<NN, FULL, 1>), dim3(nw), dim3(OP_NT), 0, s, g, iw0, hk, siw, dc, out);
}

// The k sums of gloc inside the box, where Sigma is sigma_sum(:, :, iw, k): lanes over the frequencies, which are
// next to one another in memory for one k, the waves of KB_CH workgroups over k; then the sum of the partials.
// (One workgroup per frequency with lanes over k read one n x n block in a whole box per lane: 478 us of 60 late
// workgroups for 60 of 2000 frequencies at 20^3 k, three orbitals, where the others take 124.)
constexpr int KB_CH = 128;

template <int NN>
__global__ void __launch_bounds__(OP_NT) k_op_kbox(Geom g, int nw, const z64* __restrict__ hk,
                                                   const z64* __restrict__ siw, const z64* __restrict__ dc,
                                                   const z64* __restrict__ ssum, bool own, z64* __restrict__ part) {
  constexpr int NW = OP_NT / 64;
  __shared__ z64 red[NW][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int iw = blockIdx.x * 64 + lane;
  z64 acc[NN * NN];
#pragma unroll
  for (int e = 0; e < NN * NN; ++e) acc[e] = mk(0.0, 0.0);
  for (int k = blockIdx.y * NW + wave; k < g.nkp && iw < nw; k += KB_CH * NW) {
    z64 a[NN][NN];
    ginv<NN>(g, hk, k, iw, siw, dc, ssum + ((long)k * g.nf + (iw + g.iwf)) * NN * NN, own, a);
    inv_small<NN>(a);
#pragma unroll
    for (int i = 0; i < NN; ++i)
#pragma unroll
      for (int j = 0; j < NN; ++j) acc[i + j * NN] = cadd(acc[i + j * NN], a[i][j]);
  }
#pragma unroll
  for (int e = 0; e < NN * NN; ++e) {
    __syncthreads();
    red[wave][lane] = acc[e];
    __syncthreads();
    if (wave == 0 && iw < nw) {
      z64 s = red[0][lane];
      for (int w = 1; w < NW; ++w) s = cadd(s, red[w][lane]);
      part[((long)blockIdx.y * NN * NN + e) * nw + iw] = s;
    }
  }
}

// gloc(iw, a, b) = (1/nkp) of the partials' sum and gloc(-iw-1) = gloc(iw)^H; a wave per element (e, iw)
__global__ void __launch_bounds__(64) k_op_kbox_sum(Geom g, int nw, const z64* __restrict__ part,
                                                    z64* __restrict__ gloc) {
  const int iw = blockIdx.x, e = blockIdx.y, lane = threadIdx.x;
  z64 s = mk(0.0, 0.0);
  for (int c = lane; c < KB_CH; c += 64) s = cadd(s, part[((long)c * g.n2 + e) * nw + iw]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s.re += __shfl_xor(s.re, off);
    s.im += __shfl_xor(s.im, off);
  }
  if (lane == 0) {
    const z64 v = mk(s.re / (double)g.nkp, s.im / (double)g.nkp);
    const long w2 = 2L * g.iwmax;
    const int i = e % g.n, j = e / g.n;
    gloc[(iw + g.iwmax) + i * w2 + j * w2 * g.n] = v;
    gloc[(-iw - 1 + g.iwmax) + j * w2 + i * w2 * g.n] = mk(v.re, -v.im);
  }
}

// frequency sums at fixed k (blockIdx.x = index into the k list), threads over nu_0 .. nu_{iwmax-1}:
// out(kk, a, b) = 2/beta sum_nu Re G_ab + delta_ab / 2 (complex, zero imaginary part).
//   DGA = false: k = kk on the full grid, Sigma = siw (get_nfock).
//   DGA = true:  k = k_data_eom(kk), Sigma = sigma_sum(:, :, iw, kk) for iw < iwfmax_small, siw
//                outside (get_ndga).
template <int NN, bool DGA>
__global__ void __launch_bounds__(OP_NT) k_op_wsum(Geom g, int nk, const z64* __restrict__ hk, const z64* __restrict__ siw,
                                                   const z64* __restrict__ dc, const int* __restrict__ keom,
                                                   const z64* __restrict__ ssum, bool own, z64* __restrict__ out) {
  __shared__ z64 red[OP_NT / 64];
  const int kk = blockIdx.x, t = threadIdx.x;
  const int k = DGA ? keom[kk] - 1 : kk;
  double acc[NN * NN];
#pragma unroll
  for (int e = 0; e < NN * NN; ++e) acc[e] = 0.0;
  for (int iw = t; iw < g.iwmax; iw += OP_NT) {
    const z64* sf = (DGA && iw < g.iwf) ? ssum + ((long)kk * g.nf + (iw + g.iwf)) * NN * NN : nullptr;
    z64 a[NN][NN];
    ginv<NN>(g, hk, k, iw, siw, dc, sf, own, a);
    inv_small<NN>(a);
#pragma unroll
    for (int i = 0; i < NN; ++i)
#pragma unroll
      for (int j = 0; j < NN; ++j) acc[i + j * NN] += a[i][j].re;
  }
#pragma unroll
  for (int e = 0; e < NN * NN; ++e) {
    const z64 s = wg_sum(mk(acc[e], 0.0), red);
    if (t == 0) {
      const int i = e % NN, j = e / NN;
      double v = 2.0 * s.re / g.beta;
      if (i == j) v += 0.5;
      out[kk + (long)i * nk + (long)j * nk * NN] = mk(v, 0.0);
    }
  }
}

// n_dga(i) = (1/nk) sum_kk n_dga_k(kk, i, i) (get_ndga 383-389); one workgroup per orbital.
__global__ void __launch_bounds__(OP_NT) k_op_ndga_mean(int n, int nk, const z64* __restrict__ ndk, z64* __restrict__ nd) {
  __shared__ z64 red[OP_NT / 64];
  const int i = blockIdx.x, t = threadIdx.x;
  double s = 0.0;
  for (int kk = t; kk < nk; kk += OP_NT) s += ndk[kk + (long)i * nk + (long)i * nk * n].re;
  const z64 r = wg_sum(mk(s, 0.0), red);
  if (t == 0) nd[i] = mk(r.re / nk, 0.0);
}

// sigma_loc(a, b, iw) = (1/nkp) sum_k sigma_sum(a, b, iw, k) over the whole box (get_sigma_g_loc 145-150),
// in two passes: partial sums over SL_KCH chunks of k (a wave reads 64 consecutive elements of one
// k, four waves take every fourth k of the chunk), then the sum of the partials.  own: ssum is the accumulated
// Sigma_nl, of which the frequencies from 0 on are read: those below are Sigma(a, b, -nu) = conj Sigma(b, a, nu) as
// adga_get_sigma fills them, and siw is added on the diagonal as add_siw_dmft does (eom_module.f90:237-251).
constexpr int SL_KCH = 32;

__global__ void __launch_bounds__(OP_NT) k_op_sigma_loc_part(Geom g, const z64* __restrict__ ssum, bool own,
                                                             const z64* __restrict__ siw, z64* __restrict__ part) {
  __shared__ z64 red[OP_NT / 64][64];
  const int t = threadIdx.x, el = t & 63, ks = t >> 6;
  const long ne = (long)g.n2 * g.nf;
  const long e = (long)blockIdx.x * 64 + el;
  const int kper = (g.nkp + SL_KCH - 1) / SL_KCH;
  const int k0 = blockIdx.y * kper, k1 = min(g.nkp, k0 + kper);
  z64 s = mk(0.0, 0.0);
  if (e < ne) {
    const int d = (int)(e / g.n2), ab = (int)(e % g.n2), ca = ab % g.n, cb = ab / g.n;
    const bool neg = own && d < g.iwf;
    const long src = neg ? cb + ca * g.n + (long)(g.nf - 1 - d) * g.n2 : e;
    const z64 add = own && ca == cb ? siw[(d - g.iwf + g.iwmax) + (long)ca * 2 * g.iwmax] : mk(0.0, 0.0);
    for (int k = k0 + ks; k < k1; k += OP_NT / 64) {
      const z64 v = ssum[(long)k * ne + src];
      s = cadd(s, cadd(mk(v.re, neg ? -v.im : v.im), add));
    }
  }
  red[ks][el] = s;
  __syncthreads();
  if (ks == 0 && e < ne) {
    z64 r = red[0][el];
    for (int w = 1; w < OP_NT / 64; ++w) r = cadd(r, red[w][el]);
    part[(long)blockIdx.y * ne + e] = r;
  }
}

__global__ void k_op_sigma_loc_sum(Geom g, const z64* __restrict__ part, z64* __restrict__ sloc) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ne = (long)g.n2 * g.nf;
  if (e >= ne) return;
  z64 s = mk(0.0, 0.0);
  for (int c = 0; c < SL_KCH; ++c) s = cadd(s, part[(long)c * ne + e]);
  sloc[e] = mk(s.re / g.nkp, s.im / g.nkp);
}

}  // namespace

#define ADGA_OP_SWITCH(F)                       \
  switch (g.n) {                               \
    case 1: F(1); break;                       \
    case 2: F(2); break;                       \
    case 3: F(3); break;                       \
    case 4: F(4); break;                       \
    case 5: F(5); break;                       \
    case 6: F(6); break;                       \
    case 7: F(7); break;                       \
    case 8: F(8); break;                       \
    default: return false;                     \
  }

bool launch_op_giw(const Geom& g, const z64* hk, const z64* siw, const z64* dc, z64* giw, hipStream_t s) {
#define F(NN) op_ksum<NN, false>(g, 0, hk, siw, dc, giw, s)
  ADGA_OP_SWITCH(F)
#undef F
  return true;
}

bool launch_op_nfock(const Geom& g, const z64* hk, const z64* siw, const z64* dc, z64* nfock, hipStream_t s) {
#define F(NN)                                                                                                 \
  hipLaunchKernelGGL((k_op_wsum<NN, false>), dim3(g.nkp), dim3(OP_NT), 0, s, g, g.nkp, hk, siw, dc, nullptr, \
                     nullptr, false, nfock)
  ADGA_OP_SWITCH(F)
#undef F
  return true;
}

size_t op_sigma_loc_scratch(const Geom& g) {
  return (size_t)g.n2 * std::max(SL_KCH * g.nf, KB_CH * std::min(g.iwf, g.iwmax));
}

bool launch_op_sigma_g_loc(const Geom& g, const z64* hk, const z64* siw, const z64* dc, const z64* ssum, bool own,
                           z64* sloc, z64* gloc, z64* scratch, hipStream_t s) {
  const long ne = (long)g.n2 * g.nf;
  hipLaunchKernelGGL(k_op_sigma_loc_part, dim3((unsigned)((ne + 63) / 64), SL_KCH), dim3(OP_NT), 0, s, g, ssum, own,
                     siw, scratch);
  hipLaunchKernelGGL(k_op_sigma_loc_sum, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, s, g, scratch, sloc);
  const int nw = std::min(g.iwf, g.iwmax);
#define F(NN)                                                                                                         \
  hipLaunchKernelGGL((k_op_kbox<NN>), dim3((nw + 63) / 64, KB_CH), dim3(OP_NT), 0, s, g, nw, hk, siw, dc, ssum, own, \
                     scratch);                                                                                        \
  op_ksum<NN, true>(g, nw, hk, siw, dc, gloc, s)
  ADGA_OP_SWITCH(F)
#undef F
  hipLaunchKernelGGL(k_op_kbox_sum, dim3(nw, g.n2), dim3(64), 0, s, g, nw, scratch, gloc);
  return true;
}

bool launch_op_ndga(const Geom& g, const z64* hk, const z64* siw, const z64* dc, const int* keom, const z64* ssum,
                    bool own, z64* ndk, z64* nd, hipStream_t s) {
#define F(NN)                                                                                                   \
  hipLaunchKernelGGL((k_op_wsum<NN, true>), dim3(g.nkp_eom), dim3(OP_NT), 0, s, g, g.nkp_eom, hk, siw, dc, keom, \
                     ssum, own, ndk)
  ADGA_OP_SWITCH(F)
#undef F
  hipLaunchKernelGGL(k_op_ndga_mean, dim3(g.n), dim3(OP_NT), 0, s, g.n, g.nkp_eom, ndk, nd);
  return true;
}

}  // namespace adga
