// Column kernels of the LDS path for power-of-two columns of 64 .. 8192 points
// (columns of 16384: the register kernels of kern_lds.h).  The transform is
// RegFft: N / 16 threads per column, first and last stages in registers.
#pragma once
#include "fft_reg.h"
#include "kern_lds.h"

namespace curig {

// Threads of a column workgroup at most (the plan's cpw, cpw_inv keep to them).
// The lanes of a wavefront take the workgroup's columns in turn, so those of a
// tile read and write the pieces of a chunk of H together.
//   forward: 256 threads, or one column's N / 16; FP64 columns of 4096 in pairs
//   (512 threads, 1.13 against 1.22 ms per 30 planes of 2048 columns; in FP32
//   pairs lost, 0.71 against 0.62 ms: longer barriers);
//   inverse: whole tiles of four columns where 1024 threads (FP64: 512) allow
//   (FP32, 4096 points: 0.86 ms, pairs 1.02 ms).
// Prefetch (forward): the next plane's column in flight during the transform;
// it pays where two wavefronts per SIMD are all the registers allow (FP64:
// 1.13 against 1.22 ms), in FP32 the third wavefront hides as much (0.63
// against 0.62 ms).
template <typename T, int N> struct ColCfg {
  static constexpr bool dbl = sizeof(T) == 8;
  static constexpr int top = dbl ? 512 : 1024;
  static constexpr int fwd_threads = dbl && N >= 4096 ? 512 : N / 16 > 256 ? N / 16 : 256;
  static constexpr int inv_threads = N / 4 > top ? top : N / 4 > 256 ? N / 4 : 256;
  static constexpr bool prefetch = dbl && N <= 4096;
  static constexpr int fwd_waves = dbl ? 2 : N <= 4096 ? 3 : 4;
  static constexpr int fwd_tw = dbl || N > 4096 ? kTwPair : kTwHeld;
  static constexpr int inv_waves = dbl ? 2 : N <= 1024 ? 3 : 4;
  static constexpr int inv_tw = dbl ? kTwPair : N >= 2048 ? kTwFull : kTwHeld;
  using Fwd = RegFft<T, N, +1, fwd_tw>;
  using Inv = RegFft<T, N, -1, inv_tw>;
  static size_t fwd_lds(int cpw) { return sizeof(cpx<T>) * (size_t)(cpw * Fwd::kStride + Fwd::kTwLds); }
  static size_t inv_lds(int cpw) { return sizeof(cpx<T>) * (size_t)(cpw * Inv::kStride + Inv::kTwLds); }
};

// ms2dirty column pass fused with the w-accumulation (w_term_dft, cuft.cu:520-572):
// a workgroup owns cpw columns and walks planes [blockIdx.y pchunk, + pchunk) of
// the batch's nb, last to first: load the row-transformed columns, FFT over nf2,
// then by Horner's rule in FP64 acc = acc e^{i z'} + F_p for the image rows, and
// once at the end the phase e^{i z' (p_first - P/2)}.  Four FP64 multiply-adds
// per image cell and plane took the place of a phase reduction, two polynomials
// and four multiply-adds (about 40 instructions; the 4096-point column pass,
// 30 planes of 2048 columns, was bound by them and by index arithmetic at 92%
// VALU).  Small images leave the chip idle with one workgroup for all planes of
// its columns: each plane chunk then sums into its own accumulator
// (accT + blockIdx.y npix), added by the epilogue.
template <typename T, int N>
__global__ void __launch_bounds__((ColCfg<T, N>::fwd_threads), (ColCfg<T, N>::fwd_waves)) col_fwd_kernel(
    const cpx<T> *__restrict__ H, double2 *__restrict__ accT, const cpx<T> *__restrict__ tw, Geom g, int p0, int nb,
    int first, int cpw_lg, int pchunk) {
  using F = typename ColCfg<T, N>::Fwd;
  constexpr int G = F::G;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int cpw = 1 << cpw_lg, s = threadIdx.x & (cpw - 1), j = threadIdx.x >> cpw_lg, N2 = g.N2;
  cpx<T> *ltw = reinterpret_cast<cpx<T> *>(smem_raw), *buf = ltw + F::kTwLds + s * F::kStride;
  const int sl = xcd_group(blockIdx.x, gridDim.x) * cpw + s;  // column slot
  const int col = sl < g.nslot ? slot_column(sl, g) : -1;
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  if (__syncthreads_or(col >= 0) == 0) return;
  F fft;
  fft.init(tw, j, ltw);
  double ar[8], ai[8], er[8], ei[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    ar[q] = ai[q] = 0.0;
    const int row = image_index(j + G * image_elem(q), N2, N);
    double sn, cs;
    sincos_cw(row >= 0 && col >= 0 ? pixel_zp(row, col, g) : 0.0, &sn, &cs);
    er[q] = cs;
    ei[q] = sn;
  }
  // byte offset of this thread's first element in a plane (< 4 GiB: uniform
  // base, 32-bit offset); threads without a column read the first one's and
  // store nothing
  const unsigned off = sizeof(cpx<T>) * (unsigned)((col >= 0 ? h_slot(g, sl) : 0) + (j << kTileLog2));
  // a wavefront's rows j + G e lie in one block of Geom::occ for each e; the rows
  // of blocks without records are zero and not in H
  const int jw = __builtin_amdgcn_readfirstlane(j);
  auto load = [&](cpx<T> *v, int k) {
    const cpx<T> *hk = H + h_plane(g, k);
    const uint64_t occ = occ_mask(g, p0 + k);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if (occ_row(occ, jw + G * e, g))
        v[e] = *reinterpret_cast<const cpx<T> *>(reinterpret_cast<const char *>(hk + ((G * e) << kTileLog2)) + off);
      else
        v[e] = fftc::mk((T)0, (T)0);
    }
  };
  cpx<T> nx[16];
  if (ColCfg<T, N>::prefetch) load(nx, k1 - 1);
  for (int k = k1 - 1; k >= k0; --k) {
    cpx<T> v[16];
    if (ColCfg<T, N>::prefetch) {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = nx[e];
      if (k > k0) load(nx, k - 1);
    } else {
      load(v, k);
    }
    __syncthreads();  // the previous plane's LDS reads are done
    fft.template run<false>(v, buf, j);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const cpx<T> f = v[image_elem(q)];
      const double t = ar[q] * er[q] - ai[q] * ei[q] + (double)f.x;
      ai[q] = ar[q] * ei[q] + ai[q] * er[q] + (double)f.y;
      ar[q] = t;
    }
  }
  if (col < 0) return;
  double2 *out = accT + (size_t)blockIdx.y * g.N1 * N2 + (size_t)col * N2;
  const double m = (double)(p0 + k0 - g.P / 2);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int row = image_index(j + G * image_elem(q), N2, N);
    if (row >= 0) {
      double sn, cs;
      sincos_cw(pixel_zp(row, col, g) * m, &sn, &cs);
      double2 r = make_double2(ar[q] * cs - ai[q] * sn, ar[q] * sn + ai[q] * cs);
      if (!first) {
        const double2 o = out[row];
        r.x += o.x;
        r.y += o.y;
      }
      out[row] = r;
    }
  }
}

// dirty2ms column pass fused with the w-fill (w_term_idft, cuft.cu:575-612): a
// workgroup owns cpw columns and, for each plane p of its chunk, transforms
// gT[col][row] e^{-i z' (p - P/2)} at the image rows (zeros elsewhere) and
// writes the full columns to the column-tiled H.  The phased values are carried
// from plane to plane in FP64 (times e^{-i z'}: four multiply-adds).  FP32
// workgroups own whole or half column tiles where they fit (Geom::cpw_inv), so
// each 32-byte chunk of H is written by one workgroup.
template <typename T, int N>
__global__ void __launch_bounds__((ColCfg<T, N>::inv_threads), (ColCfg<T, N>::inv_waves)) col_inv_kernel(
    const cpx<T> *__restrict__ gT, cpx<T> *__restrict__ H, const cpx<T> *__restrict__ tw, Geom g, int p0, int nb,
    int cpw_lg, int pchunk) {
  using F = typename ColCfg<T, N>::Inv;
  constexpr int G = F::G;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int cpw = 1 << cpw_lg, s = threadIdx.x & (cpw - 1), j = threadIdx.x >> cpw_lg, N2 = g.N2;
  cpx<T> *ltw = reinterpret_cast<cpx<T> *>(smem_raw), *buf = ltw + F::kTwLds + s * F::kStride;
  const int sl = xcd_group(blockIdx.x, gridDim.x) * cpw + s;  // column slot
  const int col = sl < g.nslot ? slot_column(sl, g) : -1;
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  if (__syncthreads_or(col >= 0) == 0) return;
  F fft;
  fft.init(tw, j, ltw);
  double xr[8], xi[8], er[8], ei[8];
  const double m = (double)(p0 + k0 - g.P / 2);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    xr[q] = xi[q] = 0.0;
    er[q] = ei[q] = 0.0;
    const int row = image_index(j + G * image_elem(q), N2, N);
    if (row >= 0 && col >= 0) {
      const double zp = pixel_zp(row, col, g);
      double sn, cs;
      sincos_cw(-zp, &sn, &cs);
      er[q] = cs;
      ei[q] = sn;
      sincos_cw(-zp * m, &sn, &cs);
      const cpx<T> gv = gT[(size_t)col * N2 + row];
      xr[q] = (double)gv.x * cs - (double)gv.y * sn;
      xi[q] = (double)gv.x * sn + (double)gv.y * cs;
    }
  }
  const unsigned off = sizeof(cpx<T>) * (unsigned)((col >= 0 ? ht_slot(g, sl) : 0) + ht_row(j));
  const int jw = __builtin_amdgcn_readfirstlane(j);  // col_fwd_kernel: rows outside Geom::occ are not read
  for (int k = k0; k < k1; ++k) {
    cpx<T> v[16];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      v[image_elem(q)] = fftc::mk((T)xr[q], (T)xi[q]);
      const double t = xr[q] * er[q] - xi[q] * ei[q];
      xi[q] = xr[q] * ei[q] + xi[q] * er[q];
      xr[q] = t;
    }
    __syncthreads();  // the previous plane's LDS reads are done
    fft.template run<true>(v, buf, j);
    // keeps the last butterflies out of the store's branch (there they spill)
#pragma unroll
    for (int e = 0; e < 16; ++e) __asm__ volatile("" : "+v"(v[e].x), "+v"(v[e].y));
    cpx<T> *hk = H + h_plane(g, k);
    const uint64_t occ = occ_mask(g, p0 + k);
    if (col >= 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (occ_row(occ, jw + G * e, g))
          *reinterpret_cast<cpx<T> *>(reinterpret_cast<char *>(hk + ((G * e) << kTileLog2)) + off) = v[e];
    }
  }
}

inline int col_groups(const Geom &g, int cpw) { return (g.nslot + cpw - 1) / cpw; }
inline int plane_chunks(int nb, int pchunk) { return (nb + pchunk - 1) / pchunk; }

// ms2dirty, one batch on the LDS path: column FFT + w-accumulation into accT
template <typename T>
void lds_cols_forward(const Geom &g, int p0, int nb, const cpx<T> *H, double2 *accT, const cpx<T> *tw2, int first,
                      hipStream_t st) {
  if (g.colreg) {
    col_fwd_reg_kernel<T><<<col_groups(g, 1), colr::NT, g.lds_col_bytes, st>>>(H, accT, tw2, g, p0, nb, first);
    return;
  }
  const dim3 grd(col_groups(g, g.cpw), plane_chunks(nb, g.pch_fwd));
  with_reg_fft(g.nf2, [&](auto N) {
    col_fwd_kernel<T, N.value><<<grd, g.cpw * N.value / 16, ColCfg<T, N.value>::fwd_lds(g.cpw), st>>>(
        H, accT, tw2, g, p0, nb, first, 31 - __builtin_clz(g.cpw), g.pch_fwd);
  });
}

// dirty2ms, one batch on the LDS path: w-fill + inverse column FFT -> H (column-tiled)
template <typename T>
void lds_cols_backward(const Geom &g, int p0, int nb, const cpx<T> *gT, cpx<T> *H, const cpx<T> *tw2,
                       hipStream_t st) {
  if (g.colreg) {
    const dim3 grd(col_groups(g, 1), plane_chunks(nb, g.pch_inv));
    col_inv_reg_kernel<T><<<grd, colr::NT, g.lds_col_bytes, st>>>(gT, H, tw2, g, p0, nb, g.pch_inv);
    return;
  }
  const dim3 grd(col_groups(g, g.cpw_inv), plane_chunks(nb, g.pch_inv));
  with_reg_fft(g.nf2, [&](auto N) {
    col_inv_kernel<T, N.value><<<grd, g.cpw_inv * N.value / 16, ColCfg<T, N.value>::inv_lds(g.cpw_inv), st>>>(
        gT, H, tw2, g, p0, nb, 31 - __builtin_clz(g.cpw_inv), g.pch_inv);
  });
}

template <typename T>
int allow_cols(const Geom &g) {
  if (g.colreg) {
    CURIG_TRY(allow_lds(col_fwd_reg_kernel<T>, g.lds_col_bytes));
    CURIG_TRY(allow_lds(col_inv_reg_kernel<T>, g.lds_col_bytes));
    return kOk;
  }
  int ier = kErrArg;
  const bool known = with_reg_fft(g.nf2, [&](auto N) {
    constexpr int n = N.value;
    using C = ColCfg<T, n>;
    auto pow2 = [](int c) { return c >= 1 && (c & (c - 1)) == 0; };
    if (!pow2(g.cpw) || !pow2(g.cpw_inv) || g.cpw * n / 16 > C::fwd_threads || g.cpw_inv * n / 16 > C::inv_threads ||
        g.pch_fwd < 1 || g.pch_inv < 1)
      return;
    ier = allow_lds(col_fwd_kernel<T, n>, (int)C::fwd_lds(g.cpw));
    if (ier == kOk) ier = allow_lds(col_inv_kernel<T, n>, (int)C::inv_lds(g.cpw_inv));
  });
  if (!known || ier == kErrArg)
    set_error("column pass of %d points: %d and %d columns, %d and %d planes per workgroup", g.nf2, g.cpw, g.cpw_inv,
              g.pch_fwd, g.pch_inv);
  return ier;
}

#define CURIG_LDS_COLS_INST(T)                                                                                     \
  template void lds_cols_forward<T>(const Geom &, int, int, const cpx<T> *, double2 *, const cpx<T> *, int,        \
                                    hipStream_t);                                                                  \
  template void lds_cols_backward<T>(const Geom &, int, int, const cpx<T> *, cpx<T> *, const cpx<T> *,             \
                                     hipStream_t);                                                                 \
  template int allow_cols<T>(const Geom &);

}  // namespace curig
