// Row and column kernels of the LDS path for grids whose axes are 2^a 3^b 5^c
// but not powers of two with the image inside half the grid (those run the
// kernels of kern_lds.h and kern_cols.h).  The same passes over the same
// column-tiled planes H, with the mixed-radix LDS transform of fft_mix.h: the
// full grid planes of the rocFFT path (written and read five times per plane)
// are never formed.  Each workgroup keeps its rows or columns and walks a chunk
// of the batch's planes.
//
// What bounds them: VALU issue of the transform (about 100 instructions per
// element: butterflies, twiddles and the run-time index arithmetic) and its LDS
// passes, with one workgroup's memory phases behind another's transform.
#pragma once
#include "kern_rows.h"

#include "fft_mix.h"

namespace curig {

template <typename T> struct MixThreads { static constexpr int value = sizeof(T) == 8 ? 512 : 1024; };

// stages [s0, P.ns) of the transform; the caller's barrier precedes it, a
// barrier ends it
template <typename T, int SIGN, typename Tw>
__device__ __forceinline__ void mix_stages(cpx<T> *buf, const fftm::Plan &P, const Tw &tw, int s0, int Ns) {
  for (int s = s0; s < P.ns; ++s) {
    const int R = P.R[s];
    // opaque copy of the thread id: every radix's addresses are formed where
    // they are used (hoisted out of the plane loop they spill)
    int tid = threadIdx.x;
    __asm__ volatile("" : "+v"(tid));
    fftm::with_radix(R, [&](auto tag) {
      constexpr int RR = decltype(tag)::value;
      cpx<T> v[RR * fftm::radix_nb(RR)];
      fftm::stage_load<T, RR, SIGN>([&](int q, int k) { return buf[q * P.stride + fftc::pad(k)]; }, v, P, s, Ns, tw, tid);
      __syncthreads();
      fftm::stage_store<T, RR>([&](int q, int k, cpx<T> x) { buf[q * P.stride + fftc::pad(k)] = x; }, v, P, s, Ns, tid);
    });
    __syncthreads();
    Ns *= R;
  }
}

// f(element of the register array, offset in the buffer) for this thread's inputs
// of the first stage, f(butterfly's first element) after each butterfly's
template <int RR, typename F, typename B>
__device__ __forceinline__ void mix_first_inputs(const fftm::Plan &P, int tid, F f, B each) {
  const int nbf = P.n / RR, total = nbf * P.count;
#pragma unroll
  for (int b = 0; b < fftm::radix_nb(RR); ++b) {
    const int jg = tid + b * P.nt;
    if (jg < total) {
      const int seq = P.count > 1 ? fftm::quot(jg, P.bf_magic[0]) : 0, j = jg - seq * nbf;
#pragma unroll
      for (int r = 0; r < RR; ++r) f(b * RR + r, seq * P.stride + fftc::pad(j + r * nbf));
      each(b * RR);
    }
  }
}

constexpr int kMixElems = 20;  // inputs of a stage per thread at most

// the real parts of this thread's inputs of the first stage, their cells cleared
template <typename T> __device__ __forceinline__ void mix_take_real(double *cells, const fftm::Plan &P, T *re) {
  int tid = threadIdx.x;
  __asm__ volatile("" : "+v"(tid));
  fftm::with_radix(P.R[0], [&](auto tag) {
    constexpr int RR = decltype(tag)::value;
    mix_first_inputs<RR>(
        P, tid,
        [&](int e, int at) {
          re[e] = (T)cells[at];
          cells[at] = 0.0;
        },
        [](int) {});
    // ends each radix's case differently: its stores to re, merged with another's, would go to memory
    __asm__ volatile("; %0" ::"i"(RR));
  });
}

// the first stage on the spread's sums, in whose place (complex cells: first half)
// the transform then runs
template <typename T, int SIGN, typename Cell>
__device__ __forceinline__ void mix_first_cells(cpx<T> *buf, const Cell *acc, const T *re, const fftm::Plan &P) {
  int tid = threadIdx.x;
  __asm__ volatile("" : "+v"(tid));
  fftm::with_radix(P.R[0], [&](auto tag) {
    constexpr int RR = decltype(tag)::value;
    cpx<T> v[RR * fftm::radix_nb(RR)];
    mix_first_inputs<RR>(
        P, tid,
        [&](int e, int at) {
          if constexpr (std::is_same<Cell, double>::value)
            v[e] = fftc::mk(re[e], (T)acc[at]);
          else
            v[e] = fftc::mk((T)acc[at].x, (T)acc[at].y);
        },
        [&](int e) {
          fftm::dft<T, RR, SIGN>(v + e);
          __builtin_amdgcn_sched_barrier(0);
        });
    __syncthreads();
    fftm::stage_store<T, RR>([&](int q, int k, cpx<T> x) { buf[q * P.stride + fftc::pad(k)] = x; }, v, P, 0, 1, tid);
  });
  __syncthreads();
}

// ms2dirty: spread into the workgroup's rows (LDS), row FFT, image columns to H.
// Accumulation as RowAcc says; outputs added to H where gridDim.z workgroups share
// the rows' records.
template <typename T, int KWM, bool ACC64>
__global__ void __launch_bounds__(MixThreads<T>::value) spread_row_mix_kernel(
    const Rec<T> *__restrict__ recs, const T *__restrict__ taps, const int *__restrict__ off, cpx<T> *__restrict__ H,
    const cpx<T> *__restrict__ tw, Geom g, fftm::Plan P, int p0, int nb, int pchunk) {
  using Cell = typename RowAcc<T, ACC64>::cell;
  constexpr bool kParts = RowAcc<T, ACC64>::parts;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ WalkTable wt[2];
  const int nf1 = g.nf1, nf2 = g.nf2, N1 = g.N1, nt = blockDim.x, tid = threadIdx.x, rpw = g.rpw;
  const int nbuf = P.count * P.stride, h1 = N1 / 2;
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw);
  Cell *acc = reinterpret_cast<Cell *>(smem_raw);
  cpx<T> *ltw = reinterpret_cast<cpx<T> *>(acc + nbuf);
  const int row0 = row_group(g) * rpw, nrows = min(rpw, nf2 - row0);
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  const bool add = gridDim.z > 1;
  // planes whose blocks of rows (two at most, rpw <= 64) hold no record are passed over
  PlaneWalk<> pw(g, p0, k0, k1, row0, row0 + nrows - 1);
  int pn = pw.next();
  if (pn >= k1) return;
  const auto tv = lds_twiddles<T>(ltw, tw, nf1);
  if (tid < 64) walk_table_build(wt[0], off, g, p0 + pn, row0, nrows);
  for (int i = tid; i < nbuf; i += nt) acc[i] = Cell{};
  __syncthreads();
  int cur = 0;
  for (int pl = pn; pl < k1; pl = pn, cur ^= 1) {
    const int p = p0 + pl, total = wt[cur].total;
    pn = pw.next();
    const bool more = pn < k1;
    WalkAhead wa;
    if (tid < 64 && more) walk_issue(wa, off, g, p0 + pn, row0, nrows);
    T re[kParts ? kMixElems : 1];
    if constexpr (kParts) {
      if (total > 0) {
        spread_records<kReal, T, KWM>(wt[cur], total, recs, taps, g, p, row0, nrows, acc, P.stride);
        __syncthreads();
        mix_take_real<T>(acc, P, re);
        __syncthreads();
      }
    }
    spread_records<kParts ? kImag : kBoth, T, KWM>(wt[cur], total, recs, taps, g, p, row0, nrows, acc, P.stride);
    if (tid < 64 && more) walk_finish(wt[cur ^ 1], wa);
    __syncthreads();  // spread done; the next plane's walk table is complete
    cpx<T> *hb = H + h_plane(g, pl) + row0 * kTile;
    if (total == 0) {
      // no visibility reaches these rows of this plane (and the LDS is still clear)
      const uint64_t occ = occ_mask(g, p);
      for (int r = 0; r < nrows && !add; ++r)
        for (int i = occ_row(occ, row0 + r, g) ? tid : N1; i < N1; i += nt) hb[h_slot(g, i) + (r << kTileLog2)] = fftc::mk((T)0, (T)0);
      continue;
    }
    if constexpr (kParts || ACC64) {
      mix_first_cells<T, +1>(buf, acc, re, P);
      mix_stages<T, +1>(buf, P, tv, 1, P.R[0]);
    } else {
      mix_stages<T, +1>(buf, P, tv, 0, 1);
    }
    for (int r = 0; r < nrows; ++r)
      for (int i = tid; i < N1; i += nt) {
        const int k = i >= h1 ? i - h1 : nf1 + i - h1;
        put_row(hb + h_slot(g, i) + (r << kTileLog2), buf[r * P.stride + fftc::pad(k)], add);
      }
    __syncthreads();  // every output read: clear for the next plane
    for (int i = tid; i < nbuf; i += nt) acc[i] = Cell{};
    __syncthreads();
  }
}

// rows [row0, row0 + nrows) of a dirty2ms plane into LDS, expanded to nf1 cells
template <typename T>
__device__ __forceinline__ void mix_load_rows(cpx<T> *buf, const cpx<T> *hb, const Geom &g, const fftm::Plan &P, int row0,
                                              int nrows, int N1) {
  const int nt = blockDim.x, nf1 = g.nf1;
  for (int r = 0; r < nrows; ++r) {
    const cpx<T> *hr = hb + ht_row(row0 + r);
    constexpr int B = 8;  // loads in flight
    for (int i0 = threadIdx.x; i0 < nf1; i0 += B * nt) {
      cpx<T> v[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int i = i0 + b * nt, col = i < nf1 ? image_index(i, N1, nf1) : -1;
        v[b] = col >= 0 ? hr[ht_slot(g, col)] : fftc::mk((T)0, (T)0);
      }
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int i = i0 + b * nt;
        if (i < nf1) buf[r * P.stride + fftc::pad(i)] = v[b];
      }
    }
  }
}

// dirty2ms: rows of H expanded to the grid, inverse row FFT, interpolation of
// every record that touches the rows (FP64 atomics on its accumulator).
template <typename T, int KWM>
__global__ void __launch_bounds__(MixThreads<T>::value) row_interp_mix_kernel(
    const cpx<T> *__restrict__ H, const Rec<T> *__restrict__ recs, const T *__restrict__ taps,
    const int *__restrict__ off, double2 *__restrict__ vacc, const cpx<T> *__restrict__ tw, Geom g, fftm::Plan P, int p0,
    int nb, int pchunk) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ WalkTable wt[2];
  const int nf1 = g.nf1, nf2 = g.nf2, N1 = g.N1, nt = blockDim.x, tid = threadIdx.x, rpw = g.rpw;
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw);
  const int row0 = row_group(g) * rpw, nrows = min(rpw, nf2 - row0);
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  PlaneWalk<> pw(g, p0, k0, k1, row0, row0 + nrows - 1);
  int pn = pw.next();
  if (pn >= k1) return;
  const auto tv = lds_twiddles<T>(buf + P.count * P.stride, tw, nf1);
  if (tid < 64) walk_table_build(wt[0], off, g, p0 + pn, row0, nrows);
  // rows past the grid (the last workgroup): zero sequences, transformed along
  for (int i = tid; i < P.count * P.stride; i += nt) buf[i] = fftc::mk((T)0, (T)0);
  __syncthreads();
  int cur = 0;
  for (int pl = pn; pl < k1; pl = pn, cur ^= 1) {
    const int p = p0 + pl, total = wt[cur].total;
    pn = pw.next();
    const bool more = pn < k1;
    WalkAhead wa;
    if (tid < 64 && more) walk_issue(wa, off, g, p0 + pn, row0, nrows);
    if (total > 0) {
      mix_load_rows<T>(buf, H + h_plane(g, pl), g, P, row0, nrows, N1);
      __syncthreads();
      mix_stages<T, -1>(buf, P, tv, 0, 1);
      interp_records<T, KWM>(wt[cur], total, recs, taps, g, p, row0, nrows, buf, P.stride, vacc);
    }
    if (tid < 64 && more) walk_finish(wt[cur ^ 1], wa);
    __syncthreads();  // the rows are free; the next plane's walk table is complete
  }
}

// dirty2ms where the records are dense on the grid (Geom::gather): the rows are
// written out as full planes, and interp_gather_kernel reads each record's cells
// from there, once per record, where the fused row pass would visit the record
// in every row and plane of its support and add two FP64 atomics each time.
template <typename T>
__global__ void __launch_bounds__(MixThreads<T>::value) row_planes_mix_kernel(const cpx<T> *__restrict__ H,
                                                                             cpx<T> *__restrict__ grid,
                                                                             const cpx<T> *__restrict__ tw, Geom g,
                                                                             fftm::Plan P, int p0, int nb, int pchunk) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int nf1 = g.nf1, nf2 = g.nf2, N1 = g.N1, nt = blockDim.x, tid = threadIdx.x, rpw = g.rpw;
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw);
  const int row0 = row_group(g) * rpw, nrows = min(rpw, nf2 - row0);
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  const auto tv = lds_twiddles<T>(buf + P.count * P.stride, tw, nf1);
  for (int i = tid; i < P.count * P.stride; i += nt) buf[i] = fftc::mk((T)0, (T)0);
  PlaneWalk<> pw(g, p0, k0, k1, row0, row0 + nrows - 1);
  for (int pl = pw.next(); pl < k1; pl = pw.next()) {
    __syncthreads();  // the previous plane's rows are written
    mix_load_rows<T>(buf, H + h_plane(g, pl), g, P, row0, nrows, N1);
    __syncthreads();
    mix_stages<T, -1>(buf, P, tv, 0, 1);
    for (int r = 0; r < nrows; ++r) {
      cpx<T> *out = grid + ((size_t)pl * nf2 + row0 + r) * nf1;
      for (int i = tid; i < nf1; i += nt) out[i] = buf[r * P.stride + fftc::pad(i)];
    }
  }
}

// ms2dirty column pass (col_fwd_kernel's work): cpw columns, planes of a chunk
// last to first, Horner's rule in FP64; NO image cells per thread, MT threads at
// most (long FP32 columns only take more than 512, whose registers they halve).
template <typename T, int NO, int MT>
__global__ void __launch_bounds__(MT) col_fwd_mix_kernel(const cpx<T> *__restrict__ H,
                                                                          double2 *__restrict__ accT,
                                                                          const cpx<T> *__restrict__ tw, Geom g,
                                                                          fftm::Plan P, int p0, int nb, int first,
                                                                          int cpw_lg, int pchunk) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw);
  const int nf2 = g.nf2, N2 = g.N2, nt = blockDim.x, tid = threadIdx.x, cpw = 1 << cpw_lg;
  const int s0 = xcd_group(blockIdx.x, gridDim.x) << cpw_lg, cols = min(cpw, g.N1 - s0);
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk), nout = N2 << cpw_lg, nin = nf2 << cpw_lg;
  const auto tv = lds_twiddles<T>(buf + P.count * P.stride, tw, nf2);
  double ar[NO], ai[NO], er[NO], ei[NO];
#pragma unroll
  for (int q = 0; q < NO; ++q) {
    ar[q] = ai[q] = 0.0;
    const int o = tid + q * nt, c = o & (cpw - 1), row = o >> cpw_lg;
    sincos_cw(o < nout && c < cols ? pixel_zp(row, s0 + c, g) : 0.0, &ei[q], &er[q]);
  }
  for (int k = k1 - 1; k >= k0; --k) {
    const cpx<T> *hk = H + h_plane(g, k);
    const uint64_t occ = occ_mask(g, p0 + k);  // rows outside it are zero and not in H
    __syncthreads();  // the previous plane's LDS reads are done
    constexpr int B = 8;  // loads in flight
    auto load = [&](auto all) {
      for (int i0 = tid; i0 < nin; i0 += B * nt) {
        cpx<T> v[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int i = i0 + b * nt, c = i & (cpw - 1);
          const bool on = i < nin && c < cols && (all.value || occ_row(occ, i >> cpw_lg, g));
          v[b] = on ? hk[h_slot(g, s0 + c) + ((i >> cpw_lg) << kTileLog2)] : fftc::mk((T)0, (T)0);
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int i = i0 + b * nt;
          if (i < nin) buf[(i & (cpw - 1)) * P.stride + fftc::pad(i >> cpw_lg)] = v[b];
        }
      }
    };
    // the test of every row costs as much as the reads it saves on a fully occupied plane
    if (occ_full(occ, g))
      load(std::true_type());
    else
      load(std::false_type());
    __syncthreads();
    mix_stages<T, +1>(buf, P, tv, 0, 1);
#pragma unroll
    for (int q = 0; q < NO; ++q) {
      const int o = tid + q * nt;
      if (o < nout) {
        const cpx<T> f = buf[(o & (cpw - 1)) * P.stride + fftc::pad(grid_index(o >> cpw_lg, N2, nf2))];
        const double t = ar[q] * er[q] - ai[q] * ei[q] + (double)f.x;
        ai[q] = ar[q] * ei[q] + ai[q] * er[q] + (double)f.y;
        ar[q] = t;
      }
    }
  }
  double2 *out = accT + (size_t)blockIdx.y * g.N1 * N2;
  const double m = (double)(p0 + k0 - g.P / 2);
#pragma unroll
  for (int q = 0; q < NO; ++q) {
    const int o = tid + q * nt, c = o & (cpw - 1), row = o >> cpw_lg;
    if (o < nout && c < cols) {
      double sn, cs;
      sincos_cw(pixel_zp(row, s0 + c, g) * m, &sn, &cs);
      double2 r = make_double2(ar[q] * cs - ai[q] * sn, ar[q] * sn + ai[q] * cs);
      double2 *d = out + (size_t)(s0 + c) * N2 + row;
      if (!first) {
        r.x += d->x;
        r.y += d->y;
      }
      *d = r;
    }
  }
}

// dirty2ms column pass (col_inv_kernel's work): phased image cells carried from
// plane to plane in FP64, inverse FFT, full columns to H.
template <typename T, int NO, int MT>
__global__ void __launch_bounds__(MT) col_inv_mix_kernel(const cpx<T> *__restrict__ gT,
                                                                          cpx<T> *__restrict__ H,
                                                                          const cpx<T> *__restrict__ tw, Geom g,
                                                                          fftm::Plan P, int p0, int nb, int cpw_lg,
                                                                          int pchunk) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw);
  const int nf2 = g.nf2, N2 = g.N2, h2 = N2 / 2, nt = blockDim.x, tid = threadIdx.x, cpw = 1 << cpw_lg;
  const int s0 = xcd_group(blockIdx.x, gridDim.x) << cpw_lg, cols = min(cpw, g.N1 - s0);
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk), nin = N2 << cpw_lg, nout = nf2 << cpw_lg;
  const auto tv = lds_twiddles<T>(buf + P.count * P.stride, tw, nf2);
  double xr[NO], xi[NO], er[NO], ei[NO];
  const double m = (double)(p0 + k0 - g.P / 2);
#pragma unroll
  for (int q = 0; q < NO; ++q) {
    xr[q] = xi[q] = er[q] = ei[q] = 0.0;
    const int o = tid + q * nt, c = o & (cpw - 1), row = o >> cpw_lg;
    if (o < nin && c < cols) {
      const double zp = pixel_zp(row, s0 + c, g);
      double sn, cs;
      sincos_cw(-zp, &ei[q], &er[q]);
      sincos_cw(-zp * m, &sn, &cs);
      const cpx<T> gv = gT[(size_t)(s0 + c) * N2 + row];
      xr[q] = (double)gv.x * cs - (double)gv.y * sn;
      xi[q] = (double)gv.x * sn + (double)gv.y * cs;
    }
  }
  for (int k = k0; k < k1; ++k) {
    __syncthreads();  // the previous plane's LDS reads are done
#pragma unroll
    for (int q = 0; q < NO; ++q) {
      const int o = tid + q * nt;
      if (o < nin) {
        buf[(o & (cpw - 1)) * P.stride + fftc::pad(grid_index(o >> cpw_lg, N2, nf2))] = fftc::mk((T)xr[q], (T)xi[q]);
        const double t = xr[q] * er[q] - xi[q] * ei[q];
        xi[q] = xr[q] * ei[q] + xi[q] * er[q];
        xr[q] = t;
      }
    }
    for (int z = tid; z < (nf2 - N2) << cpw_lg; z += nt)
      buf[(z & (cpw - 1)) * P.stride + fftc::pad(N2 - h2 + (z >> cpw_lg))] = fftc::mk((T)0, (T)0);
    __syncthreads();
    mix_stages<T, -1>(buf, P, tv, 0, 1);
    cpx<T> *hk = H + h_plane(g, k);
    const uint64_t occ = occ_mask(g, p0 + k);
    for (int i = tid; i < nout; i += nt) {
      const int c = i & (cpw - 1), k2 = i >> cpw_lg;
      if (c < cols && occ_row(occ, k2, g)) hk[ht_slot(g, s0 + c) + ht_row(k2)] = buf[c * P.stride + fftc::pad(k2)];
    }
  }
}

// --------------------------------------------------------------------------
// launchers
// --------------------------------------------------------------------------
template <typename T> inline int mix_row_lds(const Geom &g, bool spread) {
  const int cells = g.rpw * fftm::seq_stride(g.nf1);
  return cells * (int)(spread && g.acc64 ? sizeof(double2) : sizeof(cpx<T>)) +
         fftc::twiddle_entries(g.nf1) * (int)sizeof(cpx<T>);
}
template <typename T> inline int mix_col_lds(const Geom &g, int cpw) {
  return (int)sizeof(cpx<T>) * (cpw * fftm::seq_stride(g.nf2) + fftc::twiddle_entries(g.nf2));
}
// f(cells per thread 8 or 16, threads at most 512 or 1024)
template <typename T, typename F> inline void with_cells(int cells, int nt, F f) {
  using std::integral_constant;
  if constexpr (sizeof(T) == 4) {
    if (nt > 512) {
      if (cells <= 8)
        f(integral_constant<int, 8>(), integral_constant<int, 1024>());
      else
        f(integral_constant<int, 16>(), integral_constant<int, 1024>());
      return;
    }
  }
  if (cells <= 8)
    f(integral_constant<int, 8>(), integral_constant<int, 512>());
  else
    f(integral_constant<int, 16>(), integral_constant<int, 512>());
}
inline int mix_cells(int cpw, int N2, int nt) { return (cpw * N2 + nt - 1) / nt; }

template <typename T>
void mix_spread_rows(const Rec<T> *recs, const T *taps, const int *off, const ChanPlan &cp, int p0, int nb, cpx<T> *H,
                     const cpx<T> *tw1, hipStream_t st) {
  const Geom &g = cp.g;
  const dim3 grd((g.nf2 + g.rpw - 1) / g.rpw, (nb + g.pch_row - 1) / g.pch_row, g.zrow);
  const int lb = mix_row_lds<T>(g, true), nt = cp.rowf.nt;
  if (g.zrow > 1) zero_planes<T>(H, g, nb, st);
  with_acc64<T>(g.acc64, [&](auto A) {
    if (g.kw <= 8)
      spread_row_mix_kernel<T, 8, A.value><<<grd, nt, lb, st>>>(recs, taps, off, H, tw1, g, cp.rowf, p0, nb, g.pch_row);
    else
      spread_row_mix_kernel<T, 16, A.value><<<grd, nt, lb, st>>>(recs, taps, off, H, tw1, g, cp.rowf, p0, nb, g.pch_row);
  });
}

template <typename T>
void mix_row_interp(const Rec<T> *recs, const T *taps, const int *off, const cpx<T> *H, void *grid, double2 *vacc,
                    const cpx<T> *tw1, const ChanPlan &cp, int p0, int nb, hipStream_t st) {
  const Geom &g = cp.g;
  const dim3 grd((g.nf2 + g.rpw - 1) / g.rpw, (nb + g.pch_row - 1) / g.pch_row);
  const int lb = mix_row_lds<T>(g, false), nt = cp.rowf.nt;
  if (g.gather) {
    cpx<T> *planes = (cpx<T> *)grid;
    row_planes_mix_kernel<T><<<grd, nt, lb, st>>>(H, planes, tw1, g, cp.rowf, p0, nb, g.pch_row);
    launch_gather<T>(recs, taps, off, planes, vacc, g, cp.nvalid, p0, nb, st);
    return;
  }
  if (g.kw <= 8)
    row_interp_mix_kernel<T, 8><<<grd, nt, lb, st>>>(H, recs, taps, off, vacc, tw1, g, cp.rowf, p0, nb, g.pch_row);
  else
    row_interp_mix_kernel<T, 16><<<grd, nt, lb, st>>>(H, recs, taps, off, vacc, tw1, g, cp.rowf, p0, nb, g.pch_row);
}

template <typename T>
void mix_cols_forward(const ChanPlan &cp, int p0, int nb, const cpx<T> *H, double2 *accT, const cpx<T> *tw2, int first,
                      hipStream_t st) {
  const Geom &g = cp.g;
  const int nt = cp.colf.nt, lb = mix_col_lds<T>(g, g.cpw), lg = 31 - __builtin_clz(g.cpw);
  const dim3 grd((g.N1 + g.cpw - 1) / g.cpw, (nb + g.pch_fwd - 1) / g.pch_fwd);
  with_cells<T>(mix_cells(g.cpw, g.N2, nt), nt, [&](auto NO, auto MT) {
    col_fwd_mix_kernel<T, NO.value, MT.value><<<grd, nt, lb, st>>>(H, accT, tw2, g, cp.colf, p0, nb, first, lg, g.pch_fwd);
  });
}

template <typename T>
void mix_cols_backward(const ChanPlan &cp, int p0, int nb, const cpx<T> *gT, cpx<T> *H, const cpx<T> *tw2,
                       hipStream_t st) {
  const Geom &g = cp.g;
  const int nt = cp.colf.nt, lb = mix_col_lds<T>(g, g.cpw), lg = 31 - __builtin_clz(g.cpw);
  const dim3 grd((g.N1 + g.cpw - 1) / g.cpw, (nb + g.pch_inv - 1) / g.pch_inv);
  with_cells<T>(mix_cells(g.cpw, g.N2, nt), nt, [&](auto NO, auto MT) {
    col_inv_mix_kernel<T, NO.value, MT.value><<<grd, nt, lb, st>>>(gT, H, tw2, g, cp.colf, p0, nb, lg, g.pch_inv);
  });
}

template <typename T> int allow_mix(const ChanPlan &cp) {
  const Geom &g = cp.g;
  const int top = MixThreads<T>::value, rows = cp.rowf.nt, cols = cp.colf.nt;
  // what the kernels assume of their launches
  if (cp.rowf.n != g.nf1 || cp.rowf.count != g.rpw || g.rpw > 64 || cp.colf.n != g.nf2 || cp.colf.count != g.cpw || rows < 64 ||
      rows > top || cols < 64 || cols > top || mix_cells(g.cpw, g.N2, cols) > 16 || g.pch_row < 1 || g.pch_fwd < 1 ||
      g.pch_inv < 1 || g.zrow < 1 || (g.cpw & (g.cpw - 1)) != 0) {
    set_error("mixed-radix plan of grid %d x %d does not fit its kernels", g.nf2, g.nf1);
    return kErrArg;
  }
  const int ls = mix_row_lds<T>(g, true), lr = mix_row_lds<T>(g, false), lc = mix_col_lds<T>(g, g.cpw);
  int ier = kOk;
  with_acc64<T>(g.acc64, [&](auto A) {
    ier = allow_lds(spread_row_mix_kernel<T, 8, A.value>, ls);
    if (ier == kOk) ier = allow_lds(spread_row_mix_kernel<T, 16, A.value>, ls);
  });
  CURIG_TRY(ier);
  CURIG_TRY((allow_lds(row_interp_mix_kernel<T, 8>, lr)));
  CURIG_TRY((allow_lds(row_interp_mix_kernel<T, 16>, lr)));
  CURIG_TRY((allow_lds(row_planes_mix_kernel<T>, lr)));
  with_cells<T>(mix_cells(g.cpw, g.N2, cols), cols, [&](auto NO, auto MT) {
    ier = allow_lds(col_fwd_mix_kernel<T, NO.value, MT.value>, lc);
    if (ier == kOk) ier = allow_lds(col_inv_mix_kernel<T, NO.value, MT.value>, lc);
  });
  return ier;
}

#define CURIG_MIX_INST(T)                                                                                          \
  template void mix_spread_rows<T>(const Rec<T> *, const T *, const int *, const ChanPlan &, int, int, cpx<T> *,   \
                                   const cpx<T> *, hipStream_t);                                                   \
  template void mix_row_interp<T>(const Rec<T> *, const T *, const int *, const cpx<T> *, void *, double2 *,       \
                                  const cpx<T> *, const ChanPlan &, int, int, hipStream_t);                        \
  template void mix_cols_forward<T>(const ChanPlan &, int, int, const cpx<T> *, double2 *, const cpx<T> *, int,    \
                                    hipStream_t);                                                                  \
  template void mix_cols_backward<T>(const ChanPlan &, int, int, const cpx<T> *, cpx<T> *, const cpx<T> *,         \
                                     hipStream_t);                                                                 \
  template int allow_mix<T>(const ChanPlan &);

}  // namespace curig
