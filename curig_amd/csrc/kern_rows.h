// Record passes of the row kernels that hold one or several whole grid rows in
// LDS (padded, fftc::pad): the spread of every record that touches the rows in
// one plane, with its block-floating-point scaling in FP32, and the interpolation
// from them; and the gather of whole records from full planes.
#pragma once
#include "kern_lds.h"

namespace curig {

// Row group of this workgroup: blocks of four rows (whole lines of H), of 16 on
// grids of 2048 rows and more (they share most of their records), are dealt to the
// XCDs in turn.  Most records lie in the rows around 0, the grid's first and last,
// which a contiguous range each gave to two XCDs of the eight: 1024^2 gradient, rows
// 796 -> 706 us; 3000 x 2500 FP64 prediction 10.97 -> 9.5 ms; 20M uniform points
// 2.69 -> 2.73 ms.
__device__ __forceinline__ int row_group(const Geom &g) {
  const int rows = g.nf2 >= 2048 ? 16 : 4;
  return xcd_interleave(blockIdx.x, gridDim.x, max(1, rows / g.rpw));
}

// blocks of the block-floating-point spread per row
__host__ __device__ inline int fix_row_blocks(int nf1) { return (nf1 + (1 << kFixBlkLog2) - 1) >> kFixBlkLog2; }

// Blocks of the cells ix .. ix + kw - 1 (cyclic, kw <= 16): at most b0, the
// row's last block (when they wrap) and the last cell's.
struct FixBlocks {
  int b0, bm, b1;
};
__device__ __forceinline__ FixBlocks fix_blocks(int ix, int kw, int nf1) {
  FixBlocks f;
  const int last = ix + kw - 1;
  f.b0 = ix >> kFixBlkLog2;
  f.bm = last >= nf1 ? (nf1 - 1) >> kFixBlkLog2 : f.b0;
  f.b1 = (last >= nf1 ? last - nf1 : last) >> kFixBlkLog2;
  return f;
}

// plane tap of a record in plane p, or -1
__device__ __forceinline__ int plane_tap(int iw, int p, const Geom &g) {
  int k = p - iw;
  if (k < 0) k += g.P;
  return k < g.kww ? k : -1;
}

// How the spread accumulates: kAccFix (FP32; a bound pass over the records, then
// integers), or FP64 sums: in FP64, and in FP32 where the records are dense
// (Geom::acc64), whose rows read every record from far memory and would read it
// twice for the bounds.
template <typename T, bool ACC64> struct RowAcc {
  static constexpr bool fix = sizeof(T) == 4 && !ACC64;
  using cell = cpx<typename std::conditional<ACC64, double, T>::type>;  // a cell's LDS element
};

// Record t of a walk is handled by this thread for t = walk_first(), + walk_step():
// the grid's z workgroups of a row share its records.
__device__ __forceinline__ int walk_first() { return threadIdx.x + blockIdx.z * blockDim.x; }
__device__ __forceinline__ int walk_step() { return blockDim.x * gridDim.z; }

// Bound pass of the block-floating-point spread (bound_row_part's bound) over
// the workgroup's rows: bsum[r * nblk + block].
template <typename T, int KWM>
__device__ __forceinline__ void bound_records(const WalkTable &wt, int total, const Rec<T> *__restrict__ recs,
                                              const T *__restrict__ taps, const Geom &g, int p, int row0, int nrows,
                                              float *fixt, int nblk) {
  const int kw = g.kw, nf1 = g.nf1, nf2 = g.nf2;
  for (int t = walk_first(); t < total; t += walk_step()) {
    const int ia = walk_record(wt, t);
    const Rec<T> rc = recs[ia];
    const int k = plane_tap(rc.iw, p, g);
    if (k < 0) continue;
    const T *tq = taps + (size_t)ia * (3 * KWM);
    const float a = (fabsf((float)rc.re) + fabsf((float)rc.im)) * fabsf((float)tq[2 * KWM + k]);
    const FixBlocks f = fix_blocks(rc.ix, kw, nf1);
    for (int r = 0; r < nrows; ++r) {
      int jj = row0 + r - rc.iy;
      if (jj < 0) jj += nf2;
      if (jj >= kw) continue;
      const float b = a * fabsf((float)tq[KWM + jj]);
      float *bs = fixt + r * nblk;
      atomicAdd(bs + f.b0, b);
      if (f.bm != f.b0) atomicAdd(bs + f.bm, b);
      if (f.b1 != f.b0 && f.b1 != f.bm) atomicAdd(bs + f.b1, b);
    }
  }
}

// the blocks' exponents for the first FFT stage, published by the caller's next
// barrier; *fixnan set when a bound is not finite
__device__ __forceinline__ void block_exponents(const float *fixt, short *fixe, int n, int *fixnan) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int e = fix_block_exp(fixt[i]);
    fixe[i] = (short)(e == kFixNaN ? 0 : e);
    if (e == kFixNaN) *fixnan = 1;
  }
}

// Spread into rows [row0, row0 + nrows) of plane p at buf + r * stride, as
// RowAcc accumulates (integers after bound_records).
template <typename T, int KWM, bool ACC64>
__device__ __forceinline__ void spread_records(const WalkTable &wt, int total, const Rec<T> *__restrict__ recs,
                                               const T *__restrict__ taps, const Geom &g, int p, int row0, int nrows,
                                               typename RowAcc<T, ACC64>::cell *buf, int stride, const float *fixt, int nblk) {
  using Cell = typename RowAcc<T, ACC64>::cell;
  constexpr bool kFix = RowAcc<T, ACC64>::fix;
  const int kw = g.kw, nf1 = g.nf1, nf2 = g.nf2;
  for (int t = walk_first(); t < total; t += walk_step()) {
    const int ia = walk_record(wt, t);
    const Rec<T> rc = recs[ia];
    const int k = plane_tap(rc.iw, p, g);
    if (k < 0) continue;
    const T *tq = taps + (size_t)ia * (3 * KWM);
    T kx[KWM];
#pragma unroll
    for (int i = 0; i < KWM; ++i) kx[i] = tq[i];
    const T kz = tq[2 * KWM + k];
    const FixBlocks f = kFix ? fix_blocks(rc.ix, kw, nf1) : FixBlocks{};
    for (int r = 0; r < nrows; ++r) {
      int jj = row0 + r - rc.iy;
      if (jj < 0) jj += nf2;
      if (jj >= kw) continue;
      const T a = kz * tq[KWM + jj], vre = rc.re * a, vim = rc.im * a;
      Cell *row = buf + r * stride;
      int e0 = 0, em = 0, e1 = 0;
      if (kFix) {
        const float *bs = fixt + r * nblk;
        e0 = fix_block_exp(bs[f.b0]);
        em = fix_block_exp(bs[f.bm]);
        e1 = fix_block_exp(bs[f.b1]);
        e0 = e0 == kFixNaN ? 0 : e0;
        em = em == kFixNaN ? 0 : em;
        e1 = e1 == kFixNaN ? 0 : e1;
      }
#pragma unroll
      for (int i = 0; i < KWM; ++i) {
        if (i < kw) {
          int cx = rc.ix + i;
          if (cx >= nf1) cx -= nf1;
          const T re = vre * kx[i], im = vim * kx[i];
          if (kFix) {
            const int blk = cx >> kFixBlkLog2, e = blk == f.b0 ? e0 : blk == f.bm ? em : e1;
            int *d = reinterpret_cast<int *>(row + fftc::pad(cx));
            atomicAdd(d, __float2int_rn(ldexpf((float)re, e)));
            atomicAdd(d + 1, __float2int_rn(ldexpf((float)im, e)));
          } else {
            Cell *d = row + fftc::pad(cx);
            atomicAdd(&d->x, re);
            atomicAdd(&d->y, im);
          }
        }
      }
    }
  }
}

// Interpolation of every record that touches the rows: its share, summed over
// the rows, added to its FP64 accumulator.
template <typename T, int KWM>
__device__ __forceinline__ void interp_records(const WalkTable &wt, int total, const Rec<T> *__restrict__ recs,
                                               const T *__restrict__ taps, const Geom &g, int p, int row0, int nrows,
                                               const cpx<T> *buf, int stride, double2 *__restrict__ vacc) {
  const int nt = blockDim.x, kw = g.kw, nf1 = g.nf1, nf2 = g.nf2;
  for (int t = threadIdx.x; t < total; t += nt) {
    const int ia = walk_record(wt, t);
    const Rec<T> rc = recs[ia];
    const int k = plane_tap(rc.iw, p, g);
    if (k < 0) continue;
    const T *tq = taps + (size_t)ia * (3 * KWM);
    T kx[KWM];
#pragma unroll
    for (int i = 0; i < KWM; ++i) kx[i] = tq[i];
    const T kz = tq[2 * KWM + k];
    T sr = 0, si = 0;
    bool hit = false;
    for (int r = 0; r < nrows; ++r) {
      int jj = row0 + r - rc.iy;
      if (jj < 0) jj += nf2;
      if (jj >= kw) continue;
      hit = true;
      const cpx<T> *row = buf + r * stride;
      T rr = 0, ri = 0;
#pragma unroll
      for (int i = 0; i < KWM; ++i) {
        if (i < kw) {
          int cx = rc.ix + i;
          if (cx >= nf1) cx -= nf1;
          const cpx<T> f = row[fftc::pad(cx)];
          rr += f.x * kx[i];
          ri += f.y * kx[i];
        }
      }
      const T ky = tq[KWM + jj];
      sr += rr * ky;
      si += ri * ky;
    }
    if (hit) {
      atomicAdd(&vacc[ia].x, (double)(sr * kz));
      atomicAdd(&vacc[ia].y, (double)(si * kz));
    }
  }
}

// KWM lanes per record, lane i at tap i of each row of its support: a row's
// cells are then one or two lines, where a thread per record touched a line per
// lane and load (11-wide kernel, FP64, 220,000 records on a 250 x 360 grid:
// 1,490 us in the fused row pass, 1,080 with eight lanes each at rows of their own,
// 560 so).  The x tap multiplies the lane's sum at the end.
template <typename T, int KWM>
__global__ void __launch_bounds__(256) interp_gather_kernel(const Rec<T> *__restrict__ recs,
                                                            const T *__restrict__ taps, const int *__restrict__ off,
                                                            const cpx<T> *__restrict__ grid,
                                                            double2 *__restrict__ vacc, Geom g, int p0, int nb) {
  int ra0, ra1, rb0, rb1;
  layer_ranges(off, g, imod(p0 - g.kww + 1, g.P), nb + g.kww - 1, ra0, ra1, rb0, rb1);
  const long n0 = ra1 - ra0, ntot = n0 + (rb1 - rb0);
  const int lane = threadIdx.x & (KWM - 1), kw = g.kw, nf1 = g.nf1, nf2 = g.nf2;
  const size_t plane = (size_t)nf1 * nf2;
  const long step = (long)gridDim.x * blockDim.x / KWM;
  for (long t = (blockIdx.x * (long)blockDim.x + threadIdx.x) / KWM; t < ntot; t += step) {
    const int r = t < n0 ? ra0 + (int)t : rb0 + (int)(t - n0);
    const int ix = recs[r].ix, iy = recs[r].iy, iw = recs[r].iw;
    const T *tq = taps + (size_t)r * (3 * KWM);
    const T kx = tq[lane];  // zero beyond the kernel width
    int cx = ix + lane;
    if (cx >= nf1) cx -= nf1;
    T ky[KWM];
#pragma unroll
    for (int i = 0; i < KWM; ++i) ky[i] = tq[KWM + i];
    double sr = 0.0, si = 0.0;
    for (int k = 0; k < g.kww; ++k) {
      int p = iw + k;
      if (p >= g.P) p -= g.P;
      if (p < p0 || p >= p0 + nb) continue;
      const cpx<T> *col = grid + (size_t)(p - p0) * plane + cx;
      const T kz = tq[2 * KWM + k];
      T rr = 0, ri = 0;
#pragma unroll
      for (int jj = 0; jj < KWM; ++jj) {
        if (jj < kw) {
          int cy = iy + jj;
          if (cy >= nf2) cy -= nf2;
          const cpx<T> f = col[(size_t)cy * nf1];
          rr += f.x * ky[jj];
          ri += f.y * ky[jj];
        }
      }
      sr += (double)(rr * kz);
      si += (double)(ri * kz);
    }
    sr = lane < kw ? sr * (double)kx : 0.0;
    si = lane < kw ? si * (double)kx : 0.0;
#pragma unroll
    for (int m = KWM / 2; m > 0; m >>= 1) {
      sr += __shfl_xor(sr, m, 64);
      si += __shfl_xor(si, m, 64);
    }
    if (lane == 0) {
      const double2 o = vacc[r];
      vacc[r] = make_double2(o.x + sr, o.y + si);
    }
  }
}

// f(std::integral_constant<bool, ACC64>()): the flag is set for FP32 only
template <typename T, typename F> inline void with_acc64(bool acc64, F f) {
  if constexpr (sizeof(T) == 4) {
    if (acc64) return f(std::true_type());
  }
  f(std::false_type());
}

// clears the batch's planes, for rows whose records several workgroups share
template <typename T> inline void zero_planes(cpx<T> *H, const Geom &g, int nb, hipStream_t st) {
  launch_fill_zero_c128(reinterpret_cast<double2 *>(H), (long)((size_t)nb * g.nct * g.tstride * sizeof(cpx<T>) / 16), st);
}

template <typename T>
void launch_gather(const Rec<T> *recs, const T *taps, const int *off, const cpx<T> *planes, double2 *vacc, const Geom &g,
                   long nvalid, int p0, int nb, hipStream_t st) {
  const int nbk = nblocks(nvalid * (g.kw <= 8 ? 8 : 16), 256, 1 << 16);
  if (g.kw <= 8)
    interp_gather_kernel<T, 8><<<nbk, 256, 0, st>>>(recs, taps, off, planes, vacc, g, p0, nb);
  else
    interp_gather_kernel<T, 16><<<nbk, 256, 0, st>>>(recs, taps, off, planes, vacc, g, p0, nb);
}

// output x of a row pass: stored, or added where several workgroups share the row
template <typename T> __device__ __forceinline__ void put_row(cpx<T> *d, cpx<T> x, bool add) {
  if (add) {
    atomicAdd(&d->x, x.x);
    atomicAdd(&d->y, x.y);
  } else {
    *d = x;
  }
}

}  // namespace curig
