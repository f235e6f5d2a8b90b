// Record passes of the row kernels that hold one or several whole grid rows in
// LDS (padded, fftc::pad): the spread of every record that touches the rows in
// one plane, summed in FP64, and the interpolation from them; and the gather of
// whole records from full planes.
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

// plane tap of a record in plane p, or -1
__device__ __forceinline__ int plane_tap(int iw, int p, const Geom &g) {
  int k = p - iw;
  if (k < 0) k += g.P;
  return k < g.kww ? k : -1;
}

// The spread sums in FP64 in LDS.  FP32 rows either in complex cells (ACC64:
// twice the LDS of a row, each record read once), or one component after the
// other in cells of one double (parts: the LDS of a row, each record read twice).
// Sums in FP32 and in integers scaled by a block's bound lose digits as records
// share its cells: 47,000 rows of noise within 4 cells of the centre of a 1200^2
// grid, error against 64 bits 1.1e-6 (float), 1.3e-5 (int32, 30 bits of a 16-cell
// block's bound), 1.4e-7 (FP64).  Integers / FP64 components: 1500 x 1100 image,
// 43 record visits per row and plane, 1.05 / 1.11 ms per 32 planes; 1024^2, 94
// visits, 0.26 / 0.24 ms.
template <typename T, bool ACC64> struct RowAcc {
  static constexpr bool parts = sizeof(T) == 4 && !ACC64;
  using cell = typename std::conditional<parts, double, cpx<double>>::type;
};
enum { kBoth = 0, kReal = 1, kImag = 2 };  // what a pass of the spread adds to the cells

// Record t of a walk is handled by this thread for t = walk_first(), + walk_step():
// the grid's z workgroups of a row share its records.
__device__ __forceinline__ int walk_first() { return threadIdx.x + blockIdx.z * blockDim.x; }
__device__ __forceinline__ int walk_step() { return blockDim.x * gridDim.z; }

// Spread into rows [row0, row0 + nrows) of plane p at buf + r * stride: complex
// cells (COMP kBoth) or one component.
template <int COMP, typename T, int KWM, typename Cell>
__device__ __forceinline__ void spread_records(const WalkTable &wt, int total, const Rec<T> *__restrict__ recs,
                                               const T *__restrict__ taps, const Geom &g, int p, int row0, int nrows,
                                               Cell *buf, int stride) {
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
    for (int r = 0; r < nrows; ++r) {
      int jj = row0 + r - rc.iy;
      if (jj < 0) jj += nf2;
      if (jj >= kw) continue;
      const T a = kz * tq[KWM + jj], vre = rc.re * a, vim = rc.im * a;
      Cell *row = buf + r * stride;
#pragma unroll
      for (int i = 0; i < KWM; ++i) {
        if (i < kw) {
          int cx = rc.ix + i;
          if (cx >= nf1) cx -= nf1;
          if constexpr (COMP == kBoth) {
            Cell *d = row + fftc::pad(cx);
            atomicAdd(&d->x, vre * kx[i]);
            atomicAdd(&d->y, vim * kx[i]);
          } else {
            atomicAdd(row + fftc::pad(cx), (double)((COMP == kReal ? vre : vim) * kx[i]));
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
