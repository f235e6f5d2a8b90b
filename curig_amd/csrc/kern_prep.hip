// Preparation kernels: w range of the rows, binning of rows into sorted
// records (count, scan, scatter), fills.
#include "dev_common.h"

namespace curig {

// --------------------------------------------------------------------------
// prep kernels
// --------------------------------------------------------------------------
// Per-block min / max of w (metres) over unflagged rows.
__global__ void __launch_bounds__(256) w_minmax_kernel(const double *__restrict__ uvw, int nrow,
                                                        const uint8_t *__restrict__ flag, long fs,
                                                        double *__restrict__ part, int *__restrict__ cnt) {
  __shared__ double smin[256], smax[256];
  __shared__ int scnt[256];
  double lo = INFINITY, hi = -INFINITY;
  int n = 0;
  for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < nrow; j += (long)gridDim.x * blockDim.x) {
    if (row_skipped(flag, fs, j)) continue;
    double w = uvw[3 * j + 2];
    // NaN propagates to the host check through the sum of |u|+|v|+|w|
    double a = uvw[3 * j] + uvw[3 * j + 1];
    if (!(fabs(a) < INFINITY) || !(fabs(w) < INFINITY)) {
      lo = NAN;
      hi = NAN;
    } else if (lo == lo) {
      lo = fmin(lo, w);
      hi = fmax(hi, w);
    }
    ++n;
  }
  smin[threadIdx.x] = lo;
  smax[threadIdx.x] = hi;
  scnt[threadIdx.x] = n;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      double a = smin[threadIdx.x], b = smin[threadIdx.x + s];
      smin[threadIdx.x] = (a != a || b != b) ? NAN : fmin(a, b);
      a = smax[threadIdx.x];
      b = smax[threadIdx.x + s];
      smax[threadIdx.x] = (a != a || b != b) ? NAN : fmax(a, b);
      scnt[threadIdx.x] += scnt[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = smin[0];
    part[2 * blockIdx.x + 1] = smax[0];
    cnt[blockIdx.x] = scnt[0];
  }
}

// uvw = scale * columns (null: zeros)
__global__ void __launch_bounds__(256) pack_columns_kernel(Columns c, double *__restrict__ uvw, int n) {
  for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x)
#pragma unroll
    for (int i = 0; i < 3; ++i) uvw[3 * j + i] = c.c[i] ? c.scale * c.c[i][j] : 0.0;
}

__global__ void fill_int_kernel(int *__restrict__ p, long n, int v) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void fill_zero_c128_kernel(double2 *__restrict__ p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    p[i] = make_double2(0.0, 0.0);
}

// Count rows per bin; each row keeps its rank inside the bin (GM-sort idea).
__global__ void __launch_bounds__(256) bin_count_kernel(const double *__restrict__ uvw, int nrow,
                                                         const uint8_t *__restrict__ flag, long fs, Geom g,
                                                         int *__restrict__ hist, int2 *__restrict__ binrank) {
  for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < nrow; j += (long)gridDim.x * blockDim.x) {
    if (row_skipped(flag, fs, j)) {
      binrank[j] = make_int2(-1, 0);
      continue;
    }
    Coords c = row_coords(uvw, j, g);
    int b = row_bin(c, g);
    int r = atomicAdd(&hist[b], 1);
    binrank[j] = make_int2(b, r);
  }
}

// The same for rows that are several to a bin, where the atomics on few addresses
// bound the count: a workgroup counts its chunk of rows in LDS, adds its bins to
// the histogram once and gives its rows their ranks from there.  bin_count_kernel
// and here: 20M points in 4096 bins 1.32 and 0.18 ms; 1.03M rows of an array (most
// of them in few bins) in 9216 bins 86 and 28 us; 31,744 in 1024 bins 15 and 5 us.
__global__ void __launch_bounds__(1024) bin_count_lds_kernel(const double *__restrict__ uvw, int nrow,
                                                              const uint8_t *__restrict__ flag, long fs, Geom g,
                                                              int nbins, int chunk, int *__restrict__ hist,
                                                              int2 *__restrict__ binrank) {
  extern __shared__ int cnt[];
  const long j0 = blockIdx.x * (long)chunk, j1 = j0 + chunk < nrow ? j0 + chunk : nrow;
  for (int i = threadIdx.x; i < nbins; i += blockDim.x) cnt[i] = 0;
  __syncthreads();
  for (long j = j0 + threadIdx.x; j < j1; j += blockDim.x) {
    int2 br = make_int2(-1, 0);
    if (!row_skipped(flag, fs, j)) {
      br.x = row_bin(row_coords(uvw, j, g), g);
      br.y = atomicAdd(&cnt[br.x], 1);
    }
    binrank[j] = br;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nbins; i += blockDim.x) {
    const int c = cnt[i];
    cnt[i] = c ? atomicAdd(&hist[i], c) : 0;
  }
  __syncthreads();
  for (long j = j0 + threadIdx.x; j < j1; j += blockDim.x) {  // the rows this thread counted
    const int2 br = binrank[j];
    if (br.x >= 0) binrank[j].y = br.y + cnt[br.x];
  }
}

// Exclusive scan of n ints: three passes (block sums, scan of sums, apply).

__global__ void __launch_bounds__(kScanBlock) scan_reduce_kernel(const int *__restrict__ in, long n,
                                                                  int *__restrict__ bsum) {
  __shared__ int s[kScanBlock];
  long base = (long)blockIdx.x * kScanTile;
  int acc = 0;
  for (int k = 0; k < kScanItems; ++k) {
    long i = base + (long)k * kScanBlock + threadIdx.x;
    if (i < n) acc += in[i];
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int st = kScanBlock / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = s[0];
}

// single block: exclusive scan of nb block sums in place
__global__ void __launch_bounds__(1024) scan_sums_kernel(int *__restrict__ bsum, int nb) {
  __shared__ int s[1024];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nb; base += 1024) {
    int i = base + threadIdx.x;
    int v = i < nb ? bsum[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      int t = threadIdx.x >= off ? s[threadIdx.x - off] : 0;
      __syncthreads();
      s[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nb) bsum[i] = carry + s[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry += s[1023];
    __syncthreads();
  }
}

// out[i] = bsum[block] + exclusive scan within the tile; out[n] = total
__global__ void __launch_bounds__(kScanBlock) scan_apply_kernel(const int *__restrict__ in, long n,
                                                                 const int *__restrict__ bsum,
                                                                 int *__restrict__ out, int total) {
  __shared__ int s[kScanBlock];
  long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
  int loc[kScanItems];
  int sum = 0;
  for (int k = 0; k < kScanItems; ++k) {
    long i = base + k;
    loc[k] = i < n ? in[i] : 0;
    sum += loc[k];
  }
  s[threadIdx.x] = sum;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    int t = threadIdx.x >= off ? s[threadIdx.x - off] : 0;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  int run = bsum[blockIdx.x] + s[threadIdx.x] - sum;
  for (int k = 0; k < kScanItems; ++k) {
    long i = base + k;
    if (i < n) out[i] = run;
    run += loc[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = total;
}

// Whether any of the bins [s0, s1] of layer l holds a record
__device__ __forceinline__ bool strips_hold(const int *off, const Geom &g, int l, int s0, int s1) {
  return off[l * g.ntiles + s1 + 1] > off[l * g.ntiles + s0];
}

// Geom::occ of plane p from the bin offsets (full-width row strips, LDS path), by a
// wavefront, a lane per block of rows.  The records that reach rows [r0, r1] of
// plane p have iy in [r0 - kw + 1, r1] and iw in [p - kww + 1, p], both cyclic;
// the answer is that of their bins, so it holds every row and plane whose walk
// (walk_table_build) finds a record.
// An observation leaves rows of the grid empty: a 128-antenna, 5 km array on
// 8192^2 pixels of 6 degrees reaches 63% of its rows and planes.  The row passes
// leave the empty ones out and H without them, and the column passes neither read
// nor write them: 32 planes of 16384^2, image rows 21.0 -> 13.5 ms and columns 14.4
// -> 12.4, prediction rows 14.1 -> 10.7; 8192^2, 66% occupied, rows 5.05 -> 3.97
// ms, columns 3.13 -> 2.86 per 26 planes.
__device__ __forceinline__ void occ_plane(const int *off, const Geom &g, int p, uint64_t *__restrict__ occ) {
  const int b = threadIdx.x & 63;
  const int r0 = b << g.occ_lg, r1 = min(g.nf2, r0 + (1 << g.occ_lg)) - 1;
  bool any = false;
  if (r0 < g.nf2) {
    // [lo, hi] and, wrapped below row 0, [wl, nf2 - 1]
    const int lo = r0 - g.kw + 1, wl = lo < 0 ? max(lo + g.nf2, 0) : g.nf2;
    const int a0 = max(lo, 0) / g.T2, a1 = r1 / g.T2, b0 = wl / g.T2, b1 = (g.nf2 - 1) / g.T2;
    // layers of planes pl .. p, and wrapped ones wp .. P - 1
    const int pl = p - g.kww + 1, wp = pl < 0 ? max(pl + g.P, 0) : g.P;
    for (int l = max(pl, 0) / g.Pbin; l <= p / g.Pbin; ++l)
      any = any || strips_hold(off, g, l, a0, a1) || (wl < g.nf2 && strips_hold(off, g, l, b0, b1));
    if (wp < g.P)
      for (int l = wp / g.Pbin; l <= (g.P - 1) / g.Pbin; ++l)
        any = any || strips_hold(off, g, l, a0, a1) || (wl < g.nf2 && strips_hold(off, g, l, b0, b1));
  }
  const uint64_t m = __ballot(any);
  if (b == 0) occ[p] = m;
}

__global__ void __launch_bounds__(256) occ_kernel(const int *__restrict__ off, Geom g, uint64_t *__restrict__ occ) {
  const int p = (int)((blockIdx.x * (long)blockDim.x + threadIdx.x) >> 6);
  if (p < g.P) occ_plane(off, g, p, occ);
}

// The scan of few bins (kSmallScan at most) and the occupied blocks, in one
// workgroup: a small image's call is as long as its launches, and four were here
// (256^2 image 151 -> 138 us a call, prediction 120 -> 110).
constexpr int kSmallScan = 16384;
__global__ void __launch_bounds__(1024) scan_small_kernel(const int *__restrict__ in, int n, int *out, int total, Geom g,
                                                           uint64_t *__restrict__ occ) {
  __shared__ int ws[16];
  const int items = (n + 1023) / 1024, base = threadIdx.x * items, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int loc[kSmallScan / 1024], sum = 0;
#pragma unroll
  for (int k = 0; k < kSmallScan / 1024; ++k) {
    loc[k] = k < items && base + k < n ? in[base + k] : 0;
    sum += loc[k];
  }
  int run = sum;  // inclusive over the wavefront
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(run, d);
    if (lane >= d) run += t;
  }
  if (lane == 63) ws[wave] = run;
  __syncthreads();
  run -= sum;
  for (int w = 0; w < wave; ++w) run += ws[w];
#pragma unroll
  for (int k = 0; k < kSmallScan / 1024; ++k) {
    if (k < items && base + k < n) out[base + k] = run;
    run += loc[k];
  }
  if (threadIdx.x == 0) out[n] = total;
  if (!occ) return;
  __threadfence_block();
  __syncthreads();
  for (int p = wave; p < g.P; p += 16) occ_plane(out, g, p, occ);
}

// Scatter rows into bin order; slot[j] (dirty2ms): row j's record, or -1; the
// value carries the weight and e^{+i D w}
// (ms2dirty pre-stages, src/astro/ra_exec.cu:98-110).
// taps (LDS path, else null): each record's kernel values at its KP cells per
// axis, [nrec][3][KP] (x, y, w; zero beyond the kernel width; the w taps are
// 1, 0, ... in the 2-D form), evaluated from the rounded offsets stored in the
// record, so the row kernels read what they would compute.
template <typename T, int KP>
__global__ void __launch_bounds__(256) bin_scatter_kernel(const double *__restrict__ uvw, int nrow,
                                                           const void *__restrict__ vis, long vs,
                                                           const void *__restrict__ wgt, long ws, Geom g,
                                                           const int2 *__restrict__ binrank,
                                                           const int *__restrict__ off, Rec<T> *__restrict__ recs,
                                                           int *__restrict__ slot, int with_value,
                                                           T *__restrict__ taps) {
  for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < nrow; j += (long)gridDim.x * blockDim.x) {
    int2 br = binrank[j];
    int dst = br.x < 0 ? -1 : off[br.x] + br.y;
    if (!with_value) slot[j] = dst;
    if (dst < 0) continue;
    Coords c = row_coords(uvw, j, g);
    Rec<T> r;
    r.ix = c.ix;
    r.iy = c.iy;
    r.iw = c.iw;
    r.dx = (T)c.dx;
    r.dy = (T)c.dy;
    r.dw = (T)c.dw;
    if (with_value) {
      double2 v = load_c<T>(vis, j * vs);
      double wt = wgt ? load_r<T>(wgt, j * ws) : 1.0;
      double s, co;
      sincos(g.D * c.we, &s, &co);
      r.re = (T)(wt * (v.x * co - v.y * s));
      r.im = (T)(wt * (v.x * s + v.y * co));
    } else {
      r.re = 0;
      r.im = 0;
    }
    recs[dst] = r;
    if (taps) {
      const Ker<T> K = make_ker<T>(g);
      T kx[KP], ky[KP], kz[KP];
      K.template taps<KP>(r.dx, kx);
      K.template taps<KP>(r.dy, ky);
      if (g.kww == 1) {
#pragma unroll
        for (int i = 0; i < KP; ++i) kz[i] = i == 0 ? (T)1 : (T)0;
      } else {
        K.template taps<KP>(r.dw, kz);
      }
      T *o = taps + (size_t)dst * (3 * KP);
#pragma unroll
      for (int i = 0; i < KP; ++i) {
        o[i] = kx[i];
        o[KP + i] = ky[i];
        o[2 * KP + i] = kz[i];
      }
    }
  }
}

// Whether the block of rows blockIdx.y of plane blockIdx.x is crowded (Geom::crowd; the
// others that occ has are Geom::plain's): more than kFixRecords records reach a row
// of it in one block of 16 cells (of a row part: m cells).  A sample of the records
// that reach the block's rows is counted by cell block and by groups of eight first
// rows; a row's records lie in two neighbouring groups, three for kernels beyond 8.
constexpr int kCrowdSample = 1024, kCrowdGroups = (256 + 15 + 7) / 8;
__global__ void __launch_bounds__(256) crowd_kernel(const int *__restrict__ off, const Rec<float> *__restrict__ recs,
                                                    Geom g, int m, const uint64_t *__restrict__ occ,
                                                    uint64_t *__restrict__ crowd, uint64_t *__restrict__ plain) {
  __shared__ int hist[kCrowdGroups][256];
  const int p = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  if (!(occ[p] >> b & 1)) return;
  const int r0 = b << g.occ_lg, rows = min(g.nf2 - r0, 1 << g.occ_lg), s1 = (r0 + rows - 1) / g.T2;
  // the runs of records in bins of strips [a, s1], [w, nty - 1], planes [pl, p], [wp, P - 1] (occ_plane)
  const int lo = r0 - g.kw + 1, a = max(lo, 0) / g.T2, w = lo < 0 ? max(lo + g.nf2, 0) / g.T2 : g.nty;
  const int pl = p - g.kww + 1, wp = pl < 0 ? max(pl + g.P, 0) : g.P;
  auto runs = [&](auto f) {
    auto layer = [&](int l) {
      const int *o = off + l * g.ntiles;
      f(o[a], o[s1 + 1]);
      if (w < g.nty) f(o[w], o[g.nty]);
    };
    for (int l = max(pl, 0) / g.Pbin; l <= p / g.Pbin; ++l) layer(l);
    if (wp < g.P)
      for (int l = wp / g.Pbin; l <= (g.P - 1) / g.Pbin; ++l) layer(l);
  };
  long n = 0;
  runs([&](int i0, int i1) { n += i1 - i0; });
  bool full = false;
  if (n > kFixRecords) {
    const int groups = (rows + g.kw + 6) >> 3, step = (int)((n + kCrowdSample - 1) / kCrowdSample);
    for (int i = 0; i < groups; ++i) hist[i][tid] = 0;
    __syncthreads();
    long at = 0;  // records before the run: every step-th of all runs is taken
    runs([&](int i0, int i1) {
      for (long i = (at + step - 1) / step + tid; i * step < at + i1 - i0; i += blockDim.x) {
        const Rec<float> &rc = recs[i0 + (i * step - at)];
        const int dy = imod(rc.iy - lo, g.nf2), dz = imod(p - rc.iw, g.P), ix = rc.ix;
        if (dy >= rows + g.kw - 1 || dz >= g.kww) continue;
        const int c0 = (ix & (m - 1)) >> 4, c1 = ((ix + g.kw - 1) & (m - 1)) >> 4;
        atomicAdd(&hist[dy >> 3][c0], 1);
        if (c1 != c0) atomicAdd(&hist[dy >> 3][c1], 1);
      }
      at += i1 - i0;
    });
    __syncthreads();
    const long most = kFixRecords / step;
    int x = 0, y = 0;
    for (int i = 0; i < groups; ++i) {
      const int z = hist[i][tid];
      full = full || (g.kw > 8 ? x : 0) + y + z > most;
      x = y;
      y = z;
    }
  }
  full = __syncthreads_or(full);
  if (tid == 0) atomicOr((unsigned long long *)(full ? crowd : plain) + p, 1ull << b);
}

// --------------------------------------------------------------------------
// launchers
// --------------------------------------------------------------------------
void launch_w_minmax(int nblk, const double *uvw, int nrow, const uint8_t *flag, long fs, double *part, int *cnt,
                     hipStream_t st) {
  w_minmax_kernel<<<nblk, 256, 0, st>>>(uvw, nrow, flag, fs, part, cnt);
}

void launch_pack_columns(const Columns &c, double *uvw, int n, hipStream_t st) {
  pack_columns_kernel<<<nblocks(n), 256, 0, st>>>(c, uvw, n);
}

void launch_fill_zero_c128(double2 *p, long n, hipStream_t st) {
  fill_zero_c128_kernel<<<nblocks(n), 256, 0, st>>>(p, n);
}

// Phase 3: binning of one problem (kernels only).
template <typename T>
void enqueue_binning(const Problem &pb, const ChanPlan &cp, const Bufs &b, hipStream_t st, bool with_value) {
  const Geom &g = cp.g;
  const long nbins = (long)g.nlayer * g.ntiles;
  const long nscan = (nbins + kScanTile - 1) / kScanTile;
  fill_int_kernel<<<nblocks(nbins), 256, 0, st>>>(b.hist, nbins, 0);
  // Counted in LDS where that leaves 16 workgroups of a row a bin each: fewer rows
  // a bin and the additions to the histogram are as many as the rows
  const long groups = std::min<long>(512, pb.nrow / nbins);
  const int chunk = groups > 0 ? (int)((pb.nrow + groups - 1) / groups) : 0;
  if (nbins <= 12288 && groups >= 16)
    bin_count_lds_kernel<<<(pb.nrow + chunk - 1) / chunk, 1024, sizeof(int) * nbins, st>>>(
        pb.uvw, pb.nrow, pb.flag, pb.flag_stride, g, (int)nbins, chunk, b.hist, b.binrank);
  else if (pb.nrow > 0)
    bin_count_kernel<<<nblocks(pb.nrow), 256, 0, st>>>(pb.uvw, pb.nrow, pb.flag, pb.flag_stride, g, b.hist,
                                                       b.binrank);
  uint64_t *occ = g.occ ? b.occ : nullptr;
  if (nbins <= kSmallScan) {
    scan_small_kernel<<<1, 1024, 0, st>>>(b.hist, (int)nbins, b.off, (int)cp.nvalid, g, occ);
  } else {
    scan_reduce_kernel<<<(int)nscan, kScanBlock, 0, st>>>(b.hist, nbins, b.bsum);
    scan_sums_kernel<<<1, 1024, 0, st>>>(b.bsum, (int)nscan);
    scan_apply_kernel<<<(int)nscan, kScanBlock, 0, st>>>(b.hist, nbins, b.bsum, b.off, (int)cp.nvalid);
    if (occ) occ_kernel<<<(g.P + 3) / 4, 256, 0, st>>>(b.off, g, occ);
  }
  if (pb.nrow > 0) {
    T *taps = g.fft_lds ? (T *)b.taps : nullptr;
    if (tap_width(g.kw) == 8)
      bin_scatter_kernel<T, 8><<<nblocks(pb.nrow), 256, 0, st>>>(pb.uvw, pb.nrow, pb.vis, pb.vis_stride, pb.wgt,
                                                                  pb.wgt_stride, g, b.binrank, b.off,
                                                                  (Rec<T> *)b.recs, b.slot, with_value ? 1 : 0, taps);
    else
      bin_scatter_kernel<T, 16><<<nblocks(pb.nrow), 256, 0, st>>>(pb.uvw, pb.nrow, pb.vis, pb.vis_stride, pb.wgt,
                                                                   pb.wgt_stride, g, b.binrank, b.off,
                                                                   (Rec<T> *)b.recs, b.slot, with_value ? 1 : 0,
                                                                   taps);
  }
  if (sizeof(T) == 4 && g.crowd) {
    fill_int_kernel<<<nblocks(4 * g.P), 256, 0, st>>>((int *)b.crowd, 4L * g.P, 0);  // and plain behind it
    const dim3 grd(g.P, ((g.nf2 - 1) >> g.occ_lg) + 1);
    crowd_kernel<<<grd, 256, 0, st>>>(b.off, (const Rec<float> *)b.recs, g, g.nf1 / std::max(g.rsplit, 1), occ, b.crowd,
                                      b.crowd + g.P);
  }
}

template void enqueue_binning<float>(const Problem &, const ChanPlan &, const Bufs &, hipStream_t, bool);
template void enqueue_binning<double>(const Problem &, const ChanPlan &, const Bufs &, hipStream_t, bool);

}  // namespace curig
