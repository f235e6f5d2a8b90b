// Row kernels of the LDS path for whole power-of-two rows of 64 .. 2048 points
// (4096 and parts of 4096: the plane-loop kernels of kern_lds.h; FP32 rows of
// 8192 kept whole).  A workgroup holds rpw rows in LDS, N / 16 threads each
// (RegFft), and walks a chunk of the batch's planes: the stage twiddles are set
// up once, the spread accumulates in FP64 (RowAcc) and the first and last stages
// of the transform stay in registers.
#pragma once
#include "fft_reg.h"
#include "kern_rows.h"

namespace curig {

template <int N> struct RowThreads { static constexpr int value = N / 16 > 256 ? N / 16 : 256; };

// Slots of the image columns that thread j of a row holds: element e (first or
// last quarter) is column j + h1 + G e, less N in the last quarter; its slot
// steps by G / kTile tiles per element (whole rows: slot = column).
template <int G> __device__ __forceinline__ long elem_step(const Geom &g, int e) {
  return (long)(G / kTile) * g.tstride * (e < 8 ? e : e - 16);
}
template <int N> __device__ __forceinline__ bool elem_image(int j, int e, int N1) {
  return image_index(j + (N / 16) * e, N1, N) >= 0;
}

// ms2dirty: spread into the workgroup's rows, row FFT, image columns to H (added
// to it where gridDim.z workgroups share the rows' records)
template <typename T, int KWM, int N, bool ACC64>
__global__ void __launch_bounds__(RowThreads<N>::value) spread_row_reg_kernel(
    const Rec<T> *__restrict__ recs, const T *__restrict__ taps, const int *__restrict__ off, cpx<T> *__restrict__ H,
    const cpx<T> *__restrict__ tw, Geom g, int p0, int nb, int pchunk) {
  using F = RegFft<T, N, +1>;
  constexpr int G = F::G;
  using Cell = typename RowAcc<T, ACC64>::cell;
  constexpr bool kParts = RowAcc<T, ACC64>::parts;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ WalkTable wt[2];
  const int tid = threadIdx.x, nt = blockDim.x, rpw = g.rpw, s = tid / G, j = tid % G, N1 = g.N1, h1 = N1 / 2;
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw), *own = buf + s * F::kStride;
  // the cells; in FP32 the transform runs in their place (complex cells: in their first half)
  Cell *acc = reinterpret_cast<Cell *>(smem_raw), *ownc = acc + s * F::kStride;
  const int row0 = row_group(g) * rpw;
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  const bool add = gridDim.z > 1;
  // planes whose block of rows holds no record are passed over (rpw, a power of
  // two of at most 64, keeps to a block)
  PlaneWalk<> pw(g, p0, k0, k1, row0, row0);
  int pn = pw.next();
  if (pn >= k1) return;
  if (tid < 64) walk_table_build(wt[0], off, g, p0 + pn, row0, rpw);
  for (int i = tid; i < rpw * F::kStride; i += nt) acc[i] = Cell{};
  F fft;
  fft.init(tw, j, nullptr);
  __syncthreads();
  int cur = 0;
  for (int pl = pn; pl < k1; pl = pn, cur ^= 1) {
    const int p = p0 + pl, total = wt[cur].total;
    pn = pw.next();
    const bool more = pn < k1;
    WalkAhead wa;
    if (tid < 64 && more) walk_issue(wa, off, g, p0 + pn, row0, rpw);
    cpx<T> v[16];
    if constexpr (kParts) {
      if (total > 0) {
        spread_records<kReal, T, KWM>(wt[cur], total, recs, taps, g, p, row0, rpw, acc, F::kStride);
        __syncthreads();
        Cell *in = ownc + F::pos0(j);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          v[e].x = (T)in[F::pos(e)];
          in[F::pos(e)] = 0.0;
        }
        __syncthreads();
      }
    }
    spread_records<kParts ? kImag : kBoth, T, KWM>(wt[cur], total, recs, taps, g, p, row0, rpw, acc, F::kStride);
    if (tid < 64 && more) walk_finish(wt[cur ^ 1], wa);
    __syncthreads();  // spread done; the next plane's walk table is complete
    if (total > 0) {
      const Cell *in = ownc + F::pos0(j);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if constexpr (kParts)
          v[e].y = (T)in[F::pos(e)];
        else
          v[e] = fftc::mk((T)in[F::pos(e)].x, (T)in[F::pos(e)].y);
      }
      __syncthreads();
      fft.template run<false>(v, own, j);
    } else {
      // no visibility reaches these rows of this plane (and the LDS is still clear)
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = fftc::mk((T)0, (T)0);
    }
    cpx<T> *hb = H + h_plane(g, pl) + (row0 + s) * kTile + h_slot(g, j + h1);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = image_elem(q);
      if (elem_image<N>(j, e, N1) && (total > 0 || !add)) put_row(hb + elem_step<G>(g, e), v[e], add);
    }
    if (total == 0) continue;
    __syncthreads();  // the transform's LDS reads are done: clear for the next plane
#pragma unroll
    for (int e = 0; e < 16; ++e) (ownc + F::pos0(j))[F::pos(e)] = Cell{};
    __syncthreads();
  }
}

// a row of a dirty2ms plane into the registers of its threads: elements 0..3
// and 12..15 (the others are zero)
template <typename T, int N>
__device__ __forceinline__ void load_row_elems(cpx<T> *v, const cpx<T> *__restrict__ H, const Geom &g, int pl, int row,
                                               int j) {
  constexpr int G = N / 16;
  const cpx<T> *hb = H + h_plane(g, pl) + ht_row(row) + ht_slot(g, j + g.N1 / 2);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int e = image_elem(q);
    v[e] = elem_image<N>(j, e, g.N1) ? hb[elem_step<G>(g, e)] : fftc::mk((T)0, (T)0);
  }
}

// dirty2ms: inverse row FFT and interpolation of every record that touches the rows
template <typename T, int KWM, int N>
__global__ void __launch_bounds__(RowThreads<N>::value) row_interp_reg_kernel(
    const cpx<T> *__restrict__ H, const Rec<T> *__restrict__ recs, const T *__restrict__ taps,
    const int *__restrict__ off, double2 *__restrict__ vacc, const cpx<T> *__restrict__ tw, Geom g, int p0, int nb,
    int pchunk) {
  using F = RegFft<T, N, -1>;
  constexpr int G = F::G;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ WalkTable wt[2];
  const int tid = threadIdx.x, rpw = g.rpw, s = tid / G, j = tid % G;
  cpx<T> *buf = reinterpret_cast<cpx<T> *>(smem_raw), *own = buf + s * F::kStride;
  const int row0 = row_group(g) * rpw;
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  PlaneWalk<> pw(g, p0, k0, k1, row0, row0);
  int pn = pw.next();
  if (pn >= k1) return;
  if (tid < 64) walk_table_build(wt[0], off, g, p0 + pn, row0, rpw);
  F fft;
  fft.init(tw, j, nullptr);
  __syncthreads();
  int cur = 0;
  for (int pl = pn; pl < k1; pl = pn, cur ^= 1) {
    const int p = p0 + pl, total = wt[cur].total;
    pn = pw.next();
    const bool more = pn < k1;
    WalkAhead wa;
    if (tid < 64 && more) walk_issue(wa, off, g, p0 + pn, row0, rpw);
    if (total > 0) {
      cpx<T> v[16];
      load_row_elems<T, N>(v, H, g, pl, row0 + s, j);
      fft.template run<true>(v, own, j);
      __syncthreads();  // the transform's LDS reads are done
#pragma unroll
      for (int e = 0; e < 16; ++e) (own + F::pos0(j))[F::pos(e)] = v[e];
      __syncthreads();
      interp_records<T, KWM>(wt[cur], total, recs, taps, g, p, row0, rpw, buf, F::kStride, vacc);
    }
    if (tid < 64 && more) walk_finish(wt[cur ^ 1], wa);
    __syncthreads();  // the rows are free; the next plane's walk table is complete
  }
}

// dirty2ms with dense records (Geom::gather): the rows written out as full planes
template <typename T, int N>
__global__ void __launch_bounds__(RowThreads<N>::value) row_planes_reg_kernel(const cpx<T> *__restrict__ H,
                                                                             cpx<T> *__restrict__ grid,
                                                                             const cpx<T> *__restrict__ tw, Geom g,
                                                                             int p0, int nb, int pchunk) {
  using F = RegFft<T, N, -1>;
  constexpr int G = F::G;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int tid = threadIdx.x, rpw = g.rpw, s = tid / G, j = tid % G;
  cpx<T> *own = reinterpret_cast<cpx<T> *>(smem_raw) + s * F::kStride;
  const int row = row_group(g) * rpw + s;
  const int k0 = blockIdx.y * pchunk, k1 = min(nb, k0 + pchunk);
  PlaneWalk<> pw(g, p0, k0, k1, row & ~(rpw - 1), row & ~(rpw - 1));
  F fft;
  fft.init(tw, j, nullptr);
  for (int pl = pw.next(); pl < k1; pl = pw.next()) {
    cpx<T> v[16];
    load_row_elems<T, N>(v, H, g, pl, row, j);
    __syncthreads();  // the previous plane's LDS reads are done
    fft.template run<true>(v, own, j);
    cpx<T> *out = grid + ((size_t)pl * g.nf2 + row) * N + j;
#pragma unroll
    for (int e = 0; e < 16; ++e) out[G * e] = v[e];
  }
}

// --------------------------------------------------------------------------
// launchers
// --------------------------------------------------------------------------
// f(std::integral_constant<int, N>()) for the lengths of whole rows that run
// here: up to 2048 points, FP32 also 8192, and 4096 where the rows are gathered
template <typename T, typename F> inline bool with_row_len(int n, F f) {
  using std::integral_constant;
  switch (n) {
    case 64: f(integral_constant<int, 64>()); return true;
    case 128: f(integral_constant<int, 128>()); return true;
    case 256: f(integral_constant<int, 256>()); return true;
    case 512: f(integral_constant<int, 512>()); return true;
    case 1024: f(integral_constant<int, 1024>()); return true;
    case 2048: f(integral_constant<int, 2048>()); return true;
    case 4096: f(integral_constant<int, 4096>()); return true;
  }
  if constexpr (sizeof(T) == 4) {
    if (n == 8192) {
      f(integral_constant<int, 8192>());
      return true;
    }
  }
  return false;
}

// whether a plan sums rows of N cells so (ACC64: Geom::acc64): FP32 rows of 2048
// and 8192 both ways, shorter ones and 4096 in complex cells only
template <typename T, int N, bool ACC64> constexpr bool row_acc() {
  return sizeof(T) == 8 ? N != 4096 : ACC64 || N == 2048 || N == 8192;
}

template <typename T> inline int rowreg_lds(const Geom &g, bool spread) {
  const int cells = g.rpw * (g.nf1 + g.nf1 / 16 + 16);
  return cells * (int)(spread && g.acc64 ? sizeof(double2) : sizeof(cpx<T>));
}

template <typename T>
void rowreg_spread(const Rec<T> *recs, const T *taps, const int *off, const Geom &g, int p0, int nb, cpx<T> *H,
                   const cpx<T> *tw1, hipStream_t st) {
  const dim3 grd(g.nf2 / g.rpw, (nb + g.pch_row - 1) / g.pch_row, g.zrow);
  const int lb = rowreg_lds<T>(g, true), nt = g.rpw * g.nf1 / 16;
  if (g.zrow > 1) zero_planes<T>(H, g, nb, st);
  with_row_len<T>(g.nf1, [&](auto N) {
    with_acc64<T>(g.acc64, [&](auto A) {
      if constexpr (row_acc<T, N.value, A.value>()) {
        if (g.kw <= 8)
          spread_row_reg_kernel<T, 8, N.value, A.value><<<grd, nt, lb, st>>>(recs, taps, off, H, tw1, g, p0, nb, g.pch_row);
        else
          spread_row_reg_kernel<T, 16, N.value, A.value><<<grd, nt, lb, st>>>(recs, taps, off, H, tw1, g, p0, nb, g.pch_row);
      }
    });
  });
}

template <typename T>
void rowreg_interp(const Rec<T> *recs, const T *taps, const int *off, const cpx<T> *H, void *grid, double2 *vacc,
                   const cpx<T> *tw1, const Geom &g, long nvalid, int p0, int nb, hipStream_t st) {
  const dim3 grd(g.nf2 / g.rpw, (nb + g.pch_row - 1) / g.pch_row);
  const int lb = rowreg_lds<T>(g, false), nt = g.rpw * g.nf1 / 16;
  with_row_len<T>(g.nf1, [&](auto N) {
    if (g.gather) {
      row_planes_reg_kernel<T, N.value><<<grd, nt, lb, st>>>(H, (cpx<T> *)grid, tw1, g, p0, nb, g.pch_row);
    } else if constexpr (N.value != 4096) {
      if (g.kw <= 8)
        row_interp_reg_kernel<T, 8, N.value><<<grd, nt, lb, st>>>(H, recs, taps, off, vacc, tw1, g, p0, nb, g.pch_row);
      else
        row_interp_reg_kernel<T, 16, N.value><<<grd, nt, lb, st>>>(H, recs, taps, off, vacc, tw1, g, p0, nb, g.pch_row);
    }
  });
  if (g.gather) launch_gather<T>(recs, taps, off, (const cpx<T> *)grid, vacc, g, nvalid, p0, nb, st);
}

// checks a plan against the kernels' launch limits and raises their dynamic LDS
template <typename T> int allow_rowreg(const Geom &g, bool spread) {
  const int lb = rowreg_lds<T>(g, spread), nt = g.rpw * g.nf1 / 16;
  int ier = kErrArg;
  const bool known = with_row_len<T>(g.nf1, [&](auto N) {
    constexpr int n = N.value;
    if (g.rpw < 1 || g.rpw > 64 || (g.rpw & (g.rpw - 1)) || nt < 64 || nt > RowThreads<n>::value || g.nf2 % g.rpw || g.pch_row < 1 || g.zrow < 1) return;
    if (spread) {
      with_acc64<T>(g.acc64, [&](auto A) {
        if constexpr (row_acc<T, n, A.value>()) {
          ier = allow_lds(spread_row_reg_kernel<T, 8, n, A.value>, lb);
          if (ier == kOk) ier = allow_lds(spread_row_reg_kernel<T, 16, n, A.value>, lb);
        }
      });
    } else if (g.gather) {
      ier = allow_lds(row_planes_reg_kernel<T, n>, lb);
    } else if constexpr (n != 4096) {
      ier = allow_lds(row_interp_reg_kernel<T, 8, n>, lb);
      if (ier == kOk) ier = allow_lds(row_interp_reg_kernel<T, 16, n>, lb);
    }
  });
  if (!known || ier == kErrArg) set_error("row pass of %d points: %d rows, %d planes per workgroup", g.nf1, g.rpw, g.pch_row);
  return ier;
}

#define CURIG_ROWREG_INST(T)                                                                                       \
  template void rowreg_spread<T>(const Rec<T> *, const T *, const int *, const Geom &, int, int, cpx<T> *,         \
                                 const cpx<T> *, hipStream_t);                                                     \
  template void rowreg_interp<T>(const Rec<T> *, const T *, const int *, const cpx<T> *, void *, double2 *,        \
                                 const cpx<T> *, const Geom &, long, int, int, hipStream_t);                       \
  template int allow_rowreg<T>(const Geom &, bool);

}  // namespace curig
