// Power-of-two FFT of N = 64 .. 8192 points by G = N / 16 threads, 16 elements
// each in registers: thread j enters with x[j + G e] in v[e] and leaves with
// X[j + G e] there.  Stockham stages of radix 16 and a last stage of N's
// remainder (2, 4, 8 or 16); between them the elements pass through LDS
// (padded, fftc::pad), so a transform of 4096 stores and loads each element
// twice, and the first stage's inputs and the last stage's outputs never pass
// through LDS.  A thread's stage twiddles are the same for every transform it
// runs: they are read once and held.  One workgroup may run several
// transforms side by side (its barriers cover all of them).
#pragma once
#include <type_traits>

#include "dev_common.h"

namespace curig {

// Where a thread finds its stage twiddles:
//   kTwHeld  registers, read once (the plane loops: 2 to 4 complex values per stage);
//   kTwPair  the axis' two-level table in LDS, one product per value (short of registers);
//   kTwFull  an LDS table of every stage's values (short of registers, LDS to spare).
enum { kTwHeld = 0, kTwPair = 1, kTwFull = 2 };

template <typename T, int N, int SIGN, int TW = kTwHeld> struct RegFft {
  static_assert(N >= 64 && N <= 8192 && (N & (N - 1)) == 0, "power of two, 64 .. 8192");
  static constexpr int G = N / 16;
  // complex LDS elements of one transform; transforms of one workgroup whose
  // threads interleave lie 16 elements further apart, half of the banks
  static constexpr int kStride = N + N / 16 + 16;
  static constexpr int radix(int NS) { return NS * 16 <= N ? 16 : N / NS; }
  static constexpr int tw_count(int R) { return R == 16 ? 4 : R == 8 ? 3 : R == 4 ? 2 : 1; }
  static constexpr int tw_base(int NS) { return NS <= 16 ? 0 : tw_base(NS / 16) + tw_count(radix(NS / 16)); }
  static constexpr int last_ns() {
    int ns = 1;
    while (ns * radix(ns) < N) ns *= radix(ns);
    return ns;
  }
  static constexpr int kTw = tw_base(last_ns()) + tw_count(radix(last_ns()));
  // twiddles of a stage are indexed by k < span: j mod NS, or j in a last stage of radix < 16
  static constexpr int span(int NS) { return NS < G ? NS : G; }
  static constexpr int full_base(int NS) {
    return NS <= 16 ? 0 : full_base(NS / 16) + span(NS / 16) * tw_count(radix(NS / 16));
  }
  static constexpr int pair_entries() { return fftc::twiddle_entries_c(N); }
  // LDS elements of the twiddles of one workgroup
  static constexpr int kTwLds = TW == kTwPair   ? pair_entries()
                                : TW == kTwFull ? full_base(last_ns()) + span(last_ns()) * tw_count(radix(last_ns()))
                                                : 0;
  cpx<T> held[TW == kTwHeld ? kTw : 1];
  const cpx<T> *lds;

  // value i (w^(2^i)) of stage NS for index k
  template <int NS, typename Tab> __device__ __forceinline__ static cpx<T> value(const Tab &t, int k, int i) {
    constexpr int step = N / (NS * radix(NS));
    const cpx<T> w = t[((k << i) * step) & (N - 1)];
    return fftc::mk(w.x, (T)SIGN * w.y);
  }
  template <int NS, typename Tab> __device__ __forceinline__ void load_stage(const Tab &t, int j, cpx<T> *out) {
    constexpr int R = radix(NS), C = tw_count(R);
    if constexpr (TW == kTwHeld) {
#pragma unroll
      for (int i = 0; i < C; ++i) held[tw_base(NS) + i] = value<NS>(t, j & (span(NS) - 1), i);
    } else {
      for (int m = threadIdx.x; m < span(NS) * C; m += blockDim.x) out[full_base(NS) + m] = value<NS>(t, m / C, m % C);
    }
    if constexpr (NS * R < N) load_stage<NS * R>(t, j, out);
  }
  // table: the axis' two-level table (global); ltw: kTwLds elements of LDS,
  // complete after the next barrier
  __device__ __forceinline__ void init(const cpx<T> *__restrict__ table, int j, cpx<T> *ltw) {
    lds = ltw;
    if constexpr (TW == kTwPair) {
      for (int m = threadIdx.x; m < pair_entries(); m += blockDim.x) ltw[m] = table[m];
    } else {
      const int lb = fftc::twiddle_split(N);
      const fftc::TwoLevel<T, const cpx<T> *> t{table, table + (N >> lb), lb};
      load_stage<16>(t, j, ltw);
    }
  }
  template <int NS> __device__ __forceinline__ void stage_twiddles(cpx<T> *q, int j) const {
    constexpr int C = tw_count(radix(NS));
    const int k = j & (span(NS) - 1);
    if constexpr (TW == kTwPair) {
      constexpr int lb = fftc::twiddle_split_c(N);
      const fftc::TwoLevel<T, const cpx<T> *> t{lds, lds + (N >> lb), lb};
#pragma unroll
      for (int i = 0; i < C; ++i) q[i] = value<NS>(t, k, i);
    } else if constexpr (TW == kTwFull) {
      const cpx<T> *p = lds + full_base(NS) + k * C;
#pragma unroll
      for (int i = 0; i < C; ++i) q[i] = p[i];
    } else {
#pragma unroll
      for (int i = 0; i < C; ++i) {
        // the products of powers stay at their use (hoisted out of a plane
        // loop they would hold 22 more registers)
        q[i] = held[tw_base(NS) + i];
        __asm__ volatile("" : "+v"(q[i].x), "+v"(q[i].y));
      }
    }
  }

  // position of element j + G e: one address plus constants
  __device__ __forceinline__ static int pos0(int j) { return G >= 16 ? fftc::pad(j) : j; }
  static constexpr int pos(int e) { return G >= 16 ? e * (G + G / 16) : fftc::pad(e * G); }

  template <int NS> __device__ __forceinline__ void stage(cpx<T> *v, cpx<T> *buf, int j) const {
    constexpr int R = radix(NS), NB = 16 / R;
    constexpr bool last = NS * R == N;
    const cpx<T> *in = buf + pos0(j);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = in[pos(e)];
    cpx<T> q[4];
    stage_twiddles<NS>(q, j);
    if constexpr (R == 16) {
#pragma unroll
      for (int r = 1; r < 16; ++r) {
        const int lo = __builtin_ctz(r);
        cpx<T> w = q[lo];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (((r >> i) & 1) && i != lo) w = fftc::mul(w, q[i]);
        v[r] = fftc::mul(v[r], w);
      }
      fftc::dft_small<T, 16>(v, SIGN);
    } else {
      // the last stage: butterfly b of thread j has k = j + G b, so its
      // twiddles are W_N^{j r} W_16^{b r}
      static_assert(last, "a radix below 16 ends the transform");
      cpx<T> w[R];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const int lo = __builtin_ctz(r);
        w[r] = q[lo];
#pragma unroll
        for (int i = 0; i < 3; ++i)
          if (((r >> i) & 1) && i != lo) w[r] = fftc::mul(w[r], q[i]);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        cpx<T> u[R];
        u[0] = v[b];
#pragma unroll
        for (int r = 1; r < R; ++r) u[r] = fftc::rot16(fftc::mul(v[b + r * NB], w[r]), (b * r) & 15, SIGN);
        fftc::dft_small<T, R>(u, SIGN);
#pragma unroll
        for (int r = 0; r < R; ++r) v[b + r * NB] = u[r];
      }
    }
    if constexpr (!last) {
      __syncthreads();  // every input of this stage is read
      const int k = j & (NS - 1);
      cpx<T> *out = buf + fftc::pad((j - k) * 16 + k);
#pragma unroll
      for (int r = 0; r < 16; ++r) out[r * (NS + NS / 16)] = v[r];
      __syncthreads();
      stage<NS * 16>(v, buf, j);
    }
  }

  // The caller has made buf free (a barrier after its last reader); after the
  // transform the threads may still be reading it.  HALF_IN: only v[0..3] and
  // v[12..15] are nonzero on entry (the others are not read).
  template <bool HALF_IN> __device__ __forceinline__ void run(cpx<T> *v, cpx<T> *buf, int j) const {
    if (HALF_IN) {
      // first radix-2 level with one zero input each: copies
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r + 8] = v[r];
        v[r + 4] = v[r + 12];
        v[r + 12] = fftc::mk(-v[r + 12].x, -v[r + 12].y);
      }
      fftc::dft16_from_pairs<T>(v, SIGN);
    } else {
      fftc::dft_small<T, 16>(v, SIGN);
    }
    cpx<T> *out = buf + 17 * j;  // pad(16 j + r)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[r] = v[r];
    __syncthreads();
    stage<16>(v, buf, j);
  }
};

// element e = q or q + 8 of RegFft's sixteen that can be an image row or column:
// with the image at most half the grid, its grid indices lie in the first and
// last quarter
__device__ __forceinline__ constexpr int image_elem(int q) { return q < 4 ? q : q + 8; }

// f(std::integral_constant<int, N>()) for the supported lengths
template <typename F> inline bool with_reg_fft(int n, F f) {
  switch (n) {
    case 64: f(std::integral_constant<int, 64>()); return true;
    case 128: f(std::integral_constant<int, 128>()); return true;
    case 256: f(std::integral_constant<int, 256>()); return true;
    case 512: f(std::integral_constant<int, 512>()); return true;
    case 1024: f(std::integral_constant<int, 1024>()); return true;
    case 2048: f(std::integral_constant<int, 2048>()); return true;
    case 4096: f(std::integral_constant<int, 4096>()); return true;
    case 8192: f(std::integral_constant<int, 8192>()); return true;
  }
  return false;
}

}  // namespace curig
