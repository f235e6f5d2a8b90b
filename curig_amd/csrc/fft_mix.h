// Mixed-radix Stockham FFT over a padded LDS buffer, for lengths 2^a 3^b 5^c
// chosen at run time: stages of radix 2 .. 16 whose radices and sub-sizes come
// from a plan, each radix's butterfly a compile-time function of the registers.
//
// Host+device code, as fft_core.h: the kernels run it with a workgroup's
// threads, the CPU check (tests/native/fft_mix_check.cpp) with a loop over
// thread ids and a bounds-checked buffer.
//
// A buffer holds `count` sequences of length n, element k of sequence s at
// s * stride + pad(k).  A stage of radix R has count * n / R butterflies, dealt
// to the threads in turn, at most radix_nb(R) each: every thread loads and
// transforms its butterflies, all threads wait, then it stores them, so one
// buffer suffices.
#pragma once
#include <cstdint>
#include <initializer_list>

#include "fft_core.h"

namespace curig {
namespace fftm {

using fftc::cpx;

constexpr int kMaxStages = 14;

// butterflies per thread and stage at most: 16 to 20 elements in registers
FC_HD constexpr int radix_nb(int R) {
  return R == 16 || R == 15 || R == 12 ? 1 : R == 10 || R == 9 || R == 8 ? 2 : R == 6 ? 3 : R == 5 || R == 4 ? 4 : R == 3 ? 6 : 8;
}

struct Plan {
  int n = 0, count = 0;  // length, sequences side by side
  int ns = 0, nt = 0;    // stages, threads
  int stride = 0;        // elements from one sequence to the next
  uint8_t R[kMaxStages] = {};
  uint32_t ns_magic[kMaxStages] = {};  // quotient by the stage's sub-size (product of the radices before it)
  uint32_t bf_magic[kMaxStages] = {};  // quotient by its butterflies per sequence, n / R
};

FC_HD constexpr int seq_stride(int n) { return n + (n >> 4) + 1; }

// x / d as the high half of x * magic(d): exact for x d < 2^32 (d = 1: magic 0)
FC_HD uint32_t magic(uint32_t d) { return d == 1 ? 0 : (uint32_t)((uint64_t(1) << 32) / d) + 1; }
FC_HD int quot(int x, uint32_t m) {
  if (m == 0) return x;
#if defined(__HIP_DEVICE_COMPILE__)
  return (int)__umulhi((unsigned)x, m);
#else
  return (int)(((uint64_t)(uint32_t)x * m) >> 32);
#endif
}

// ---- butterflies: X[q] = sum_r v[r] e^{SIGN 2 pi i q r / R} in place --------
template <typename T, int SIGN> FC_HD void dft3(cpx<T> &a, cpx<T> &b, cpx<T> &c) {
  const T s = (T)(SIGN * 0.86602540378443864676);
  const cpx<T> t = fftc::add(b, c), u = fftc::mk(a.x - (T)0.5 * t.x, a.y - (T)0.5 * t.y);
  const cpx<T> d = fftc::mk(s * (b.x - c.x), s * (b.y - c.y));
  a = fftc::add(a, t);
  b = fftc::mk(u.x - d.y, u.y + d.x);
  c = fftc::mk(u.x + d.y, u.y - d.x);
}
template <typename T, int SIGN> FC_HD void dft5(cpx<T> &a, cpx<T> &b, cpx<T> &c, cpx<T> &d, cpx<T> &e) {
  const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
  const T s1 = (T)(SIGN * 0.95105651629515357212), s2 = (T)(SIGN * 0.58778525229247312917);
  const cpx<T> p = fftc::add(b, e), q = fftc::add(c, d), m = fftc::sub(b, e), o = fftc::sub(c, d);
  const cpx<T> u = fftc::mk(a.x + c1 * p.x + c2 * q.x, a.y + c1 * p.y + c2 * q.y);
  const cpx<T> w = fftc::mk(a.x + c2 * p.x + c1 * q.x, a.y + c2 * p.y + c1 * q.y);
  const cpx<T> g = fftc::mk(s1 * m.x + s2 * o.x, s1 * m.y + s2 * o.y);
  const cpx<T> h = fftc::mk(s2 * m.x - s1 * o.x, s2 * m.y - s1 * o.y);
  a = fftc::mk(a.x + p.x + q.x, a.y + p.y + q.y);
  b = fftc::mk(u.x - g.y, u.y + g.x);
  e = fftc::mk(u.x + g.y, u.y - g.x);
  c = fftc::mk(w.x - h.y, w.y + h.x);
  d = fftc::mk(w.x + h.y, w.y - h.x);
}

template <typename T, int R, int SIGN> FC_HD void dft(cpx<T> *v);

// R = A B with A, B coprime (prime-factor mapping, no twiddles)
template <typename T, int A, int B, int SIGN> FC_HD void dft_coprime(cpx<T> *v) {
  constexpr int R = A * B;
  cpx<T> w[R];
#pragma unroll
  for (int i = 0; i < A; ++i) {
#pragma unroll
    for (int k = 0; k < B; ++k) w[i * B + k] = v[(B * i + A * k) % R];
    dft<T, B, SIGN>(w + i * B);
  }
#pragma unroll
  for (int k = 0; k < B; ++k) {
    cpx<T> u[A];
#pragma unroll
    for (int i = 0; i < A; ++i) u[i] = w[i * B + k];
    dft<T, A, SIGN>(u);
    // output q with q = i' mod A and q = k mod B, i' the A-point frequency
#pragma unroll
    for (int i = 0; i < A; ++i) {
      int q = k;
      while (q % A != i) q += B;
      v[q] = u[i];
    }
  }
}

template <typename T, int SIGN> FC_HD void dft9(cpx<T> *v) {
  // 3 x 3 with twiddles W9^{i k}
  const T c1 = (T)0.76604444311897803520, s1 = (T)(SIGN * 0.64278760968653932632);
  const T c2 = (T)0.17364817766693034885, s2 = (T)(SIGN * 0.98480775301220805937);
  const T c4 = (T)-0.93969262078590838405, s4 = (T)(SIGN * 0.34202014332566873304);
#pragma unroll
  for (int i = 0; i < 3; ++i) dft3<T, SIGN>(v[i], v[i + 3], v[i + 6]);
  v[4] = fftc::mulw(v[4], c1, s1);
  v[7] = fftc::mulw(v[7], c2, s2);
  v[5] = fftc::mulw(v[5], c2, s2);
  v[8] = fftc::mulw(v[8], c4, s4);
#pragma unroll
  for (int k = 0; k < 3; ++k) dft3<T, SIGN>(v[3 * k], v[3 * k + 1], v[3 * k + 2]);
  // v[3 k + q] holds X[k + 3 q]: transpose
  cpx<T> t;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int k = i + 1; k < 3; ++k) {
      t = v[3 * i + k];
      v[3 * i + k] = v[3 * k + i];
      v[3 * k + i] = t;
    }
}

template <typename T, int R, int SIGN> FC_HD void dft(cpx<T> *v) {
  if constexpr (R == 1) return;
  else if constexpr (R == 3) dft3<T, SIGN>(v[0], v[1], v[2]);
  else if constexpr (R == 5) dft5<T, SIGN>(v[0], v[1], v[2], v[3], v[4]);
  else if constexpr (R == 6) dft_coprime<T, 2, 3, SIGN>(v);
  else if constexpr (R == 9) dft9<T, SIGN>(v);
  else if constexpr (R == 10) dft_coprime<T, 2, 5, SIGN>(v);
  else if constexpr (R == 12) dft_coprime<T, 4, 3, SIGN>(v);
  else if constexpr (R == 15) dft_coprime<T, 3, 5, SIGN>(v);
  else fftc::dft_small<T, R>(v, SIGN);
}

// ---- one stage --------------------------------------------------------------
// Phase 1: load and transform this thread's butterflies of stage s (radix R,
// sub-size Ns).  ld(seq, k): element k of sequence seq; tw: table of n entries.
template <typename T, int R, int SIGN, typename Ld, typename Tw>
FC_HD void stage_load(const Ld &ld, cpx<T> *v, const Plan &P, int s, int Ns, const Tw &tw, int tid) {
  const int nbf = P.n / R, total = nbf * P.count, step = nbf / Ns;
#pragma unroll
  for (int b = 0; b < radix_nb(R); ++b) {
    const int jg = tid + b * P.nt;
    if (jg < total) {
      const int seq = P.count > 1 ? quot(jg, P.bf_magic[s]) : 0, j = jg - seq * nbf;
      cpx<T> *u = v + b * R;
#pragma unroll
      for (int r = 0; r < R; ++r) u[r] = ld(seq, j + r * nbf);
      if (Ns > 1) {
        const int k = j - quot(j, P.ns_magic[s]) * Ns, base = k * step;
        cpx<T> w[R];
        // w, w^2, w^4, w^8 from the table, the others as products
#pragma unroll
        for (int r = 1; r < R; ++r) {
          int hi = 1;
          while (2 * hi <= r) hi *= 2;
          w[r] = r == hi ? tw[base * r] : fftc::mul(w[hi], w[r - hi]);
          u[r] = fftc::mulw(u[r], w[r].x, (T)SIGN * w[r].y);
        }
      }
      dft<T, R, SIGN>(u);
    }
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
  }
}

// Phase 2: st(seq, k, value) of this thread's butterflies.
template <typename T, int R, typename St>
FC_HD void stage_store(const St &st, const cpx<T> *v, const Plan &P, int s, int Ns, int tid) {
  const int nbf = P.n / R, total = nbf * P.count;
#pragma unroll
  for (int b = 0; b < radix_nb(R); ++b) {
    const int jg = tid + b * P.nt;
    if (jg < total) {
      const int seq = P.count > 1 ? quot(jg, P.bf_magic[s]) : 0, j = jg - seq * nbf;
      const int k = Ns > 1 ? j - quot(j, P.ns_magic[s]) * Ns : 0, d = (j - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) st(seq, d + r * Ns, v[b * R + r]);
    }
  }
}

// f(std::integral_constant-like tag with ::value = R) for the radices a plan uses
template <int N> struct Rad { static constexpr int value = N; };
template <typename F> FC_HD void with_radix(int R, const F &f) {
  switch (R) {
    case 16: f(Rad<16>()); break;
    case 15: f(Rad<15>()); break;
    case 12: f(Rad<12>()); break;
    case 10: f(Rad<10>()); break;
    case 9: f(Rad<9>()); break;
    case 8: f(Rad<8>()); break;
    case 6: f(Rad<6>()); break;
    case 5: f(Rad<5>()); break;
    case 4: f(Rad<4>()); break;
    case 3: f(Rad<3>()); break;
    default: f(Rad<2>()); break;
  }
}

// ---- plan (host) --------------------------------------------------------------
inline bool smooth235(int n) {
  if (n < 2) return false;
  for (int p : {2, 3, 5})
    while (n % p == 0) n /= p;
  return n == 1;
}

// Instructions of one butterfly, about: its transform, twiddles and addresses.
inline double radix_cost(int R) {
  switch (R) {
    case 16: return 168 + 15 * 4 + 16 * 6 + 80;
    case 15: return 162 + 14 * 4 + 15 * 6 + 76;
    case 12: return 96 + 11 * 4 + 12 * 6 + 60;
    case 10: return 100 + 9 * 4 + 10 * 6 + 56;
    case 9: return 80 + 8 * 4 + 9 * 6 + 52;
    case 8: return 64 + 7 * 4 + 8 * 6 + 48;
    case 6: return 36 + 5 * 4 + 6 * 6 + 40;
    case 5: return 36 + 4 * 4 + 5 * 6 + 40;
    case 4: return 16 + 3 * 4 + 4 * 6 + 36;
    case 3: return 14 + 2 * 4 + 3 * 6 + 30;
    default: return 4 + 4 + 2 * 6 + 24;
  }
}

// The cheapest radices of n for `count` sequences on nt threads (wavefronts of
// 64, whole ones counted), stages in descending radix.  False when no
// factorisation keeps every thread within radix_nb butterflies.
inline bool make_plan(Plan &out, int n, int count, int nt) {
  if (!smooth235(n) || count < 1 || nt < 64 || (long)n * count > (1 << 16)) return false;
  const int rad[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
  int best[kMaxStages], cur[kMaxStages], nbest = 0;
  double bestc = 1e300;
  struct Search {
    const int *rad;
    int n, count, nt, *best, *cur, *nbest;
    double *bestc;
    void go(int rest, int from, int depth, double c) {
      if (c >= *bestc) return;
      if (rest == 1) {
        *bestc = c;
        *nbest = depth;
        for (int i = 0; i < depth; ++i) best[i] = cur[i];
        return;
      }
      if (depth == kMaxStages) return;
      for (int i = from; i < 11; ++i) {
        const int R = rad[i];
        if (rest % R) continue;
        const long bf = (long)count * (n / R);
        if (bf > (long)radix_nb(R) * nt) continue;
        cur[depth] = R;
        // 40: a stage's two barriers, per wavefront of the workgroup
        go(rest / R, i, depth + 1, c + (double)((bf + 63) / 64) * radix_cost(R) + 40.0 * (nt / 64));
      }
    }
  } search{rad, n, count, nt, best, cur, &nbest, &bestc};
  search.go(n, 0, 0, 0.0);
  if (nbest == 0) return false;
  out = Plan();
  out.n = n;
  out.count = count;
  out.nt = nt;
  out.ns = nbest;
  out.stride = seq_stride(n);
  int Ns = 1;
  for (int s = 0; s < nbest; ++s) {
    out.R[s] = (uint8_t)best[s];
    out.ns_magic[s] = magic((uint32_t)Ns);
    out.bf_magic[s] = magic((uint32_t)(n / best[s]));
    Ns *= best[s];
  }
  return true;
}

}  // namespace fftm
}  // namespace curig
