// Host run of the mixed-radix LDS FFT (fft_mix.h) with the workgroup's threads
// emulated by loops: same code, same indexing, plus bounds checks on every
// buffer and table access.  Built with g++ by tests/test_fft_mix.py.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "fft_mix.h"

using namespace curig;
using fftc::cpx;

namespace {

template <typename T> struct Checked {
  cpx<T> *p;
  long n;
  const char *what;
  cpx<T> &operator[](long i) const {
    if (i < 0 || i >= n) {
      fprintf(stderr, "fft_mix_check: %s index %ld outside [0, %ld)\n", what, i, n);
      abort();
    }
    return p[i];
  }
};

template <typename T, int SIGN> void run(const fftm::Plan &P, double *data) {
  const int n = P.n, lb = fftc::twiddle_split(n), nhi = fftc::twiddle_hi(n), nlo = 1 << lb;
  std::vector<cpx<T>> hv(nhi), lv(nlo), buf((size_t)P.count * P.stride);
  for (int j = 0; j < nhi; ++j)
    hv[j] = fftc::mk((T)std::cos(2 * M_PI * ((double)j * nlo) / n), (T)std::sin(2 * M_PI * ((double)j * nlo) / n));
  for (int j = 0; j < nlo; ++j) lv[j] = fftc::mk((T)std::cos(2 * M_PI * j / n), (T)std::sin(2 * M_PI * j / n));
  fftc::TwoLevel<T, Checked<T>> tw{Checked<T>{hv.data(), nhi, "hi"}, Checked<T>{lv.data(), nlo, "lo"}, lb};
  Checked<T> b{buf.data(), (long)buf.size(), "buffer"};
  auto at = [&](int seq, int k) {
    if (seq < 0 || seq >= P.count || k < 0 || k >= n) {
      fprintf(stderr, "fft_mix_check: element (%d, %d) of %d x %d\n", seq, k, P.count, n);
      abort();
    }
    return (long)seq * P.stride + fftc::pad(k);
  };
  for (int s = 0; s < P.count; ++s)
    for (int k = 0; k < n; ++k) b[at(s, k)] = fftc::mk((T)data[2 * ((long)s * n + k)], (T)data[2 * ((long)s * n + k) + 1]);
  std::vector<cpx<T>> regs((size_t)P.nt * 20);
  int Ns = 1;
  for (int s = 0; s < P.ns; ++s) {
    fftm::with_radix(P.R[s], [&](auto tag) {
      constexpr int R = decltype(tag)::value;
      static_assert(R * fftm::radix_nb(R) <= 20, "registers per thread");
      for (int t = 0; t < P.nt; ++t)
        fftm::stage_load<T, R, SIGN>([&](int q, int k) { return b[at(q, k)]; }, &regs[(size_t)t * 20], P, s, Ns, tw, t);
      for (int t = 0; t < P.nt; ++t)
        fftm::stage_store<T, R>([&](int q, int k, cpx<T> v) { b[at(q, k)] = v; }, &regs[(size_t)t * 20], P, s, Ns, t);
    });
    Ns *= P.R[s];
  }
  for (int s = 0; s < P.count; ++s)
    for (int k = 0; k < n; ++k) {
      data[2 * ((long)s * n + k)] = b[at(s, k)].x;
      data[2 * ((long)s * n + k) + 1] = b[at(s, k)].y;
    }
}

}  // namespace

// 0: transformed; 1: no plan.  radices: up to 14 of the plan's, then 0.
extern "C" int fftm_check_run(int n, int count, int nt, int sign, int dbl, double *data, int *radices) {
  fftm::Plan P;
  if (!fftm::make_plan(P, n, count, nt)) return 1;
  for (int i = 0; i < fftm::kMaxStages; ++i) radices[i] = i < P.ns ? P.R[i] : 0;
  if (dbl)
    sign > 0 ? run<double, 1>(P, data) : run<double, -1>(P, data);
  else
    sign > 0 ? run<float, 1>(P, data) : run<float, -1>(P, data);
  return 0;
}
