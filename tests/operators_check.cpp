// Host check of the kernels' operator images (local-dg_amd/csrc/ldg_kernels.hpp
// fill_image), built with hipcc for the host only by tests/test_operators.py.
// On constants the FP32 operators keep what the FP64 ones do, up to the
// rounding unit of the row's smallest coefficient: I reproduces them, D, Dg and
// the normal derivative (with the neighbour's weight) give zero, and Dh
// balances the lifted face terms a (eta' - eta).  No coefficient is further
// from its FP64 value than the roundings of its row together, and the FP64
// image holds the operators as they are.
#include <cmath>
#include <cstdio>
#include <vector>

#include "operators.hpp"

using namespace ldg;

static long bad = 0, rows = 0;

static double ulp(double x) { return std::ldexp(1.0, std::ilogb((float)x) - 23); }

// sum weight c = target up to the unit of the smallest c that is not zero (it
// may have doubled; weight 2, half a unit of rounding)
static void check_sum(const char *what, int N, const std::vector<double> &c, const std::vector<double> &w, double target) {
  double s = -target, lo = 1e300, hi = 0.0;
  for (size_t i = 0; i < c.size(); ++i) {
    s += w[i] * c[i];
    if (c[i] != 0.0) lo = std::fmin(lo, std::fabs(c[i]));
    hi = std::fmax(hi, std::fabs(c[i]));
  }
  ++rows;
  if (std::fabs(s) > 2 * ulp(lo) + 1e-14 * hi) {
    ++bad;
    std::printf("%s N=%d: sum off by %.2e, smallest coefficient %.2e\n", what, N, s, lo);
  }
}

template <int N, typename T>
static void check_rows(const char *what, const SymMat<N, T> &m, int S, const double (&target)[N]) {
  for (int q = 0; q < N; ++q) {
    std::vector<double> c, w;
    if (SymMat<N, T>::SPLIT) {
      if (q >= (N + 1) / 2 || (S < 0 && 2 * q + 1 == N)) continue;
      for (int j = 0; j < N / 2; ++j) { c.push_back(m.P[q][j]); w.push_back(2.0); }
      if (N & 1) { c.push_back(m.C[q]); w.push_back(1.0); }
    } else {
      for (int j = 0; j < N; ++j) { c.push_back(m.A[q][j]); w.push_back(1.0); }
    }
    check_sum(what, N, c, w, target[q]);
  }
}

template <int N, typename T>
static void check_close(const char *what, const SymMat<N, T> &m, const SymMat<N, double> &s, double f, double eps) {
  const T *a = reinterpret_cast<const T *>(&m);
  const double *b = reinterpret_cast<const double *>(&s);
  double hi = 0.0;
  const int n = sizeof(s) / sizeof(double);
  for (int i = 0; i < n; ++i) hi = std::fmax(hi, std::fabs(b[i] * f));
  for (int i = 0; i < n; ++i)
    if (std::fabs((double)a[i] - b[i] * f) > eps * hi) {
      ++bad;
      std::printf("%s N=%d: coefficient %d is %.9e, not %.9e\n", what, N, i, (double)a[i], b[i] * f);
    }
}

template <int N>
static void check(const double a[3]) {
  double asym = 0.0;
  const Ops<N, double> o = ldg_host::make_ops<N>(make_basis(N - 1), asym);
  if (!(asym < 1e-13)) ++bad;
  std::vector<double> img(GImage<N>::BYTES / sizeof(double) + 1);
  fill_image<N>(reinterpret_cast<unsigned char *>(img.data()), o, a);
  const unsigned char *b = reinterpret_cast<const unsigned char *>(img.data());
  const auto &f = *reinterpret_cast<const GOps<N, float> *>(b + GImage<N>::OF);
  const auto &d = *reinterpret_cast<const GOps<N, double> *>(b + GImage<N>::OD);
  double one[N], zero[N], dh[N];
  for (int q = 0; q < N; ++q) one[q] = 1.0, zero[q] = 0.0;
  check_rows<N, float>("I", f.I, 1, one);
  check_rows<N, float>("D", f.D, -1, zero);
  const double e32 = N * std::ldexp(1.0, -23);
  check_close<N, float>("I", f.I, o.sI, 1.0, e32);
  check_close<N, float>("D", f.D, o.sD, 1.0, e32);
  check_close<N, double>("I64", d.I, o.sI, 1.0, 0.0);
  for (int l = 0; l < 3; ++l) {
    check_rows<N, float>("Dg", f.Dg[l], -1, zero);
    for (int q = 0; q < N; ++q) dh[q] = (double)f.a[l] * ((double)f.eta[N - 1 - q] - (double)f.eta[q]);
    check_rows<N, float>("Dh", f.Dh[l], -1, dh);
    std::vector<double> c(f.nrm[l], f.nrm[l] + N), w(N + 1, 1.0);
    c.push_back(f.nbr[l]);
    check_sum("normal", N, c, w, 0.0);
    check_close<N, float>("Dg", f.Dg[l], o.sDg, a[l], e32);
    check_close<N, float>("Dh", f.Dh[l], o.sDh, a[l], e32);
    check_close<N, double>("Dg64", d.Dg[l], o.sDg, a[l], 0.0);
    check_close<N, double>("Dh64", d.Dh[l], o.sDh, a[l], 0.0);
    for (int q = 0; q < N; ++q)
      if (d.eta[q] != o.eta[q] || f.eta[q] != (float)o.eta[q]) ++bad;
  }
}

int main() {
  const double as[][3] = {{64 / M_PI, 64 / M_PI, 64 / M_PI}, {31 / M_PI, 17 / M_PI, 23 / M_PI}, {8.0, 2.0 / 0.3, 0.01},
                          {1234.5, 24 / M_PI, 1.0 / 3.0}};
  for (const auto &a : as) {
    check<2>(a);
    check<3>(a);
    check<4>(a);
    check<5>(a);
    check<6>(a);
  }
  std::printf("%ld operator rows, %ld failures\n%s\n", rows, bad, bad ? "FAILED" : "ok");
  return bad ? 1 : 0;
}
