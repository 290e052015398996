// operators.hpp -- the 1D operators of the kernels (host, FP64) from the basis.
#pragma once

#include <algorithm>
#include <cmath>

#include "basis.hpp"
#include "ldg_kernels.hpp"

namespace ldg_host {

using namespace ldg;

// largest change made by symmetrize (A is replaced by its symmetric part)
template <int N>
double symmetrize_checked(double (&A)[N][N], int S) {
  double B[N][N], dev = 0.0;
  for (int a = 0; a < N; ++a)
    for (int b = 0; b < N; ++b) B[a][b] = A[a][b];
  symmetrize<N>(A, S);
  for (int a = 0; a < N; ++a)
    for (int b = 0; b < N; ++b) dev = std::max(dev, std::fabs(A[a][b] - B[a][b]));
  return dev;
}

template <int N>
Ops<N, double> make_ops(const Basis1D &B, double &asym) {
  Ops<N, double> o;
  for (int a = 0; a < N; ++a) {
    for (int b = 0; b < N; ++b) {
      o.I[a][b] = B.at(B.I, a, b);
      o.D[a][b] = B.at(B.D, a, b);
      o.Dn[a][b] = B.at(B.Dn, a, b);
      o.Minv[a][b] = B.at(B.M1inv, a, b);
    }
    o.L0[a] = B.at(B.M1inv, a, 0);
    o.w[a] = B.w[a];
  }
  // Gauss form: Lagrange polynomials L_q of the Gauss points at the nodes
  // (I^-1) and their derivatives at the Gauss points (Dg; barycentric, each
  // diagonal minus its row, so that constants are annihilated)
  double I[N][N], D[N][N], Ii[N][N], Dg[N][N], Dh[N][N], bw[N];
  for (int q = 0; q < N; ++q) {
    bw[q] = 1.0;
    for (int j = 0; j < N; ++j)
      if (j != q) bw[q] /= (B.g[q] - B.g[j]);
  }
  for (int a = 0; a < N; ++a) {
    double sum = 0.0;
    for (int b = 0; b < N; ++b) {
      I[a][b] = o.I[a][b];
      D[a][b] = o.D[a][b];
      double v = 1.0;
      for (int j = 0; j < N; ++j)
        if (j != b) v *= (B.r[a] - B.g[j]) / (B.g[b] - B.g[j]);
      Ii[a][b] = v;
      if (b != a) {
        Dg[a][b] = bw[b] / bw[a] / (B.g[a] - B.g[b]);
        sum += Dg[a][b];
      }
    }
    Dg[a][a] = -sum;
  }
  for (int q = 0; q < N; ++q) {
    o.eta[q] = Ii[0][q] / B.w[q];   // the first node is the - face
    for (int j = 0; j < N; ++j) Dh[q][j] = Dg[j][q] * B.w[j] / B.w[q];
  }
  // sweep operators in even/odd split form, from their (anti-)centro-symmetric
  // parts (the node sets are symmetric; this removes construction round-off)
  asym = std::max(std::max(symmetrize_checked<N>(I, 1), symmetrize_checked<N>(Ii, 1)),
                  std::max(symmetrize_checked<N>(D, -1), symmetrize_checked<N>(Dg, -1)));
  asym = std::max(asym, symmetrize_checked<N>(Dh, -1));
  for (int q = 0; q < N; ++q) {     // the lifts of the two faces mirror each other
    const double lo = Ii[0][q] / B.w[q];
    asym = std::max(asym, std::fabs(lo - o.eta[q]));
    o.eta[q] = lo;
  }
  make_symmat<N, double>(I, o.sI);
  make_symmat<N, double>(D, o.sD);
  make_symmat<N, double>(Ii, o.sIi);
  make_symmat<N, double>(Dg, o.sDg);
  make_symmat<N, double>(Dh, o.sDh);
  return o;
}

}  // namespace ldg_host
