// wave_kernels.hpp -- the gradient and right-hand-side kernels for small
// meshes (gfx950).
//
// ldg_kernels.hpp's kernels give a thread one line of an element for all five
// variables.  That is what large meshes want (few instructions, many
// elements in flight); a mesh of a few hundred elements leaves most of the
// chip idle, and the time of a launch is the length of one thread's
// instruction stream: about 2,700 vector instructions issued one wave at a
// time.  Here a workgroup of the same E elements has five waves, wave s
// doing the lines of variable s.  Every sweep stays within one variable, so
// the waves run on their own between the two places where the variables
// meet: the pointwise volume flux (one Gauss point per thread, over all five
// waves) and the face flux (wave D: direction D).  The stream of a thread is
// about a fifth as long.
//
// Measured, us per RK4 step (8 of these launches and the kinetic energy), these
// kernels / ldg_kernels.hpp's: FP64 8^3 p = 2 51 / 86, 8^3 p = 4 61 / 108, mixed
// 8^3 p = 4 54 / 94, 8^3 p = 5 64 / 115.  What is left there is the launches themselves (about 5 us
// each) and HBM latency.  On large meshes these kernels take longer (64-lane
// waves hold 50 lines at p = 4, every wave repeats the index arithmetic).
//
// The arithmetic of every value is that of ldg_kernels.hpp, operation by
// operation, and the kinetic-energy sum is taken in the same order (from the
// same partial sums: ke_per_element), so a launch's choice between these
// kernels and ldg_kernels.hpp's default does not show in its results.
#pragma once

#include "ldg_kernels.hpp"

namespace ldg {

// Orders the LDS accesses of a wave's lanes (the LDS executes a wave's
// operations in order; this only keeps the compiler from moving them).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Elements per workgroup: as many lines as fit one wave.
template <int N> struct WaveE { static constexpr int value = 64 / (N * N); };
constexpr int WAVE_NTH = 64 * NSTATE;

// line i of `count`, 64 lanes at a time
#define LDG_WAVE_LINES(i, count) _Pragma("unroll") for (int i0 = 0; i0 < (count); i0 += 64) if (const int i = i0 + l; i < (count))

template <int N, typename T, typename UT>
__global__ void __launch_bounds__(WAVE_NTH)
ldg_grad_wave_kernel(const UT *__restrict__ U, T *__restrict__ FF, LaunchArgs la, const unsigned char *__restrict__ img) {
  constexpr int E = WaveE<N>::value;
  using S = Shape<N, E>;
  static_assert(S::NTH == 64, "one wave per variable");
  constexpr int NN = S::NN, NF = S::NF, EV = S::EV, FS = E * NF, EN = E * N;
  __shared__ T su[NSTATE][E * NN];           // the block's state
  __shared__ T snb[3][NSTATE][FS];           // the -d neighbours' nodal traces
  __shared__ T swk[3][21][FS];               // face fields as in ldg_grad_kernel
  __shared__ T sedge[NSTATE][3][EN];         // per variable and direction: the second sweep's edge line
  const int lb = logical_block(la);
  if (lb < 0) return;
  int kl, ne;
  const InstDesc &d = block_span(la, lb, E, kl, ne);
  if (ne <= 0) return;
  const long k0 = d.elem_off + kl;
  const int t = threadIdx.x, l = t & 63, s = __builtin_amdgcn_readfirstlane(t >> 6);
  const int e = l / NF, ab = l - e * NF, b = ab / N, a = ab - b * N;
  const bool act = e < ne;
  const GOps<N, T> *const op = reinterpret_cast<const GOps<N, T> *>(img + (long)instance_of(la, lb) * GImage<N>::BYTES +
                                                                    GImage<N>::template offset<T>());
  const double rho0 = d.ph.rho0, E0 = d.ph.E0;
  struct Vec { T r[N]; };
  const SymMat<N, T> I = uniform_load<SymMat<N, T>, T>(&op->I);
  const SymMat<N, T> Dm = uniform_load<SymMat<N, T>, T>(&op->D);
  const Vec eta = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->eta));
  struct Sc { T r[3]; };
  const Sc sc = uniform_load<Sc, T>(reinterpret_cast<const Sc *>(op->a));
  int c[3];
  element_coords(d, kl + (act ? e : 0), c);

  // loads: variable s of the block, and its -d neighbours' traces
  constexpr int UL = (E * NN + 63) / 64;
  UT v[UL], vn[3];
#pragma unroll
  for (int i = 0; i < UL; ++i) {
    const int w = l + 64 * i < ne * NN ? l + 64 * i : ne * NN - 1;
    v[i] = U[k0 * EV + (w / NN * EV + s * NN + w % NN)];
  }
  {
    const int node[3] = {N - 1 + N * ab, a + N * (N - 1) + NF * b, ab + NF * (N - 1)};
#pragma unroll
    for (int D = 0; D < 3; ++D)
      vn[D] = U[(k0 + (act ? e : 0) + neighbor_step(d, c, D, -1)) * EV + s * NN + (act ? node[D] : 0)];
  }
#pragma unroll
  for (int i = 0; i < UL; ++i)
    if (l + 64 * i < ne * NN) su[s][l + 64 * i] = fluctuation<T>(v[i], s, rho0, E0);
  wave_sync();

  // own trace, neighbour's trace and normal derivative at the face nodes
  if (act) {
    const int base[3] = {N * ab, a + NF * b, ab};
    constexpr int ST[3] = {1, N, NF};
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      struct Row { T r[N]; };
      const Row nrm = uniform_load<Row, T>(reinterpret_cast<const Row *>(op->nrm[D]));
      const T nw = uniform_load<T, T>(&op->nbr[D]);
      const T *us = su[s] + e * NN + base[D];
      const T nbr = fluctuation<T>(vn[D], s, rho0, E0);
      T q = nw * nbr;
#pragma unroll
      for (int j = 0; j < N; ++j) q = fma_(nrm.r[j], us[j * ST[D]], q);
      swk[D][s][l] = us[0];
      swk[D][2 * NSTATE + s][l] = q;
      snb[D][s][l] = nbr;
    }
  }
  wave_sync();

  // which in-face derivative variable s carries along l on a -D face, -1: none
  auto deriv = [&](int D, int l_) -> int { return s == 0 ? 0 : s == 1 + D ? 1 : s == 1 + l_ ? 2 : -1; };
  auto dir_a = [](int D) { return D == 0 ? 1 : 0; };
  auto dir_b = [](int D) { return D == 2 ? 1 : 2; };
  auto scale = [&](int l_) -> T { return l_ == 0 ? sc.r[0] : l_ == 1 ? sc.r[1] : sc.r[2]; };
  // in-face derivative along a (before the first sweep overwrites the trace)
  LDG_WAVE_LINES(i, 3 * EN) {
    const int D = i / EN, x0 = i - D * EN, l_ = dir_a(D), f = deriv(D, l_);
    if (f >= 0) {
      const int at = D < 2 ? N * x0 : x0 / N * NF + x0 % N;
      T x[N], o[N];
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = swk[D][s][N * x0 + j];
      const T jmp = x[0] - snb[l_][s][at], al = scale(l_);
      sym_apply<N, -1, T>(Dm, x, o);
#pragma unroll
      for (int j = 0; j < N; ++j) swk[D][15 + f][N * x0 + j] = al * fma_(eta.r[j], jmp, o[j]);
    }
  }
  // the second sweep's edge lines
  LDG_WAVE_LINES(i, 3 * E) {
    const int D = i / E, ee = i - D * E, l_ = dir_b(D);
    if (deriv(D, l_) >= 0) {
      T x[N], o[N];
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = snb[l_][s][ee * NF + (D == 0 ? N * j : j)];
      sym_apply<N, 1, T>(I, x, o);
#pragma unroll
      for (int j = 0; j < N; ++j) sedge[s][D][ee * N + j] = o[j];
    }
  }
  wave_sync();
  // first sweep: the own trace, the neighbour's (from its nodal copy), the
  // normal derivative
  LDG_WAVE_LINES(i, 9 * EN) {
    const int g = i / (3 * EN), r = i - g * (3 * EN), D = r / EN, x0 = r - D * EN;
    T *const dst = &swk[D][g * NSTATE + s][N * x0];
    const T *const src = g == 1 ? &snb[D][s][N * x0] : dst;
    T x[N], o[N];
#pragma unroll
    for (int j = 0; j < N; ++j) x[j] = src[j];
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int j = 0; j < N; ++j) dst[j] = o[j];
  }
  wave_sync();
  // in-face derivative along b, and the second sweep of the one along a
  LDG_WAVE_LINES(i, 3 * EN) {
    const int D = i / EN, x0 = i - D * EN, at = x0 / N * NF + x0 % N, l_ = dir_b(D);
    const int fa = deriv(D, dir_a(D)), fb = deriv(D, l_);
    T x[N], o[N];
    if (fa >= 0) {
      T *const p = &swk[D][15 + fa][at];
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = p[N * j];
      sym_apply<N, 1, T>(I, x, o);
#pragma unroll
      for (int j = 0; j < N; ++j) p[N * j] = o[j];
    }
    if (fb >= 0) {
      const T *const p = &swk[D][s][at];
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = p[N * j];
      const T jmp = x[0] - sedge[s][D][x0], be = scale(l_);
      sym_apply<N, -1, T>(Dm, x, o);
      T *const fd = &swk[D][18 + fb][at];
#pragma unroll
      for (int j = 0; j < N; ++j) fd[N * j] = be * fma_(eta.r[j], jmp, o[j]);
    }
  }
  wave_sync();
  // second sweep
  LDG_WAVE_LINES(i, 9 * EN) {
    const int g = i / (3 * EN), r = i - g * (3 * EN), D = r / EN, x0 = r - D * EN;
    T *const p = &swk[D][g * NSTATE + s][x0 / N * NF + x0 % N];
    T x[N], o[N];
#pragma unroll
    for (int j = 0; j < N; ++j) x[j] = p[N * j];
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int j = 0; j < N; ++j) p[N * j] = o[j];
  }
  __syncthreads();

  // fluxes of direction D on wave D
  if (s < 3 && act) {
    const Bg<T> bg(d.ph);
    const size_t plane = (size_t)la.nelem * NF;
    T *const f0 = FF + (size_t)k0 * NF;
    auto one = [&](auto dir) {
      constexpr int D = decltype(dir)::value;
      T oK[5], oN[5];
      face_point_flux<T, D, FS>(&swk[D][0][l], bg, oK, oN);
      const int st = l + neighbor_step(d, c, D, -1) * NF;
      const T ad = sc.r[D];
#pragma unroll
      for (int v_ = 0; v_ < NSTATE; ++v_) {
        (f0 + (2 * D * NSTATE + v_) * plane)[l] = oN[v_] * ad;
        (f0 + ((2 * D + 1) * NSTATE + v_) * plane)[st] = oK[v_] * ad;
      }
    };
    if (s == 0) one(std::integral_constant<int, 0>());
    else if (s == 1) one(std::integral_constant<int, 1>());
    else one(std::integral_constant<int, 2>());
  }
}

// LDS of the right-hand side: per variable four sets A, B, C, D of E x N^3
// (element stride padded as in RhsLds), A and B together the FP64 rates in
// the mixed path, C and D first the jumps' face fields.
template <int N, typename T>
struct RhsWaveLds {
  static constexpr int E = WaveE<N>::value;
  static constexpr int ES = N * N * N + (N == 2 ? 0 : N == 3 ? 5 : N == 4 ? 4 : N == 5 ? 8 : 8);   // element stride
  static constexpr int SET = (E * ES + 1) / 2 * 2;
  static_assert(3 * E * N * N <= 2 * SET, "the jumps fit sets C and D");
};

template <int N, typename T, typename UT>
__global__ void __launch_bounds__(WAVE_NTH)
ldg_rhs_wave_kernel(const UT *__restrict__ U, const T *__restrict__ FF, LaunchArgs la,
                    const unsigned char *__restrict__ img, StageArgs st) {
  using L = RhsWaveLds<N, T>;
  constexpr int E = L::E, ES = L::ES, SET = L::SET;
  using S = Shape<N, E>;
  static_assert(S::NTH == 64, "one wave per variable");
  constexpr int NN = S::NN, NF = S::NF, EV = S::EV, FS = E * NF, EN = E * N;
  static_assert(E * NN <= WAVE_NTH, "one Gauss point per thread");
  __shared__ __align__(16) T sbuf[NSTATE][4][SET];
  const int lb = logical_block(la);
  if (lb < 0) return;
  const int t = threadIdx.x, l = t & 63, s = __builtin_amdgcn_readfirstlane(t >> 6);
  int kl, ne;
  const InstDesc &d = block_span(la, lb, E, kl, ne);
  if (ne <= 0) return;
  const long k0 = d.elem_off + kl;
  const int e = l / NF, ab = l - e * NF, b = ab / N, a = ab - b * N;
  const bool act = e < ne;
  const unsigned char *const im = img + (long)instance_of(la, lb) * GImage<N>::BYTES;
  const GOps<N, T> *const op = reinterpret_cast<const GOps<N, T> *>(im + GImage<N>::template offset<T>());
  const GOpsD<N> *const opd = reinterpret_cast<const GOpsD<N> *>(im);
  struct Vec { T r[N]; };
  T *const sA = sbuf[s][0], *const sB = sbuf[s][1], *const sC = sbuf[s][2], *const sD = sbuf[s][3], *const sJ = sC;
  double *const md = reinterpret_cast<double *>(sA);   // FP64: set A; mixed: sets A and B
  const int lx = N * ab, ly = a + NF * b, lz = ab;
  const int bx = e * ES + lx, by = e * ES + ly, bz = e * ES + lz;
  int c[3];
  element_coords(d, kl + (act ? e : 0), c);

  // ---- all loads of the variable: x-lines, jumps, face fluxes, and the
  // epilogue's operands
  UT v[N], vy, vz, nx, ny, nz;
  T fm[3], fp[3];
  const size_t plane = (size_t)la.nelem * NF;
  if (act) {
    const UT *const ue = U + (k0 + e) * EV + s * NN;
    const UT *const ux = ue + (long)neighbor_step(d, c, 0, -1) * EV + (N - 1 + N * ab);
    const UT *const uy = ue + (long)neighbor_step(d, c, 1, -1) * EV + (a + N * (N - 1) + NF * b);
    const UT *const uz = ue + (long)neighbor_step(d, c, 2, -1) * EV + (ab + NF * (N - 1));
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = ue[lx + q];
    vy = ue[ly];
    vz = ue[lz];
    nx = ux[0];
    ny = uy[0];
    nz = uz[0];
    const T *const ffo = FF + (size_t)k0 * NF;
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      fm[D] = (ffo + (2 * D * NSTATE + s) * plane)[l];
      fp[D] = (ffo + ((2 * D + 1) * NSTATE + s) * plane)[l];
    }
  }
  const bool need_u0 = (st.acc && st.acc_init) || st.unext || st.unext32;
  const bool need_acc = st.acc && !st.acc_init;
  constexpr int EPI = (E * NN + 63) / 64;
  unsigned ew[EPI], lw[EPI];
  double ru[EPI], ra[EPI];
#pragma unroll
  for (int it = 0; it < EPI; ++it) {
    const int i = l + it * 64, j = i < ne * NN ? i : ne * NN - 1;
    ew[it] = (unsigned)(j + j / NN * (EV - NN) + s * NN);
    lw[it] = (unsigned)(j + j / NN * (ES - NN));
    ru[it] = need_u0 ? (st.u0 + k0 * EV)[ew[it]] : 0.0;
    ra[it] = need_acc ? (st.acc + k0 * EV)[ew[it]] : 0.0;
  }

  const SymMat<N, T> I = uniform_load<SymMat<N, T>, T>(&op->I);
  // ---- x
  if (act) {
    const double rho0 = d.ph.rho0, E0 = d.ph.E0;
    auto fl = [&](UT x) -> T { return fluctuation<T>(x, s, rho0, E0); };
    T x[N], o[N];
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = fl(v[q]);
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int q = 0; q < N; ++q) sA[bx + q] = o[q];
    sJ[0 * FS + l] = x[0] - fl(nx);
    sJ[1 * FS + l] = fl(vy) - fl(ny);
    sJ[2 * FS + l] = fl(vz) - fl(nz);
  }
  wave_sync();
  // ---- y, and the jumps along a
  if (act) {
    T *p = sA + by;
    T x[N], o[N];
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = p[N * q];
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int q = 0; q < N; ++q) p[N * q] = o[q];
  }
  LDG_WAVE_LINES(i, 3 * EN) {
    T *p = sJ + N * i;
    T x[N], o[N];
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = p[q];
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int q = 0; q < N; ++q) p[q] = o[q];
  }
  wave_sync();
  // ---- z, and the jumps along b
  T ug[N];
  if (act) {
    T *p = sA + bz;
    T x[N];
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = p[NF * q];
    sym_apply<N, 1, T>(I, x, ug);
#pragma unroll
    for (int q = 0; q < N; ++q) p[NF * q] = ug[q];
  }
  LDG_WAVE_LINES(i, 3 * EN) {
    T *p = sJ + (i / N) * NF + i % N;
    T x[N], o[N];
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = p[N * q];
    sym_apply<N, 1, T>(I, x, o);
#pragma unroll
    for (int q = 0; q < N; ++q) p[N * q] = o[q];
  }
  wave_sync();
  // ---- d: the gradient of the variable into B, C, D (the jumps are read first)
  {
    T jmp[3];
#pragma unroll
    for (int D = 0; D < 3; ++D) jmp[D] = act ? sJ[D * FS + l] : T(0);
    wave_sync();
    if (act) {
#pragma unroll
      for (int D = 0; D < 3; ++D) {
        const SymMat<N, T> Dg = uniform_load<SymMat<N, T>, T>(&op->Dg[D]);
        const Vec ae = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->aeta[D]));
        const int at = D == 0 ? bx : D == 1 ? by : bz, stp = D == 0 ? 1 : D == 1 ? N : NF;
        T *const out = D == 0 ? sB : D == 1 ? sC : sD;
        T x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = D == 2 ? ug[q] : sA[at + stp * q];
        sym_apply<N, -1, T>(Dg, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) o[q] = fma_(ae.r[q], jmp[D], o[q]);
#pragma unroll
        for (int q = 0; q < N; ++q) out[at + stp * q] = o[q];
      }
    }
  }
  __syncthreads();
  // ---- p: one Gauss point per thread
  if (t < ne * NN) {
    const int pe = t / NN, pt = pe * ES + (t - pe * NN);
    const Bg<T> bg(d.ph);
    T w[NSTATE], g[NGRAD], F[NGRAD];
#pragma unroll
    for (int v_ = 0; v_ < NSTATE; ++v_) {
      w[v_] = sbuf[v_][0][pt];
      g[v_] = sbuf[v_][1][pt];
      g[NSTATE + v_] = sbuf[v_][2][pt];
      g[2 * NSTATE + v_] = sbuf[v_][3][pt];
    }
    volume_flux<T>(w, g, bg, F);
#pragma unroll
    for (int v_ = 0; v_ < NSTATE; ++v_) {
      sbuf[v_][1][pt] = F[v_];
      sbuf[v_][2][pt] = F[NSTATE + v_];
      sbuf[v_][3][pt] = F[2 * NSTATE + v_];
    }
  }
  __syncthreads();
  // ---- t: Dh F_l minus the faces; the z-line stays in registers
  T kz[N];
  if (act) {
    const Vec et = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->eta));
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      const SymMat<N, T> Dh = uniform_load<SymMat<N, T>, T>(&op->Dh[D]);
      const int at = D == 0 ? bx : D == 1 ? by : bz, stp = D == 0 ? 1 : D == 1 ? N : NF;
      T *const p = (D == 0 ? sB : D == 1 ? sC : sD) + at;
      T x[N], o[N];
#pragma unroll
      for (int q = 0; q < N; ++q) x[q] = p[stp * q];
      sym_apply<N, -1, T>(Dh, x, o);
#pragma unroll
      for (int q = 0; q < N; ++q) {
        const T r = o[q] - fma_(et.r[q], fm[D], et.r[N - 1 - q] * fp[D]);
        if (D < 2) p[stp * q] = r;
        else kz[q] = r;
      }
    }
  }
  wave_sync();
  // ---- zi, yi, xi (FP64)
  {
    const SymMat<N, double> Ii = uniform_load<SymMat<N, double>, double>(&opd->Ii);
    double r[N];
    if (act) {
      double x[N];
#pragma unroll
      for (int q = 0; q < N; ++q) x[q] = (double)(kz[q] + (sB[bz + NF * q] + sC[bz + NF * q]));
      sym_apply<N, 1, double>(Ii, x, r);
    }
    wave_sync();
    if (act) {
#pragma unroll
      for (int q = 0; q < N; ++q) md[bz + NF * q] = r[q];
    }
    wave_sync();
#pragma unroll
    for (int D = 1; D >= 0; --D) {
      if (act) {
        double *const p = md + (D == 1 ? by : bx);
        const int stp = D == 1 ? N : 1;
        double x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[stp * q];
        sym_apply<N, 1, double>(Ii, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[stp * q] = o[q];
      }
      wave_sync();
    }
  }
  // ---- epilogue of the variable
  {
    const double dtb = d.dt * st.cb, dta = d.dt * st.ca;
    const double bg = s == 0 ? d.ph.rho0 : s == NSTATE - 1 ? d.ph.E0 : 0.0;
    const long gofs = k0 * EV;
#pragma unroll
    for (int it = 0; it < EPI; ++it) {
      if (l + it * 64 < ne * NN) {
        const unsigned w = ew[it];
        double k = md[lw[it]];
        if (st.corr && st.gate[k0 + w / EV]) k += (st.corr + gofs)[w];
        if (st.kout) (st.kout + gofs)[w] = k;
        if (st.unext) (st.unext + gofs)[w] = ru[it] + dta * k;
        if (st.unext32) (st.unext32 + gofs)[w] = (float)(ru[it] + dta * k - bg);
        if (st.acc) {
          double x = st.acc_init ? ru[it] : ra[it];
          x += dtb * k;
          (st.acc + gofs)[w] = x;
          if (st.next32) (st.next32 + gofs)[w] = (float)(x - bg);
          if (st.ke_part) md[lw[it]] = x;
        }
      }
    }
  }
  if (st.ke_part) {
    __syncthreads();
    if (s == 0) {
      double kel = 0.0;
      if (act) {
        auto at = [&](int v_, int q) { return reinterpret_cast<const double *>(sbuf[v_][0])[bz + NF * q]; };
#pragma unroll
        for (int q = 0; q < N; ++q) {
          const double rho = at(0, q), m1 = at(1, q), m2 = at(2, q), m3 = at(3, q);
          kel += opd->w[a] * opd->w[b] * opd->w[q] * fma_(m3, m3, fma_(m2, m2, m1 * m1)) / (2.0 * rho);
        }
      }
      const double x = group_sum<64>(kel, nullptr);
      static_assert(E == 1 || !ke_per_element(N), "one element to a partial sum");
      if (t == 0) st.ke_part[ke_per_element(N) ? k0 : lb] = x;
    }
  }
}

#undef LDG_WAVE_LINES

}  // namespace ldg
