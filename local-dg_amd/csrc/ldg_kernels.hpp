// ldg_kernels.hpp -- HIP kernels of the LDG right-hand side for gfx950.
//
// One RK4 stage is two launches over the whole periodic mesh:
//   ldg_grad_kernel  auxiliary gradient Q_l = (1/alpha_l)(Dn U + L0 jump_l)
//                    (Solver::rk4Rhs first half, solver.cpp:490-508) on the
//                    faces and the Roe + one-sided viscous face fluxes of both
//                    elements of every face (solver.cpp:643-698, 750-814,
//                    891-921, 1194-1374)
//   ldg_rhs_kernel   the volume gradient and volume integrals, minus the
//                    face terms, the return to the nodes (with W^-1 in the
//                    operators: the inverse mass) and the fused RK4 stage
//                    epilogue (solver.cpp:510-535 and 410-434)
// Both stage a block of E consecutive elements in LDS, work in 1D "lines"
// of N = p+1 values owned by one thread (in-place sum-factorised sweeps in
// Gauss form, see GOps, with the even/odd split of the centro-symmetric 1D
// operators, symop.hpp), and read the periodic neighbours' face slices
// straight from HBM (the on-device form of the single-rank halo exchange,
// solver.cpp:929-998).
//
// Precision: the state, the RK4 combination, the return to the nodes (I^-1
// along three directions) and every reduction are FP64.  The interpolation,
// flux evaluation, derivatives and face terms (Dh, eta, which hold the
// inverse mass's W^-1) run in the compute type T (double for the plain path,
// float for the mixed path), on fluctuations about the constant background
// (rho0, 0, 0, 0, E0 = p0/(gamma-1)): the background is subtracted in FP64
// when U is loaded (exact, both values are close), so the O(1/M0^2) part of
// the energy never enters the T-precision arithmetic.  A constant state is a
// discrete steady state, so the fluctuation form changes nothing but
// rounding.
//
// Data in HBM:
//   u0, acc, unext : FP64 (node, state, element) -- the reference layout
//   U (stage input): the same, or in the mixed path (RK stages 2-4) FP32
//                    fluctuations about the background in that layout
//   FF             : T, [direction][side][state][element][face Gauss point]:
//                    the face fluxes (gradient kernel -> rhs kernel)
//   Q              : TQ (node, s + 5*l, element) -- the nodal gradient, 15
//                    fields per element, written only when asked for
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

#include "symop.hpp"

namespace ldg {

constexpr int NSTATE = 5;
constexpr int NGRAD = 15;
constexpr int NT = 256;          // threads per workgroup

// 1D operators (row-major [row][col]), FP64, in device memory.
template <int N, typename T>
struct Ops {
  T I[N][N];      // I[q][i]  = l_i(g_q)
  T D[N][N];      // D[q][i]  = l_i'(g_q)
  T Dn[N][N];     // Dn[i][j] = l_j'(r_i)
  T Minv[N][N];   // inverse 1D mass matrix
  T L0[N];        // Minv[:, 0]: lift of the jump at the left face
  T w[N];         // Gauss weights
  T eta[N];       // L_q(-1) / w_q: that lift in Gauss form (I L0)
  // sweep operators in even/odd split form: I, D = I Dn, I^-1, the
  // derivative Dg at the Gauss points of the polynomial through them, and
  // W^-1 Dg^T W
  SymMat<N, T> sI, sD, sIi, sDg, sDh;
};

struct MeshArgs {
  int nx, ny, nz;
  double ialpha[3];      // 2 / dx_l
};

struct PhysArgs {
  double gamma, gm1, mu, kappa;   // kappa = mu gamma / Pr acting on grad(e)
  double rho0, E0, H0;            // background: E0 = p0/(gamma-1), H0 = E0 + p0
};

struct StageArgs {
  const double *u0;   // u^n (RK base state)
  double *acc;        // running u^n + dt sum b_s k_s
  double *unext;      // next stage input u^n + dt a_s k_s
  float *unext32;     // or, in the mixed path, that input as FP32 fluctuations about the background
  float *next32;      // stage 4 (mixed): the new running sum u^{n+1} as FP32 fluctuations, the
                      // next step's stage-1 input when that step follows in the same call
  double *kout;       // raw k (parity / single RHS)
  double cb, ca;      // RK4 coefficients b_s, a_s (times each instance's dt)
  int acc_init;       // 1: acc = u0 + dt b k   0: acc += dt b k
  double *ke_part;    // per-workgroup partial sums of the reference KE of acc
  double *diag_part;  // or those of the diagnostics (reference KE, Gauss KE, enstrophy)
  const double *corr;          // learned closure: k += corr where gate[element] != 0
  const unsigned char *gate;
};

// One solver instance inside a launch.  A launch covers the elements of all
// instances of one order (an ensemble); a single solver is a launch of one
// instance.  Instances are stored back to back in the launch's arrays.
// n / d for 0 <= n < 2^31 by one 32x32->64-bit multiply and a shift
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994): with l = ceil(log2 d), s = 31 + l and
// m = ceil(2^s / d) < 2^32, floor(n m / 2^s) = floor(n / d) because the
// error n (m d - 2^s) / (d 2^s) < n / 2^s <= 2^-l <= 1/d.  Built on the host;
// with uniform operands the device evaluates it on the scalar unit, where a
// plain division by a run-time value would take a dozen vector instructions.
struct FastDiv {
  unsigned m;
  int s;
  __host__ __device__ inline int div(int n) const {
    return (int)(((unsigned long long)(unsigned)n * m) >> s);
  }
};
inline FastDiv make_fastdiv(int d) {
  int l = 0;
  while ((1LL << l) < d) ++l;
  FastDiv f;
  f.s = 31 + l;
  f.m = (unsigned)(((1ULL << f.s) + (unsigned long long)d - 1) / (unsigned long long)d);
  return f;
}

struct InstDesc {
  int nx, ny, nz;
  int nblocks;           // its logical workgroups (whole bricks, see block_elements)
  long nelem;            // elements of this instance
  long elem_off;         // its first element in the launch's arrays
  int block_off;         // its first logical workgroup
  int nbx;               // element blocks per x-row: ceil(nx / E)
  int tb[3];             // brick of tb[0] x tb[1] x tb[2] blocks (x blocks, y rows, z planes)
  int nbrick[3];         // bricks per direction
  FastDiv div_bs, div_nb0, div_nb1, div_tb0, div_tb1;   // by tb0 tb1 tb2, nbrick[0], nbrick[1], tb[0], tb[1]
  // spans (see span_elements): ncy strips of `rows` rows (the last one of the
  // rest); nbr workgroups per strip plane, main_blocks in all strips but the last
  int ncy, rows, nbr, main_blocks;
  FastDiv div_nx, div_ny, div_nz;
  FastDiv div_nbr, div_last;             // by nbr, and by the last strip's workgroups per plane
  double ialpha[3];      // 2 / dx_l
  double dt;             // its time step
  PhysArgs ph;
};

// Elements of an instance's logical workgroup lbl (0-based within the
// instance): blocks are E consecutive elements of one x-row, and blocks are
// visited brick by brick (tb blocks per brick, bricks x-fastest), so that the
// workgroups resident at the same time on an XCD cover a compact region and
// their face neighbours in y and z are mostly in that XCD's L2.  Returns the
// coordinates of the first element and the count, 0 for a padding block of
// a partial brick.
__host__ __device__ inline void block_elements(const InstDesc &d, int E, int lbl, int ec[3], int &ne) {
  const int bs = d.tb[0] * d.tb[1] * d.tb[2];
  const int brick = d.div_bs.div(lbl), off = lbl - brick * bs;
  const int t = d.div_nb0.div(brick), Bx = brick - t * d.nbrick[0];
  const int Bz = d.div_nb1.div(t), By = t - Bz * d.nbrick[1];
  const int u = d.div_tb0.div(off), ox = off - u * d.tb[0];
  const int oz = d.div_tb1.div(u), oy = u - oz * d.tb[1];
  const int bx = Bx * d.tb[0] + ox, ey = By * d.tb[1] + oy, ez = Bz * d.tb[2] + oz;
  ec[0] = ec[1] = ec[2] = 0;
  ne = 0;
  if (bx >= d.nbx || ey >= d.ny || ez >= d.nz) return;
  ec[0] = bx * E; ec[1] = ey; ec[2] = ez;
  ne = (d.nx - ec[0]) < E ? (d.nx - ec[0]) : E;
}

// Elements of an instance's logical workgroup lbl in the span numbering of
// the gradient and right-hand-side kernels: E consecutive elements kl ..
// kl + ne - 1 (ne < E only at the end of a run; there are no empty
// workgroups).  The mesh is cut into strips of whole rows in y that are walked
// plane by plane along z; a strip's part of a plane is a run of consecutive
// elements.  The traces a workgroup gathers from its -y and -z neighbours were
// read one row and one plane of the strip earlier and are still in the XCD's
// L2 (or, where a plane is large, in the memory-side cache).
__host__ __device__ inline void span_elements(const InstDesc &d, int E, int lbl, int &kl, int &ne) {
  int st, z, j;
  if (lbl < d.main_blocks) {
    const int run = d.div_nbr.div(lbl);
    j = lbl - run * d.nbr;
    st = d.div_nz.div(run);
    z = run - st * d.nz;
  } else {
    const int r = lbl - d.main_blocks, last = d.ny - (d.ncy - 1) * d.rows, nb = (last * d.nx + E - 1) / E;
    st = d.ncy - 1;
    z = d.div_last.div(r);
    j = r - z * nb;
  }
  const int y0 = st * d.rows;
  const int len = (d.ny - y0 < d.rows ? d.ny - y0 : d.rows) * d.nx;
  kl = (z * d.ny + y0) * d.nx + j * E;
  ne = len - j * E < E ? len - j * E : E;
}

// Sets d's span numbering (d.nx, ny, nz, nelem given) for workgroups of E
// elements with n nodes per direction; returns the number of workgroups.  An
// eighth of the rows to a strip: logical_block gives each of the 8 XCDs an
// eighth of the workgroups, so that an XCD walks a strip of its own.  Below
// 96 MB of state a strip's part of a plane is about 1 MB, a quarter of an
// XCD's L2: the same time alone, and 0.5 % less in an ensemble, where an XCD
// walks whole instances (48 of them, 2 steps 5.64 ms).  Measured against
// columns of about 16 x 16 elements (p = 4, 1 MB of a plane) and against strips
// of 2 to 12 rows, ms per step mixed / FP64: 64^3 p = 4 8 rows 6.28 / 10.15,
// columns 6.58 / 10.39, 4 rows 6.46 / 10.28, 12 rows 6.41 / 10.21; 80^3 p = 4
// 12.2 / 19.7 against 13.2 / 20.3; 100^3 p = 2 6.43 / 10.0 against 6.93 / 10.6;
// 61x37x29 p = 4 1.65 / 2.54 against 1.75 / 2.64; planes of 10 MB (128 x 128)
// 6.31 / 9.88 against 6.67 / 10.1; 24^3 p = 5 2 % less.
// More rows where the runs' last workgroups would be more than 2 % of all:
// 24^3, p = 2 has 2112 instead of 1992 with 3 rows, 8.25 instead of 7.8 per CU,
// and took 9 % longer; 31x17x23, p = 3, mixed takes 449 us for 2 steps instead
// of 506 with two strips of 9 and 8 rows.
inline long make_spans(InstDesc &d, int n, int E) {
  const double el = 8.0 * NSTATE * n * n * n;
  long nbr, nl, main, nb;
  int r = el * d.nx * d.ny * d.nz > 96e6 ? (d.ny + 7) / 8 : std::min(d.ny, std::max(1, (int)(1048576.0 / (el * d.nx))));
  for (;; ++r) {
    d.ncy = (d.ny + r - 1) / r;
    d.rows = (d.ny + d.ncy - 1) / d.ncy;
    d.ncy = (d.ny + d.rows - 1) / d.rows;
    const int last = d.ny - (d.ncy - 1) * d.rows;
    nbr = ((long)d.rows * d.nx + E - 1) / E;
    nl = ((long)last * d.nx + E - 1) / E;
    main = (long)(d.ncy - 1) * d.nz * nbr;
    nb = main + nl * d.nz;
    if (r >= d.ny || nb * E <= 1.02 * d.nx * d.ny * d.nz) break;
  }
  if (nb > (1L << 30)) return nb;
  d.nbr = (int)nbr;
  d.main_blocks = (int)main;
  d.div_last = make_fastdiv((int)nl);
  d.div_nbr = make_fastdiv(d.nbr);
  d.div_nx = make_fastdiv(d.nx);
  d.div_ny = make_fastdiv(d.ny);
  d.div_nz = make_fastdiv(d.nz);
  return nb;
}

struct LaunchArgs {
  const InstDesc *inst;
  const int *blk_inst;   // logical workgroup -> instance (nullptr: one instance)
  int nblocks;           // logical workgroups of the launch
  int per_xcd;           // ceil(nblocks / 8)
  long nelem;            // elements of the launch (all instances)
};

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of element blocks so that face neighbours share that
// XCD's L2.  Returns -1 for padding workgroups.
__device__ inline int logical_block(const LaunchArgs &la) {
  const int b = blockIdx.x;
  const int lb = (b & 7) * la.per_xcd + (b >> 3);
  return lb < la.nblocks ? lb : -1;
}

__device__ inline int instance_of(const LaunchArgs &la, int lb) { return la.blk_inst ? la.blk_inst[lb] : 0; }

// The instance of logical workgroup lb and the block's span of elements
// (local to the instance).
__device__ inline const InstDesc &block_span(const LaunchArgs &la, int lb, int E, int &kl, int &ne) {
  const InstDesc &d = la.inst[instance_of(la, lb)];
  span_elements(d, E, lb - d.block_off, kl, ne);
  return d;
}

// The instance of logical workgroup lb, its mesh, and the block's first
// element (coordinates ec and index kl, local to the instance) and element
// count.
template <int E>
__device__ inline const InstDesc &block_instance(const LaunchArgs &la, int lb, MeshArgs &m, int ec[3], long &kl,
                                                 int &ne) {
  const InstDesc &d = la.inst[la.blk_inst ? la.blk_inst[lb] : 0];
  m.nx = d.nx; m.ny = d.ny; m.nz = d.nz;
  m.ialpha[0] = d.ialpha[0]; m.ialpha[1] = d.ialpha[1]; m.ialpha[2] = d.ialpha[2];
  block_elements(d, E, lb - d.block_off, ec, ne);
  kl = ec[0] + (long)d.nx * (ec[1] + (long)d.ny * ec[2]);
  return d;
}

// c + dir (dir = +-1) on a periodic axis of n elements
__device__ inline int wrap_step(int c, int dir, int n) {
  c += dir;
  return c < 0 ? c + n : (c >= n ? c - n : c);
}

// Face neighbours of the block's elements (periodic; the reference builds
// the same table as eToE, mesh.cpp:201-315, with ghost slots on the faces),
// computed once per workgroup from the first element's coordinates ec:
// nb[e][f] for faces f = -x,+x,-y,+y,-z,+z.
__device__ inline void fill_neighbors(const MeshArgs &m, const int ec[3], long off, int ne, long (*nb)[6], int tid) {
  if (tid < ne * 6) {
    const int e = tid / 6, f = tid % 6, dim = f >> 1, dir = (f & 1) ? 1 : -1;
    int x = ec[0] + e, y = ec[1], z = ec[2];
    if (dim == 0) x = wrap_step(x, dir, m.nx);
    else if (dim == 1) y = wrap_step(y, dir, m.ny);
    else z = wrap_step(z, dir, m.nz);
    nb[e][f] = off + x + (long)m.nx * (y + (long)m.ny * z);
  }
}

// ---------------------------------------------------------------------
// Pointwise physics in fluctuation form, textbook forms of
// solver.cpp:1040-1374.  A state w = (rho - rho0, rho u, rho v, rho w,
// E - E0); p' = p - p0 = (gamma-1)(w4 - |m|^2/(2 rho)) and
// E + p = H0 + w4 + p'.
// ---------------------------------------------------------------------
// Reciprocal and square root: correctly rounded in FP64; in FP32 (the
// mixed path, whose error budget is set by FP32 rounding anyway) the
// hardware approximations v_rcp_f32 / v_sqrt_f32 (1 ulp).
__device__ inline double rcp(double x) { return 1.0 / x; }
__device__ inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double sqrt_(double x) { return sqrt(x); }
__device__ inline float sqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }

// The pointwise physics says itself where a multiply-add is fused, and the
// compiler fuses nothing else there (fp contract(off)): which product of a
// sum it picks depends on the code around, and the kernels of this file and
// of wave_kernels.hpp are to agree bit by bit.
__device__ inline double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <typename T>
struct Bg {
  T rho0, E0, H0, gm1, mu, kappa;
  __device__ inline explicit Bg(const PhysArgs &p)
      : rho0(T(p.rho0)), E0(T(p.E0)), H0(T(p.H0)), gm1(T(p.gm1)), mu(T(p.mu)), kappa(T(p.kappa)) {}
};

// Velocity gradient gv[i][l] and internal-energy gradient ge[l] from the
// state (density rho = 1/ir, velocity v, total energy E) and the conserved
// gradients g[s + 5 l].
template <typename T>
__device__ inline void prim_grads(T ir, T E, const T v[3], const T *g, T gv[3][3], T ge[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const T drho = g[5 * l];
#pragma unroll
    for (int i = 0; i < 3; ++i) gv[i][l] = fma_(-v[i], drho, g[1 + i + 5 * l]) * ir;
    const T dEr = fma_(-(E * ir), drho, g[4 + 5 * l]) * ir;
    ge[l] = dEr - fma_(v[2], gv[2][l], fma_(v[1], gv[1][l], v[0] * gv[0][l]));
  }
}

// p - p0 of the fluctuation w with velocity v
template <typename T>
__device__ inline T pressure(const T w[5], const T v[3], const Bg<T> &b) {
#pragma clang fp contract(off)
  return b.gm1 * fma_(T(-0.5), fma_(w[3], v[2], fma_(w[2], v[1], w[1] * v[0])), w[4]);
}

// Volume flux F[s + 5 l] = Fc_l(u) - Fv_l(u, g) (fluxC minus fluxV,
// solver.cpp:1040-1188).  The momentum flux carries p' = p - p0: a constant
// pressure contributes exactly nothing to the discrete residual (the Gauss
// rules integrate d(phi)/dx and the face traces of phi exactly).
template <typename T>
__device__ inline void volume_flux(const T w[5], const T *g, const Bg<T> &b, T F[15]) {
#pragma clang fp contract(off)
  const T rho = b.rho0 + w[0];
  const T ir = rcp(rho);
  const T v[3] = {w[1] * ir, w[2] * ir, w[3] * ir};
  const T pf = pressure(w, v, b);
  const T hv = b.H0 + w[4] + pf;   // E + p
  T gv[3][3], ge[3], tau[3][3];
  prim_grads<T>(ir, b.E0 + w[4], v, g, gv, ge);
  const T m23 = (b.mu * T(2.0 / 3.0)) * (gv[0][0] + gv[1][1] + gv[2][2]);
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int i = 0; i <= l; ++i)
      tau[i][l] = tau[l][i] = i == l ? fma_(b.mu, gv[i][l] + gv[l][i], -m23) : b.mu * (gv[i][l] + gv[l][i]);
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    F[5 * l] = w[1 + l];
#pragma unroll
    for (int i = 0; i < 3; ++i) F[1 + i + 5 * l] = fma_(w[1 + i], v[l], i == l ? pf - tau[i][l] : -tau[i][l]);
    F[4 + 5 * l] =
        fma_(hv, v[l], -fma_(b.kappa, ge[l], fma_(v[2], tau[2][l], fma_(v[1], tau[1][l], v[0] * tau[0][l]))));
  }
}

// Fluxes of one face, for both elements that share it.  The face has the
// element K on its - side and the element N on its + side (normal +e_D out
// of K); wK, wN are the two traces and q the gradient trace chosen by the
// one-sided switch, which is N's own on this face for both sides (the
// switch takes the + side element's gradient: the neighbour's for K, whose
// normal sum is positive, and N's own for N).  Returns K's flux
//   outK = Roe(uN, uK, +e_D) - Fv_D(uK, q)
// (numericalFluxC, solver.cpp:1194-1374; numericalFluxV, solver.cpp:891-921)
// and N's flux on the same face, whose normal is -e_D,
//   outN = Roe(uK, uN, -e_D) + Fv_D(uN, q) = -Roe(uN, uK, +e_D) + Fv_D(uN, q):
// the Roe flux is evaluated once and enters the two sides with opposite
// signs (F*(a, b, n) = -F*(b, a, -n): the Roe average is symmetric in the
// two states and |A(-n)| = |A(n)|), while the viscous flux is evaluated on
// each side's own trace, as the reference does.
template <typename T, int D>
__device__ inline void visc_face(const T w[5], T ir, const T v[3], const T *q, const Bg<T> &b, T fv[4]) {
#pragma clang fp contract(off)
  T gv[3][3], ge[3];
  prim_grads<T>(ir, b.E0 + w[4], v, q, gv, ge);
  const T m23 = (b.mu * T(2.0 / 3.0)) * (gv[0][0] + gv[1][1] + gv[2][2]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
    fv[i] = i == D ? fma_(b.mu, gv[i][D] + gv[D][i], -m23) : b.mu * (gv[i][D] + gv[D][i]);
  fv[3] = fma_(b.kappa, ge[D], fma_(v[2], fv[2], fma_(v[1], fv[1], v[0] * fv[0])));
}

// Whether the Roe flux between the traces wK and wN is a number: the squared
// sound speed of their Roe average (face_flux_pair's c2) is positive and finite.
template <typename T>
__device__ inline bool roe_defined(const T wK[5], const T wN[5], const Bg<T> &b) {
#pragma clang fp contract(off)
  const T irN = rcp(b.rho0 + wN[0]), irK = rcp(b.rho0 + wK[0]);
  const T vN[3] = {wN[1] * irN, wN[2] * irN, wN[3] * irN};
  const T vK[3] = {wK[1] * irK, wK[2] * irK, wK[3] * irK};
  const T HN = (b.H0 + wN[4] + pressure(wN, vN, b)) * irN, HK = (b.H0 + wK[4] + pressure(wK, vK, b)) * irK;
  const T s = sqrt_((b.rho0 + wN[0]) * irK);
  T vt[3];   // times s + 1, as the velocities of the average
#pragma unroll
  for (int i = 0; i < 3; ++i) vt[i] = fma_(s, vN[i], vK[i]);
  const T q2 = fma_(vt[2], vt[2], fma_(vt[1], vt[1], vt[0] * vt[0]));
  const T c2 = fma_(T(-0.5), q2, fma_(s, HN, HK) * (s + T(1)));   // times (s + 1)^2 / (gamma - 1)
  return c2 > T(0) && c2 <= std::numeric_limits<T>::max();
}

template <typename T, int D>
__device__ inline void face_flux_pair(const T wK[5], const T wN[5], const T *q, const Bg<T> &b, T outK[5],
                                      T outN[5]) {
#pragma clang fp contract(off)
  const T rN = b.rho0 + wN[0], rK = b.rho0 + wK[0];
  const T irN = rcp(rN), irK = rcp(rK);
  const T vN[3] = {wN[1] * irN, wN[2] * irN, wN[3] * irN};
  const T vK[3] = {wK[1] * irK, wK[2] * irK, wK[3] * irK};
  const T pN = pressure(wN, vN, b), pK = pressure(wK, vK, b);                               // p - p0
  const T hN = b.H0 + wN[4] + pN, hK = b.H0 + wK[4] + pK;                                   // E + p
  const T HN = hN * irN, HK = hK * irK;
  const T qN = vN[D], qK = vK[D];
  const T s = sqrt_(rN * irK);
  const T iden = rcp(s + T(1));
  T vt[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) vt[i] = fma_(s, vN[i], vK[i]) * iden;
  const T ht = fma_(s, HN, HK) * iden;
  const T q2 = fma_(vt[2], vt[2], fma_(vt[1], vt[1], vt[0] * vt[0]));
  const T qt = vt[D];
  const T c2 = b.gm1 * fma_(T(-0.5), q2, ht);
  const T c = sqrt_(c2), ic = rcp(c);
  const T l0 = fabs(qt), lp = fabs(qt + c), lm = fabs(qt - c);
  T dd[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) dd[k] = wN[k] - wK[k];
  const T dp = b.gm1 * (fma_(T(0.5) * q2, dd[0], -fma_(vt[2], dd[3], fma_(vt[1], dd[2], vt[0] * dd[1]))) + dd[4]);
  const T dV = fma_(-qt, dd[0], dd[1 + D]);
  const T s1 = fma_(T(0.5), lp + lm, -l0), s2 = T(0.5) * (lp - lm);
  const T dpi = dp * ic;
  const T A = fma_(s1, dpi, s2 * dV) * ic;
  const T B = fma_(s2, dpi, s1 * dV);
  // R = (F(N) + F(K) - |A| (uN - uK)) / 2 along D
  T R[5];
  R[0] = T(0.5) * (fma_(rN, qN, rK * qK) - fma_(l0, dd[0], A));
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const T x = fma_(wN[1 + i], qN, wK[1 + i] * qK), y = fma_(l0, dd[1 + i], A * vt[i]);
    R[1 + i] = T(0.5) * (i == D ? (x + (pN + pK)) - (y + B) : x - y);
  }
  R[4] = T(0.5) * (fma_(hN, qN, hK * qK) - fma_(l0, dd[4], fma_(A, ht, B * qt)));
  T fK[4], fN[4];
  visc_face<T, D>(wK, irK, vK, q, b, fK);
  visc_face<T, D>(wN, irN, vN, q, b, fN);
  outK[0] = R[0];
  outN[0] = -R[0];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    outK[1 + i] = R[1 + i] - fK[i];
    outN[1 + i] = fN[i] - R[1 + i];
  }
}

// ---------------------------------------------------------------------
// The element's operators in Gauss form.
//
// A basis polynomial is as well given by its values at the N Gauss points
// (u_g = I u) as by those at the nodes, and in that form every operator of
// the scheme is a 1D derivative, a rank-1 face term, or I and its inverse:
//   LDG gradient     Q_l = a_l (Dg u_g + eta J_l)             a_l = 2/dx_l
//   volume + faces   k_g = sum_l a_l (Dh F_l) - eta f_l^- - eta' f_l^+
//   rate             k   = (I^-1 (x) I^-1 (x) I^-1) k_g
// with Dg the derivative at the Gauss points of the polynomial through
// them, Dh = W^-1 Dg^T W, eta_q = L_q(-1) / w_q (L_q: Lagrange polynomial of
// Gauss point q; eta'_q = eta_{N-1-q} for the + face), J_l the jump u - u_nbr
// on the -l face and f_l the face fluxes times a_l, both at the face Gauss
// points.  It is the weak form of the nodal scheme, exactly: M1 = I^T W I
// (the rule integrates products of two basis polynomials exactly), so
// M1^-1 I^T = I^-1 W^-1 turns the test functions and the inverse mass into
// W^-1 in Gauss form, D^T = I^T Dg^T, and M1^-1 e_0 = I^-1 eta.
// Against sweeping with I, D, I^T, D^T and M1^-1 at the nodes it needs 60
// field sweeps of a line instead of 100, no weights at the points, and the
// face fluxes stay at the face Gauss points (no lift).
// ---------------------------------------------------------------------
template <int N, typename T>
struct GOps {
  SymMat<N, T> I;                          // nodes -> Gauss points
  SymMat<N, T> Dg[3], Dh[3];               // a_l Dg, a_l Dh (l = x, y, z)
  T eta[N];
  T aeta[3][N];                            // a_l eta: the lift of J_l
  // the face kernel: D = I Dn along the face (unscaled), the derivative
  // along the normal at the - face node, a_d (Dn[0][:] + L0[0] e_0), and the
  // neighbour's weight in it, -a_d L0[0]
  SymMat<N, T> D;
  T nrm[3][N];
  T nbr[3];
  T a[3];
};
template <int N>
struct GOpsD {                             // FP64 in every path
  SymMat<N, double> Ii;                    // Gauss points -> nodes
  double w[N];                             // Gauss weights
};

// An FP32 operator is rounded once, and what its coefficients miss acts alike
// on every element in every step.  What acts on constants matters most, since a
// field is nearly constant over an element: I has to reproduce them, the
// derivatives have to give zero, and Dh has to balance the face terms of a
// constant flux.  So in each row the smallest coefficient, whose rounding unit
// is the finest, takes up the sum of the others' rounding.  64^3, p = 4, mixed
// against FP64 at t = 1, coefficients rounded one by one / like this: kinetic
// energy 1.5e-7 / 2.0e-9, -dEk/dt 3.7e-3 / 2.4e-4, momentum 2.4e-7 / 7.3e-8.

// Moves the smallest of the coefficients c that are not zero so that
// sum_i weight[i] c[i] is `target` as nearly as its precision allows.
template <typename T>
void fit_sum(T *const *c, const double *weight, int n, double target) {
  double r = target;
  int k = -1;
  for (int i = 0; i < n; ++i) {
    r -= weight[i] * (double)*c[i];
    if (*c[i] != T(0) && (k < 0 || std::fabs((double)*c[i]) < std::fabs((double)*c[k]))) k = i;
  }
  if (k >= 0) *c[k] = T((double)*c[k] + r / weight[k]);
}

// The same for the rows of an operator (symmetry S) applied to constants.
template <int N, typename T>
void fit_rows(SymMat<N, T> &m, int S, const double (&target)[N]) {
  T *c[N];
  double w[N];
  for (int q = 0; q < (N + 1) / 2; ++q) {
    int n = 0;
    if constexpr (SymMat<N, T>::SPLIT) {
      if (S < 0 && 2 * q + 1 == N) break;    // the even part of the middle row is zero
      for (int j = 0; j < N / 2; ++j) { c[n] = &m.P[q][j]; w[n++] = 2.0; }
      if (N & 1) { c[n] = &m.C[q]; w[n++] = 1.0; }
      fit_sum(c, w, n, target[q]);
    } else {
      for (int i : {q, N - 1 - q}) {
        for (n = 0; n < N; ++n) { c[n] = &m.A[i][n]; w[n] = 1.0; }
        fit_sum(c, w, n, target[i]);
      }
    }
  }
}

template <int N, typename T>
void fill_gops(GOps<N, T> &g, const Ops<N, double> &op, const double a[3]) {
  constexpr int MS = sizeof(SymMat<N, T>) / sizeof(T);
  static_assert(sizeof(SymMat<N, double>) == MS * sizeof(double), "operators are plain coefficient arrays");
  auto put = [&](SymMat<N, T> &d, const SymMat<N, double> &s, double f) {
    for (int i = 0; i < MS; ++i) reinterpret_cast<T *>(&d)[i] = T(reinterpret_cast<const double *>(&s)[i] * f);
  };
  put(g.I, op.sI, 1.0);
  put(g.D, op.sD, 1.0);
  for (int l = 0; l < 3; ++l) {
    put(g.Dg[l], op.sDg, a[l]);
    put(g.Dh[l], op.sDh, a[l]);
    for (int q = 0; q < N; ++q) {
      g.aeta[l][q] = T(op.eta[q] * a[l]);
      g.nrm[l][q] = T((op.Dn[0][q] + (q == 0 ? op.L0[0] : 0.0)) * a[l]);
    }
    g.nbr[l] = T(-op.L0[0] * a[l]);
    g.a[l] = T(a[l]);
  }
  for (int q = 0; q < N; ++q) g.eta[q] = T(op.eta[q]);
  if constexpr (sizeof(T) < sizeof(double)) {
    double one[N], zero[N], dh[N];
    for (int q = 0; q < N; ++q) { one[q] = 1.0; zero[q] = 0.0; }
    fit_rows<N, T>(g.I, 1, one);
    fit_rows<N, T>(g.D, -1, zero);
    for (int l = 0; l < 3; ++l) {
      fit_rows<N, T>(g.Dg[l], -1, zero);
      for (int q = 0; q < N; ++q) dh[q] = (double)g.a[l] * ((double)g.eta[N - 1 - q] - (double)g.eta[q]);
      fit_rows<N, T>(g.Dh[l], -1, dh);
      T *c[N + 1];
      double w[N + 1];
      for (int q = 0; q < N; ++q) { c[q] = &g.nrm[l][q]; w[q] = 1.0; }
      c[N] = &g.nbr[l];
      w[N] = 1.0;
      fit_sum(c, w, N + 1, 0.0);
    }
  }
}

// Operator image of one instance: FP64-only part, FP32 and FP64 operators,
// each padded to 16 bytes.
template <int N>
struct GImage {
  static constexpr int pad(size_t b) { return (int)((b + 15) / 16 * 16); }
  static constexpr int OF = pad(sizeof(GOpsD<N>)), OD = OF + pad(sizeof(GOps<N, float>));
  static constexpr int BYTES = OD + pad(sizeof(GOps<N, double>));
  template <typename T>
  __host__ __device__ static constexpr int offset() { return sizeof(T) == sizeof(double) ? OD : OF; }
};
template <int N>
void fill_image(unsigned char *b, const Ops<N, double> &op, const double a[3]) {
  GOpsD<N> &d = *reinterpret_cast<GOpsD<N> *>(b);
  d.Ii = op.sIi;
  for (int q = 0; q < N; ++q) d.w[q] = op.w[q];
  fill_gops<N, float>(*reinterpret_cast<GOps<N, float> *>(b + GImage<N>::OF), op, a);
  fill_gops<N, double>(*reinterpret_cast<GOps<N, double> *>(b + GImage<N>::OD), op, a);
}

// A wave-uniform constant object (an operator) through the scalar cache:
// its coefficients become scalar registers, one of which a vector
// instruction reads as an operand, so a sweep holds no coefficients in
// vector registers and reads none from LDS.
template <typename S, typename T>
__device__ inline S uniform_load(const S *p) {
  static_assert(sizeof(S) % sizeof(T) == 0, "whole words");
  S s;
  const __attribute__((address_space(4))) T *src = (const __attribute__((address_space(4))) T *)(unsigned long long)p;
  T *d = reinterpret_cast<T *>(&s);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(S) / sizeof(T)); ++i) d[i] = src[i];
  return s;
}

// Workgroup shape of the two kernels: E elements, one thread per (element,
// line) with N^2 lines per element; a thread works on the five variables of
// its line at once, so a phase's addresses are computed once and all its
// LDS and register accesses are at compile-time offsets from them.
template <int N, int E>
struct Shape {
  static constexpr int NN = N * N * N, NF = N * N, EV = NSTATE * NN;
  static constexpr int NTH = (E * NF + 63) / 64 * 64;
};

// Sum of one double per thread over a workgroup of NTH threads -> thread 0
// (fixed order: butterfly in each wave, then the waves in order).
template <int NTH>
__device__ inline double group_sum(double v, double *sw) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if constexpr (NTH > 64) {
    if ((threadIdx.x & 63) == 0) sw[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sw[0];
#pragma unroll
    for (int w = 1; w < NTH / 64; ++w) v += sw[w];
    __syncthreads();
  }
  return v;
}

// Kinetic-energy partial sums: one per workgroup, or at p = 5 one per element.
// Without the autotuner a launch takes its kernels by its number of elements
// (an ensemble's together), and an instance's energy must not depend on which:
// at p <= 4 both take the same elements to a workgroup and number them alike,
// at p = 5 the large kernel takes 3 and the wave kernel 1.
__host__ __device__ constexpr bool ke_per_element(int n) { return n == 6; }

// Sum over an element of the values its N^2 lines left at v, by one wave (the
// butterfly of group_sum, idle lanes zero).
template <int N>
__device__ inline double element_sum(const double *v) {
  const int l = threadIdx.x & 63;
  double x = l < N * N ? v[l] : 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// Face-flux array FF, T: 30 planes (direction 2 d + side, state), each of
// the launch's elements x N^2 face Gauss points: the fluxes times a_d, side 0
// the element's own -d face, side 1 its +d face (written by the +d
// neighbour's workgroup, see ldg_grad_kernel).  Plane-major, so that a
// workgroup's threads (element, point) read and write each plane in one
// contiguous piece.
__host__ __device__ constexpr int ff_chunk(int n) { return NSTATE * n * n; }

// Coordinates of element kl of an instance.
__host__ __device__ inline void element_coords(const InstDesc &d, int kl, int c[3]) {
  const int row = d.div_nx.div(kl);
  c[0] = kl - row * d.nx;
  c[2] = d.div_ny.div(row);
  c[1] = row - c[2] * d.ny;
}
// Element number difference to the periodic neighbour along axis l (dir +-1).
__host__ __device__ inline int neighbor_step(const InstDesc &d, const int c[3], int l, int dir) {
  const int n = l == 0 ? d.nx : l == 1 ? d.ny : d.nz, st = l == 0 ? 1 : l == 1 ? d.nx : d.nx * d.ny;
  const bool wrap = dir > 0 ? c[l] == n - 1 : c[l] == 0;
  return wrap ? -dir * (n - 1) * st : dir * st;
}

// The stage input as the fluctuation about the background in type T.  An
// FP64 input in the mixed path (RK stage 1 of a call) is rounded to the
// FP32 fluctuation the other stages read, so a step's result does not depend
// on which form its input came in.
template <typename T, typename UT>
__device__ inline T fluctuation(UT x, int s, double rho0, double E0) {
  if constexpr (sizeof(UT) == 4) return T(x);
  else return T((double)x - (s == 0 ? rho0 : s == 4 ? E0 : 0.0));
}

// ---------------------------------------------------------------------
// Kernel A: the fluxes of the elements' -d faces, for both sides.
//
// The face between an element N and its -d neighbour K needs K's trace, N's
// trace and N's gradient trace (the one-sided switch picks it for both
// sides), so the workgroup that owns N evaluates that face once for both
// elements: the two traces, the normal derivative at the face nodes
// (a_d (Dn u + L0 J)_0) and, along the face, the derivatives of the
// variables the viscous flux reads (rho, m_D and the momentum along that
// direction), each interpolated or differentiated to the face Gauss points
// by two sweeps in the face plane, then Roe + viscous fluxes
// (face_flux_pair).  A derivative along l in the face plane carries the lift
// of the jump on the element's -l face, at the edge the two faces share: for
// the first sweep direction that is the neighbour's nodal trace there, for
// the second the same interpolated along the first (sedge).
//
// Threads: at nodes and points (element, point); the sweeps of one
// direction are (variable, line) items over the whole workgroup, each doing
// the line of the own trace, of the neighbour's trace, of the normal
// derivative and of the in-face derivative, which share their addresses.
// The three directions take turns in one set of face fields, with the own
// traces and normal derivatives waiting in registers: against all three at
// once the LDS footprint is 915 instead of 1620 values per element (p = 4;
// 0.56 -> 0.41 ms mixed, 1.20 -> 0.89 ms FP64 at 64^3).
//
// Measured at 64^3, p = 4: mixed 0.41 ms (0.68 with the gradient at the face
// nodes, 21 interpolated fields and lifted fluxes), bound by vector issue (95 %
// of it); FP64 0.89 ms (1.22), vector issue and LDS at 53 % each.
// ---------------------------------------------------------------------
template <int N, int E, typename T>
struct GradLds {
  using S = Shape<N, E>;
  static constexpr int FS = E * S::NF;                     // one field
  static constexpr int NFIELD = 21;                        // own 0-4, nbr 5-9, normal 10-14, d/da 15-17, d/db 18-20
  static constexpr int NB = 3 * NSTATE * FS;               // the neighbours' nodal traces
  static constexpr int BUF = NB + NFIELD * FS > E * S::EV ? NB + NFIELD * FS : E * S::EV;
  static constexpr int EDGE = 3 * E * N;
  static constexpr int WAVES = sizeof(T) == 4 ? 4 : 2;
};

// Fluxes of direction D at one face point: fp points at the point in field
// 0 of the direction, fields FS apart.
template <typename T, int D, int FS>
__device__ inline void face_point_flux(const T *fp, const Bg<T> &bg, T outK[5], T outN[5]) {
  constexpr int la = D == 0 ? 1 : 0, lb = D == 2 ? 1 : 2;
  T wN[5], wK[5], q[NGRAD];
#pragma unroll
  for (int s = 0; s < NSTATE; ++s) { wN[s] = fp[s * FS]; wK[s] = fp[(NSTATE + s) * FS]; }
#pragma unroll
  for (int k = 0; k < NGRAD; ++k) q[k] = T(0);   // the rest is not read by the direction-D flux
#pragma unroll
  for (int s = 0; s < NSTATE; ++s) q[s + NSTATE * D] = fp[(2 * NSTATE + s) * FS];
  q[0 + NSTATE * la] = fp[15 * FS];
  q[1 + D + NSTATE * la] = fp[16 * FS];
  q[1 + la + NSTATE * la] = fp[17 * FS];
  q[0 + NSTATE * lb] = fp[18 * FS];
  q[1 + D + NSTATE * lb] = fp[19 * FS];
  q[1 + lb + NSTATE * lb] = fp[20 * FS];
  face_flux_pair<T, D>(wK, wN, q, bg, outK, outN);
}

template <int N, int E, typename T, typename UT>
__global__ void __launch_bounds__((Shape<N, E>::NTH), (GradLds<N, E, T>::WAVES))
ldg_grad_kernel(const UT *__restrict__ U, T *__restrict__ FF, LaunchArgs la, const unsigned char *__restrict__ img) {
  using S = Shape<N, E>;
  using L = GradLds<N, E, T>;
  constexpr int NN = S::NN, NF = S::NF, EV = S::EV, NTH = S::NTH, FS = L::FS;
  __shared__ __align__(16) T sb[L::BUF];     // the block's state, then the neighbours' traces and the face fields
  __shared__ T sedge[L::EDGE];               // edge values of the second sweep direction's -l neighbour
  const int lb = logical_block(la);
  if (lb < 0) return;
  int kl, ne;
  const InstDesc &d = block_span(la, lb, E, kl, ne);
  if (ne <= 0) return;
  const long k0 = d.elem_off + kl;
  const int t = threadIdx.x, e = t / NF, ab = t - e * NF, b = ab / N, a = ab - b * N;
  const bool act = e < ne;
  const GOps<N, T> *const op =
      reinterpret_cast<const GOps<N, T> *>(img + (long)instance_of(la, lb) * GImage<N>::BYTES + GImage<N>::template offset<T>());
  const double rho0 = d.ph.rho0, E0 = d.ph.E0;

  // loads: the block's state (contiguous), and each thread's point of the -d
  // neighbours' traces on their +d faces
  constexpr int UL = (E * EV + NTH - 1) / NTH;
  UT v[UL], vn[3][NSTATE];
  const int tot = ne * EV;
#pragma unroll
  for (int i = 0; i < UL; ++i) {
    const int w = t + i * NTH;
    v[i] = U[k0 * EV + (w < tot ? w : tot - 1)];
  }
  {
    int c[3];
    element_coords(d, kl + (act ? e : 0), c);
    const int node[3] = {N - 1 + N * ab, a + N * (N - 1) + NF * b, ab + NF * (N - 1)};
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      const UT *src = U + (k0 + (act ? e : 0) + neighbor_step(d, c, D, -1)) * EV + node[D];
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) vn[D][s] = src[s * NN];
    }
  }
#pragma unroll
  for (int i = 0; i < UL; ++i) {
    const int w = t + i * NTH;
    const int s = sizeof(UT) == 4 ? 0 : (w % EV) / NN;
    if (w < tot) sb[w] = fluctuation<T>(v[i], s, rho0, E0);
  }
  __syncthreads();

  // own trace and normal derivative at the thread's node of the three faces
  T own[3][NSTATE], nbr[3][NSTATE], qn[3][NSTATE];
  if (act) {
    const int base[3] = {N * ab, a + NF * b, ab};
    constexpr int ST[3] = {1, N, NF};
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      struct Row { T r[N]; };
      const Row nrm = uniform_load<Row, T>(reinterpret_cast<const Row *>(op->nrm[D]));
      const T nw = uniform_load<T, T>(&op->nbr[D]);
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        const T *us = sb + e * EV + s * NN + base[D];
        nbr[D][s] = fluctuation<T>(vn[D][s], s, rho0, E0);
        own[D][s] = us[0];
        T q = nw * nbr[D][s];
#pragma unroll
        for (int j = 0; j < N; ++j) q = fma_(nrm.r[j], us[j * ST[D]], q);
        qn[D][s] = q;
      }
    }
  }
  __syncthreads();
  T *const nb = sb, *const wk = sb + L::NB;   // nb: field 5 D + s
  if (act) {
#pragma unroll
    for (int D = 0; D < 3; ++D)
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) nb[(NSTATE * D + s) * FS + t] = nbr[D][s];
  }
  int c[3];
  element_coords(d, kl + (act ? e : 0), c);
  const size_t plane = (size_t)la.nelem * NF;
  const Bg<T> bg(d.ph);
  struct Vec { T r[N]; };

  auto direction = [&](auto dir) {
    constexpr int D = decltype(dir)::value;
    constexpr int la_ = D == 0 ? 1 : 0, lb_ = D == 2 ? 1 : 2;   // the directions of a and b
    // items of the sweeps: (variable s, line x = e N + position); the in-face
    // derivative of variable s along l is one of three (rho, m_D, m_l)
    constexpr int IT = NSTATE * E * N, PASS = (IT + NTH - 1) / NTH;
    auto deriv = [&](int s, int l) -> int { return s == 0 ? 0 : s == 1 + D ? 1 : s == 1 + l ? 2 : -1; };
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        wk[s * FS + t] = own[D][s];
        wk[(2 * NSTATE + s) * FS + t] = qn[D][s];
      }
    }
    __syncthreads();
    {
      const SymMat<N, T> I = uniform_load<SymMat<N, T>, T>(&op->I);
      const SymMat<N, T> Dm = uniform_load<SymMat<N, T>, T>(&op->D);
      const Vec eta = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->eta));
      const T al = uniform_load<T, T>(&op->a[la_]), be = uniform_load<T, T>(&op->a[lb_]);
      // first sweep (along a)
#pragma unroll
      for (int p = 0; p < PASS; ++p) {
        const int i = t + p * NTH;
        if (i < IT) {
          const int s = i / (E * N), x0 = i - s * (E * N);
          T *f0 = wk + s * FS + N * x0;
          T x[N], o[N];
#pragma unroll
          for (int j = 0; j < N; ++j) x[j] = f0[j];
          sym_apply<N, 1, T>(I, x, o);
#pragma unroll
          for (int j = 0; j < N; ++j) f0[j] = o[j];
          const int f = deriv(s, la_);
          if (f >= 0) {
            // the -l neighbour's trace at the edge: l = y on the -x face: -y
            // trace at (x, z) = (0, b); l = x on the -y face: -x trace at
            // (y, z) = (0, b); l = x on the -z face: at (b, 0)
            const int at = D < 2 ? N * x0 : x0 / N * NF + x0 % N;
            const T jmp = x[0] - nb[(NSTATE * la_ + s) * FS + at];
            sym_apply<N, -1, T>(Dm, x, o);
            T *fd = wk + (15 + f) * FS + N * x0;
#pragma unroll
            for (int j = 0; j < N; ++j) fd[j] = al * fma_(eta.r[j], jmp, o[j]);
          }
          const T *g = nb + (NSTATE * D + s) * FS + N * x0;
#pragma unroll
          for (int j = 0; j < N; ++j) x[j] = g[j];
          sym_apply<N, 1, T>(I, x, o);
#pragma unroll
          for (int j = 0; j < N; ++j) (f0 + NSTATE * FS)[j] = o[j];
          T *fg = f0 + 2 * NSTATE * FS;
#pragma unroll
          for (int j = 0; j < N; ++j) x[j] = fg[j];
          sym_apply<N, 1, T>(I, x, o);
#pragma unroll
          for (int j = 0; j < N; ++j) fg[j] = o[j];
        }
      }
      // the second sweep's edge lines: the -l neighbour's trace along a
      for (int i = t; i < 3 * E; i += NTH) {
        const int f = i / E, ee = i - f * E, s = f == 0 ? 0 : f == 1 ? 1 + D : 1 + lb_;
        const T *p = nb + (NSTATE * lb_ + s) * FS + ee * NF;
        T x[N], o[N];
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = p[D == 0 ? N * j : j];
        sym_apply<N, 1, T>(I, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) sedge[i * N + q] = o[q];
      }
      __syncthreads();
      // second sweep (along b, in place)
#pragma unroll
      for (int p = 0; p < PASS; ++p) {
        const int i = t + p * NTH;
        if (i < IT) {
          const int s = i / (E * N), x0 = i - s * (E * N), at = x0 / N * NF + x0 % N;
          T *f0 = wk + s * FS + at;
          T x[N], o[N];
          auto interp = [&](T *f) {
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = f[N * j];
            sym_apply<N, 1, T>(I, x, o);
#pragma unroll
            for (int j = 0; j < N; ++j) f[N * j] = o[j];
          };
          interp(f0 + NSTATE * FS);
          interp(f0 + 2 * NSTATE * FS);
          const int fa = deriv(s, la_), fb = deriv(s, lb_);
          if (fa >= 0) interp(wk + (15 + fa) * FS + at);
          interp(f0);   // x: the own trace before it
          if (fb >= 0) {
            const T jmp = x[0] - sedge[fb * (E * N) + x0];
            sym_apply<N, -1, T>(Dm, x, o);
            T *fd = wk + (18 + fb) * FS + at;
#pragma unroll
            for (int j = 0; j < N; ++j) fd[N * j] = be * fma_(eta.r[j], jmp, o[j]);
          }
        }
      }
    }
    __syncthreads();
    // fluxes of both sides at the thread's point; side 1 goes to the -d
    // neighbour's record
    if (act) {
      T oK[5], oN[5];
      face_point_flux<T, D, FS>(wk + t, bg, oK, oN);
      T *const f0 = FF + (size_t)k0 * NF;
      const int st = t + neighbor_step(d, c, D, -1) * NF;
      const T ad = uniform_load<T, T>(&op->a[D]);
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        (f0 + (2 * D * NSTATE + s) * plane)[t] = oN[s] * ad;
        (f0 + ((2 * D + 1) * NSTATE + s) * plane)[st] = oK[s] * ad;
      }
    }
  };
  direction(std::integral_constant<int, 0>());
  __syncthreads();
  direction(std::integral_constant<int, 1>());
  __syncthreads();
  direction(std::integral_constant<int, 2>());
}

// ---------------------------------------------------------------------
// Nodal LDG gradient Q_l = a_l (Dn u + L0 J_l) (solver.cpp:490-508, restated
// in strong form: -M1^{-1} S1 + face lifts = Dn + M1^{-1} e_0 e_0^T, exactly),
// for ldg_rhs's gradient output and the closure's features.  One thread per
// node computes all 15 components and stores them straight to HBM
// (consecutive threads -> consecutive nodes, coalesced).
// ---------------------------------------------------------------------
template <int N, int E, typename TQ, typename UT>
__global__ void __launch_bounds__(NT) ldg_nodal_grad_kernel(const UT *__restrict__ U, TQ *__restrict__ Q, LaunchArgs la,
                                                            const Ops<N, double> *__restrict__ opp) {
  constexpr int NN = N * N * N, NF = N * N;
  using C = TQ;
  __shared__ C su[E][NSTATE][NN];
  __shared__ C sf[E][3][NSTATE][NF];   // the -d neighbours' traces on their +d faces
  __shared__ C sD[N][N + 1];
  __shared__ long snb[E][6];
  const int lb = logical_block(la);
  if (lb < 0) return;
  MeshArgs m;
  long kl;
  int ne, ec[3];
  const InstDesc &d = block_instance<E>(la, lb, m, ec, kl, ne);
  if (ne == 0) return;                // padding block of a partial brick
  const long k0 = d.elem_off + kl;
  const unsigned tid = threadIdx.x;
  fill_neighbors(m, ec, d.elem_off, ne, snb, tid);
  // the own trace u_0 is the line's first node, so its lift joins column 0
  // of Dn and only the neighbour's trace enters separately, with weight
  // -L0(i) in column N
  if (tid < N * (N + 1)) {
    const int i = tid / (N + 1), j = tid % (N + 1);
    sD[i][j] = C(j < N ? opp->Dn[i][j] + (j == 0 ? opp->L0[i] : 0.0) : -opp->L0[i]);
  }
  __syncthreads();
  const double rho0 = d.ph.rho0, E0 = d.ph.E0;
  for (unsigned w = tid; w < (unsigned)ne * NN; w += NT) {
    const unsigned e = w / NN, node = w - e * NN;
#pragma unroll
    for (int s = 0; s < NSTATE; ++s)
      su[e][s][node] = fluctuation<C>(U[(k0 + e) * (NSTATE * NN) + s * NN + node], s, rho0, E0);
  }
  for (unsigned w = tid; w < (unsigned)ne * 3 * NF; w += NT) {
    const unsigned ed = w / NF, ab = w - ed * NF, e = ed / 3, dd = ed - 3 * e, b = ab / N, a = ab - b * N;
    const unsigned node = (dd == 0 ? N : 1) * a + (dd == 2 ? N : NF) * b + (dd == 0 ? 1 : dd == 1 ? N : NF) * (N - 1);
#pragma unroll
    for (int s = 0; s < NSTATE; ++s)
      sf[e][dd][s][ab] = fluctuation<C>(U[snb[e][2 * dd] * (NSTATE * NN) + s * NN + node], s, rho0, E0);
  }
  __syncthreads();
  for (unsigned w = tid; w < (unsigned)ne * NN; w += NT) {
    const unsigned e = w / NN, node = w - e * NN;
    const unsigned iz = node / NF, rem = node - iz * NF;
    const unsigned iy = rem / N, ix = rem - iy * N;
    C rx[N + 1], ry[N + 1], rz[N + 1];
#pragma unroll
    for (int j = 0; j <= N; ++j) { rx[j] = sD[ix][j]; ry[j] = sD[iy][j]; rz[j] = sD[iz][j]; }
    TQ *Qe = Q + (k0 + e) * NGRAD * NN + node;
#pragma unroll
    for (int s = 0; s < NSTATE; ++s) {
      const C *us = su[e][s];
      C qx = rx[N] * sf[e][0][s][iy + N * iz];
      C qy = ry[N] * sf[e][1][s][ix + N * iz];
      C qz = rz[N] * sf[e][2][s][ix + N * iy];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        qx += rx[j] * us[j + N * iy + NF * iz];
        qy += ry[j] * us[ix + N * j + NF * iz];
        qz += rz[j] * us[ix + N * iy + NF * j];
      }
      Qe[(0 * NSTATE + s) * NN] = qx * C(m.ialpha[0]);
      Qe[(1 * NSTATE + s) * NN] = qy * C(m.ialpha[1]);
      Qe[(2 * NSTATE + s) * NN] = qz * C(m.ialpha[2]);
    }
  }
}

// ---------------------------------------------------------------------
// Kernel B: volume gradient and integrals, the face terms, inverse mass,
// RK epilogue, in Gauss form (GOps above).
//
// A thread owns one line (element e, face position ab) for all five
// variables; x-lines (y, z) = (a, b), y-lines (x, z) = (a, b), z-lines
// (x, y) = (a, b).  LDS holds two sets of five fields per element (A, B), at
// the end the FP64 rates.  Phases, with the values a thread keeps in
// registers between them in brackets:
//   x    nodes from HBM, I -> A; the jumps J_l at the face nodes
//   y    I on A; J along a
//   z    I on A [u_g on the thread's z-line]; J along b
//   d    Qx = a (Dg u + eta J) on A's x-lines, Qy on its y-lines -> A, B
//   p    Qz on the z-line; fluxes at its points: Fx, Fy -> A, B; [Dh Fz - faces]
//   t    Dh Fx - faces on A's x-lines, Dh Fy - faces on B's y-lines
//   zi   sum of the three, I^-1 along z in FP64 -> the FP64 buffer
//   yi   I^-1 along y;   xi   along x
//   epilogue: rate, running sum, next stage input (flat, coalesced)
//
// Measured at 64^3, p = 4, average of the four stages: mixed 1.13 ms (1.42
// with sweeps at the nodes and one line of one variable per thread), 5.1 TB/s
// of HBM traffic where a streaming kernel with two reads to a write
// reaches 5.8; FP64 1.56 ms (2.26), 4.9 TB/s, LDS busy for 60 %.
// ---------------------------------------------------------------------
template <int N, int E, typename T>
struct RhsLds {
  using S = Shape<N, E>;
  // the jumps' face fields: in FP64 in set B, which is free until phase d
  // stores Qy (the smaller footprint lets more workgroups share a CU)
  static constexpr bool JB = N >= 3;
  // element stride in a set: padded so that the lines of a wave's elements
  // fall on different LDS banks (p = 4: the x, y and z lines of 32 lanes in
  // 12 instead of 20 cycles per wave and value)
  static constexpr int PAD = N == 2 ? 0 : N == 3 ? 6 : N == 4 ? 20 : N == 5 ? 8 : 5;
  static constexpr int ES = S::EV + PAD;
  static constexpr int SET = E * ES, JS = 3 * NSTATE * E * S::NF;
  static constexpr int BUF = JB ? 2 * SET : 2 * SET + JS;
  static constexpr int WAVES = sizeof(T) == 4 && N <= 5 ? 3 : 2;
};

// DIAG: instead of the rate, the diagnostics of the state U to st.diag_part
// (the nodal and the two Gauss-point sums), from the state and its gradient at
// the Gauss points; no face fluxes are read.  A sum is NaN if the state has no
// right-hand side, although kinetic energy and enstrophy may be finite then
// (a NaN or infinite energy, a negative density): the pressure has to be
// finite at every Gauss point, and the Roe average of every face to have a
// sound speed.  The traces for that come from the element's own lines and the
// jumps, at the points the face kernel evaluates the flux at.
template <int N, int E, typename T, typename UT, bool DIAG>
__global__ void __launch_bounds__((Shape<N, E>::NTH), (RhsLds<N, E, T>::WAVES))
ldg_rhs_kernel(const UT *__restrict__ U, const T *__restrict__ FF, LaunchArgs la,
               const unsigned char *__restrict__ img, StageArgs st) {
  using S = Shape<N, E>;
  using L = RhsLds<N, E, T>;
  constexpr int NN = S::NN, NF = S::NF, EV = S::EV, ES = L::ES, NTH = S::NTH;
  __shared__ __align__(16) T sbuf[L::BUF];
  __shared__ double sred[NTH / 64];
  const int lb = logical_block(la);
  if (lb < 0) return;
  const int t = threadIdx.x;
  int kl, ne;
  const InstDesc &d = block_span(la, lb, E, kl, ne);
  // (no span is empty; without this line the compiler moves the loads up and
  // the mixed kernel takes 144 instead of 140 registers, 0.5 % more at 64^3, p = 4)
  if (ne <= 0) return;
  const long k0 = d.elem_off + kl;
  const int e = t / NF, ab = t - e * NF, b = ab / N, a = ab - b * N;
  const bool act = e < ne;
  const unsigned char *const im = img + (long)instance_of(la, lb) * GImage<N>::BYTES;
  const GOps<N, T> *const op = reinterpret_cast<const GOps<N, T> *>(im + GImage<N>::template offset<T>());
  const GOpsD<N> *const opd = reinterpret_cast<const GOpsD<N> *>(im);
  struct Vec { T r[N]; };
  T *const sA = sbuf, *const sB = sbuf + L::SET, *const sJ = L::JB ? sB : sbuf + 2 * L::SET;
  double *const md = reinterpret_cast<double *>(sbuf);
  const int lx = N * ab, ly = a + NF * b, lz = ab;                                // the thread's lines
  const int bx = e * ES + lx, by = e * ES + ly, bz = e * ES + lz;                // in a set
  int c[3];
  element_coords(d, kl + (act ? e : 0), c);

  // ---- x
  double dkn = 0.0, dke = 0.0, dens = 0.0;   // (DIAG)
  bool defined = true;
  if (act) {
    const double rho0 = d.ph.rho0, E0 = d.ph.E0;
    const UT *const ue = U + (k0 + e) * EV;
    UT v[NSTATE][N], vy[NSTATE], vz[NSTATE], nx[NSTATE], ny[NSTATE], nz[NSTATE];
    const UT *const ux = U + (k0 + e + neighbor_step(d, c, 0, -1)) * EV + (N - 1 + N * ab);
    const UT *const uy = U + (k0 + e + neighbor_step(d, c, 1, -1)) * EV + (a + N * (N - 1) + NF * b);
    const UT *const uz = U + (k0 + e + neighbor_step(d, c, 2, -1)) * EV + (ab + NF * (N - 1));
#pragma unroll
    for (int s = 0; s < NSTATE; ++s) {
#pragma unroll
      for (int q = 0; q < N; ++q) v[s][q] = (ue + lx)[s * NN + q];
      vy[s] = (ue + ly)[s * NN];
      vz[s] = (ue + lz)[s * NN];
      nx[s] = ux[s * NN];
      ny[s] = uy[s * NN];
      nz[s] = uz[s * NN];
    }
    if constexpr (DIAG) {
#pragma unroll
      for (int q = 0; q < N; ++q)
        dkn += opd->w[a] * opd->w[b] * opd->w[q] *
               (v[1][q] * v[1][q] + v[2][q] * v[2][q] + v[3][q] * v[3][q]) / (2.0 * v[0][q]);
    }
    const SymMat<N, T> I = uniform_load<SymMat<N, T>, T>(&op->I);
#pragma unroll
    for (int s = 0; s < NSTATE; ++s) {
      auto fl = [&](UT x) -> T { return fluctuation<T>(x, s, rho0, E0); };
      T x[N], o[N];
#pragma unroll
      for (int q = 0; q < N; ++q) x[q] = fl(v[s][q]);
      sym_apply<N, 1, T>(I, x, o);
#pragma unroll
      for (int q = 0; q < N; ++q) sA[bx + s * NN + q] = o[q];
      sJ[(0 * NSTATE + s) * (E * NF) + t] = x[0] - fl(nx[s]);
      sJ[(1 * NSTATE + s) * (E * NF) + t] = fl(vy[s]) - fl(ny[s]);
      sJ[(2 * NSTATE + s) * (E * NF) + t] = fl(vz[s]) - fl(nz[s]);
    }
  }
  __syncthreads();
  // ---- y, and the jumps along a
  T ug[NSTATE][N];
  {
    const SymMat<N, T> I = uniform_load<SymMat<N, T>, T>(&op->I);
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        T *p = sA + by + s * NN;
        T x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[N * q];
        sym_apply<N, 1, T>(I, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[N * q] = o[q];
      }
    }
    constexpr int JL = 3 * NSTATE * E * N;
#pragma unroll
    for (int i0 = 0; i0 < JL; i0 += NTH) {
      const int i = i0 + t;
      if (i < JL) {
        T *p = sJ + N * i;
        T x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[q];
        sym_apply<N, 1, T>(I, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[q] = o[q];
      }
    }
    __syncthreads();
    // ---- z, and the jumps along b
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        T *p = sA + bz + s * NN;
        T x[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[NF * q];
        sym_apply<N, 1, T>(I, x, ug[s]);
#pragma unroll
        for (int q = 0; q < N; ++q) p[NF * q] = ug[s][q];
      }
    }
#pragma unroll
    for (int i0 = 0; i0 < JL; i0 += NTH) {
      const int i = i0 + t;
      if (i < JL) {
        T *p = sJ + (i / N) * NF + i % N;
        T x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[N * q];
        sym_apply<N, 1, T>(I, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[N * q] = o[q];
      }
    }
  }
  __syncthreads();
  // ---- d
  // (the face fluxes are loaded a phase before they are used)
  const size_t plane = (size_t)la.nelem * NF;
  const T *const ffo = FF + (size_t)k0 * NF;
  T fz[2][NSTATE], fx[2][NSTATE], fy[2][NSTATE];
  auto load_faces = [&](T (&f)[2][NSTATE], int l) {
    if (act) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int s = 0; s < NSTATE; ++s) f[g][s] = (ffo + ((2 * l + g) * NSTATE + s) * plane)[(unsigned)t];
    }
  };
  if constexpr (!DIAG) {
    load_faces(fz, 2);
  } else if (act) {
    // the thread's point of the three - faces: a line's polynomial there is
    // sum_q L_q(-1) u_q (32^3, p = 4, FP64: 114 us without this check, 130 with;
    // taken from the sweeps below, whose lines these are, it is 125, but FP64 then
    // needs 256 registers instead of 174 at p = 4 and spills at p = 5)
    const Bg<T> bg(d.ph);
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const T *const p = sA + (l == 0 ? bx : l == 1 ? by : bz);
      const int stp = l == 0 ? 1 : l == 1 ? N : NF;
      T wN[NSTATE], wK[NSTATE];
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        wN[s] = T(0);
#pragma unroll
        for (int q = 0; q < N; ++q) wN[s] = fma_(op->eta[q] * T(opd->w[q]), p[s * NN + stp * q], wN[s]);
        wK[s] = wN[s] - sJ[(l * NSTATE + s) * (E * NF) + t];
      }
      defined = defined && roe_defined<T>(wK, wN, bg);
    }
  }
  T jz[NSTATE];
  {
    T qx[NSTATE][N], qy[NSTATE][N];
    if (act) {
      T jx[NSTATE], jy[NSTATE];
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        jx[s] = sJ[(0 * NSTATE + s) * (E * NF) + t];
        jy[s] = sJ[(1 * NSTATE + s) * (E * NF) + t];
        jz[s] = sJ[(2 * NSTATE + s) * (E * NF) + t];
      }
      {
        const SymMat<N, T> Dx = uniform_load<SymMat<N, T>, T>(&op->Dg[0]);
        const Vec ax = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->aeta[0]));
#pragma unroll
        for (int s = 0; s < NSTATE; ++s) {
          const T *p = sA + bx + s * NN;
          T x[N];
#pragma unroll
          for (int q = 0; q < N; ++q) x[q] = p[q];
          sym_apply<N, -1, T>(Dx, x, qx[s]);
#pragma unroll
          for (int q = 0; q < N; ++q) qx[s][q] = fma_(ax.r[q], jx[s], qx[s][q]);
        }
      }
      {
        const SymMat<N, T> Dy = uniform_load<SymMat<N, T>, T>(&op->Dg[1]);
        const Vec ay = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->aeta[1]));
#pragma unroll
        for (int s = 0; s < NSTATE; ++s) {
          const T *p = sA + by + s * NN;
          T x[N];
#pragma unroll
          for (int q = 0; q < N; ++q) x[q] = p[N * q];
          sym_apply<N, -1, T>(Dy, x, qy[s]);
#pragma unroll
          for (int q = 0; q < N; ++q) {
            qy[s][q] = fma_(ay.r[q], jy[s], qy[s][q]);
            if (!L::JB) sB[by + s * NN + N * q] = qy[s][q];
          }
        }
      }
    }
    __syncthreads();
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s)
#pragma unroll
        for (int q = 0; q < N; ++q) {
          sA[bx + s * NN + q] = qx[s][q];
          if (L::JB) sB[by + s * NN + N * q] = qy[s][q];
        }
    }
  }
  __syncthreads();
  // ---- p
  T kz[NSTATE][N];
  if (act) {
    {
      const SymMat<N, T> Dz = uniform_load<SymMat<N, T>, T>(&op->Dg[2]);
      const Vec az = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->aeta[2]));
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        sym_apply<N, -1, T>(Dz, ug[s], kz[s]);
#pragma unroll
        for (int q = 0; q < N; ++q) kz[s][q] = fma_(az.r[q], jz[s], kz[s][q]);
      }
    }
    const Bg<T> bg(d.ph);
#pragma unroll
    for (int q = 0; q < N; ++q) {
      T w[NSTATE], g[NGRAD], F[NGRAD];
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        w[s] = ug[s][q];
        g[s] = sA[bz + s * NN + NF * q];
        g[NSTATE + s] = sB[bz + s * NN + NF * q];
        g[2 * NSTATE + s] = kz[s][q];
      }
      if constexpr (DIAG) {
        const double rho = d.ph.rho0 + (double)w[0];
        const double ir = 1.0 / rho;
        const double vv[3] = {(double)w[1] * ir, (double)w[2] * ir, (double)w[3] * ir};
        double gd[15], gv[3][3], ge[3];
#pragma unroll
        for (int k = 0; k < 15; ++k) gd[k] = g[k];
        prim_grads<double>(ir, d.ph.E0 + (double)w[4], vv, gd, gv, ge);
        const double w1 = gv[2][1] - gv[1][2], w2 = gv[0][2] - gv[2][0], w3 = gv[1][0] - gv[0][1];
        const double wq = opd->w[a] * opd->w[b] * opd->w[q];
        const T irt = rcp(bg.rho0 + w[0]), vt[3] = {w[1] * irt, w[2] * irt, w[3] * irt};
        defined = defined && fabs(pressure(w, vt, bg)) <= std::numeric_limits<T>::max();
        dke += wq * 0.5 * ((double)w[1] * vv[0] + (double)w[2] * vv[1] + (double)w[3] * vv[2]);
        dens += wq * 0.5 * rho * (w1 * w1 + w2 * w2 + w3 * w3);
        continue;
      }
      volume_flux<T>(w, g, bg, F);
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        sA[bz + s * NN + NF * q] = F[s];
        sB[bz + s * NN + NF * q] = F[NSTATE + s];
        kz[s][q] = F[2 * NSTATE + s];
      }
    }
    if constexpr (!DIAG) {
      load_faces(fx, 0);
      load_faces(fy, 1);
    }
    const SymMat<N, T> Dz = uniform_load<SymMat<N, T>, T>(&op->Dh[2]);
    const Vec eta = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->eta));
#pragma unroll
    for (int s = 0; s < NSTATE; ++s) {
      T o[N];
      sym_apply<N, -1, T>(Dz, kz[s], o);
#pragma unroll
      for (int q = 0; q < N; ++q) kz[s][q] = o[q] - fma_(eta.r[q], fz[0][s], eta.r[N - 1 - q] * fz[1][s]);
    }
  }
  if constexpr (DIAG) {
    if (!defined) dke = std::numeric_limits<double>::quiet_NaN();
    const double n = group_sum<NTH>(dkn, sred), x = group_sum<NTH>(dke, sred), y = group_sum<NTH>(dens, sred);
    if (t == 0) {
      st.diag_part[3 * lb] = n;
      st.diag_part[3 * lb + 1] = x;
      st.diag_part[3 * lb + 2] = y;
    }
    return;
  }
  __syncthreads();
  // ---- t
  if (act) {
    const Vec eta = uniform_load<Vec, T>(reinterpret_cast<const Vec *>(op->eta));
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const SymMat<N, T> Dh = uniform_load<SymMat<N, T>, T>(&op->Dh[l]);
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        T *p = l == 0 ? sA + bx + s * NN : sB + by + s * NN;
        T x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[l == 0 ? q : N * q];
        sym_apply<N, -1, T>(Dh, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q)
          p[l == 0 ? q : N * q] =
              o[q] - fma_(eta.r[q], (l == 0 ? fx : fy)[0][s], eta.r[N - 1 - q] * (l == 0 ? fx : fy)[1][s]);
      }
    }
  }
  __syncthreads();
  // ---- zi, yi, xi (FP64)
  const bool need_u0 = (st.acc && st.acc_init) || st.unext || st.unext32;
  const bool need_acc = st.acc && !st.acc_init;
  const long gofs = k0 * EV;
  // Epilogue items: word it NTH + t of the block's values of one variable
  // (element after element), for variable 0 at `ew` past the block's base in
  // every (node, state, element) array and at `lw` in the FP64 buffer, and s
  // N^3 further for variable s.  (Coalesced, through LDS: with the epilogue on
  // the thread's own x-lines, lanes 8 N bytes apart, the mixed kernel was 5 %
  // slower at 64^3, p = 4, the FP64 kernel the same.)
  constexpr int EPI = (E * NN + NTH - 1) / NTH;
  unsigned ew[EPI], lw[EPI];
#pragma unroll
  for (int it = 0; it < EPI; ++it) {
    const int i = t + it * NTH, j = i < ne * NN ? i : ne * NN - 1;
    ew[it] = (unsigned)(j + j / NN * (EV - NN));
    lw[it] = (unsigned)(j + j / NN * (ES - NN));
  }
  // (a uniform base and a 32-bit byte offset: no 64-bit address per item)
  auto at = [&](auto *p, int it) {
    return reinterpret_cast<decltype(p)>((char *)p + ew[it] * (unsigned)sizeof(*p));
  };
  double ru[EPI][NSTATE], ra[EPI][NSTATE];
  {
    const SymMat<N, double> Ii = uniform_load<SymMat<N, double>, double>(&opd->Ii);
    constexpr bool INPLACE = sizeof(T) == sizeof(double);   // a thread's FP64 results replace its own A values
    {
      double r[NSTATE][N];
      if (act) {
#pragma unroll
        for (int s = 0; s < NSTATE; ++s) {
          double x[N];
#pragma unroll
          for (int q = 0; q < N; ++q)
            x[q] = (double)(kz[s][q] + (sA[bz + s * NN + NF * q] + sB[bz + s * NN + NF * q]));
          sym_apply<N, 1, double>(Ii, x, r[s]);
        }
      }
      if (!INPLACE) __syncthreads();
      if (act) {
#pragma unroll
        for (int s = 0; s < NSTATE; ++s)
#pragma unroll
          for (int q = 0; q < N; ++q) md[bz + s * NN + NF * q] = r[s][q];
      }
    }
    // the epilogue's HBM operands, covered by the sweeps below
    if (need_u0) {
      const double *const p = st.u0 + gofs;
#pragma unroll
      for (int it = 0; it < EPI; ++it)
#pragma unroll
        for (int v = 0; v < NSTATE; ++v) ru[it][v] = at(p, it)[v * NN];
    }
    __syncthreads();
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        double *p = md + by + s * NN;
        double x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[N * q];
        sym_apply<N, 1, double>(Ii, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[N * q] = o[q];
      }
    }
    if (need_acc) {
      const double *const p = st.acc + gofs;
#pragma unroll
      for (int it = 0; it < EPI; ++it)
#pragma unroll
        for (int v = 0; v < NSTATE; ++v) ra[it][v] = at(p, it)[v * NN];
    }
    __syncthreads();
    if (act) {
#pragma unroll
      for (int s = 0; s < NSTATE; ++s) {
        double *p = md + bx + s * NN;
        double x[N], o[N];
#pragma unroll
        for (int q = 0; q < N; ++q) x[q] = p[q];
        sym_apply<N, 1, double>(Ii, x, o);
#pragma unroll
        for (int q = 0; q < N; ++q) p[q] = o[q];
      }
    }
    __syncthreads();
  }

  // ---- epilogue (FP64): k, RK4 accumulation and next stage input
  {
    const double dtb = d.dt * st.cb, dta = d.dt * st.ca;
    // background of variable v (the FP32 copies are fluctuations)
    const double bg[NSTATE] = {d.ph.rho0, 0.0, 0.0, 0.0, d.ph.E0};
    auto items = [&](auto &&body) {
#pragma unroll
      for (int it = 0; it < EPI; ++it)
        if (t + it * NTH < ne * NN) {
#pragma unroll
          for (int v = 0; v < NSTATE; ++v) body(it, v, md + lw[it] + v * NN);
        }
    };
    if (st.corr) {
      const double *const p = st.corr + gofs;
      const unsigned char *const gate = st.gate + k0;
      items([&](int it, int v, double *k) {
        if (gate[ew[it] / EV]) *k += at(p, it)[v * NN];
      });
    }
    if (st.kout) {
      double *const p = st.kout + gofs;
      items([&](int it, int v, double *k) { at(p, it)[v * NN] = *k; });
    }
    if (st.acc_init) {
#pragma unroll
      for (int it = 0; it < EPI; ++it)
#pragma unroll
        for (int v = 0; v < NSTATE; ++v) ra[it][v] = ru[it][v];
    }
    // one branch-free loop per combination of outputs
    auto step = [&](auto acc, auto un, auto un32, auto nx32) {
      double *const pa = st.acc + gofs, *const pu = st.unext + gofs;
      float *const pu32 = st.unext32 + gofs, *const pn32 = st.next32 + gofs;
      items([&](int it, int v, double *kp) {
        const double k = *kp;
        if constexpr (un) at(pu, it)[v * NN] = ru[it][v] + dta * k;
        if constexpr (un32) at(pu32, it)[v * NN] = (float)(ru[it][v] + dta * k - bg[v]);
        if constexpr (acc) {
          ra[it][v] += dtb * k;
          at(pa, it)[v * NN] = ra[it][v];
        }
        if constexpr (nx32) at(pn32, it)[v * NN] = (float)(ra[it][v] - bg[v]);
      });
    };
    constexpr std::true_type Y;
    constexpr std::false_type X;
    if (st.acc) {
      if (st.unext) step(Y, Y, X, X);
      else if (st.unext32) step(Y, X, Y, X);
      else if (st.next32) step(Y, X, X, Y);
      else step(Y, X, X, X);
    } else if (st.unext32) {
      step(X, X, Y, X);
    }
    if (st.ke_part) items([&](int it, int v, double *k) { *k = ra[it][v]; });
  }
  if (st.ke_part) {
    __syncthreads();
    double kel = 0.0;
    if (act) {
#pragma unroll
      for (int q = 0; q < N; ++q) {
        const double *x = md + bz + NF * q;
        const double rho = x[0], m1 = x[NN], m2 = x[2 * NN], m3 = x[3 * NN];
        kel += opd->w[a] * opd->w[b] * opd->w[q] * fma_(m3, m3, fma_(m2, m2, m1 * m1)) / (2.0 * rho);
      }
    }
    if constexpr (ke_per_element(N)) {
      __syncthreads();
      if (act) md[t] = kel;
      __syncthreads();
      for (int i = t >> 6; i < ne; i += NTH / 64) {
        const double x = element_sum<N>(md + i * NF);
        if ((t & 63) == 0) st.ke_part[k0 + i] = x;
      }
    } else {
      const double x = group_sum<NTH>(kel, sred);
      if (t == 0) st.ke_part[lb] = x;
    }
  }
}

// Ordered per-instance sums of partials, one workgroup per instance i and
// partial j of `stride`: out[(row * row_stride + i) * stride + j] = scale_i * (sum
// over the instance's partials b of part[b * stride + j]).  The partials are the
// instance's workgroups' or (BY_ELEM) its elements'.  With `step` a row of a
// history: row >= 0 is the row, row < 0 (graph replays) the instance's own
// counter step[i], which is left at the row after it; without it row 0.
//
// One workgroup reads every partial, so what counts is the loads in flight:
// 128 KB (64^3, p = 4: 131,072 partials in 27 us; 33 with 256 threads).
constexpr int FIN_NT = 1024;
template <bool BY_ELEM>
static __global__ void __launch_bounds__(FIN_NT) ldg_finalize_kernel(const double *__restrict__ part, int stride,
                                                            const InstDesc *__restrict__ inst, int row_stride,
                                                            const double *__restrict__ scale, double *__restrict__ out,
                                                            int row, int *__restrict__ step) {
  __shared__ double sred[FIN_NT / 64];
  const int i = blockIdx.x, j = blockIdx.y;
  const int b0 = BY_ELEM ? (int)inst[i].elem_off : inst[i].block_off;
  const int b1 = b0 + (BY_ELEM ? (int)inst[i].nelem : inst[i].nblocks);
  const long r = !step ? 0 : row >= 0 ? row : step[i];
  constexpr int A = 16;   // accumulators per thread
  // thread t sums partials b0 + t + k FIN_NT into accumulator k mod A; the
  // order depends only on b - b0
  double acc[A];
#pragma unroll
  for (int k = 0; k < A; ++k) acc[k] = 0.0;
  for (int base = b0 + threadIdx.x; base < b1; base += A * FIN_NT) {
    double x[A];
#pragma unroll
    for (int k = 0; k < A; ++k) {
      const int b = base + k * FIN_NT;
      x[k] = b < b1 ? part[(long)b * stride + j] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < A; ++k) acc[k] += x[k];
  }
#pragma unroll
  for (int h = A / 2; h > 0; h /= 2)
#pragma unroll
    for (int k = 0; k < h; ++k) acc[k] += acc[k + h];
  const double t = group_sum<FIN_NT>(acc[0], sred);
  if (threadIdx.x == 0) out[(r * row_stride + i) * stride + j] = t * scale[i];
  if (step && threadIdx.x == 0) step[i] = (int)r + 1;
}

// Taylor-Green initial state at the CGL nodes (solver.cpp:194-236).
struct TGVArgs {
  int n, nx, ny, nz;
  long nelem;
  double xmin[3], xmax[3];
  double r[8];
  double L, p0, rho0, V0, RT0, gamma;
  double phase[3];       // the field is evaluated at x + phase (0 for the reference case)
};

static __global__ void ldg_tgv_kernel(double *__restrict__ u, TGVArgs t) {
  const int dofs = t.n * t.n * t.n;
  const long total = t.nelem * dofs;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < total; w += (long)gridDim.x * blockDim.x) {
    const long k = w / dofs;
    const int iN = (int)(w - k * dofs);
    const long ie[3] = {k % t.nx, (k / t.nx) % t.ny, k / ((long)t.nx * t.ny)};
    const int in[3] = {iN % t.n, (iN / t.n) % t.n, iN / (t.n * t.n)};
    const int ns[3] = {t.nx, t.ny, t.nz};
    double X[3];
    for (int l = 0; l < 3; ++l) {
      const double lo = ie[l] * (t.xmax[l] - t.xmin[l]) / ns[l] + t.xmin[l];
      const double hi = (ie[l] + 1) * (t.xmax[l] - t.xmin[l]) / ns[l] + t.xmin[l];
      X[l] = lo + .5 * (t.r[in[l]] + 1.0) * (hi - lo);
    }
    const double x = X[0] + t.phase[0], y = X[1] + t.phase[1], z = X[2] + t.phase[2], L = t.L;
    const double pr = t.p0 + (t.rho0 * t.V0 * t.V0 / 16.0) * (cos(2 * x / L) + cos(2 * y / L)) * (cos(2 * z / L) + 2);
    const double rho = pr / t.RT0;
    const double m1 = t.rho0 * t.V0 * sin(x / L) * cos(y / L) * cos(z / L);
    const double m2 = -t.rho0 * t.V0 * cos(x / L) * sin(y / L) * cos(z / L);
    const double m3 = 0.0;
    double *uk = u + k * NSTATE * dofs;
    uk[iN] = rho;
    uk[iN + dofs] = m1;
    uk[iN + 2 * dofs] = m2;
    uk[iN + 3 * dofs] = m3;
    uk[iN + 4 * dofs] = pr / (t.gamma - 1) + (m1 * m1 + m2 * m2 + m3 * m3) / (2.0 * rho);
  }
}

}  // namespace ldg
