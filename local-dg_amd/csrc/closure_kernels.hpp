// closure_kernels.hpp -- device code of the learned per-element closure:
// L2 projection between orders, feature/target assembly, a BF16-input MFMA
// GEMM with fused bias + SiLU, and the elementwise pieces of the MLP's
// backward pass and Adam.
//
// The network maps one element's state and LDG gradient (5 + 15 fields at
// the (p+1)^3 nodes; 540 values at p = 2) to a correction of its
// right-hand side (5 fields at the nodes; 135 values):
//   H1 = silu(X W1^T + b1), H2 = silu(H1 W2^T + b2), Y = H2 W3^T + b3.
// Weights are kept in FP32 and enter the matrix cores rounded to BF16, with
// FP32 accumulation.
#pragma once

#include <hip/hip_runtime.h>

#include "ldg_kernels.hpp"

namespace ldg_mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// FP32 -> BF16, round to nearest even (inputs here are finite).
__device__ inline unsigned short to_bf16(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ inline float silu(float z) { return z / (1.0f + __expf(-z)); }

constexpr int GT = 64;       // output tile (rows and columns) per workgroup
constexpr int GK = 32;       // K chunk staged in LDS
constexpr int GPAD = 8;      // LDS row padding (BF16 elements)
enum { EPI_NONE = 0, EPI_BIAS = 1, EPI_BIAS_SILU = 2 };

// C[m][n] = epi( sum_k A(m,k) B(k,n) ), FP32 in memory, BF16 x BF16 -> FP32
// on v_mfma_f32_32x32x16_bf16.  A(m,k) = TA ? A[k*lda+m] : A[m*lda+k];
// B(k,n) = TB ? B[n*ldb+k] : B[k*ldb+n].  Epilogue: + bias[n]; with SiLU the
// pre-activation goes to Z (if not null) and silu() to C.  Grid:
// (ceil(N/64), ceil(M/64)), 256 threads; four waves own 32x32 quadrants.
// Every global access is guarded by the matrix bounds (out-of-range
// operands are staged as zeros).
template <bool TA, bool TB, int EPI>
__global__ void __launch_bounds__(256) mlp_gemm(int M, int N, int K, const float *__restrict__ A, int lda,
                                                const float *__restrict__ B, int ldb, const float *__restrict__ bias,
                                                float *__restrict__ Z, float *__restrict__ C, int ldc) {
  __shared__ __align__(16) unsigned short As[GT][GK + GPAD];   // [m][k]
  __shared__ __align__(16) unsigned short Bs[GT][GK + GPAD];   // [n][k]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  floatx16 acc;
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = 0.0f;

  for (int k0 = 0; k0 < K; k0 += GK) {
    if (!TA) {
      const int r = tid >> 2, c = (tid & 3) * 8, m = m0 + r;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = k0 + c + i;
        As[r][c + i] = to_bf16((m < M && k < K) ? A[(long)m * lda + k] : 0.0f);
      }
    } else {
      const int kk = tid >> 3, c = (tid & 7) * 8, k = k0 + kk;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = m0 + c + i;
        As[c + i][kk] = to_bf16((m < M && k < K) ? A[(long)k * lda + m] : 0.0f);
      }
    }
    if (TB) {
      const int r = tid >> 2, c = (tid & 3) * 8, n = n0 + r;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = k0 + c + i;
        Bs[r][c + i] = to_bf16((n < N && k < K) ? B[(long)n * ldb + k] : 0.0f);
      }
    } else {
      const int kk = tid >> 3, c = (tid & 7) * 8, k = k0 + kk;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int n = n0 + c + i;
        Bs[c + i][kk] = to_bf16((n < N && k < K) ? B[(long)k * ldb + n] : 0.0f);
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GK; kk += 16) {
      // lane l supplies row (l mod 32) of A / column (l mod 32) of B and the
      // 8 consecutive k of half (l / 32) of the 16-deep step
      const int kb = kk + (lane >> 5) * 8;
      const u16x8 a = *reinterpret_cast<const u16x8 *>(&As[wm + (lane & 31)][kb]);
      const u16x8 b = *reinterpret_cast<const u16x8 *>(&Bs[wn + (lane & 31)][kb]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                    acc, 0, 0, 0);
    }
    __syncthreads();
  }
  // accumulator j of lane l holds row 8 (j/4) + 4 (l/32) + j%4, column l%32
  const int n = n0 + wn + (lane & 31);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int m = m0 + wm + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
    if (m < M && n < N) {
      float v = acc[j];
      if (EPI >= EPI_BIAS) v += bias[n];
      if (EPI == EPI_BIAS_SILU) {
        if (Z) Z[(long)m * ldc + n] = v;
        v = silu(v);
      }
      C[(long)m * ldc + n] = v;
    }
  }
}

// Features of elements [0, K) of one instance: X[e][j] = (x_j - mean_j) *
// istd_j with x = (state minus the background (rho0, 0, 0, 0, E0): nU
// values, then the gradient: nQ values), both in their per-element layout.
template <typename TQ, typename UT>
__global__ void mlp_features(const UT *__restrict__ U, const TQ *__restrict__ Q, long K, int dofs,
                             double rho0, double E0, const float *__restrict__ mean, const float *__restrict__ istd,
                             float *__restrict__ X) {
  const int nU = 5 * dofs, nin = 20 * dofs;
  const long total = K * nin;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < total; w += (long)gridDim.x * blockDim.x) {
    const long e = w / nin;
    const int j = (int)(w - e * nin);
    double x;
    if (j < nU) {
      const int s = j / dofs;
      x = (double)U[e * nU + j] - (s == 0 ? rho0 : s == 4 ? E0 : 0.0);
    } else {
      x = (double)Q[e * (long)(15 * dofs) + (j - nU)];
    }
    X[w] = (float)((x - (double)mean[j]) * (double)istd[j]);
  }
}

// Training targets of elements [0, K): T = Pk - k (projected fine
// right-hand side minus the coarse right-hand side of the projected state).
__global__ void mlp_targets(const double *__restrict__ Pk, const double *__restrict__ k, long n,
                            float *__restrict__ T) {
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < n; w += (long)gridDim.x * blockDim.x)
    T[w] = (float)(Pk[w] - k[w]);
}

// Rate of change of the element's nodal kinetic energy sum_j |m_j|^2 /
// (2 rho_j) caused by a correction c of (rho, m) (one wave; lanes over the
// nodes; every lane returns the sum).
// The correction is c = y * ostd + omean (y: the normalised output row).
// u: the element's state, or its fluctuation (then rho_add = rho0).
template <typename UT>
__device__ inline double ke_production(const UT *__restrict__ u, double rho_add, int dofs, const float *y,
                                       const float *__restrict__ ostd, const float *__restrict__ omean, int lane) {
  auto c = [&](int k) { return (double)y[k] * (double)ostd[k] + (double)omean[k]; };
  double pr = 0.0;
  for (int j = lane; j < dofs; j += 64) {
    const double ir = 1.0 / ((double)u[j] + rho_add);
    const double v0 = (double)u[dofs + j] * ir, v1 = (double)u[2 * dofs + j] * ir, v2 = (double)u[3 * dofs + j] * ir;
    pr += v0 * c(dofs + j) + v1 * c(2 * dofs + j) + v2 * c(3 * dofs + j) - 0.5 * (v0 * v0 + v1 * v1 + v2 * v2) * c(j);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pr += __shfl_xor(pr, o, 64);
  return pr;
}

// Closure correction of each element (one 64-thread block per element):
// corr = Y * ostd + omean, applied (gate = 1) only if the RMS of the
// normalised output Y is at most `bound` and, with `dissipative` = 1, if it
// does not raise the element's kinetic energy (= -1: does not lower it);
// else gate = 0 (plain RHS).
template <typename UT>
__global__ void __launch_bounds__(64) mlp_correction(const float *__restrict__ Y, long K, int nout,
                                                     const float *__restrict__ omean, const float *__restrict__ ostd,
                                                     double bound, int dissipative, const UT *__restrict__ U,
                                                     double rho_add, double *__restrict__ corr,
                                                     unsigned char *__restrict__ gate) {
  for (long e = blockIdx.x; e < K; e += gridDim.x) {
    const float *y = Y + e * nout;
    float ss = 0.0f;
    for (int j = threadIdx.x; j < nout; j += 64) ss += y[j] * y[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    bool on = sqrt((double)ss / nout) <= bound;
    if (on && dissipative)
      on = dissipative * ke_production(U + e * nout, rho_add, nout / 5, y, ostd, omean, threadIdx.x) <= 0.0;
    for (int j = threadIdx.x; j < nout; j += 64)
      corr[e * nout + j] = on ? (double)y[j] * (double)ostd[j] + (double)omean[j] : 0.0;
    if (threadIdx.x == 0) gate[e] = on ? 1 : 0;
  }
}

// dY = scale rw (Y - T); per-block partial sums of rw (Y - T)^2 (FP64),
// with rw the weight of the row (rows of `width` values; 1 if rw is null).
__global__ void __launch_bounds__(256) mlp_loss_grad(const float *__restrict__ Y, const float *__restrict__ T,
                                                     long n, int width, const float *__restrict__ rw, float scale,
                                                     float *__restrict__ dY, double *__restrict__ part) {
  __shared__ double red[256];
  double s = 0.0;
  for (long w = blockIdx.x * 256L + threadIdx.x; w < n; w += (long)gridDim.x * 256) {
    const float d = Y[w] - T[w];
    const float r = rw ? rw[w / width] : 1.0f;
    if (dY) dY[w] = scale * r * d;
    s += (double)r * d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// dZ = dH * silu'(Z), silu'(z) = s (1 + z (1 - s)), s = sigmoid(z).
__global__ void mlp_silu_back(const float *__restrict__ dH, const float *__restrict__ Z, long n,
                              float *__restrict__ dZ) {
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < n; w += (long)gridDim.x * blockDim.x) {
    const float z = Z[w];
    const float s = 1.0f / (1.0f + __expf(-z));
    dZ[w] = dH[w] * s * (1.0f + z * (1.0f - s));
  }
}

// Column sums of a rows x cols row-major matrix (one thread per column,
// fixed order: deterministic).
__global__ void mlp_colsum(const float *__restrict__ D, int rows, int cols, float *__restrict__ out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= cols) return;
  float s = 0.0f;
  for (int r = 0; r < rows; ++r) s += D[(long)r * cols + c];
  out[c] = s;
}

// Adam (bias-corrected), elementwise over all parameters.
__global__ void mlp_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                         float *__restrict__ v, long n, float lr, float b1, float b2, float eps, float bc1, float bc2) {
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < n; w += (long)gridDim.x * blockDim.x) {
    const float gi = g[w];
    const float mi = b1 * m[w] + (1.0f - b1) * gi;
    const float vi = b2 * v[w] + (1.0f - b2) * gi * gi;
    m[w] = mi;
    v[w] = vi;
    p[w] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  }
}

// dst[b][:] = src[idx[b]][:] (rows of `width` floats).
__global__ void mlp_gather(const float *__restrict__ src, int width, const long *__restrict__ idx, int rows,
                           float *__restrict__ dst) {
  const long total = (long)rows * width;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < total; w += (long)gridDim.x * blockDim.x) {
    const long b = w / width;
    const int j = (int)(w - b * width);
    dst[w] = src[idx[b] * width + j];
  }
}

// out[r] = mean over the row of D[r][j]^2 (one thread per row).
__global__ void mlp_rowmeansq(const float *__restrict__ D, long rows, int width, float *__restrict__ out) {
  for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < rows; r += (long)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int j = 0; j < width; ++j) s += (double)D[r * width + j] * D[r * width + j];
    out[r] = (float)(s / width);
  }
}

// Per-feature sums over a chunk of rows (FP64), for mean and spread:
// part[(chunk * 2 + 0) * width + j] = sum x, [... + 1] = sum x^2.
__global__ void mlp_moments(const float *__restrict__ D, long rows, int width, long chunk, double *__restrict__ part) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= width) return;
  const long r0 = blockIdx.y * chunk;
  const long r1 = r0 + chunk < rows ? r0 + chunk : rows;
  double s = 0.0, s2 = 0.0;
  for (long r = r0; r < r1; ++r) {
    const double x = D[r * width + j];
    s += x;
    s2 += x * x;
  }
  part[(blockIdx.y * 2L + 0) * width + j] = s;
  part[(blockIdx.y * 2L + 1) * width + j] = s2;
}

// D[r][j] = (D[r][j] - mean[j]) * scale[j], in place.
__global__ void mlp_normalize(float *__restrict__ D, long rows, int width, const float *__restrict__ mean,
                              const float *__restrict__ scale) {
  const long total = rows * width;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < total; w += (long)gridDim.x * blockDim.x) {
    const int j = (int)(w % width);
    D[w] = (D[w] - mean[j]) * scale[j];
  }
}

// An operand of the matrix cores in the order they take it: for every tile of
// 32 rows (features) and step of 16 k (samples, or columns of a weight matrix)
// 64 lanes x 8 values, so that a wave's load is one contiguous KiB.  op_at: the
// place of (row, k); ldk: the k extent, a multiple of 16.
__host__ __device__ constexpr long op_size(int rows, int ldk) { return (long)((rows + 31) / 32 * 32) * ldk; }
__device__ inline long op_at(int row, int k, int ldk) {
  return ((long)(row >> 5) * (ldk >> 4) + (k >> 4)) * 512 + (((k >> 3) & 1) * 32 + (row & 31)) * 8 + (k & 7);
}

// BF16 copies of the weight matrices for the fused kernels, in that order:
// k padded to a multiple of 16 (W1) and the rows of the output matrix to a
// multiple of 32 (W3), padding zero.
//   W1b [hid][k1p], W2b [hid][hid], W3b [noutp][hid].
__global__ void mlp_pack_bf16(const float *__restrict__ W1, const float *__restrict__ W2,
                              const float *__restrict__ W3, int nin, int hid, int nout, int k1p, int noutp,
                              unsigned short *__restrict__ W1b, unsigned short *__restrict__ W2b,
                              unsigned short *__restrict__ W3b) {
  const long n1 = (long)hid * k1p, n2 = (long)hid * hid, n3 = (long)noutp * hid;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < n1 + n2 + n3; w += (long)gridDim.x * blockDim.x) {
    if (w < n1) {
      const long r = w / k1p;
      const int c = (int)(w - r * k1p);
      W1b[op_at((int)r, c, k1p)] = c < nin ? to_bf16(W1[r * nin + c]) : 0;
    } else if (w < n1 + n2) {
      W2b[op_at((int)((w - n1) / hid), (int)((w - n1) % hid), hid)] = to_bf16(W2[w - n1]);
    } else {
      const long v = w - n1 - n2;
      const long r = v / hid;
      W3b[op_at((int)r, (int)(v - r * hid), hid)] = r < nout ? to_bf16(W3[v]) : 0;
    }
  }
}

// One wave's 32 x 32 tile of A W^T over KS steps of 16: A is 32 rows in LDS
// (stride LDA), W the tile of weight rows at w (matrix-core order).  The first
// PF steps' weights are loaded by the constructor (before the barrier that A
// waits for), the later ones PF steps ahead.
template <int KS, int PF>
struct TileProduct {
  static constexpr int P = PF < KS ? PF : KS;
  const unsigned short *w;
  u16x8 buf[P];
  __device__ inline TileProduct(const unsigned short *__restrict__ W, int tile, int lane)
      : w(W + (long)tile * KS * 512 + 8 * lane) {
#pragma unroll
    for (int p = 0; p < P; ++p) buf[p] = *reinterpret_cast<const u16x8 *>(w + 512 * p);
  }
  template <int LDA>
  __device__ inline floatx16 run(const unsigned short *A, int lr, int kh) {
    floatx16 acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u16x8 cur = buf[s % P];
      if (s + P < KS) buf[s % P] = *reinterpret_cast<const u16x8 *>(w + 512 * (s + P));
      const u16x8 av = *reinterpret_cast<const u16x8 *>(A + lr * LDA + 16 * s + kh);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, cur),
                                                    acc, 0, 0, 0);
    }
    return acc;
  }
};

// Fused inference for p = 2 elements (27 nodes: NIN = 540 inputs, NOUT =
// 135 outputs) and HID = 256: one workgroup evaluates the network on FR = 32
// elements of one instance entirely on chip -- the nodal gradient from the
// state in type C, the features (background removed, normalised, rounded to
// BF16) into LDS, three MFMA layers with hidden activations kept in LDS, then
// the gate and the correction.  Numerically identical to
// ldg_nodal_grad_kernel + mlp_features + 3 x mlp_gemm + mlp_correction (same
// roundings, same MFMA sequence over k).
//
// The gradient is formed here because a state is 5 of the 20 feature fields:
// with the gradient written by a kernel of its own and read back, 13,824
// elements moved 135 MB instead of 45 (FP64).
//
// Bound by latency: 13,824 elements are 432 workgroups, all resident at once
// (two to a CU), so the time is that of one workgroup's chain.  Measured there
// in FP64: 28.8 us, where the gradient kernel took 14.7 and the inference
// without it 28.7 (55 with four waves that loaded the features in eight
// dependent batches and rows of weights 4 steps ahead).
constexpr int FR = 32;

template <typename C, typename UT, int NIN, int HID, int NOUT>
__global__ void __launch_bounds__(512, 4) mlp_infer(const UT *__restrict__ U, const ldg::InstDesc *__restrict__ inst,
                                                    const ldg::Ops<3, double> *__restrict__ op, long K, double rho0,
                                                    double E0, const float *__restrict__ norm,
                                                    const unsigned short *__restrict__ W1b,
                                                    const unsigned short *__restrict__ W2b,
                                                    const unsigned short *__restrict__ W3b,
                                                    const float *__restrict__ b1, const float *__restrict__ b2,
                                                    const float *__restrict__ b3, double bound, int dissipative,
                                                    double rho_add, double *__restrict__ corr,
                                                    unsigned char *__restrict__ gate) {
  constexpr int N = 3, NF = N * N, DOFS = NIN / 20, NU = 5 * DOFS, NTHR = 512;
  constexpr int K1P = (NIN + 15) / 16 * 16, NOUTP = (NOUT + 31) / 32 * 32;
  constexpr int XS = K1P + 8, HS = HID + 8, YS = NOUT + 1;
  static_assert(DOFS == N * NF, "27 nodes");
  static_assert(HID == 256, "eight waves of 32 hidden columns");
  static_assert(NOUTP / 32 <= 8, "one output tile per wave");
  static_assert(XS >= HS, "the second hidden layer reuses the feature buffer");
  __shared__ __align__(16) unsigned short Xs[FR][XS];
  // the state until the features are formed, then the hidden layer and the output
  constexpr int SB = FR * NU * (int)sizeof(C), HB = FR * HS * 2, YB = FR * YS * 4;
  __shared__ __align__(16) unsigned char buf[SB > HB + YB ? SB : HB + YB];
  __shared__ float snorm[2 * NU];
  __shared__ int snb[FR][3];
  C *const su = reinterpret_cast<C *>(buf);
  unsigned short(*const Hs)[HS] = reinterpret_cast<unsigned short(*)[HS]>(buf);
  float(*const Ys)[YS] = reinterpret_cast<float(*)[YS]>(buf + HB);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long e0 = (long)blockIdx.x * FR;
  const int rows = (int)((K - e0) < FR ? (K - e0) : FR);
  const float *omean = norm + 2 * NIN, *ostd = norm + 2 * NIN + NOUT;

  // loads: the block's state (contiguous), then the -d neighbours' traces on
  // their +d faces, both all in flight at once (past the last row: the last
  // one's, whose results nothing reads).  A thread keeps one variable and face
  // position, so that its features' means and spreads are loaded once, and
  // takes the lines there of every RG-th row in all three directions.
  constexpr int UL = (FR * NU + NTHR - 1) / NTHR, VF = 5 * NF, RG = NTHR / VF, LL = (FR + RG - 1) / RG;
  UT v[UL], vn[3][LL];
  const int tot = rows * NU;
#pragma unroll
  for (int i = 0; i < UL; ++i) v[i] = U[e0 * NU + min(tid + NTHR * i, tot - 1)];
  if (tid < FR) {
    const int kl = (int)e0 + min(tid, rows - 1);
    int c[3];
    ldg::element_coords(*inst, kl, c);
#pragma unroll
    for (int D = 0; D < 3; ++D) snb[tid][D] = kl + ldg::neighbor_step(*inst, c, D, -1);
  }
  for (int w = tid; w < NU; w += NTHR) {
    snorm[w] = norm[w];
    snorm[NU + w] = norm[NIN + w];
  }
  for (int w = tid; w < FR * (K1P - NIN); w += NTHR) Xs[w / (K1P - NIN)][NIN + w % (K1P - NIN)] = 0;
  __syncthreads();
  const int g0 = tid / VF, sab = tid - g0 * VF, s = sab / NF, ab = sab - s * NF, a_ = ab % N, b_ = ab / N;
  const int base[3] = {N * ab, a_ + NF * b_, ab};
  constexpr int ST[3] = {1, N, NF};
#pragma unroll
  for (int i = 0; i < LL; ++i)
#pragma unroll
    for (int D = 0; D < 3; ++D)
      vn[D][i] = U[(long)snb[min(g0 + RG * i, FR - 1)][D] * NU + s * DOFS + base[D] + ST[D] * (N - 1)];
#pragma unroll
  for (int i = 0; i < UL; ++i) {
    const int w = tid + NTHR * i, r = w / NU, j = w - r * NU, vs = j / DOFS;
    if (w < FR * NU) {
      su[w] = ldg::fluctuation<C>(v[i], vs, rho0, E0);
      const double x = (double)v[i] - (vs == 0 ? rho0 : vs == 4 ? E0 : 0.0);
      Xs[r][j] = to_bf16((float)((x - (double)snorm[j]) * (double)snorm[NU + j]));
    }
  }
  __syncthreads();
  // nodal gradient (operations and order of ldg_nodal_grad_kernel, nothing
  // fused across the product with ialpha, which that kernel stores): the own
  // trace's lift is in column 0 of Dn, the neighbour's has weight -L0
  if (g0 < RG) {
#pragma clang fp contract(off)
    C dn[N][N + 1];
#pragma unroll
    for (int q = 0; q < N; ++q) {
#pragma unroll
      for (int j = 0; j < N; ++j) dn[q][j] = C(op->Dn[q][j] + (j == 0 ? op->L0[q] : 0.0));
      dn[q][N] = C(-op->L0[q]);
    }
#pragma unroll
    for (int D = 0; D < 3; ++D) {
      const C ia = C(inst->ialpha[D]);
      const int j = NU + (5 * D + s) * DOFS + base[D];
      double mean[N], scale[N];
#pragma unroll
      for (int q = 0; q < N; ++q) {
        mean[q] = (double)norm[j + ST[D] * q];
        scale[q] = (double)norm[NIN + j + ST[D] * q];
      }
#pragma unroll
      for (int i = 0; i < LL; ++i) {
        const int r = g0 + RG * i;
        if (r < FR) {
          const C *const us = su + r * NU + s * DOFS + base[D];
          const C nb = ldg::fluctuation<C>(vn[D][i], s, rho0, E0);
          C x[N];
#pragma unroll
          for (int k = 0; k < N; ++k) x[k] = us[ST[D] * k];
#pragma unroll
          for (int q = 0; q < N; ++q) {
            C g = dn[q][N] * nb;
#pragma unroll
            for (int k = 0; k < N; ++k) g = ldg::fma_(dn[q][k], x[k], g);
            Xs[r][j + ST[D] * q] = to_bf16((float)(((double)(g * ia) - mean[q]) * scale[q]));
          }
        }
      }
    }
  }
  // wave w owns hidden columns [32 w, 32 w + 32)
  const int lr = lane & 31, kh = (lane >> 5) * 8, c = 32 * wave + lr;
  auto row_of = [&](int j) { return 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3); };
  TileProduct<K1P / 16, 17> p1(W1b, wave, lane);
  __syncthreads();
  TileProduct<HID / 16, 16> p2(W2b, wave, lane);
  {
    const float bias = b1[c];
    const floatx16 a = p1.template run<XS>(&Xs[0][0], lr, kh);
#pragma unroll
    for (int j = 0; j < 16; ++j) Hs[row_of(j)][c] = to_bf16(silu(a[j] + bias));
  }
  __syncthreads();
  // output tiles of 32 columns, tile w on wave w
  const bool ow = wave < NOUTP / 32;
  TileProduct<HID / 16, 16> p3(W3b, ow ? wave : 0, lane);
  // layer 2 into the feature buffer
  {
    const float bias = b2[c];
    const floatx16 a = p2.template run<HS>(&Hs[0][0], lr, kh);
#pragma unroll
    for (int j = 0; j < 16; ++j) Xs[row_of(j)][c] = to_bf16(silu(a[j] + bias));
  }
  __syncthreads();
  constexpr int OT = (NOUT + 63) / 64;
  float os[OT], om[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    os[t] = ostd[min(lane + 64 * t, NOUT - 1)];
    om[t] = omean[min(lane + 64 * t, NOUT - 1)];
  }
  if (ow) {
    const floatx16 a = p3.template run<XS>(&Xs[0][0], lr, kh);
    if (c < NOUT) {
#pragma unroll
      for (int j = 0; j < 16; ++j) Ys[row_of(j)][c] = a[j] + b3[c];
    }
  }
  __syncthreads();
  // gate and correction, one wave per row
#pragma unroll
  for (int i = 0; i < FR / (NTHR / 64); ++i) {
    const int r = wave + i * (NTHR / 64);
    if (r >= rows) break;
    float ss = 0.0f;
    for (int j = lane; j < NOUT; j += 64) ss += Ys[r][j] * Ys[r][j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    bool on = sqrt((double)ss / NOUT) <= bound;
    const long e = e0 + r;
    if (on && dissipative)
      on = dissipative * ke_production(U + e * NU, rho_add, DOFS, &Ys[r][0], ostd, omean, lane) <= 0.0;
#pragma unroll
    for (int t = 0; t < OT; ++t) {
      const int j = lane + 64 * t;
      if (j < NOUT) corr[e * NOUT + j] = on ? (double)Ys[r][j] * (double)os[t] + (double)om[t] : 0.0;
    }
    if (lane == 0) gate[e] = on ? 1 : 0;
  }
}

// L2 projection between orders, element by element: dst (nc^3 nodes per
// field) = (P (x) P (x) P) src (nf^3 nodes), P = nc x nf row-major, for 5
// fields per element.  One thread per (element, field, coarse node).
__global__ void mlp_project(int nf, int nc, long K, const double *__restrict__ P, const double *__restrict__ src,
                            double *__restrict__ dst) {
  const int df = nf * nf * nf, dc = nc * nc * nc;
  const long total = K * 5 * dc;
  for (long w = blockIdx.x * (long)blockDim.x + threadIdx.x; w < total; w += (long)gridDim.x * blockDim.x) {
    const long es = w / dc;                 // element * 5 + field
    const int node = (int)(w - es * dc);
    const int i = node % nc, j = (node / nc) % nc, k = node / (nc * nc);
    const double *s = src + es * df;
    double acc = 0.0;
    for (int c = 0; c < nf; ++c) {
      double accb = 0.0;
      for (int b = 0; b < nf; ++b) {
        double acca = 0.0;
        for (int a = 0; a < nf; ++a) acca += P[i * nf + a] * s[a + nf * (b + nf * c)];
        accb += P[j * nf + b] * acca;
      }
      acc += P[k * nf + c] * accb;
    }
    dst[w] = acc;
  }
}

}  // namespace ldg_mlp
