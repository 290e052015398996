// closure_train.hpp -- one training step of the p = 2 closure with 256 hidden
// units in two launches (device code).
//
//   mlp_train_rows     32 samples per workgroup, everything that is local to a
//                      sample on chip: gather, the three layers, the loss
//                      and the backward pass down to dZ1.  Leaves the operands
//                      of the weight gradients in HBM as BF16 and dY, dZ2, dZ1
//                      in FP32 for the bias gradients (layouts: TrainOperands).
//   mlp_train_weights  a wave per 32 x 32 tile of the three weight gradients:
//                      both operands are read as 16-byte vectors of 8 samples
//                      straight into the matrix cores' registers; then Adam
//                      on the tile and its BF16 copies.  Other workgroups sum
//                      the bias gradients.
// Bound by latency: 2,048 samples are 64 workgroups (22 us, the weights of
// three layers there and back through each; 30 us with weights in plain
// rows), and the operands of the weight gradients that the other XCDs just
// wrote (14 us, see mlp_train_weights).  As separate launches,
// 17 per batch with a device synchronisation for the loss, a batch took
// 1.85 ms, 1.2 ms of it column sums by 135 or 256 threads.
//
// The arithmetic is that of the layer-by-layer kernels (closure_kernels.hpp):
// operands rounded to BF16 at the same places, the same matrix instructions
// over k in the same order, the same FP32 operations in Adam, bias gradients
// summed sample by sample.  Trained parameters came out equal bit by bit to
// those kernels' (3 epochs on 700 to 20,480 samples, batches of 32, 129, 300
// and 2048, with and without weights); only the loss record is summed in
// another order (FP64).
#pragma once

#include "closure_kernels.hpp"

namespace ldg_mlp {

constexpr int TIN = 540, THID = 256, TOUT = 135;
constexpr int TINP = 544, TOUTP = 144;      // k extents padded to the matrix step of 16
constexpr int TROWS = 32;                   // samples per workgroup

// BF16 copies of the weights in matrix-core order (op_at): W1 [hid][TINP],
// W2 [hid][hid], W3 [160][hid] for the forward pass (those of the fused
// inference), and W2^T [hid][hid], W3^T [hid][TOUTP] for the backward pass.
struct TrainWeights {
  unsigned short *W1, *W2, *W3, *W2T, *W3T;
};
// Operands of the weight gradients, BF16, in the same order (rows: features, k:
// samples; with a plain row per feature, 32 rows of 2,048 samples side by side,
// mlp_train_weights took 38 us, not 17).  Operands of the bias gradients, FP32:
// per tile of 64 features [sample][64] (bias_at).
// ldb: the samples rounded up to TPAD; the rest are zero in dY, dZ2, dZ1.
constexpr int TPAD = 128;
__host__ __device__ constexpr long bias_size(int features, int ldb) { return (long)((features + 63) / 64 * 64) * ldb; }
__device__ inline long bias_at(int f, int r, int ldb) { return ((long)(f >> 6) * ldb + r) * 64 + (f & 63); }
struct TrainOperands {
  unsigned short *X, *H1, *H2, *dY, *dZ2, *dZ1;
  float *fY, *fZ2, *fZ1;
};

// Four consecutive samples (accumulator entries 4 g .. 4 g + 3) of one feature.
__device__ inline void store4(unsigned short *p, const unsigned short v[4]) {
  typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<u16x4 *>(p) = u16x4{v[0], v[1], v[2], v[3]};
}
// Rows [32 b, 32 b + 32) of a batch of B samples (sample r: dataset row
// idx[r]).  GRAD: also the backward pass and the operands; without it only
// the loss.  part[b] = sum of rw (Y - T)^2.
template <bool GRAD>
__global__ void __launch_bounds__(512) mlp_train_rows(const float *__restrict__ Xd, const float *__restrict__ Td,
                                                      const float *__restrict__ Wd, const long *__restrict__ idx, int B,
                                                      int ldb, TrainWeights W, const float *__restrict__ b1,
                                                      const float *__restrict__ b2, const float *__restrict__ b3,
                                                      float scale, TrainOperands out, double *__restrict__ part) {
  constexpr int XS = TINP + 8, HS = THID + 8, YS = TOUTP + 8;
  __shared__ __align__(16) unsigned short Xs[TROWS][XS];
  __shared__ __align__(16) unsigned short Hs[TROWS][HS];    // H1, then dZ2
  __shared__ __align__(16) unsigned short Gs[TROWS][HS];    // H2
  __shared__ __align__(16) unsigned short Ys[TROWS][YS];    // dY
  __shared__ long srow[TROWS];
  __shared__ float srw[TROWS];
  __shared__ double sred[8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = blockIdx.x * TROWS;
  // wave w owns hidden columns [32 w, 32 w + 32); accumulator j of lane l
  // holds row 8 (j/4) + 4 (l/32) + j%4, column l%32
  const int lr = lane & 31, kh = (lane >> 5) * 8, c = 32 * wave + lr;
  auto row_of = [&](int j) { return 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3); };
  TileProduct<TINP / 16, 17> p1(W.W1, wave, lane);
  if (tid < TROWS) {
    const bool in = r0 + tid < B;
    const long row = in ? idx[r0 + tid] : -1;
    srow[tid] = row;
    srw[tid] = in ? (Wd ? Wd[row] : 1.0f) : 0.0f;
  }
  for (int w = tid; w < TROWS * (TINP - TIN); w += 512) Xs[w / (TINP - TIN)][TIN + w % (TINP - TIN)] = 0;
  if (GRAD)
    for (int w = tid; w < TROWS * (TOUTP - TOUT); w += 512) Ys[w / (TOUTP - TOUT)][TOUT + w % (TOUTP - TOUT)] = 0;
  __syncthreads();
  // the samples, 4 features a time (a row is 135 of them), and the targets of
  // the output tile; all of a thread's loads before the first is used
  constexpr int V = TIN / 4, XL = (TROWS * V + 511) / 512;
  float4 xv[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int w = tid + 512 * i < TROWS * V ? tid + 512 * i : TROWS * V - 1, r = w / V;
    const long row = srow[r];
    xv[i] = reinterpret_cast<const float4 *>(Xd + (row >= 0 ? row : 0) * TIN)[w - r * V];
  }
  float tv[16];
  if (c < TOUT) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const long row = srow[row_of(j)];
      tv[j] = Td[(row >= 0 ? row : 0) * TOUT + c];
    }
  }
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int w = tid + 512 * i, r = w / V;
    if (w < TROWS * V) {
      const bool in = srow[r] >= 0;
      const unsigned short v[4] = {to_bf16(in ? xv[i].x : 0.f), to_bf16(in ? xv[i].y : 0.f),
                                   to_bf16(in ? xv[i].z : 0.f), to_bf16(in ? xv[i].w : 0.f)};
      store4(&Xs[r][4 * (w - r * V)], v);
    }
  }
  __syncthreads();
  float z1[16], z2[16];
  TileProduct<THID / 16, 16> p2(W.W2, wave, lane);
  {
    const float bias = b1[c];
    const floatx16 a = p1.template run<XS>(&Xs[0][0], lr, kh);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned short h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * g + i;
        z1[j] = a[j] + bias;
        h[i] = to_bf16(silu(z1[j]));
        Hs[row_of(j)][c] = h[i];
      }
      if (GRAD) store4(out.H1 + op_at(c, r0 + row_of(4 * g), ldb), h);
    }
  }
  if (GRAD) {   // X^T
    for (int w = tid; w < TINP * (TROWS / 8); w += 512) {
      const int o = w / TINP, f = w - o * TINP;
      u16x8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = Xs[8 * o + j][f];
      *reinterpret_cast<u16x8 *>(out.X + op_at(f, r0 + 8 * o, ldb)) = v;
    }
  }
  __syncthreads();
  const bool ow = wave < (TOUT + 31) / 32;   // the output layer: tile w (columns [32 w, 32 w + 32) of 135) on wave w
  TileProduct<THID / 16, 16> p3(W.W3, ow ? wave : 0, lane);
  {
    const float bias = b2[c];
    const floatx16 a = p2.template run<HS>(&Hs[0][0], lr, kh);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned short h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * g + i;
        z2[j] = a[j] + bias;
        h[i] = to_bf16(silu(z2[j]));
        Gs[row_of(j)][c] = h[i];
      }
      if (GRAD) store4(out.H2 + op_at(c, r0 + row_of(4 * g), ldb), h);
    }
  }
  __syncthreads();
  TileProduct<TOUTP / 16, TOUTP / 16> p4(GRAD ? W.W3T : W.W1, GRAD ? wave : 0, lane);
  double loss = 0.0;
  if (ow) {
    const floatx16 a = p3.template run<HS>(&Gs[0][0], lr, kh);
    if (c < TOUT) {
      const float bias = b3[c];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        unsigned short hb[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = 4 * g + i, r = row_of(j);
          const float y = a[j] + bias;
          const float d = srow[r] >= 0 ? y - tv[j] : 0.0f;
          loss += (double)srw[r] * d * d;
          const float hf = scale * srw[r] * d;
          hb[i] = to_bf16(hf);
          if (GRAD) {
            Ys[r][c] = hb[i];
            out.fY[bias_at(c, r0 + r, ldb)] = hf;
          }
        }
        if (GRAD) store4(out.dY + op_at(c, r0 + row_of(4 * g), ldb), hb);
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
  if (lane == 0) sred[wave] = loss;
  __syncthreads();
  if (tid == 0) {
    double s = 0.0;
    for (int w = 0; w < 8; ++w) s += sred[w];
    part[blockIdx.x] = s;
  }
  if (!GRAD) return;

  // dZ = dH silu'(Z), silu'(z) = s (1 + z (1 - s)), s = sigmoid(z)
  auto back = [](float dh, float z) -> float {
    const float s = 1.0f / (1.0f + __expf(-z));
    return dh * s * __builtin_fmaf(z, 1.0f - s, 1.0f);
  };
  TileProduct<THID / 16, 16> p5(W.W2T, wave, lane);
  {
    const floatx16 a = p4.template run<YS>(&Ys[0][0], lr, kh);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned short hb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * g + i;
        const float hf = back(a[j], z2[j]);
        hb[i] = to_bf16(hf);
        out.fZ2[bias_at(c, r0 + row_of(j), ldb)] = hf;
        Hs[row_of(j)][c] = hb[i];
      }
      store4(out.dZ2 + op_at(c, r0 + row_of(4 * g), ldb), hb);
    }
  }
  __syncthreads();
  {
    const floatx16 a = p5.template run<HS>(&Hs[0][0], lr, kh);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned short hb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * g + i;
        const float hf = back(a[j], z1[j]);
        hb[i] = to_bf16(hf);
        out.fZ1[bias_at(c, r0 + row_of(j), ldb)] = hf;
      }
      store4(out.dZ1 + op_at(c, r0 + row_of(4 * g), ldb), hb);
    }
  }
}

// Parameters, moments and Adam's constants of a step (the FP32 operations of
// mlp_adam).
struct AdamArgs {
  float *p, *m, *v;
  float lr, b1, b2, eps, bc1, bc2;
};
struct AdamState { float p, m, v; };
__device__ inline AdamState adam_load(const AdamArgs &a, long w) { return AdamState{a.p[w], a.m[w], a.v[w]}; }
__device__ inline float adam_update(const AdamArgs &a, long w, const AdamState &s, float g) {
  const float mi = __builtin_fmaf(1.0f - a.b1, g, a.b1 * s.m);
  const float vi = __builtin_fmaf(g, (1.0f - a.b2) * g, a.b2 * s.v);
  a.m[w] = mi;
  a.v[w] = vi;
  const float p = s.p - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
  a.p[w] = p;
  return p;
}

constexpr int T1M = THID / 32, T1N = (TIN + 31) / 32, T2 = THID / 32, T3M = (TOUT + 31) / 32;
constexpr int TRAIN_TILES = T1M * T1N + T2 * T2 + T3M * T2;
constexpr int TBF = 32;                     // bias gradients per workgroup
constexpr int TRAIN_BIAS_BLOCKS = 2 * (THID / TBF) + (TOUT + TBF - 1) / TBF;

// Offsets of W1, b1, W2, b2, W3, b3 in the parameter vector.
constexpr long TO_B1 = (long)THID * TIN, TO_W2 = TO_B1 + THID, TO_B2 = TO_W2 + (long)THID * THID, TO_W3 = TO_B2 + THID,
               TO_B3 = TO_W3 + (long)TOUT * THID;

// Workgroups [0, TRAIN_TILES): one wave on a tile of dW = (rows of one
// operand) x (rows of the other) summed over the samples; the rest: TBF bias
// gradients each.  Either the Adam update, and the weights' BF16 copies.
//
// A tile reads 256 KB (2,048 samples) for 1.7 us of matrix instructions, so
// its time is the rate at which a CU takes operands: a tile per CU (the bias
// workgroups are why there are four waves; three leave at once).  Workgroups
// go to the 8 XCDs in turn; each XCD gets an eighth of every layer's tiles,
// those of the same columns, so that its L2 fetches 3 MB of operands instead
// of nearly all 6.6.  Measured at 2,048 samples: 14.2 us (tiles alone 11.4, bias
// gradients alone 12.1); 17.2 with four tiles per workgroup in any order and
// bias workgroups of 64 features whose additions each waited for LDS.
__global__ void __launch_bounds__(256, 1) mlp_train_weights(TrainOperands in, int ldb, TrainWeights W, AdamArgs ad) {
  // bias: BS samples of TBF features at a time through LDS, summed sample by
  // sample by one lane per feature while the next BG - 1 pieces are loaded
  constexpr int BS = TPAD, BG = 4, BL = BS * TBF / 4 / 256;
  __shared__ __align__(16) float sbias[2][BS][TBF];
  static_assert(T1M == 8 && T2 == 8, "each layer's tiles in 8 equal shares");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if ((int)blockIdx.x >= TRAIN_TILES) {
    // dZ1 (256 features), dZ2 (256), dY (135)
    constexpr int HB = THID / TBF;
    const int tile = (int)blockIdx.x - TRAIN_TILES;
    const float *d = tile < HB ? in.fZ1 : tile < 2 * HB ? in.fZ2 : in.fY;
    const int f0 = TBF * (tile < 2 * HB ? tile % HB : tile - 2 * HB), f = f0 + lane;
    d += (long)(f0 >> 6) * ldb * 64 + (f0 & 63);
    using f4 = float __attribute__((ext_vector_type(4)));
    f4 buf[BG][BL];
    constexpr int Q = TBF / 4;                 // 16-byte pieces of a sample
    float s = 0.0f;
    const f4 *const src = reinterpret_cast<const f4 *>(d) + tid / Q * 16 + tid % Q;
    auto load = [&](f4 (&v)[BL], int k0) {
#pragma unroll
      for (int i = 0; i < BL; ++i) v[i] = src[(long)(min(k0, ldb - BS) + i * (256 / Q)) * 16];
    };
    auto piece = [&](f4 (&v)[BL], int g, auto then) {
#pragma unroll
      for (int i = 0; i < BL; ++i) reinterpret_cast<f4 *>(&sbias[g & 1][0][0])[tid + 256 * i] = v[i];
      __syncthreads();   // (the sums of two pieces ago, from the same buffer, ended before it)
      then();
      if (wave == 0) {
        // 32 values on their way while 32 are added (left to the scheduler,
        // every two additions wait for their own read: 38 us)
        constexpr int R = 32;
        float x[2][R];
#pragma unroll
        for (int k = 0; k < R; ++k) x[0][k] = sbias[g & 1][k][lane & (TBF - 1)];
#pragma unroll
        for (int c = 0; c < BS / R; ++c) {
          if (c + 1 < BS / R) {
#pragma unroll
            for (int k = 0; k < R; ++k) x[(c + 1) & 1][k] = sbias[g & 1][(c + 1) * R + k][lane & (TBF - 1)];
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < R; ++k) s += x[c & 1][k];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
#pragma unroll
    for (int g = 0; g < BG; ++g) load(buf[g], g * BS);
    int k0 = 0;
    // (no condition inside the loop: at a join of paths every load is waited for)
    for (; k0 + BG * BS <= ldb; k0 += BG * BS) {
#pragma unroll
      for (int g = 0; g < BG; ++g) piece(buf[g], g, [&] { load(buf[g], k0 + (g + BG) * BS); });
    }
#pragma unroll
    for (int g = 0; g < BG - 1; ++g)
      if (k0 + g * BS < ldb) piece(buf[g], g, [] {});
    if (wave == 0 && lane < TBF && f < (tile < 2 * HB ? THID : TOUT)) {
      const long w = (tile < HB ? TO_B1 : tile < 2 * HB ? TO_B2 : TO_B3) + f;
      adam_update(ad, w, adam_load(ad, w), s);
    }
    return;
  }
  if (wave > 0) return;
  const unsigned short *A, *Bp;
  int m0, n0, M, N;
  long o;
  int layer;
  const int xcd = (int)blockIdx.x & 7, i = (int)blockIdx.x >> 3;   // i: tile of the XCD's share
  if (i < T1N) {
    layer = 1;
    const int k = T1N * xcd + i;
    m0 = k % T1M * 32;
    n0 = k / T1M * 32;
    A = in.dZ1; Bp = in.X; M = THID; N = TIN; o = 0;
  } else if (i < T1N + T2) {
    layer = 2;
    m0 = (i - T1N) * 32;
    n0 = xcd * 32;
    A = in.dZ2; Bp = in.H1; M = THID; N = THID; o = TO_W2;
  } else {
    layer = 3;
    m0 = (i - T1N - T2) * 32;
    n0 = xcd * 32;
    A = in.dY; Bp = in.H2; M = TOUT; N = THID; o = TO_W3;
  }
  const int lr = lane & 31;
  const unsigned short *pa = A + (long)m0 * ldb + 8 * lane, *pb = Bp + (long)n0 * ldb + 8 * lane;
  floatx16 acc;
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
  // Adam's operands, loaded now (one parameter's loads after the stores of the
  // one before would cost a memory round trip each, 16 times)
  const int n = n0 + lr;
  auto row_of = [&](int j) { return m0 + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3); };
  AdamState st[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int m = row_of(j) < M ? row_of(j) : M - 1;
    st[j] = adam_load(ad, o + (long)m * N + (n < N ? n : N - 1));
  }
  // PG groups of PF matrix steps in flight: the operands were just written by
  // the other XCDs, so every read goes past the L2
  constexpr int PF = TPAD / 16, PG = 2;
  u16x8 ba[PG][PF], bb[PG][PF];
  auto load = [&](int g, int k0) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      ba[g][p] = *reinterpret_cast<const u16x8 *>(pa + 32 * k0 + 512 * p);
      bb[g][p] = *reinterpret_cast<const u16x8 *>(pb + 32 * k0 + 512 * p);
    }
  };
  auto product = [&](int g) {
#pragma unroll
    for (int p = 0; p < PF; ++p)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ba[g][p]),
                                                    __builtin_bit_cast(bf16x8, bb[g][p]), acc, 0, 0, 0);
  };
  const int last = ldb - TPAD;
#pragma unroll
  for (int g = 0; g < PG; ++g) {
    load(g, min(g * TPAD, last));
    __builtin_amdgcn_sched_barrier(0);
  }
  int k0 = 0;
  for (; k0 + PG * TPAD <= ldb; k0 += PG * TPAD) {   // (no condition inside, as above)
#pragma unroll
    for (int g = 0; g < PG; ++g) {
      product(g);
      __builtin_amdgcn_sched_barrier(0);   // keep the groups in order: their loads are waited for in order
      load(g, min(k0 + (g + PG) * TPAD, last));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int g = 0; g < PG - 1; ++g)
    if (k0 + g * TPAD < ldb) product(g);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int m = row_of(j);
    if (m < M && n < N) {
      const unsigned short h = to_bf16(adam_update(ad, o + (long)m * N + n, st[j], acc[j]));
      if (layer == 1) {
        W.W1[op_at(m, n, TINP)] = h;
      } else if (layer == 2) {
        W.W2[op_at(m, n, THID)] = h;
        W.W2T[op_at(n, m, THID)] = h;
      } else {
        W.W3[op_at(m, n, THID)] = h;
        W.W3T[op_at(n, m, TOUTP)] = h;
      }
    }
  }
}

// W2^T and W3^T from the packed W2 and W3 (rows of W3^T padded with zeros).
__global__ void mlp_pack_transposed(TrainWeights W) {
  for (int w = blockIdx.x * blockDim.x + threadIdx.x; w < THID * (THID + TOUTP); w += gridDim.x * blockDim.x) {
    if (w < THID * THID) {
      const int r = w / THID, k = w - r * THID;
      W.W2T[op_at(r, k, THID)] = W.W2[op_at(k, r, THID)];
    } else {
      const int v = w - THID * THID, r = v / TOUTP, k = v - r * TOUTP;
      W.W3T[op_at(r, k, TOUTP)] = k < TOUT ? W.W3[op_at(k, r, THID)] : 0;
    }
  }
}

}  // namespace ldg_mlp
