// Training of the learned HLLD surrogate: one Adam step in two launches.
//
//   k_train_tile   a block takes 32 samples through the whole network: minibatch
//                  draw, forward, loss and backward on the matrix cores, the
//                  layers handed on in LDS.  It leaves each layer's activations
//                  and gradients as bf16 MFMA operands (K = its 32 samples) and
//                  the gradients also in FP32 for the bias sums
//   k_train_grad   one wavefront per 16x16 tile of a weight gradient (144 of
//                  them), 16 columns of a bias gradient (25) and the loss: it
//                  walks the batch tile by tile and applies Adam to its own
//                  parameters, packed for the next step's tiles
//
// What bounds it: a step of 8192 samples is 1.8 GFLOP, 1.5 us of the matrix
// cores.  What is left is the latency of eight dependent layers in the first
// launch and, in the second, 256 dependent MFMAs a wavefront fed by 512 KB of
// operands, loaded GU tiles ahead.  The sums over the batch stay in one chain
// in batch order, as a layer-by-layer product with K steps of 32 adds them
// (bias sums: four chains of every fourth sample): splitting them over blocks
// measured the same time but moved the trained parameters by 2e-5.
//
// Measured, 8192 samples: 41 us a step (k_train_tile 14.9 us, k_train_grad 18.7 us);
// as 22 launches of one 64x64-tile product or elementwise kernel each it was
// 5.26 ms, most of it the weight gradients, whose K loop over the batch ran on
// four blocks with one tile of loads in flight.
// Included by fvm_surrogate.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "fvm_mlp.h"

namespace fvm {
namespace sg {

constexpr int TS = 32;       // samples per tile: the K of one gradient MFMA
constexpr int TB = 256;      // threads per tile block: 4 wavefronts, 32 of the 128 features each
constexpr int SP = TS + 8;   // [feature][sample] row, bf16: 80 bytes, conflict-free 16-byte reads
constexpr int FP = NH + 8;   // [sample][feature] row, bf16: 272 bytes

// weight fragments in the lane order of the MFMA A operand (16x16x32: lane
// holds row lane % 16, K 8 (lane / 16) .. + 8)
//   forward  rows = output features, K = input features: W0 (K padded to 32), W1, W2, W3 (rows padded to 16)
//   backward rows = input features, K = output features: W3 (K padded to 32), W2, W1
constexpr int TF0 = 0, TF1 = TF0 + 8 * 512, TF2 = TF1 + 32 * 512, TF3 = TF2 + 32 * 512, TB3 = TF3 + 4 * 512,
              TB2 = TB3 + 8 * 512, TB1 = TB2 + 32 * 512, T_FRAG = TB1 + 32 * 512;
// what a tile leaves for k_train_grad, per tile:
//   operands, 1 KB each (lane: row lane % 16, 8 samples from 8 (lane / 16)):
//     the inputs, 8 row tiles of H0, H1, H2 and of the gradients D0, D1, D2, dL/dy
//   FP32 gradients by 16 columns, 2 KB each: [sample % 4][column][sample / 4]
constexpr int OX = 0, OH0 = 1, OH1 = 9, OH2 = 17, OD0 = 25, OD1 = 33, OD2 = 41, ODY = 49, N_OP = 50;
constexpr int CD0 = 0, CD1 = 8, CD2 = 16, CDY = 24, N_COL = 25;
constexpr size_t OP_E = 512, COL_E = 512;  // elements of an operand (bf16) and of a column group (float)

struct LossW {
  float w[7];
};
struct TrainArgs {
  int B;
  const float *X, *T;            // the training set (draw) or the batch itself
  long long nsamp;               // draw: samples of the training set
  unsigned long long seed, step;
  const __bf16 *frag;            // [T_FRAG]
  const float *P;                // parameters (biases)
  float lam;
  LossW lw;
  __bf16 *ops;                   // [tile][N_OP][OP_E]
  float *cols;                   // [tile][N_COL][COL_E]
  float *tloss;                  // [tile]
  float *Y;                      // batch outputs [B][8], or null
};

__device__ __forceinline__ unsigned long long splitmix(unsigned long long z) {
  z += 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

// LDS of a tile block
struct TrainLds {
  __bf16 xs[TS][SP];         // inputs [sample][feature], features 16..31 zero
  __bf16 xt[NIN][SP];        // inputs [feature][sample]
  __bf16 hs[2][TS][FP];      // the layer being read / written, [sample][feature]
  __bf16 dys[TS][SP];        // dL/dy [sample][output], outputs 8..31 zero
  __bf16 dyt[16][SP];        // dL/dy [output][sample], rows 8..15 zero
  float y[TS][NOUT], t[TS][NOUT];
  float dyc[COL_E];          // dL/dy as a column group, columns 8..15 zero
  struct {                   // each wavefront's own 32 features on their way out
    __bf16 t[32][SP];        // [feature][sample]
    float c[2][COL_E];       // column groups
  } wave[TB / 64];
};
static_assert(sizeof(TrainLds) <= 64 * 1024, "LDS budget");

// weight fragments of this wavefront's two row tiles, NC K steps each
template <int NC> __device__ __forceinline__ void load_frag(const __bf16 *frag, int w, int lane, bf16x8 (&a)[2][NC]) {
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int c = 0; c < NC; c++)
      a[i][c] = *reinterpret_cast<const bf16x8 *>(frag + ((size_t)((2 * w + i) * NC + c) * 64 + lane) * 8);
}
// rows (features of this wavefront) x 32 samples: acc[i][j], row tile 2w + i, sample tile j
template <int NC, int STRIDE>
__device__ __forceinline__ void layer(const bf16x8 (&a)[2][NC], const __bf16 (*src)[STRIDE], int lane, f32x4 (&acc)[2][2]) {
  const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < NC; c++) {
    bf16x8 b[2];
#pragma unroll
    for (int j = 0; j < 2; j++) b[j] = *reinterpret_cast<const bf16x8 *>(&src[16 * j + r16][32 * c + 8 * g]);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][c], b[j], acc[i][j], 0, 0, 0);
  }
}
// a layer's values: to LDS [sample][feature] for the next layer, and out as the
// operands of this wavefront's two row tiles
__device__ __forceinline__ void put(const f32x4 (&v)[2][2], __bf16 (*s)[FP], __bf16 (*t)[SP], __bf16 *op, int w, int lane) {
  const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      bf16x4 b;
#pragma unroll
      for (int r = 0; r < 4; r++) b[r] = (__bf16)v[i][j][r];
      const int f = 16 * i + 4 * g, q = 16 * j + r16;
      *reinterpret_cast<bf16x4 *>(&s[q][32 * w + f]) = b;
#pragma unroll
      for (int r = 0; r < 4; r++) t[f + r][q] = b[r];
    }
  wave_sync();
#pragma unroll
  for (int i = 0; i < 2; i++)
    *reinterpret_cast<bf16x8 *>(op + (size_t)(2 * w + i) * OP_E + 8 * lane) =
        *reinterpret_cast<const bf16x8 *>(&t[16 * i + r16][8 * g]);
  wave_sync();  // read before the next layer's values land
}
// hidden layer: bias, ReLU (returned mask: one bit per value)
__device__ __forceinline__ unsigned hidden(f32x4 (&v)[2][2], const float *bias, __bf16 (*s)[FP], __bf16 (*t)[SP],
                                           __bf16 *op, int w, int lane) {
  const int g = lane >> 4;
  unsigned mask = 0;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const f32x4 b = *reinterpret_cast<const f32x4 *>(bias + 16 * (2 * w + i) + 4 * g);
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float h = fmaxf(v[i][j][r] + b[r], 0.0f);
        v[i][j][r] = h;
        mask |= (h > 0.0f ? 1u : 0u) << (8 * i + 4 * j + r);
      }
  }
  put(v, s, t, op, w, lane);
  return mask;
}
// gradient of a hidden layer: ReLU mask, FP32 column groups, operands
__device__ __forceinline__ void hidden_grad(f32x4 (&v)[2][2], unsigned mask, __bf16 (*s)[FP], __bf16 (*t)[SP],
                                            float (*c)[COL_E], __bf16 *op, float *col, int w, int lane) {
  const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (!((mask >> (8 * i + 4 * j + r)) & 1u)) v[i][j][r] = 0.0f;
        c[i][((r16 & 3) * 16 + 4 * g + r) * 8 + 4 * j + (r16 >> 2)] = v[i][j][r];
      }
  put(v, s, t, op, w, lane);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int h = 0; h < 2; h++)
      *reinterpret_cast<f32x4 *>(col + (size_t)(2 * w + i) * COL_E + 256 * h + 4 * lane) =
          *reinterpret_cast<const f32x4 *>(&c[i][256 * h + 4 * lane]);
  wave_sync();
}

// DRAW: the tile's samples are drawn from the training set by the counter hash
template <bool DRAW> __global__ void __launch_bounds__(TB) k_train_tile(TrainArgs A) {
  __shared__ __attribute__((aligned(16))) TrainLds L;
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, r16 = lane & 15;
  const int tile = (int)blockIdx.x;
  __bf16 *ops = A.ops + (size_t)tile * N_OP * OP_E;
  float *cols = A.cols + (size_t)tile * N_COL * COL_E;
  auto &my = L.wave[w];

  bf16x8 f0[2][1], f1[2][4], f2[2][4];
  load_frag<1>(A.frag + TF0, w, lane, f0);
  load_frag<4>(A.frag + TF1, w, lane, f1);
  load_frag<4>(A.frag + TF2, w, lane, f2);
  {
    // inputs and targets: 8 threads a sample; samples past the batch are zero
    // and get no gradient
    const int q = t >> 3, part = t & 7, smp = tile * TS + q;
    float2 x = make_float2(0.0f, 0.0f);
    float tv = 0.0f;
    if (smp < A.B) {
      long long src = smp;
      if constexpr (DRAW)
        src = (long long)(splitmix(A.seed ^ splitmix((A.step << 32) ^ (unsigned long long)smp)) %
                          (unsigned long long)A.nsamp);
      x = *reinterpret_cast<const float2 *>(A.X + (size_t)src * NIN + 2 * part);
      tv = A.T[(size_t)src * NOUT + part];
    }
    // zero padding of the K and row directions
    for (int i = t; i < TS * SP; i += TB) (&L.dys[0][0])[i] = (__bf16)0.0f;
    for (int i = t; i < 16 * SP; i += TB) (&L.dyt[0][0])[i] = (__bf16)0.0f;
    for (int i = t; i < (int)COL_E; i += TB) L.dyc[i] = 0.0f;
    L.xs[q][16 + 2 * part] = L.xs[q][17 + 2 * part] = (__bf16)0.0f;
    L.xs[q][2 * part] = (__bf16)x.x;
    L.xs[q][2 * part + 1] = (__bf16)x.y;
    L.xt[2 * part][q] = (__bf16)x.x;
    L.xt[2 * part + 1][q] = (__bf16)x.y;
    L.t[q][part] = tv;
  }
  __syncthreads();
  f32x4 v[2][2];
  layer<1, SP>(f0, L.xs, lane, v);
  const unsigned m0 = hidden(v, A.P + OB0, L.hs[0], my.t, ops + OH0 * OP_E, w, lane);
  __syncthreads();
  layer<4, FP>(f1, L.hs[0], lane, v);
  bf16x8 f3[4], b3[2][1], b2[2][4], b1[2][4];
#pragma unroll
  for (int c = 0; c < 4; c++) f3[c] = *reinterpret_cast<const bf16x8 *>(A.frag + TF3 + (size_t)(c * 64 + lane) * 8);
  load_frag<1>(A.frag + TB3, w, lane, b3);
  load_frag<4>(A.frag + TB2, w, lane, b2);
  const unsigned m1 = hidden(v, A.P + OB1, L.hs[1], my.t, ops + OH1 * OP_E, w, lane);
  __syncthreads();
  layer<4, FP>(f2, L.hs[1], lane, v);
  load_frag<4>(A.frag + TB1, w, lane, b1);
  const unsigned m2 = hidden(v, A.P + OB2, L.hs[0], my.t, ops + OH2 * OP_E, w, lane);
  __syncthreads();
  // outputs: wavefronts 0 and 1 take 16 samples each
  if (w < 2) {
    f32x4 o = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const bf16x8 b = *reinterpret_cast<const bf16x8 *>(&L.hs[0][16 * w + r16][32 * c + 8 * g]);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f3[c], b, o, 0, 0, 0);
    }
    if (g < 2) {
      const f32x4 b = *reinterpret_cast<const f32x4 *>(A.P + OB3 + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; r++) L.y[16 * w + r16][4 * g + r] = o[r] + b[r];
    }
  }
  __syncthreads();
  // loss and dL/dy, one lane a sample
  float loss = 0.0f;
  if (t < TS && tile * TS + t < A.B) {
    const int s = tile * TS + t;
    float dy[NOUT], e2 = 0.0f, d[7];
#pragma unroll
    for (int k = 0; k < 7; k++) {
      d[k] = L.y[t][k] - L.t[t][k];
      e2 += A.lw.w[k] * d[k] * d[k];
    }
    const float c = log10f(e2 + 1e-10f);
    const float dc = L.y[t][7] - c;
    const float iB = 1.0f / (float)A.B;
#pragma unroll
    for (int k = 0; k < 7; k++) dy[k] = 2.0f * A.lw.w[k] * d[k] * iB;
    dy[7] = 2.0f * A.lam * dc * iB;
    loss = (e2 + A.lam * dc * dc) * iB;
    if (A.Y) {
#pragma unroll
      for (int k = 0; k < NOUT; k++) A.Y[(size_t)s * NOUT + k] = L.y[t][k];
    }
#pragma unroll
    for (int k = 0; k < NOUT; k++) {
      L.dys[t][k] = (__bf16)dy[k];
      L.dyt[k][t] = (__bf16)dy[k];
      L.dyc[((t & 3) * 16 + k) * 8 + (t >> 2)] = dy[k];
    }
  }
  __syncthreads();
  layer<1, SP>(b3, L.dys, lane, v);
  hidden_grad(v, m2, L.hs[1], my.t, my.c, ops + OD2 * OP_E, cols + CD2 * COL_E, w, lane);
  __syncthreads();
  layer<4, FP>(b2, L.hs[1], lane, v);
  hidden_grad(v, m1, L.hs[0], my.t, my.c, ops + OD1 * OP_E, cols + CD1 * COL_E, w, lane);
  __syncthreads();
  layer<4, FP>(b1, L.hs[0], lane, v);
  hidden_grad(v, m0, L.hs[1], my.t, my.c, ops + OD0 * OP_E, cols + CD0 * COL_E, w, lane);
  // inputs, dL/dy and the loss, a wavefront each
  if (w == 0)
    *reinterpret_cast<bf16x8 *>(ops + OX * OP_E + 8 * lane) = *reinterpret_cast<const bf16x8 *>(&L.xt[r16][8 * g]);
  if (w == 1)
    *reinterpret_cast<bf16x8 *>(ops + ODY * OP_E + 8 * lane) = *reinterpret_cast<const bf16x8 *>(&L.dyt[r16][8 * g]);
  if (w == 2)
#pragma unroll
    for (int h = 0; h < 2; h++)
      *reinterpret_cast<f32x4 *>(cols + CDY * COL_E + 256 * h + 4 * lane) =
          *reinterpret_cast<const f32x4 *>(&L.dyc[256 * h + 4 * lane]);
  if (w == 0) {
    for (int o = 16; o > 0; o >>= 1) loss += __shfl_xor(loss, o);  // lanes 0..31
    if (lane == 0) A.tloss[tile] = loss;
  }
}

// the places of weight i in the packed fragments
__device__ __forceinline__ int afrag(int nc, int row, int k) {  // A operand: row, K index
  return (((row >> 4) * nc + (k >> 5)) * 64 + 16 * ((k >> 3) & 3) + (row & 15)) * 8 + (k & 7);
}
__device__ __forceinline__ void pack_weight(__bf16 *frag, int i, float v) {
  const __bf16 b = (__bf16)v;
  if (i < OB0) {
    const int k = (i - OW0) / NH, n = (i - OW0) % NH;
    frag[TF0 + afrag(1, n, k)] = b;
  } else if (i >= OW1 && i < OB1) {
    const int k = (i - OW1) / NH, n = (i - OW1) % NH;
    frag[TF1 + afrag(4, n, k)] = b;
    frag[TB1 + afrag(4, k, n)] = b;
  } else if (i >= OW2 && i < OB2) {
    const int k = (i - OW2) / NH, n = (i - OW2) % NH;
    frag[TF2 + afrag(4, n, k)] = b;
    frag[TB2 + afrag(4, k, n)] = b;
  } else if (i >= OW3 && i < OB3) {
    const int k = (i - OW3) / NOUT, n = (i - OW3) % NOUT;
    frag[TF3 + afrag(4, n, k)] = b;
    frag[TB3 + afrag(1, k, n)] = b;
  }
}
// fragments of the current parameters (the padding was cleared at allocation)
__global__ void k_train_pack(const float *P, __bf16 *frag) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < NPARAM) pack_weight(frag, i, P[i]);
}

struct GradArgs {
  int ntile;
  const __bf16 *ops;
  const float *cols, *tloss;
  float *G;     // gradients (no update)
  float *loss;  // the step's loss
  float *P, *M, *V;
  float lr, b1, b2, eps, c1, c2;
  __bf16 *frag;
};
constexpr int GRAD_BLOCKS = 64 + 64 + 8 + 8 + N_COL + 1;
constexpr int GU = 16;  // tiles loaded ahead: 32 loads of 1 KB in flight

template <bool ADAM> __device__ __forceinline__ void take_grad(const GradArgs &A, int i, float g) {
  if constexpr (ADAM) {
    const float m = A.b1 * A.M[i] + (1.0f - A.b1) * g;
    const float v = A.b2 * A.V[i] + (1.0f - A.b2) * g * g;
    A.M[i] = m;
    A.V[i] = v;
    const float pn = A.P[i] - A.lr * (m / A.c1) / (sqrtf(v / A.c2) + A.eps);
    A.P[i] = pn;
    pack_weight(A.frag, i, pn);
  } else {
    A.G[i] = g;
  }
}
// every tile's 16 bytes of this lane at a and at b (tile strides sa, sb bytes)
// through f, in tile order, the next GU tiles' loads in flight
template <typename F>
__device__ __forceinline__ void walk(int ntile, const char *a, size_t sa, const char *b, size_t sb, F f) {
  int4 va[GU], vb[GU];
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < GU; u++) {
      const int t = min(t0 + u, ntile - 1);  // past the end: the last tile again, not used
      va[u] = *reinterpret_cast<const int4 *>(a + (size_t)t * sa);
      vb[u] = *reinterpret_cast<const int4 *>(b + (size_t)t * sb);
    }
  };
  load(0);
  for (int t0 = 0; t0 < ntile; t0 += GU) {
    int4 ca[GU], cb[GU];
#pragma unroll
    for (int u = 0; u < GU; u++) {
      ca[u] = va[u];
      cb[u] = vb[u];
    }
    load(t0 + GU);
#pragma unroll
    for (int u = 0; u < GU; u++)
      if (t0 + u < ntile) f(ca[u], cb[u]);
  }
}

template <bool ADAM> __global__ void __launch_bounds__(64) k_train_grad(GradArgs A) {
  const int lane = (int)threadIdx.x, g = lane >> 4, r16 = lane & 15;
  int q = (int)blockIdx.x;
  if (q < 144) {
    // a 16x16 tile of a weight gradient: rows (inputs of the layer) x columns
    int oa, ob, base, ld, row0, col0, ncol = 16;
    if (q < 128) {
      const bool l2 = q >= 64;
      q &= 63;
      oa = (l2 ? OH1 : OH0) + (q >> 3);
      ob = (l2 ? OD2 : OD1) + (q & 7);
      base = l2 ? OW2 : OW1;
      ld = NH;
      row0 = 16 * (q >> 3);
      col0 = 16 * (q & 7);
    } else if (q < 136) {
      oa = OH2 + q - 128;
      ob = ODY;
      base = OW3;
      ld = ncol = NOUT;
      row0 = 16 * (q - 128);
      col0 = 0;
    } else {
      oa = OX;
      ob = OD0 + q - 136;
      base = OW0;
      ld = NH;
      row0 = 0;
      col0 = 16 * (q - 136);
    }
    const char *ops = reinterpret_cast<const char *>(A.ops) + 16 * lane;
    const size_t st = N_OP * OP_E * sizeof(__bf16);
    f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    walk(A.ntile, ops + oa * OP_E * sizeof(__bf16), st, ops + ob * OP_E * sizeof(__bf16), st, [&](int4 a, int4 b) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                    0, 0);
    });
    if (r16 < ncol)
#pragma unroll
      for (int r = 0; r < 4; r++) take_grad<ADAM>(A, base + (row0 + 4 * g + r) * ld + col0 + r16, acc[r]);
  } else if (q < 144 + N_COL) {
    // 16 columns of a bias gradient: lane group g sums the samples s % 4 == g
    const int cg = q - 144;
    const char *p = reinterpret_cast<const char *>(A.cols) + (size_t)cg * COL_E * sizeof(float) + 32 * lane;
    const size_t st = N_COL * COL_E * sizeof(float);
    float s = 0.0f;
    walk(A.ntile, p, st, p + 16, st, [&](int4 a, int4 b) {
      s += __int_as_float(a.x);
      s += __int_as_float(a.y);
      s += __int_as_float(a.z);
      s += __int_as_float(a.w);
      s += __int_as_float(b.x);
      s += __int_as_float(b.y);
      s += __int_as_float(b.z);
      s += __int_as_float(b.w);
    });
    const float s0 = __shfl(s, r16), s1 = __shfl(s, 16 + r16), s2 = __shfl(s, 32 + r16), s3 = __shfl(s, 48 + r16);
    const float sum = (s0 + s1) + (s2 + s3);
    const int base = cg < CD1 ? OB0 + 16 * cg : cg < CD2 ? OB1 + 16 * (cg - CD1) : cg < CDY ? OB2 + 16 * (cg - CD2) : OB3;
    if (g == 0 && (cg < CDY || r16 < NOUT)) take_grad<ADAM>(A, base + r16, sum);
  } else {
    float l = 0.0f;
    for (int t = lane; t < A.ntile; t += 64) l += A.tloss[t];
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
    if (lane == 0) *A.loss = l;
  }
}

}  // namespace sg
}  // namespace fvm
