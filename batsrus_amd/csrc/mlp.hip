// mlp.hip -- training and inference of the face-flux surrogate network on
// gfx950 matrix cores (see mlp.hpp for the network and operand layouts).
//
// Training step on a minibatch of B rows (all kernels hand-written):
//   k_train_rows   a wave takes 16 rows forward and back in registers: each
//                  layer's accumulators, through SiLU and BF16, are the next
//                  layer's MFMA operand in both directions.  It leaves every
//                  layer's activations and dZ as the operands of the weight
//                  gradient, and the per-row squared errors.
//   k_train_wgrad  dW_l = A_{l-1}^T dZ_l and db_l of a chunk of rows, all
//                  layers, straight from those operands
//   k_train_update sum the chunks in a fixed order, Adam on the FP32 master
//                  weights, refresh the BF16 operand copies
// Every reduction has a fixed order, so a training run is deterministic.
// Inference (k_infer) keeps all 58 KiB of fragment-ordered BF16 weights in
// LDS and pushes 16-row tiles through the four layers per wavefront.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/bats_hip.h"
#include "mlp.hpp"
#include "mlp_host.hpp"

using namespace bats::mlp;

namespace {

// ---- training step ------------------------------------------------------
// Operands of the weight gradient.  Its MFMAs sum over rows, so a lane needs
// one feature at several rows, while a row's own chain holds one row at
// several features.  The matrix cores turn the one into the other: an
// activation fragment as the A operand times a unit matrix gives its 16 x 16
// blocks with a lane holding feature l%16 at rows 4 (l/16) .. +3, exactly
// (each sum has one term).  A 16-row tile leaves NTB blocks of 64 lanes x 4
// values; two consecutive tiles make a 32-row operand.
constexpr int TB_A0 = 0, TB_A1 = 1, TB_A2 = 9, TB_A3 = 17;   // X, A1, A2, A3
constexpr int TB_Z1 = 21, TB_Z2 = 29, TB_Z3 = 37, TB_Z4 = 41; // dZ1..dZ3, dY
constexpr int NTB = 42;
constexpr int kTrainThreads = 512, kTrainWaves = kTrainThreads / 64;

struct TrainArgs {
  const __bf16 *frag, *bfrag;  // weights, fragment order
  const float *w;              // flat FP32 parameters (biases)
  const float *X, *T;          // samples: inputs and targets
  const float *J;              // target weights or null
  float invMeanJ;
  const float *scale;          // targets are divided by scale[j] (or null)
  const int *idx;              // rows of the minibatch (null: 0 .. B-1);
  long perEpoch;               // step q takes idx[(q % perEpoch) * B ...]
  long *step;                  // [0] this step's number, copied to [1]
  int B;
  bf16x4 *ops;                 // [tile][NTB][64]
  float *rowErr;
};

// One pass instead of a matrix product per layer and direction: at 65,536
// rows a training step (this, k_train_wgrad, k_train_update) takes 34 + 26 +
// 8 us where 17 kernels with the activations in memory between them took
// 560 us.  Bound by the vector unit (two transcendentals and about 20
// instructions per activation for SiLU, its derivative and the roundings)
// and by the 21.5 KB per tile it stores (88 MB, 18 us at the card's copy
// rate); the weights of both directions stay in LDS (110 KiB, one workgroup
// per CU, two waves per SIMD).
__global__ void __launch_bounds__(kTrainThreads)
k_train_rows(TrainArgs a) {
  __shared__ __attribute__((aligned(16))) __bf16 sW[NFRAG];
  __shared__ __attribute__((aligned(16))) __bf16 sB[NBFRAG];
  __shared__ float sBias[NBIAS];
  for (int t = threadIdx.x; t < NFRAG / 8; t += kTrainThreads)
    reinterpret_cast<bf16x8 *>(sW)[t] =
        reinterpret_cast<const bf16x8 *>(a.frag)[t];
  for (int t = threadIdx.x; t < NBFRAG / 8; t += kTrainThreads)
    reinterpret_cast<bf16x8 *>(sB)[t] =
        reinterpret_cast<const bf16x8 *>(a.bfrag)[t];
  load_biases(a.w, sBias);
  __syncthreads();
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const bf16x8 *W = reinterpret_cast<const bf16x8 *>(sW) + lane;
  const bf16x8 *V = reinterpret_cast<const bf16x8 *>(sB) + lane;
  const long q = a.step ? a.step[0] : 0;
  if (a.step && blockIdx.x == 0 && threadIdx.x == 0) a.step[1] = q;
  const int *idx = a.idx ? a.idx + (q % a.perEpoch) * a.B : nullptr;
  // unit blocks in the slot orders of frag_k: natural (the inputs), and the
  // two 16-feature halves of an accumulator fragment
  bf16x8 unitX, unit[2];
#pragma unroll
  for (int t = 0; t < 8; t++) {
    unitX[t] = (__bf16)(8 * g + t == r ? 1.f : 0.f);
    unit[0][t] = (__bf16)(t < 4 && 4 * g + t == r ? 1.f : 0.f);
    unit[1][t] = (__bf16)(t >= 4 && 4 * g + t - 4 == r ? 1.f : 0.f);
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // an even number of tiles: two make an operand of k_train_wgrad
  const int nTile = (a.B + 31) / 32 * 2;
  for (int tile = blockIdx.x * kTrainWaves + (threadIdx.x >> 6); tile < nTile;
       tile += gridDim.x * kTrainWaves) {
    const int row = tile * 16 + r;
    const bool ok = row < a.B;
    const long s = ok ? (idx ? idx[row] : row) : 0;
    bf16x4 *ops = a.ops + (long)tile * NTB * 64 + lane;
    auto turn = [&](bf16x8 x, bf16x8 u, int block) {
      const f32x4 d = mfma(x, u, zero);
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = (__bf16)d[i];
      ops[block * 64] = o;
    };
    auto turn2 = [&](bf16x8 x, int block) {
      turn(x, unit[0], block);
      turn(x, unit[1], block + 1);
    };
    bf16x8 x;
#pragma unroll
    for (int t = 0; t < 8; t++)
      x[t] = (ok && g < 2) ? (__bf16)a.X[s * 16 + 8 * g + t] : (__bf16)0.f;
    turn(x, unitX, TB_A0);
    // forward: z = W^T a + b, a' = bf16(silu(z)); the derivative silu'(z)
    // of every unit stays in registers for the way back
    f32x4 acc[8], d1[8], d2[8], d3[4];
    bf16x8 f[4];
    auto act = [&](f32x4 *d, const float *b, int nb2, bf16x8 *o, int block) {
#pragma unroll
      for (int kb = 0; kb < nb2; kb++) {
        bf16x8 v;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int nb = 2 * kb + h;
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float z = acc[nb][i] + b[nb * 16 + 4 * g + i];
            const float sg = sigmoid(z);
            v[4 * h + i] = (__bf16)(z * sg);
            d[nb][i] = sg * (1.0f + z * (1.0f - sg));
          }
        }
        o[kb] = v;
        turn2(v, block + 2 * kb);
      }
    };
#pragma unroll
    for (int nb = 0; nb < 8; nb++) acc[nb] = mfma(W[(FT0 + nb) * 64], x, zero);
    act(d1, sBias + CB1, 4, f, TB_A1);
#pragma unroll
    for (int nb = 0; nb < 8; nb++) {
      acc[nb] = zero;
#pragma unroll
      for (int kb = 0; kb < 4; kb++)
        acc[nb] = mfma(W[(FT1 + nb * 4 + kb) * 64], f[kb], acc[nb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    act(d2, sBias + CB2, 4, f, TB_A2);
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      acc[nb] = zero;
#pragma unroll
      for (int kb = 0; kb < 4; kb++)
        acc[nb] = mfma(W[(FT2 + nb * 4 + kb) * 64], f[kb], acc[nb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    act(d3, sBias + CB3, 2, f, TB_A3);
    f32x4 y = mfma(W[(FT3 + 0) * 64], f[0], zero);
    y = mfma(W[(FT3 + 1) * 64], f[1], y);
    // loss (1/(8B)) sum_r W_r |Y_r - T_r|^2: the error of a row summed over
    // its outputs in order (lanes g = 0, then g = 1), and dY
    bf16x8 z4 = {};
    float dj[4], sq = 0.f;
    const float wr = (a.J && ok) ? a.J[s] * a.invMeanJ : 1.0f;
    const float sc = 2.0f * wr / (8.0f * (float)a.B);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int n = 4 * g + i;
      float t = (ok && g < 2) ? a.T[s * 8 + n] : 0.f;
      if (a.scale && g < 2) t = t / a.scale[n];
      dj[i] = (ok && g < 2) ? y[i] + sBias[CB4 + (g < 2 ? n : 0)] - t : 0.f;
      z4[i] = (__bf16)(sc * dj[i]);
    }
    if (g == 0)
#pragma unroll
      for (int i = 0; i < 4; i++) sq += dj[i] * dj[i];
    const float first = __shfl(sq, r, 64);
    if (g == 1 && ok) {
      sq = first;
#pragma unroll
      for (int i = 0; i < 4; i++) sq += dj[i] * dj[i];
      a.rowErr[row] = wr * sq;
    }
    turn(z4, unit[0], TB_Z4);
    // back: dZ = bf16((W dZ') silu'(z))
    auto back = [&](const f32x4 *d, int nb2, bf16x8 *o, int block) {
#pragma unroll
      for (int kb = 0; kb < nb2; kb++) {
        bf16x8 v;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            v[4 * h + i] = (__bf16)(acc[2 * kb + h][i] * d[2 * kb + h][i]);
        o[kb] = v;
        turn2(v, block + 2 * kb);
      }
    };
#pragma unroll
    for (int mb = 0; mb < 4; mb++) acc[mb] = mfma(V[(BT3 + mb) * 64], z4, zero);
    back(d3, 2, f, TB_Z3);
#pragma unroll
    for (int mb = 0; mb < 8; mb++) {
      acc[mb] = zero;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
        acc[mb] = mfma(V[(BT2 + mb * 2 + kb) * 64], f[kb], acc[mb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    back(d2, 4, f, TB_Z2);
#pragma unroll
    for (int mb = 0; mb < 8; mb++) {
      acc[mb] = zero;
#pragma unroll
      for (int kb = 0; kb < 4; kb++)
        acc[mb] = mfma(V[(BT1 + mb * 4 + kb) * 64], f[kb], acc[mb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    back(d1, 4, f, TB_Z1);
  }
}

// Weight and bias gradients of a chunk of rows (blockIdx.x): the four waves
// share the 108 weight tiles and the 21 bias tiles (a unit row of ones times
// dZ); every operand is 512 contiguous bytes per 16 rows, read once per wave
// that needs it (96 KB per 32 rows and workgroup, 42 KB of it distinct).
// Bound by reading them: 26 us for 88 MB at 65,536 rows.
__global__ void __launch_bounds__(256)
k_train_wgrad(const bf16x4 *ops, int nPair, int perChunk, float *partial,
              long *step) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wv = threadIdx.x >> 6;
  if (step && blockIdx.x == 0 && threadIdx.x == 0) step[0] = step[1] + 1;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 w1[2], w2[2][8], w3[2][4], w4 = zero, b1[2], b2[2], b3 = zero, b4 = zero;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    w1[i] = b1[i] = b2[i] = zero;
    for (int n = 0; n < 8; n++) w2[i][n] = zero;
    for (int n = 0; n < 4; n++) w3[i][n] = zero;
  }
  bf16x8 ones;
#pragma unroll
  for (int t = 0; t < 8; t++) ones[t] = (__bf16)1.0f;
  const int p0 = blockIdx.x * perChunk;
  const int p1 = p0 + perChunk < nPair ? p0 + perChunk : nPair;
  for (int p = p0; p < p1; p++) {
    const bf16x4 *o = ops + (long)p * 2 * NTB * 64 + lane;
    auto op = [&](int block) {
      const bf16x4 lo = o[block * 64], hi = o[(NTB + block) * 64];
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    const bf16x8 x = op(TB_A0);
    bf16x8 z[8], c[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      c[i] = op(TB_Z1 + 2 * wv + i);
      w1[i] = mfma(x, c[i], w1[i]);
      b1[i] = mfma(ones, c[i], b1[i]);
    }
#pragma unroll
    for (int n = 0; n < 8; n++) z[n] = op(TB_Z2 + n);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      c[i] = op(TB_A1 + 2 * wv + i);
#pragma unroll
      for (int n = 0; n < 8; n++) w2[i][n] = mfma(c[i], z[n], w2[i][n]);
    }
    // (a register array indexed by the wave would go to memory)
    b2[0] = mfma(ones, op(TB_Z2 + 2 * wv), b2[0]);
    b2[1] = mfma(ones, op(TB_Z2 + 2 * wv + 1), b2[1]);
#pragma unroll
    for (int n = 0; n < 4; n++) z[n] = op(TB_Z3 + n);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      c[i] = op(TB_A2 + 2 * wv + i);
#pragma unroll
      for (int n = 0; n < 4; n++) w3[i][n] = mfma(c[i], z[n], w3[i][n]);
    }
    b3 = mfma(ones, op(TB_Z3 + wv), b3);
    const bf16x8 y = op(TB_Z4);
    w4 = mfma(op(TB_A3 + wv), y, w4);
    b4 = mfma(ones, y, b4);
  }
  // tile (m, n): lane holds column n = l%16, rows m = 4 (l/16) + i
  float *P = partial + (long)blockIdx.x * NPARAM;
  auto put = [&](int l, int mb, int nb, f32x4 v) {
    const int n = nb * 16 + r;
    if (n < DIM[l + 1])
#pragma unroll
      for (int i = 0; i < 4; i++)
        P[OW[l] + (mb * 16 + 4 * g + i) * DIM[l + 1] + n] = v[i];
  };
  auto putb = [&](int l, int nb, f32x4 v) {
    const int n = nb * 16 + r;
    if (g == 0 && n < DIM[l + 1]) P[OB[l] + n] = v[0];
  };
#pragma unroll
  for (int i = 0; i < 2; i++) {
    put(0, 0, 2 * wv + i, w1[i]);
    putb(0, 2 * wv + i, b1[i]);
#pragma unroll
    for (int n = 0; n < 8; n++) put(1, 2 * wv + i, n, w2[i][n]);
    putb(1, 2 * wv + i, b2[i]);
#pragma unroll
    for (int n = 0; n < 4; n++) put(2, 2 * wv + i, n, w3[i][n]);
  }
  putb(2, wv, b3);
  put(3, wv, 0, w4);
  if (wv == 0) putb(3, 0, b4);
}

struct UpdateArgs {
  const float *partial;  // [chunk][NPARAM]
  int nChunk;
  float *grad;
  int adam;              // 0: the gradient only
  float *w, *m, *v;
  __bf16 *frag, *bfrag;  // BF16 operand copies of the weights
  float b1, b2, eps;
  // lr, 1 - b1^t, 1 - b2^t of step step[1] are sched[3 * step[1] + 0..2]
  const float *sched;
  const long *step;
};

// gradient = sum of the chunks' partials (eight runs of chunks, each in
// order, then their sums in order), and Adam (Kingma & Ba 2015) on the FP32
// master weights.  Bound by reading the partials (28 MB at 256 chunks): 128
// parameters per workgroup, 16-byte loads, eight of them in flight.
constexpr int kUpdateParams = 128;
static_assert(NPARAM % 4 == 0, "partials are read four at a time");
__global__ void __launch_bounds__(256) k_train_update(UpdateArgs a) {
  __shared__ float sSum[8][kUpdateParams];
  const int c = 4 * (threadIdx.x & 31), run = threadIdx.x >> 5;
  const int p4 = blockIdx.x * kUpdateParams + c;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  const int n0 = a.nChunk * run / 8, n1 = a.nChunk * (run + 1) / 8;
  if (p4 < NPARAM) {
#pragma unroll 8
    for (int n = n0; n < n1; n++)
      s += *reinterpret_cast<const f32x4 *>(a.partial + (long)n * NPARAM + p4);
  }
  *reinterpret_cast<f32x4 *>(&sSum[run][c]) = s;
  __syncthreads();
  const int p = blockIdx.x * kUpdateParams + threadIdx.x;
  if (threadIdx.x >= kUpdateParams || p >= NPARAM) return;
  float g = 0.f;
#pragma unroll
  for (int q = 0; q < 8; q++) g += sSum[q][threadIdx.x];
  a.grad[p] = g;
  if (!a.adam) return;
  const float *q = a.sched + 3 * a.step[1];
  const float lr = q[0], bc1 = q[1], bc2 = q[2];
  const float m = a.b1 * a.m[p] + (1.f - a.b1) * g;
  const float v = a.b2 * a.v[p] + (1.f - a.b2) * g * g;
  a.m[p] = m;
  a.v[p] = v;
  const float w = a.w[p] - lr * (m / bc1) / (sqrtf(v / bc2) + a.eps);
  a.w[p] = w;
  int l = 0;
  while (l + 1 < NL && p >= OW[l + 1]) l++;
  if (p >= OB[l]) return;  // a bias
  const int k = (p - OW[l]) / DIM[l + 1], n = (p - OW[l]) % DIM[l + 1];
  a.frag[frag_pos(l, k, n)] = (__bf16)w;
  if (l > 0) a.bfrag[bfrag_pos(l, k, n)] = (__bf16)w;
}

// per-block partial sums of squares of the 8 target columns (fixed order)
__global__ void k_col_sumsq(const float *T, long n, double *partial) {
  __shared__ double s[256][8];
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (long r = blockIdx.x * 256L + threadIdx.x; r < n; r += gridDim.x * 256L)
    for (int j = 0; j < 8; j++) acc[j] += (double)T[r * 8 + j] * T[r * 8 + j];
  for (int j = 0; j < 8; j++) s[threadIdx.x][j] = acc[j];
  __syncthreads();
  if (threadIdx.x < 8) {
    double t = 0.0;
    for (int q = 0; q < 256; q++) t += s[q][threadIdx.x];
    partial[blockIdx.x * 8 + threadIdx.x] = t;
  }
}

// last layer times (mul) or over (div) the per-output scale
__global__ void k_scale_last(float *w, const float *scale, int div) {
  const int t = threadIdx.x;  // 64*8 + 8 entries
  if (t < 64 * 8) {
    const int n = t % 8;
    w[OW4 + t] = div ? w[OW4 + t] / scale[n] : w[OW4 + t] * scale[n];
  } else if (t < 64 * 8 + 8) {
    const int n = t - 64 * 8;
    w[OB4 + n] = div ? w[OB4 + n] / scale[n] : w[OB4 + n] * scale[n];
  }
}

// fragment-ordered, zero-padded BF16 weights of both directions
__global__ void k_pack_frag(const float *w, __bf16 *frag, __bf16 *bfrag) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = (t % TILE) / 8, e = t % 8;
  if (t < NFRAG) {
    const int tile = t / TILE;
    int l = 0;
    while (l + 1 < NL && tile >= FT[l + 1]) l++;
    const int lt = tile - FT[l], nKb = KP[l] / 32;
    const int nb = lt / nKb, kb = lt % nKb;
    const int k = frag_k(l, kb, lane >> 4, e), n = nb * 16 + (lane & 15);
    const float v = (k < DIM[l] && n < DIM[l + 1])
                        ? w[OW[l] + k * DIM[l + 1] + n] : 0.0f;
    frag[t] = (__bf16)v;
  }
  if (t < NBFRAG) {
    const int tile = t / TILE;
    int l = 1;
    while (l + 1 < NL && tile >= BT[l + 1]) l++;
    const int lt = tile - BT[l], nKb = l == 3 ? 1 : DIM[l + 1] / 32;
    const int k = (lt / nKb) * 16 + (lane & 15);
    const int n = frag_k(1, lt % nKb, lane >> 4, e);
    const float v = n < DIM[l + 1] ? w[OW[l] + k * DIM[l + 1] + n] : 0.0f;
    bfrag[t] = (__bf16)v;
  }
}

}  // namespace

namespace {

// Bound by the vector unit (SiLU) on many rows and on few by the copy of the
// weights into LDS, after which each wave has one pair of tiles: 65,536 rows
// in 15.8 us, as with 16 waves of one tile each at 64 VGPRs (15.7 us), which
// spill with the pair that the surrogate's faces need.
__global__ void __launch_bounds__(kInferThreads, 4)
k_infer(const __bf16 *frag, const float *w, const float *X, float *Y,
        int rows) {
  __shared__ __attribute__((aligned(16))) __bf16 sW[NFRAG];
  __shared__ float sBias[NBIAS];
  for (int t = threadIdx.x; t < NFRAG / 8; t += kInferThreads)
    reinterpret_cast<bf16x8 *>(sW)[t] = reinterpret_cast<const bf16x8 *>(frag)[t];
  load_biases(w, sBias);
  __syncthreads();
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int nPair = (rows - 1) / 32 + 1;
  for (int pair = blockIdx.x * kInferWaves + (threadIdx.x >> 6); pair < nPair;
       pair += gridDim.x * kInferWaves) {
    bf16x8 x[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int row = pair * 32 + 16 * h + r;
#pragma unroll
      for (int t = 0; t < 8; t++)
        x[h][t] = (g < 2 && row < rows)
                      ? (__bf16)X[(long)row * 16 + 8 * g + t] : (__bf16)0.f;
    }
    infer_tiles<2>(sW, sBias, x, [&](int h, f32x4 y) {
      const int row = pair * 32 + 16 * h + r;
      if (g < 2 && row < rows)
        *reinterpret_cast<f32x4 *>(Y + (long)row * 8 + 4 * g) = y;
    });
  }
}

// the inputs of listed samples, one value per thread
__global__ void __launch_bounds__(256)
k_gather_inputs(const float *X, const int *idx, int rows, float *Xo) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t < rows * 16L) Xo[t] = X[idx[t / 16] * 16L + t % 16];
}

// The held-out errors: for output j = thread % 8 the sums over the listed
// samples of (w (Y - T))^2, (w T + B)^2 and (w T)^2 in FP64, w the sample's
// jump norm (predicted flux B + w Y against the full flux B + w T); per
// workgroup part[3][8], summed on the host in their order.  Bound by its
// reads (100 bytes per sample).  With the gathered samples copied to the host
// and summed there, a call that trains nothing on 700,001 samples took
// 2.9 ms, 1.9 ms so (four epochs of them 10.7 -> 9.8 ms).
constexpr int kErrGrid = 256;
__global__ void __launch_bounds__(256)
k_hold_err(const float *Y, const float *T, const float *B, const float *J,
           const int *idx, int rows, double *part) {
  __shared__ double sSum[4][3][8];
  const int j = threadIdx.x & 7;
  double sum[3] = {0.0, 0.0, 0.0};
  for (long r = blockIdx.x * 32L + threadIdx.x / 8; r < rows;
       r += gridDim.x * 32L) {
    const long s = idx[r];
    const double w = J[s], t = T[s * 8 + j];
    const double d = w * ((double)Y[r * 8 + j] - t);
    const double wt = w * t, f = wt + (double)B[s * 8 + j];
    sum[0] += d * d;
    sum[1] += f * f;
    sum[2] += wt * wt;
  }
#pragma unroll
  for (int q = 0; q < 3; q++) {
#pragma unroll
    for (int o = 8; o < 64; o *= 2) sum[q] += __shfl_xor(sum[q], o);
    if ((threadIdx.x & 63) < 8) sSum[threadIdx.x / 64][q][j] = sum[q];
  }
  __syncthreads();
  if (threadIdx.x < 24) {
    const double *p = &sSum[0][0][0] + threadIdx.x;
    part[blockIdx.x * 24 + threadIdx.x] = ((p[0] + p[24]) + p[48]) + p[72];
  }
}

}  // namespace

// =====================================================================
// host side: the model object
// =====================================================================
struct bats_mlp {
  hipStream_t stream;
  int dev;                   // device the model (and its stream) lives on
  float *w, *m, *v, *grad;   // FP32 master weights, Adam moments, gradient
  __bf16 *frag, *bfrag;      // fragment-ordered BF16 weights, both directions
  int step;                  // Adam steps taken
  int fragStale;             // frag, bfrag lag w (repacked before use)
  // training buffers for a minibatch of cap rows
  int cap;
  bf16x4 *ops;               // weight-gradient operands
  float *X, *T, *rowErr, *partial;
  // dataset (device): inputs (n x 16), targets (n x 8) and the baseline
  // flux the target corrects (n x 8, zero unless harvested), FP32
  float *dataX, *dataT, *dataB, *dataJ;  // + weight of each sample's target
  long nData, capData;
  // pinned memory for an epoch's permutation, and the event of its copy
  int *order;
  size_t orderCap;
  hipEvent_t orderTaken;
};

#define MCHK(x)                                                          \
  do {                                                                   \
    hipError_t e_ = (x);                                                 \
    if (e_ != hipSuccess) {                                              \
      fprintf(stderr, "bats_mlp: %s failed: %s (%s:%d)\n", #x,           \
              hipGetErrorString(e_), __FILE__, __LINE__);                \
      return e_ == hipErrorOutOfMemory ? BATS_ENOMEM : BATS_EHIP;        \
    }                                                                    \
  } while (0)

// row pairs of tiles (32 rows) per weight-gradient chunk: 256 chunks, one
// per CU, up to 256 rows each
static int chunk_pairs(int nPair) {
  const int n = (nPair + 255) / 256;
  return n < 8 ? n : 8;
}

// ---- staging memory of bats_mlp_forward_noalloc -----------------------
// bats_mlp_forward allocates device buffers for the rows it stages in and
// out on every call; the no-allocation variant stages them through this
// fixed array instead: the inputs (BATS_MLP_NOALLOC_ROWS x 16 floats), then
// the outputs (BATS_MLP_NOALLOC_ROWS x 8), 6 MiB in all.  Each device that
// runs the library holds its own copy until the process ends.  In host code
// the array's name is only a stand-in; its device address on each device
// comes from hipGetSymbolAddress, taken once per device in bats_mlp_create
// with that device current, and only that address is passed to the copies
// and kernels.
static __device__ __align__(256) float
    scratch[(size_t)BATS_MLP_NOALLOC_ROWS * (BATS_MLP_NIN + BATS_MLP_NOUT)];
static const int kMaxDevices = 64;
static std::mutex g_scratchLock;
static float *g_scratchDev[kMaxDevices];  // scratch's address per device

// record the address of this device's copy of scratch (the current device
// must be dev)
static int noalloc_setup(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return BATS_ENODEV;
  std::lock_guard<std::mutex> lock(g_scratchLock);
  if (g_scratchDev[dev]) return BATS_OK;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    fprintf(stderr, "bats_mlp: hipGetSymbolAddress(scratch) failed on "
                    "device %d: %s\n", dev, hipGetErrorString(e));
    return BATS_EHIP;
  }
  g_scratchDev[dev] = static_cast<float *>(p);
  return BATS_OK;
}

static float *noalloc_scratch(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratchLock);
  return g_scratchDev[dev];
}

static int repack(bats_mlp *m) {
  if (!m->fragStale) return BATS_OK;
  hipLaunchKernelGGL(k_pack_frag, dim3((NFRAG + 255) / 256), dim3(256), 0,
                     m->stream, m->w, m->frag, m->bfrag);
  MCHK(hipGetLastError());
  m->fragStale = 0;
  return BATS_OK;
}

extern "C" int bats_mlp_create(bats_mlp **out) {
  if (!out) return BATS_EINVAL;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return BATS_ENODEV;
  bats_mlp *m = new bats_mlp();
  memset(m, 0, sizeof *m);
  MCHK(hipGetDevice(&m->dev));
  const int st = noalloc_setup(m->dev);
  if (st) {
    delete m;
    return st;
  }
  MCHK(hipStreamCreate(&m->stream));
  MCHK(hipMalloc(&m->w, sizeof(float) * NPARAM));
  MCHK(hipMalloc(&m->m, sizeof(float) * NPARAM));
  MCHK(hipMalloc(&m->v, sizeof(float) * NPARAM));
  MCHK(hipMalloc(&m->grad, sizeof(float) * NPARAM));
  MCHK(hipMalloc(&m->frag, sizeof(__bf16) * NFRAG));
  MCHK(hipMalloc(&m->bfrag, sizeof(__bf16) * NBFRAG));
  MCHK(hipMemset(m->w, 0, sizeof(float) * NPARAM));
  MCHK(hipMemset(m->m, 0, sizeof(float) * NPARAM));
  MCHK(hipMemset(m->v, 0, sizeof(float) * NPARAM));
  MCHK(hipMemset(m->grad, 0, sizeof(float) * NPARAM));
  *out = m;
  m->fragStale = 1;
  return repack(m);
}

static void free_batch(bats_mlp *m) {
  void *p[] = {m->ops, m->X, m->T, m->rowErr, m->partial};
  for (void *q : p)
    if (q) (void)hipFree(q);
  m->ops = nullptr;
  m->X = m->T = m->rowErr = m->partial = nullptr;
  m->cap = 0;
}

extern "C" int bats_mlp_free(bats_mlp *m) {
  if (!m) return BATS_EINVAL;
  (void)hipStreamSynchronize(m->stream);
  free_batch(m);
  void *p[] = {m->w, m->m, m->v, m->grad, m->frag, m->bfrag, m->dataX, m->dataT,
               m->dataB, m->dataJ};
  for (void *q : p)
    if (q) (void)hipFree(q);
  if (m->order) (void)hipHostFree(m->order);
  if (m->orderTaken) (void)hipEventDestroy(m->orderTaken);
  (void)hipStreamDestroy(m->stream);
  delete m;
  return BATS_OK;
}

extern "C" int bats_mlp_set_params(bats_mlp *m, const float *w) {
  if (!m || !w) return BATS_EINVAL;
  MCHK(hipMemcpyAsync(m->w, w, sizeof(float) * NPARAM, hipMemcpyHostToDevice,
                      m->stream));
  MCHK(hipMemsetAsync(m->m, 0, sizeof(float) * NPARAM, m->stream));
  MCHK(hipMemsetAsync(m->v, 0, sizeof(float) * NPARAM, m->stream));
  m->step = 0;
  m->fragStale = 1;
  int st = repack(m);
  if (st) return st;
  MCHK(hipStreamSynchronize(m->stream));
  return BATS_OK;
}

extern "C" int bats_mlp_get_params(bats_mlp *m, float *w, float *grad) {
  if (!m) return BATS_EINVAL;
  MCHK(hipStreamSynchronize(m->stream));
  if (w) MCHK(hipMemcpy(w, m->w, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  if (grad)
    MCHK(hipMemcpy(grad, m->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  return BATS_OK;
}

// training buffers for a minibatch of B rows (X and T: the rows that
// bats_mlp_loss_grad takes from the host)
static int ensure_batch(bats_mlp *m, int B) {
  if (B <= m->cap) return BATS_OK;
  free_batch(m);
  const size_t b = (size_t)B;
  const int nPair = (B + 31) / 32;
  const size_t chunks = (nPair + chunk_pairs(nPair) - 1) / chunk_pairs(nPair);
  MCHK(hipMalloc(&m->ops, sizeof(bf16x4) * 2 * nPair * NTB * 64));
  MCHK(hipMalloc(&m->X, sizeof(float) * b * 16));
  MCHK(hipMalloc(&m->T, sizeof(float) * b * 8));
  MCHK(hipMalloc(&m->rowErr, sizeof(float) * b));
  // (a smaller batch may take more, smaller chunks: up to 256)
  MCHK(hipMalloc(&m->partial,
                 sizeof(float) * (chunks > 256 ? chunks : 256) * NPARAM));
  m->cap = B;
  return BATS_OK;
}

// gradient of the mean-square loss of the minibatch a describes into m->grad
// (and rowErr), and with a schedule one Adam step
static int grad_step(bats_mlp *m, TrainArgs a, const float *sched) {
  a.frag = m->frag;
  a.bfrag = m->bfrag;
  a.w = m->w;
  a.ops = m->ops;
  a.rowErr = m->rowErr;
  const int nPair = (a.B + 31) / 32, per = chunk_pairs(nPair);
  const int nChunk = (nPair + per - 1) / per;
  const int nWg = (2 * nPair + kTrainWaves - 1) / kTrainWaves;
  hipLaunchKernelGGL(k_train_rows, dim3(nWg < 256 ? nWg : 256),
                     dim3(kTrainThreads), 0, m->stream, a);
  hipLaunchKernelGGL(k_train_wgrad, dim3(nChunk), dim3(256), 0, m->stream,
                     m->ops, nPair, per, m->partial, a.step);
  UpdateArgs u;
  u.partial = m->partial;
  u.nChunk = nChunk;
  u.grad = m->grad;
  u.adam = sched != nullptr;
  u.w = m->w; u.m = m->m; u.v = m->v;
  u.frag = m->frag; u.bfrag = m->bfrag;
  u.b1 = 0.9f; u.b2 = 0.999f; u.eps = 1e-8f;
  u.sched = sched;
  u.step = a.step;
  hipLaunchKernelGGL(k_train_update,
                     dim3((NPARAM + kUpdateParams - 1) / kUpdateParams),
                     dim3(256), 0, m->stream, u);
  MCHK(hipGetLastError());
  return BATS_OK;
}

extern "C" int bats_mlp_loss_grad(bats_mlp *m, const float *X, const float *T,
                                  int B, double *Loss, float *grad) {
  if (!m || !X || !T || B <= 0) return BATS_EINVAL;
  int st = ensure_batch(m, B);
  if (st) return st;
  st = repack(m);
  if (st) return st;
  MCHK(hipMemcpyAsync(m->X, X, sizeof(float) * (size_t)B * 16,
                      hipMemcpyHostToDevice, m->stream));
  MCHK(hipMemcpyAsync(m->T, T, sizeof(float) * (size_t)B * 8,
                      hipMemcpyHostToDevice, m->stream));
  TrainArgs ta{};
  ta.X = m->X;
  ta.T = m->T;
  ta.B = B;
  st = grad_step(m, ta, nullptr);
  if (st) return st;
  std::vector<float> e(B);
  MCHK(hipMemcpyAsync(e.data(), m->rowErr, sizeof(float) * B,
                      hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  double s = 0.0;
  for (int r = 0; r < B; r++) s += e[r];
  if (Loss) *Loss = s / (8.0 * B);
  if (grad)
    MCHK(hipMemcpy(grad, m->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  return BATS_OK;
}

extern "C" int bats_mlp_forward(bats_mlp *m, const float *X, float *Y, int rows) {
  if (!m || !X || !Y || rows <= 0) return BATS_EINVAL;
  float *dX = nullptr, *dY = nullptr;
  MCHK(hipMalloc(&dX, sizeof(float) * (size_t)rows * 16));
  MCHK(hipMalloc(&dY, sizeof(float) * (size_t)rows * 8));
  MCHK(hipMemcpyAsync(dX, X, sizeof(float) * (size_t)rows * 16,
                      hipMemcpyHostToDevice, m->stream));
  int st = bats::mlp::forward_device(m, dX, dY, rows, m->stream);
  if (st == BATS_OK)
    MCHK(hipMemcpyAsync(Y, dY, sizeof(float) * (size_t)rows * 8,
                        hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  (void)hipFree(dX);
  (void)hipFree(dY);
  return st;
}

extern "C" int bats_mlp_forward_noalloc(bats_mlp *m, const float *X,
                                        float *Y, int rows) {
  if (!m || !X || !Y || rows <= 0) return BATS_EINVAL;
  if (rows > BATS_MLP_NOALLOC_ROWS) {
    fprintf(stderr, "bats_mlp_forward_noalloc: %d rows exceed the staging "
                    "limit of %d rows\n", rows, (int)BATS_MLP_NOALLOC_ROWS);
    return BATS_ELIMIT;
  }
  float *dX = noalloc_scratch(m->dev);
  if (!dX) return BATS_EHIP;
  float *dY = dX + (size_t)BATS_MLP_NOALLOC_ROWS * BATS_MLP_NIN;
  // every row written by the copy in is read, every row read by the copy
  // out is written by the kernel: nothing in scratch needs clearing
  MCHK(hipMemcpyAsync(dX, X, sizeof(float) * (size_t)rows * BATS_MLP_NIN,
                      hipMemcpyHostToDevice, m->stream));
  const int st = bats::mlp::forward_device(m, dX, dY, rows, m->stream);
  if (st == BATS_OK)
    MCHK(hipMemcpyAsync(Y, dY, sizeof(float) * (size_t)rows * BATS_MLP_NOUT,
                        hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return st;
}

int bats::mlp::forward_device(bats_mlp *m, const float *dX, float *dY,
                              int rows, hipStream_t stream) {
  if (!m || rows <= 0) return BATS_EINVAL;
  // the weights must be current on this stream
  int st = repack(m);
  if (st) return st;
  MCHK(hipStreamSynchronize(m->stream));
  const int nPair = (rows - 1) / 32 + 1;
  int grid = (nPair + kInferWaves - 1) / kInferWaves;
  if (grid > kInferGrid) grid = kInferGrid;
  hipLaunchKernelGGL(k_infer, dim3(grid), dim3(kInferThreads), 0, stream, m->frag, m->w,
                     dX, dY, rows);
  MCHK(hipGetLastError());
  return BATS_OK;
}

// ---- dataset and training loop ----------------------------------------
static int ensure_data(bats_mlp *m, long n) {
  if (n <= m->capData) return BATS_OK;
  float *x = nullptr, *t = nullptr, *b = nullptr, *jw = nullptr;
  MCHK(hipMalloc(&x, sizeof(float) * (size_t)n * 16));
  MCHK(hipMalloc(&t, sizeof(float) * (size_t)n * 8));
  MCHK(hipMalloc(&b, sizeof(float) * (size_t)n * 8));
  MCHK(hipMalloc(&jw, sizeof(float) * (size_t)n));
  if (m->nData > 0) {
    MCHK(hipMemcpyAsync(x, m->dataX, sizeof(float) * (size_t)m->nData * 16,
                        hipMemcpyDeviceToDevice, m->stream));
    MCHK(hipMemcpyAsync(t, m->dataT, sizeof(float) * (size_t)m->nData * 8,
                        hipMemcpyDeviceToDevice, m->stream));
    MCHK(hipMemcpyAsync(b, m->dataB, sizeof(float) * (size_t)m->nData * 8,
                        hipMemcpyDeviceToDevice, m->stream));
    MCHK(hipMemcpyAsync(jw, m->dataJ, sizeof(float) * (size_t)m->nData,
                        hipMemcpyDeviceToDevice, m->stream));
  }
  MCHK(hipStreamSynchronize(m->stream));
  if (m->dataX) (void)hipFree(m->dataX);
  if (m->dataT) (void)hipFree(m->dataT);
  if (m->dataB) (void)hipFree(m->dataB);
  if (m->dataJ) (void)hipFree(m->dataJ);
  m->dataX = x;
  m->dataT = t;
  m->dataB = b;
  m->dataJ = jw;
  m->capData = n;
  return BATS_OK;
}

int bats::mlp::reserve_data(bats_mlp *m, long nMore, float **X, float **T,
                            float **B, float **J) {
  int st = ensure_data(m, m->nData + nMore);
  if (st) return st;
  *X = m->dataX + (size_t)m->nData * 16;
  *T = m->dataT + (size_t)m->nData * 8;
  *B = m->dataB + (size_t)m->nData * 8;
  *J = m->dataJ + (size_t)m->nData;
  return BATS_OK;
}

__global__ void k_fill(float *x, long n, float v) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t < n) x[t] = v;
}

void bats::mlp::commit_data(bats_mlp *m, long nAdded) { m->nData += nAdded; }

bats::mlp::Weights bats::mlp::weights(bats_mlp *m) {
  (void)repack(m);
  (void)hipStreamSynchronize(m->stream);  // weights current
  return Weights{m->frag, m->w};
}

extern "C" int bats_mlp_set_data(bats_mlp *m, const float *X, const float *T,
                                 long n) {
  if (!m || n < 0 || (n > 0 && (!X || !T))) return BATS_EINVAL;
  m->nData = 0;
  int st = ensure_data(m, n);
  if (st) return st;
  if (n > 0) {
    MCHK(hipMemcpy(m->dataX, X, sizeof(float) * (size_t)n * 16,
                   hipMemcpyHostToDevice));
    MCHK(hipMemcpy(m->dataT, T, sizeof(float) * (size_t)n * 8,
                   hipMemcpyHostToDevice));
    MCHK(hipMemset(m->dataB, 0, sizeof(float) * (size_t)n * 8));
    hipLaunchKernelGGL(k_fill, dim3((n + 255) / 256), dim3(256), 0, m->stream,
                       m->dataJ, n, 1.0f);
    MCHK(hipStreamSynchronize(m->stream));
  }
  m->nData = n;
  return BATS_OK;
}

extern "C" int bats_mlp_get_data(bats_mlp *m, long *n, float *X, float *T,
                                 float *B) {
  if (!m) return BATS_EINVAL;
  MCHK(hipStreamSynchronize(m->stream));
  if (n) *n = m->nData;
  if (X && m->nData)
    MCHK(hipMemcpy(X, m->dataX, sizeof(float) * (size_t)m->nData * 16,
                   hipMemcpyDeviceToHost));
  if (T && m->nData)
    MCHK(hipMemcpy(T, m->dataT, sizeof(float) * (size_t)m->nData * 8,
                   hipMemcpyDeviceToHost));
  if (B && m->nData)
    MCHK(hipMemcpy(B, m->dataB, sizeof(float) * (size_t)m->nData * 8,
                   hipMemcpyDeviceToHost));
  return BATS_OK;
}

// splitmix64: the seeded shuffles of the training loop
static uint64_t splitmix64(uint64_t &s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static void shuffle(std::vector<int> &v, uint64_t &s) {
  for (size_t i = v.size(); i > 1; i--) {
    const size_t j = splitmix64(s) % i;
    std::swap(v[i - 1], v[j]);
  }
}

// pinned memory for a permutation of n samples (none where it cannot be had,
// without leaving the refusal behind as the thread's last error)
static int ensure_order(bats_mlp *m, size_t n) {
  if (!m->orderTaken)
    MCHK(hipEventCreateWithFlags(&m->orderTaken, hipEventDisableTiming));
  if (n <= m->orderCap) return BATS_OK;
  if (m->order) (void)hipHostFree(m->order);
  m->order = nullptr;
  m->orderCap = 0;
  if (hipHostMalloc(&m->order, sizeof(int) * n, 0) == hipSuccess) {
    m->orderCap = n;
  } else {
    (void)hipGetLastError();
    m->order = nullptr;
  }
  return BATS_OK;
}

extern "C" int bats_mlp_train(bats_mlp *m, int nEpoch, int Batch, double Lr0,
                              double HoldFrac, int Flags,
                              unsigned long long Seed, double *TrainLoss,
                              double *HeldOutRelErr_V) {
  const bool Standardize = (Flags & BATS_MLP_STANDARDIZE) != 0;
  const bool JumpWeight = (Flags & BATS_MLP_JUMP_WEIGHT) != 0;
  const bool UseGraph = (Flags & BATS_MLP_NO_GRAPH) == 0;
  if (Flags & ~(BATS_MLP_STANDARDIZE | BATS_MLP_JUMP_WEIGHT | BATS_MLP_NO_GRAPH))
    return BATS_EINVAL;
  if (!m || nEpoch < 0 || Batch <= 0 || !(Lr0 >= 0.0) || HoldFrac < 0.0 ||
      HoldFrac >= 1.0 || m->nData < 2)
    return BATS_EINVAL;
  const long n = m->nData;
  if (n > 0x7fffffffL) return BATS_EINVAL;
  const long nHold = (long)(HoldFrac * (double)n);
  const long nTrain = n - nHold;
  if (nTrain < 1) return BATS_EINVAL;
  const int B = (int)(Batch < nTrain ? Batch : nTrain);
  int st = ensure_batch(m, B);
  if (st) return st;
  // seeded split: the first nTrain of a permutation train, the rest are held
  uint64_t s = Seed;
  std::vector<int> perm(n);
  for (long i = 0; i < n; i++) perm[i] = (int)i;
  shuffle(perm, s);
  std::vector<int> train(perm.begin(), perm.begin() + nTrain);
  std::vector<int> hold(perm.begin() + nTrain, perm.end());
  int *dIdx = nullptr;
  MCHK(hipMalloc(&dIdx, sizeof(int) * (size_t)(nTrain > nHold ? nTrain : nHold)));
  // optionally standardize the targets: each output divided by its RMS
  // over the samples while training; the last layer carries the scale in
  // between calls, so the network always outputs physical targets
  float *dScale = nullptr;
  MCHK(hipMalloc(&dScale, sizeof(float) * 8));
  {
    const float one[8] = {1, 1, 1, 1, 1, 1, 1, 1};
    MCHK(hipMemcpy(dScale, one, sizeof one, hipMemcpyHostToDevice));
  }
  if (Standardize) {
    const int nb = 256;
    double *dPart = nullptr;
    MCHK(hipMalloc(&dPart, sizeof(double) * nb * 8));
    hipLaunchKernelGGL(k_col_sumsq, dim3(nb), dim3(256), 0, m->stream,
                       m->dataT, n, dPart);
    std::vector<double> part(nb * 8);
    MCHK(hipMemcpyAsync(part.data(), dPart, sizeof(double) * part.size(),
                        hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    (void)hipFree(dPart);
    float sc[8];
    for (int j = 0; j < 8; j++) {
      double t = 0.0;
      for (int q = 0; q < nb; q++) t += part[q * 8 + j];
      const double rms = sqrt(t / (double)n);
      sc[j] = rms > 0.0 ? (float)rms : 1.0f;
    }
    MCHK(hipMemcpyAsync(dScale, sc, sizeof sc, hipMemcpyHostToDevice,
                        m->stream));
    hipLaunchKernelGGL(k_scale_last, dim3(1), dim3(64 * 8 + 8), 0, m->stream,
                       m->w, dScale, 1);
    m->fragStale = 1;
  }
  st = repack(m);
  if (st) return st;
  // jump weights: each sample's squared error weighted by its jump norm
  // over the mean jump norm of the training samples
  float invMeanJ = 1.0f;
  if (JumpWeight) {
    std::vector<float> hj(n);
    MCHK(hipStreamSynchronize(m->stream));
    MCHK(hipMemcpy(hj.data(), m->dataJ, sizeof(float) * n,
                   hipMemcpyDeviceToHost));
    double sj = 0.0;
    for (long i = 0; i < nTrain; i++) sj += hj[train[i]];
    invMeanJ = sj > 0.0 ? (float)((double)nTrain / sj) : 1.0f;
  }
  const long stepsPerEpoch = nTrain / B;
  const long total = stepsPerEpoch * nEpoch;
  double lastLoss = 0.0;
  std::vector<float> e(B);
  if (total > 0) {
    // the learning rate (cosine decay) and Adam's bias corrections of every
    // step, read on the device: one training step is captured once in a
    // hipGraph and replayed (the minibatch of step q is rows q % perEpoch of
    // the epoch's permutation; a device counter advances after each step)
    std::vector<float> sched(3 * (size_t)total);
    for (long q = 0; q < total; q++) {
      const double lr = Lr0 * 0.5 * (1.0 + cos(M_PI * (double)q / (double)total));
      const float t = (float)(m->step + q + 1);
      sched[3 * q] = (float)lr;
      sched[3 * q + 1] = 1.f - powf(0.9f, t);
      sched[3 * q + 2] = 1.f - powf(0.999f, t);
    }
    float *dSched = nullptr;
    long *dStep = nullptr;
    MCHK(hipMalloc(&dSched, sizeof(float) * sched.size()));
    MCHK(hipMalloc(&dStep, 2 * sizeof(long)));
    MCHK(hipMemcpyAsync(dSched, sched.data(), sizeof(float) * sched.size(),
                        hipMemcpyHostToDevice, m->stream));
    MCHK(hipMemsetAsync(dStep, 0, 2 * sizeof(long), m->stream));
    // one training step: the same kernels whether captured or launched
    TrainArgs ta{};
    ta.X = m->dataX;
    ta.T = m->dataT;
    ta.J = JumpWeight ? m->dataJ : nullptr;
    ta.invMeanJ = invMeanJ;
    ta.scale = dScale;
    ta.idx = dIdx;
    ta.perEpoch = stepsPerEpoch;
    ta.step = dStep;
    ta.B = B;
    auto one_step = [&]() { return grad_step(m, ta, dSched); };
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    if (UseGraph) {
      MCHK(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
      st = one_step();
      const hipError_t ec = hipStreamEndCapture(m->stream, &graph);
      if (st == BATS_OK && ec == hipSuccess)
        st = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess
                 ? BATS_OK : BATS_EHIP;
      else if (st == BATS_OK)
        st = BATS_EHIP;
      if (graph) (void)hipGraphDestroy(graph);
    }
    // The permutation goes through the model's pinned memory, whose copy has
    // been read before the next epoch writes it (the event is behind the copy
    // alone: an epoch's steps run beside the next shuffle).  Without pinned
    // memory the copy is waited for before the shuffle (four epochs of
    // 700,001 samples 0.4 of 10 ms longer).
    if (st == BATS_OK) st = ensure_order(m, train.size());
    for (int ep = 0; st == BATS_OK && ep < nEpoch; ep++) {
      if (ep > 0 && !m->order &&
          hipEventSynchronize(m->orderTaken) != hipSuccess) {
        st = BATS_EHIP;
        break;
      }
      shuffle(train, s);
      const int *from = train.data();
      if (m->order) {
        if (ep > 0 && hipEventSynchronize(m->orderTaken) != hipSuccess) {
          st = BATS_EHIP;
          break;
        }
        memcpy(m->order, from, sizeof(int) * train.size());
        from = m->order;
      }
      if (hipMemcpyAsync(dIdx, from, sizeof(int) * train.size(),
                         hipMemcpyHostToDevice, m->stream) != hipSuccess ||
          hipEventRecord(m->orderTaken, m->stream) != hipSuccess) {
        st = BATS_EHIP;
        break;
      }
      for (long b = 0; st == BATS_OK && b < stepsPerEpoch; b++) {
        if (UseGraph)
          st = hipGraphLaunch(exec, m->stream) == hipSuccess ? BATS_OK : BATS_EHIP;
        else
          st = one_step();
      }
      if (st != BATS_OK) break;
      if (ep + 1 < nEpoch) continue;
      // loss of the last minibatch
      if (hipMemcpyAsync(e.data(), m->rowErr, sizeof(float) * B,
                         hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
          hipStreamSynchronize(m->stream) != hipSuccess) {
        st = BATS_EHIP;
        break;
      }
      double epLoss = 0.0;
      for (int r = 0; r < B; r++) epLoss += e[r];
      lastLoss = epLoss / (8.0 * B);
    }
    (void)hipStreamSynchronize(m->stream);
    if (exec) (void)hipGraphExecDestroy(exec);
    (void)hipFree(dSched);
    (void)hipFree(dStep);
    if (st) {
      (void)hipFree(dIdx);
      (void)hipFree(dScale);
      return st;
    }
    m->step += total;
  }
  // back to physical targets (a no-op scale of one without Standardize)
  hipLaunchKernelGGL(k_scale_last, dim3(1), dim3(64 * 8 + 8), 0, m->stream,
                     m->w, dScale, 0);
  m->fragStale = 1;
  MCHK(hipStreamSynchronize(m->stream));
  (void)hipFree(dScale);
  if (TrainLoss) *TrainLoss = lastLoss;
  // held-out relative error: ||Y - T|| / ||T|| overall and per output
  if (HeldOutRelErr_V && nHold > 0) {
    const int nWg = (int)std::min<long>((nHold + 31) / 32, kErrGrid);
    float *hx = nullptr;
    double *dPart = nullptr;
    MCHK(hipMalloc(&hx, sizeof(float) * (size_t)nHold * 24));
    MCHK(hipMalloc(&dPart, sizeof(double) * nWg * 24));
    float *hy = hx + (size_t)nHold * 16;
    MCHK(hipMemcpyAsync(dIdx, hold.data(), sizeof(int) * hold.size(),
                        hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_gather_inputs, dim3((nHold + 15) / 16), dim3(256), 0,
                       m->stream, m->dataX, dIdx, (int)nHold, hx);
    MCHK(hipGetLastError());
    st = bats::mlp::forward_device(m, hx, hy, (int)nHold, m->stream);
    if (st == BATS_OK) {
      hipLaunchKernelGGL(k_hold_err, dim3(nWg), dim3(256), 0, m->stream, hy,
                         m->dataT, m->dataB, m->dataJ, dIdx, (int)nHold, dPart);
      MCHK(hipGetLastError());
      std::vector<double> part((size_t)nWg * 24);
      MCHK(hipMemcpyAsync(part.data(), dPart, sizeof(double) * part.size(),
                          hipMemcpyDeviceToHost, m->stream));
      MCHK(hipStreamSynchronize(m->stream));
      // sum q of output j in sum[q][j + 1], of all outputs in sum[q][0]
      double sum[3][9] = {{0}};
      for (int w = 0; w < nWg; w++)
        for (int q = 0; q < 3; q++)
          for (int j = 0; j < 8; j++)
            sum[q][j + 1] += part[(w * 3 + q) * 8 + j];
      for (int q = 0; q < 3; q++)
        for (int j = 1; j < 9; j++) sum[q][0] += sum[q][j];
      for (int j = 0; j < 9; j++) {
        const double num = sum[0][j], den = sum[1][j], denT = sum[2][j];
        HeldOutRelErr_V[j] = den > 0 ? sqrt(num / den) : sqrt(num);
        HeldOutRelErr_V[9 + j] = denT > 0 ? sqrt(num / denT) : sqrt(num);
      }
    }
    (void)hipFree(hx);
    (void)hipFree(dPart);
  }
  (void)hipFree(dIdx);
  return st;
}
