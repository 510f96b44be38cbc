// mlp.hpp -- the face-flux surrogate network on gfx950 matrix cores.
//
// MLP 16 -> 128 -> 128 -> 64 -> 8 with SiLU between layers, y = x W + b.
// FP32 master weights; BF16 weights and activations feed
// v_mfma_f32_16x16x32_bf16, which accumulates in FP32.  The parameter
// vector is flat: W1 (16x128, row-major [in][out]), b1, W2, b2, W3, b3, W4,
// b4 -- 27,464 values.
//
// MFMA 16x16x32 BF16 operand layout (lane l = 0..63 of a wave):
//   A (16 x 32, rows x k): lane l holds row l%16, k = 8*(l/16) .. +7
//   B (32 x 16, k x cols): lane l holds col l%16, k = 8*(l/16) .. +7
//   D (16 x 16):           lane l holds col l%16, rows 4*(l/16) .. +3
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace bats {
namespace mlp {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int NL = 4;                       // layers
constexpr int DIM[NL + 1] = {16, 128, 128, 64, 8};
// offsets of W_l and b_l in the flat parameter vector
constexpr int OW1 = 0, OB1 = OW1 + 16 * 128;
constexpr int OW2 = OB1 + 128, OB2 = OW2 + 128 * 128;
constexpr int OW3 = OB2 + 128, OB3 = OW3 + 128 * 64;
constexpr int OW4 = OB3 + 64, OB4 = OW4 + 64 * 8;
constexpr int NPARAM = OB4 + 8;             // 27464
constexpr int OW[NL] = {OW1, OW2, OW3, OW4};
constexpr int OB[NL] = {OB1, OB2, OB3, OB4};

// fragment-ordered BF16 weights for the inference kernel.  The network runs
// transposed, Z^T = W^T A^T: a weight tile is the A operand (16 outputs n x
// 32 inputs k) and the activations are the B operand, taken straight from
// the previous layer's accumulators.  Lane l of a layer's output block nb
// holds outputs n = 16 nb + 4 (l/16) + i, i = 0..3, of activation row l%16;
// slot t of its B fragment for input block kb therefore carries input
// k = frag_k(layer, kb, l/16, t): the two output blocks 2 kb and 2 kb + 1
// of the previous layer, four values each (layer 1 reads its inputs as
// k = 8 (l/16) + t).  Layer l is padded to KP[l] x NP[l] and stored tile by
// tile (output block major, then input block), 64 lanes x 8 values each.
constexpr int KP[NL] = {32, 128, 128, 64};
constexpr int NP[NL] = {128, 128, 64, 16};
constexpr int TILE = 64 * 8;                // bf16 values per tile
constexpr int FT0 = 0;
constexpr int FT1 = FT0 + (KP[0] / 32) * (NP[0] / 16);
constexpr int FT2 = FT1 + (KP[1] / 32) * (NP[1] / 16);
constexpr int FT3 = FT2 + (KP[2] / 32) * (NP[2] / 16);
constexpr int NTILE = FT3 + (KP[3] / 32) * (NP[3] / 16);   // 58
constexpr int FT[NL] = {FT0, FT1, FT2, FT3};
constexpr int NFRAG = NTILE * TILE;         // 29696 bf16 = 58 KiB
__host__ __device__ inline int frag_k(int layer, int kb, int g, int t) {
  if (layer == 0) return kb * 32 + 8 * g + t;
  return 32 * kb + (t < 4 ? 4 * g + t : 16 + 4 * g + (t - 4));
}
// the slot (g, t) of input k within its block of 32, the inverse of frag_k
__host__ __device__ inline void frag_slot(int layer, int k, int &g, int &t) {
  const int r = k % 32;
  if (layer == 0) { g = r / 8; t = r % 8; }
  else if (r < 16) { g = r / 4; t = r % 4; }
  else { g = (r - 16) / 4; t = 4 + (r - 16) % 4; }
}
// the same for the way back: dA^T = W dZ^T of layers 2..4 takes W itself as
// the A operand (16 inputs x 32 outputs per tile, tiles input block major),
// the outputs in the order in which the layer's accumulators hold them
constexpr int BT1 = 0, BT2 = BT1 + (128 / 16) * (128 / 32);
constexpr int BT3 = BT2 + (128 / 16) * (64 / 32);
constexpr int NBTILE = BT3 + 64 / 16;       // 52
constexpr int BT[NL] = {0, BT1, BT2, BT3};
constexpr int NBFRAG = NBTILE * TILE;       // 26624 bf16 = 52 KiB
// position of parameter W_l[k][n] in the forward and the backward fragments
__host__ __device__ inline int frag_pos(int l, int k, int n) {
  int g, t;
  frag_slot(l, k, g, t);
  return ((FT[l] + (n / 16) * (KP[l] / 32) + k / 32) * 64 + 16 * g + n % 16) *
             8 + t;
}
__host__ __device__ inline int bfrag_pos(int l, int k, int n) {
  int g, t;
  frag_slot(1, n, g, t);
  const int nKb = l == 3 ? 1 : DIM[l + 1] / 32;
  return ((BT[l] + (k / 16) * nKb + n / 32) * 64 + 16 * g + k % 16) * 8 + t;
}
// the biases packed for the inference kernel's LDS copy
constexpr int CB1 = 0, CB2 = 128, CB3 = 256, CB4 = 320, NBIAS = 328;

// copy the four bias vectors of the flat parameter vector w into sBias
__device__ __forceinline__ void load_biases(const float *w, float *sBias) {
  for (int t = threadIdx.x; t < NBIAS; t += blockDim.x) {
    const int o = t < CB2 ? OB1 + t
                : t < CB3 ? OB2 + (t - CB2)
                : t < CB4 ? OB3 + (t - CB3)
                          : OB4 + (t - CB4);
    sBias[t] = w[o];
  }
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// v_exp_f32 and v_rcp_f32 (about 1 ulp each) instead of the IEEE division
// sequence: the activation is the inference kernel's VALU cost
__device__ __forceinline__ float sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }

// =====================================================================
// batched inference: Y[rows x 8] = MLP(X[rows x 16]) with fragment-ordered
// BF16 weights (flat FP32 biases); a wave takes 32 rows at a time
// =====================================================================
// inference workgroups: 8 waves share one LDS copy of the weights (59 KiB);
// two workgroups per CU, 4 waves per SIMD (at most 128 VGPRs)
constexpr int kInferThreads = 512, kInferWaves = kInferThreads / 64;
constexpr int kInferGrid = 2 * 256;

// R tiles of 16 rows through the network, x[t] the input fragment of tile t
// (lane l: inputs 8 (l/16) .. +7 of row l%16, zero from input 16 on).  sW:
// weight fragments in LDS, bias: the packed biases (load_biases) in LDS.  The
// activations never leave the registers: two output blocks of a layer,
// through SiLU and BF16, are one B fragment of the next (see frag_k), formed
// while the matrix cores work on the following two.  A weight fragment is
// read from LDS once for all R tiles.  out(t, y): lanes with l/16 < 2 hold
// outputs 4 (l/16) .. +3 of row l%16 of tile t.
template <int R, typename OUT>
__device__ __forceinline__ void infer_tiles(const __bf16 *sW,
                                            const float *bias,
                                            const bf16x8 (&x)[R], OUT out) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const bf16x8 *W = reinterpret_cast<const bf16x8 *>(sW) + lane;
  // accumulators start at the bias of their outputs 16 nb + 4 g + i
  auto bias4 = [&](const float *b, int nb) {
    const float *p = b + nb * 16 + 4 * g;
    return f32x4{p[0], p[1], p[2], p[3]};
  };
  // one layer: NK input fragments to NO output fragments per tile
  auto layer = [&](auto nk, auto no, int ft, const float *b,
                   const auto &in, auto &o) {
    constexpr int NK = decltype(nk)::value, NO = decltype(no)::value;
#pragma unroll
    for (int kb = 0; kb < NO; kb++) {
      f32x4 acc[R][2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int nb = 2 * kb + h;
        const f32x4 b4 = bias4(b, nb);
#pragma unroll
        for (int t = 0; t < R; t++) acc[t][h] = b4;
#pragma unroll
        for (int q = 0; q < NK; q++) {
          const bf16x8 w = W[(ft + nb * NK + q) * 64];
#pragma unroll
          for (int t = 0; t < R; t++) acc[t][h] = mfma(w, in[t][q], acc[t][h]);
        }
      }
#pragma unroll
      for (int t = 0; t < R; t++) {
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          v[i] = (__bf16)silu(acc[t][0][i]);
          v[4 + i] = (__bf16)silu(acc[t][1][i]);
        }
        o[t][kb] = v;
      }
      // the weight fragments of two output blocks live at a time
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using std::integral_constant;
  bf16x8 f0[R][1], f1[R][4], f2[R][4], f3[R][2];
#pragma unroll
  for (int t = 0; t < R; t++) f0[t][0] = x[t];
  layer(integral_constant<int, 1>(), integral_constant<int, 4>(), FT0,
        bias + CB1, f0, f1);
  layer(integral_constant<int, 4>(), integral_constant<int, 4>(), FT1,
        bias + CB2, f1, f2);
  layer(integral_constant<int, 4>(), integral_constant<int, 2>(), FT2,
        bias + CB3, f2, f3);
  // layer 4: 64 -> 8 (padded to 16 outputs)
#pragma unroll
  for (int t = 0; t < R; t++) {
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
    y = mfma(W[(FT3 + 0) * 64], f3[t][0], y);
    y = mfma(W[(FT3 + 1) * 64], f3[t][1], y);
    const float *p = bias + CB4 + 4 * (g & 1);
#pragma unroll
    for (int i = 0; i < 4; i++) y[i] += p[i];
    out(t, y);
  }
}

}  // namespace mlp
}  // namespace bats
