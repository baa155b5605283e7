// Learned proposal for LJ walkers: device pieces shared by the walker
// engine, the probe kernel and the training kernels.
//
// Definition (no reference counterpart; the same in the CPU restatement):
// - features of atom i at position p: f_k = sum_{j != i} exp(-(r_ij - c_k)^2
//   / (2 w^2)) with c_k = 0.9 + k (1.6/7), w = 0.2, k = 0..7, in float, r_ij
//   the float square root of the float r^2 of the double differences;
// - network 8 -> 32 -> 32 -> 1 with ReLU, BF16 weights and FP32 arithmetic,
//   parameters in the order W1[32][8], b1[32], W2[32][32], b2[32], w3[32], b3
//   (1377); output s = ln sigma clamped to [ln 0.01, 0];
// - move: atom uniform, xi ~ N(0, I3) by Box-Muller from four uniform draws,
//   p' = p + sigma(p) xi; ln H = 3 (s - s') + |xi|^2 (1 - e^{2(s - s')}) / 2
//   is the log ratio q(p' -> p) / q(p -> p') of the two Gaussian proposals
//   (sigma' evaluated at p'), added to the acceptance exponent;
// - probe record (training data): the features of a random atom and, for the
//   16 scales ln sigma_m = ln 0.01 + m ln(100)/15, the mean over 2 Gaussian
//   draws of alpha |d|^2 (alpha = the walker's acceptance probability).
#pragma once

#include "sadmc_common.h"

namespace sadmc {

constexpr int kPropNF = 8, kPropH = 32, kPropNP = 1377, kPropNS = 16, kPropR = 2, kPropRec = 24;
constexpr int kPropLds = 1384;  // the weight arrays' padded length
// The weights in LDS, widened to float once per launch (the network reads
// them twice a move): in the parameter order, but with the 32 x 32 layer's rows
// 36 floats apart, so that the 16 rows a matrix step reads as 16-byte pieces
// fall into different banks.  45 two-byte reads and shifts per evaluation
// became 15 reads.
constexpr int kPropRow = 36, kPropLdsF = 1384 + 32 * (kPropRow - 32);
constexpr float kPropC0 = 0.9f, kPropDC = 1.6f / 7.0f, kPropA = 12.5f;
constexpr float kPropSMin = -4.605170186f, kPropSMax = 0.0f;
// parameter offsets
constexpr int kW1 = 0, kB1 = 256, kW2 = 288, kB2 = 1312, kW3 = 1344, kB3 = 1376;

SADMC_HD float bf16_to_f32(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }
// Round to nearest, ties to even (finite inputs).
SADMC_HD uint16_t f32_to_bf16(float f) {
  uint32_t b = __builtin_bit_cast(uint32_t, f);
  b += 0x7FFFu + ((b >> 16) & 1u);
  return (uint16_t)(b >> 16);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sum over the G lanes of a group (the same pattern as the FP64 group sum).
__device__ __forceinline__ float group_sum_f32(float v, int G) {
  if (G >= 2) v = v + dpp_f32<0xB1>(v);
  if (G >= 4) v = v + dpp_f32<0x4E>(v);
  if (G >= 8) v = v + dpp_f32<0x141>(v);
  if (G >= 16) v = v + dpp_f32<0x140>(v);
  if (G >= 32) v = v + __shfl_xor(v, 16, 64);
  if (G >= 64) v = v + __shfl_xor(v, 32, 64);
  return v;
}

// Contribution of one neighbour at float distance r to the 8 features
// (hardware square root and exponential: the proposal only has to be the
// same function at both ends of a move, not correctly rounded).  At
// kPropFar every term is exp2 of less than -1e37, which is +0: what a slot
// without a neighbour adds.
constexpr float kPropFar = 1e18f;
__device__ __forceinline__ void feature_add(float r, float *f) {
#pragma unroll
  for (int k = 0; k < kPropNF; k++) {
    const float d = r - (kPropC0 + (float)k * kPropDC);
    f[k] += __expf(-kPropA * d * d);
  }
}

// Three standard normal draws by Box-Muller from four uniforms, with the
// hardware log2, square root and sin/cos (whose argument is in revolutions,
// so cos(2 pi u) is one instruction).  The Hastings term is computed from the
// draws actually used.
__device__ __forceinline__ void gaussian3(uint64_t &s0, uint64_t &s1, float *xi) {
  const float u1 = (float)gen_f64(s0, s1), u2 = (float)gen_f64(s0, s1);
  const float u3 = (float)gen_f64(s0, s1), u4 = (float)gen_f64(s0, s1);
  const float m2ln2 = -1.3862943611f;  // -2 ln 2
  const float r1 = __builtin_amdgcn_sqrtf(m2ln2 * __builtin_amdgcn_logf(1.0f - u1));
  const float r2 = __builtin_amdgcn_sqrtf(m2ln2 * __builtin_amdgcn_logf(1.0f - u3));
  xi[0] = r1 * __builtin_amdgcn_cosf(u2);
  xi[1] = r1 * __builtin_amdgcn_sinf(u2);
  xi[2] = r2 * __builtin_amdgcn_cosf(u4);
}

SADMC_DF double prop_lnh(float s, float s_new, float xi2) {
  const double ds = (double)s - (double)s_new;
  return 3.0 * ds + 0.5 * (double)xi2 * (1.0 - exp(2.0 * ds));
}

// Load the BF16 weights into LDS as float, in the parameter order (all 64
// lanes of the workgroup; kPropNP floats).
__device__ __forceinline__ void load_weights(const uint16_t *w, float *lw) {
  for (int i = threadIdx.x; i < kPropNP; i += 64) lw[i] = bf16_to_f32(w[i]);
  __syncthreads();
}

// The same in the padded layout above (kPropLdsF floats).
constexpr int kLW2 = 288, kLB2 = kLW2 + 32 * kPropRow, kLW3 = kLB2 + 32, kLB3 = kLW3 + 32;
__device__ __forceinline__ void load_weights_rows(const uint16_t *w, float *lw) {
  for (int i = threadIdx.x; i < kPropNP; i += 64) {
    const int k = i - kW2;
    const int at = k < 0 ? i : k < 1024 ? kLW2 + k / 32 * kPropRow + k % 32 : kLB2 + (i - kB2);
    lw[at] = bf16_to_f32(w[i]);
  }
  __syncthreads();
}

// Forward pass for one walker whose G lanes all hold the features f; lane l
// computes hidden units l, l+G, ... and the group exchanges the first layer
// through `xc` (32 floats of LDS per walker).  W: the weights in LDS
// (load_weights_rows), FP32 arithmetic.
__device__ __forceinline__ float mlp_forward(const float *W, float *xc, const float *f, int lane, int G) {
  for (int u = lane; u < kPropH; u += G) {
    const float4 *a = (const float4 *)(W + kW1 + u * kPropNF);
    const float4 a0 = a[0], a1 = a[1];
    float z = W[kB1 + u];
    z += a0.x * f[0];
    z += a0.y * f[1];
    z += a0.z * f[2];
    z += a0.w * f[3];
    z += a1.x * f[4];
    z += a1.y * f[5];
    z += a1.z * f[6];
    z += a1.w * f[7];
    xc[u] = z > 0.0f ? z : 0.0f;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const float4 *x4 = (const float4 *)xc;
  float part = 0.0f;
  for (int u = lane; u < kPropH; u += G) {
    const float4 *w2 = (const float4 *)(W + kLW2 + u * kPropRow);
    float z = W[kLB2 + u];
#pragma unroll
    for (int k = 0; k < kPropH / 4; k++) {
      const float4 w = w2[k], h = x4[k];
      z += w.x * h.x;
      z += w.y * h.y;
      z += w.z * h.z;
      z += w.w * h.w;
    }
    const float h = z > 0.0f ? z : 0.0f;
    part += W[kLW3 + u] * h;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  float s = W[kLB3] + group_sum_f32(part, G);
  return s < kPropSMin ? kPropSMin : (s > kPropSMax ? kPropSMax : s);
}

// The network on the matrix cores, for a wave whose 64 lanes all run this
// call and whose walkers have G >= 4 lanes each (at most 16 walkers: the
// columns of 16x16x4 FP32 products; v_mfma_f32_16x16x4f32 takes A[i][k] from
// lane i + 16k, B[k][j] from lane j + 16k and leaves D[4q + e][j] in element
// e of lane j + 16q).  Layer 1 is H1 = W1 X^T (two row blocks of 16 units, two
// steps of 4 features), layer 2 H2 = W2 H1 (the hidden layer stays where
// layer 1 left it: step (m, e) takes unit 16m + 4q + e from element e of
// lane j + 16q), then s = b3 + w3 . relu(H2 + b2) summed over the four lanes
// of a column.  FP32 products and sums as in mlp_forward, in another
// order.
// W: the weights in LDS (load_weights_rows); f: the walker's features in every lane of its
// group; l: the lane in the wave.
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float mlp_wave(const float *W, const float *f, int l, int G) {
  const int i = l & 15, q = l >> 4, j = l & 15;  // A row / B and D column, step
  const int g = l & (G - 1);
  const bool col = j < 64 / G;  // column j is a walker of this wave (else its source lane is wrapped and unused)
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  // both row blocks' products side by side (independent accumulators)
  f32x4 acc0 = zero, acc1 = zero;
#pragma unroll
  for (int st = 0; st < 2; st++) {
    // feature 4 st + q of walker j, from the lane of its group that holds
    // it at in-group index (4 st + q) mod G
    const float mine = G >= 8 ? f[g & 7] : f[(4 * st + g) & 7];
    const float got = __shfl(mine, (G * j + ((4 * st + q) & (G - 1))) & 63, 64);
    const float b = col ? got : 0.0f;
    const float a0 = W[kW1 + i * kPropNF + 4 * st + q];
    const float a1 = W[kW1 + (16 + i) * kPropNF + 4 * st + q];
    acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b, acc1, 0, 0, 0);
  }
  float h1[2][4];
  const f32x4 b10 = *(const f32x4 *)(W + kB1 + 4 * q), b11 = *(const f32x4 *)(W + kB1 + 16 + 4 * q);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float z0 = acc0[e] + b10[e];
    const float z1 = acc1[e] + b11[e];
    h1[0][e] = z0 > 0.0f ? z0 : 0.0f;
    h1[1][e] = z1 > 0.0f ? z1 : 0.0f;
  }
  f32x4 d0 = zero, d1 = zero;
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const f32x4 a0 = *(const f32x4 *)(W + kLW2 + i * kPropRow + 16 * m + 4 * q);
    const f32x4 a1 = *(const f32x4 *)(W + kLW2 + (16 + i) * kPropRow + 16 * m + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[e], h1[m][e], d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[e], h1[m][e], d1, 0, 0, 0);
    }
  }
  float part = 0.0f;
#pragma unroll
  for (int mo = 0; mo < 2; mo++) {
    const f32x4 b2 = *(const f32x4 *)(W + kLB2 + 16 * mo + 4 * q), w3 = *(const f32x4 *)(W + kLW3 + 16 * mo + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float z = (mo == 0 ? d0[e] : d1[e]) + b2[e];
      part += w3[e] * (z > 0.0f ? z : 0.0f);
    }
  }
  part += __shfl_xor(part, 16, 64);
  part += __shfl_xor(part, 32, 64);
  float s = W[kLB3] + part;
  s = s < kPropSMin ? kPropSMin : (s > kPropSMax ? kPropSMax : s);
  // walker l / G reads its column
  return __shfl(s, l / G, 64);
}

// The network for the walker of this lane's group: on the matrix cores when
// every lane of the wave is here and G >= 4, else mlp_forward.
__device__ __forceinline__ float mlp_eval(const float *W, float *xc, const float *f, int lane, int G) {
  if (G >= 4 && __builtin_amdgcn_read_exec() == ~0ull) return mlp_wave(W, f, (int)(threadIdx.x & 63), G);
  return mlp_forward(W, xc, f, lane, G);
}

}  // namespace sadmc
