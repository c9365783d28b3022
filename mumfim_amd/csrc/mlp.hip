// Learned surrogate: an ensemble of MLPs 10 -> 256 -> 256 -> 256 -> 6 (SiLU)
// trained and evaluated on the gfx950 matrix cores.  Weights and
// activations are BF16 (v_mfma_f32_16x16x32_bf16, FP32 accumulate); biases,
// FP32 master weights and Adam moments stay FP32.
//
// MFMA 16x16x32 operand layout (wave64): lane l supplies row (l & 15) of A
// and column (l & 15) of B, each as the 8 consecutive k values
// 8*(l >> 4) .. 8*(l >> 4) + 7; the 16x16 FP32 result leaves lane l holding
// rows 4*(l >> 4) .. 4*(l >> 4) + 3 of column (l & 15).  Every operand here
// is stored with k contiguous, so each lane's fragment is one 16-byte load.
//
// Training, three launches per mini-batch, all members in each:
//   train      per tile of samples, in LDS and registers: gather, normalise,
//              the four layers, the loss, the gradients back to layer 1;
//              leaves the transposed activations and gradients (BF16)
//   dw         D^T H over the batch, split over K into FP32 partials; the
//              transposed activations carry a row of ones, so the bias
//              gradient is one more column of the same product
//   adam       sums the partials in a fixed order (deterministic), updates
//              the FP32 masters and rewrites the BF16 copies
// Inference: one fused kernel per tile of samples keeps the activations in
// LDS through all four layers and all members; with a Jacobian it carries six
// tangent planes (d/d e_j, forward mode) through the same MFMA products.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <thread>
#include <vector>

#include "dev_util.hpp"
#include "mf_internal.hpp"
#include "mlp_internal.hpp"

namespace mf {
namespace mlpk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// BF16 copies of the weights, per member (element counts).
constexpr int kInP = 32;     // input width padded to one MFMA k step
constexpr int kOutP = 16;    // output width padded to one MFMA tile
constexpr int kTRows = 272;  // transposed hidden activations: 256 + ones row + pad
constexpr int64_t kW1 = kHid * kInP, kW2 = kHid * kHid, kW4 = kOutP * kHid;
constexpr int64_t kW4T = kHid * kInP;
constexpr int64_t kBias = 3 * kHid + kOutP;
// Position of element (row, k) of a BF16 operand of padded width kp kept in
// fragment order: the 16 rows x 32 k that one MFMA reads are one contiguous
// kilobyte, lane after lane, so a fragment load touches 8 whole 128-byte
// lines (row by row it touches 16 half lines).
__host__ __device__ constexpr int64_t frag(int64_t row, int64_t k, int64_t kp) {
  return ((row >> 4) * (kp >> 5) + (k >> 5)) * 512 + (((k & 31) >> 3) * 16 + (row & 15)) * 8 +
         (k & 7);
}
constexpr int kActLd = kHid + 8;  // LDS row stride (BF16) of the inference tile

__device__ __forceinline__ uint16_t bf(float x) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(x));
}
__device__ __forceinline__ float unbf(uint16_t b) {
  return __uint_as_float(static_cast<uint32_t>(b) << 16);
}
// two floats to BF16 (round to nearest even) in one 32-bit word, low half
// first: one v_cvt_pk_bf16_f32 (converted one at a time, each value took a
// conversion and the pair a shift and an or)
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  return make_uint2(pack2(a, b), pack2(c, d));
}
// silu(z) = z * sigmoid(z); ds = silu'(z) = sg * (1 + z * (1 - sg))
__device__ __forceinline__ float silu(float z, float &ds) {
  const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
  ds = sg * (1.0f + z * (1.0f - sg));
  return z * sg;
}
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 ld8(const uint16_t *p) {
  return *reinterpret_cast<const bf16x8 *>(p);
}

// ---------------------------------------------------------------------------
// Loss of one member from its samples' squared errors: sums of 256 samples
// (64 by a butterfly, four of those in order), added in batch order; out[mem]
// = mean, acc[mem] += mean.
__device__ void loss_sum(const float *v, int Bt, float inv, float *out, float *acc) {
  constexpr int kGroups = 64;  // 64-sample groups per pass
  __shared__ float red[kGroups];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  float s = 0.f;
  for (int64_t c = 0; c < Bt; c += 64 * kGroups) {
    float x[kGroups / 4];
#pragma unroll
    for (int j = 0; j < kGroups / 4; ++j) {
      const int64_t b = c + 64 * (w + 4 * j) + lane;
      x[j] = b < Bt ? v[b] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < kGroups / 4; ++j) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x[j] += __shfl_xor(x[j], o);
      if (lane == 0) red[w + 4 * j] = x[j];
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int g = 0; g < kGroups && c + 64 * g < Bt; g += 4)
        s += red[g] + red[g + 1] + red[g + 2] + red[g + 3];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    s *= inv;
    *out = s;
    *acc += s;
  }
}

struct AdamArgs {
  float *P, *Mo, *Ve;
  const float *part[4];
  int64_t sPart[4], sSplit[4];
  int ldp[4];
  int splits;
  uint16_t *w1, *w2, *w3, *w4, *w2t, *w3t, *w4t;
  float *bias;
  float lr, b1, b2, eps, bc1, bc2;
  float *grad;
  int mode;  // 0: Adam update, 1: gradient only, 2: refresh BF16 copies only
  // the last block of each member sums the loss, where it is asked for
  const float *loss_v;
  int Bt;
  float loss_inv, *loss_out, *loss_acc;
};

// One thread per (member, parameter): gradient = sum of the K-split
// partials of its (layer, out, in) entry, in split order.
constexpr int kAdamBlocks = (kNumParams + 255) / 256;
__global__ __launch_bounds__(256) void adam_kernel(AdamArgs a) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  const int mem = blockIdx.y;
  if (blockIdx.x == kAdamBlocks) {
    loss_sum(a.loss_v + (int64_t)mem * a.Bt, a.Bt, a.loss_inv, a.loss_out + mem,
             a.loss_acc + mem);
    return;
  }
  if (p >= kNumParams) return;
  int L, o, i;
  bool isb = false;
  if (p < kOffB1) { L = 0; o = p / kIn; i = p % kIn; }
  else if (p < kOffW2) { L = 0; o = p - kOffB1; i = kIn; isb = true; }
  else if (p < kOffB2) { L = 1; o = (p - kOffW2) / kHid; i = (p - kOffW2) % kHid; }
  else if (p < kOffW3) { L = 1; o = p - kOffB2; i = kHid; isb = true; }
  else if (p < kOffB3) { L = 2; o = (p - kOffW3) / kHid; i = (p - kOffW3) % kHid; }
  else if (p < kOffW4) { L = 2; o = p - kOffB3; i = kHid; isb = true; }
  else if (p < kOffB4) { L = 3; o = (p - kOffW4) / kHid; i = (p - kOffW4) % kHid; }
  else { L = 3; o = p - kOffB4; i = kHid; isb = true; }
  const int64_t pi = (int64_t)mem * kNumParams + p;
  float w = a.P[pi];
  if (a.mode != 2) {
    const float *part = a.part[L] + mem * a.sPart[L] + (int64_t)o * a.ldp[L] + i;
    float g = 0.f;
    int s = 0;
    for (; s + 8 <= a.splits; s += 8) {  // eight loads in flight
      float q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = part[(s + u) * a.sSplit[L]];
#pragma unroll
      for (int u = 0; u < 8; ++u) g += q[u];
    }
    for (; s < a.splits; ++s) g += part[s * a.sSplit[L]];
    if (a.mode == 1) {
      a.grad[pi] = g;
      return;
    }
    const float m = a.b1 * a.Mo[pi] + (1.f - a.b1) * g;
    const float v = a.b2 * a.Ve[pi] + (1.f - a.b2) * g * g;
    a.Mo[pi] = m;
    a.Ve[pi] = v;
    w -= a.lr * (m / a.bc1) / (sqrtf(v / a.bc2) + a.eps);
    a.P[pi] = w;
  }
  const uint16_t u = bf(w);
  if (isb) {
    a.bias[mem * kBias + L * kHid + o] = w;
    return;
  }
  switch (L) {
    case 0: a.w1[mem * kW1 + frag(o, i, kInP)] = u; break;
    case 1:
      a.w2[mem * kW2 + frag(o, i, kHid)] = u;
      a.w2t[mem * kW2 + frag(i, o, kHid)] = u;
      break;
    case 2:
      a.w3[mem * kW2 + frag(o, i, kHid)] = u;
      a.w3t[mem * kW2 + frag(i, o, kHid)] = u;
      break;
    default:
      a.w4[mem * kW4 + frag(o, i, kHid)] = u;
      a.w4t[mem * kW4T + frag(i, o, kInP)] = u;
      break;
  }
}

// Constant row of the transposed activation buffers: row `one_row` of
// every member's [rows x Bt] block is 1.
__global__ void ones_row_kernel(uint16_t *T, int64_t member_stride, int one_row, int Bt) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < Bt) T[blockIdx.y * member_stride + frag(one_row, b, Bt)] = bf(1.0f);
}

// ---------------------------------------------------------------------------
// Fused inference.  A tile holds TS = 16 Q samples; with NT > 0 it also holds
// NT of the six tangent planes (d/d e_j of every activation; blockIdx.y picks
// which), so the LDS tile has P = Q (1 + NT) blocks of 16 rows, one row per
// (plane, sample), 256 BF16 features per row.  Each layer computes the
// transposed product W (features) x act^T (rows): a wave owns 32 features and
// lane l ends up with 4 consecutive features of one row, written back as one
// 8-byte LDS store.  Plane 0 takes bias and silu, plane j the product with
// silu'(z) of the same (sample, feature), which sits in the same lane.  G
// members are evaluated at a time, eight waves each, and added in order.
//
// What bounds it: the activations' VALU work (2^20 samples, four members: 0.74 of
// the SIMD cycles, with the matrix cores at 0.39 and LDS at 0.54 beside it) and,
// with J, the LDS reads of the activations (0.78, half of it bank conflicts), then
// the matrix cores (0.57).  The weights come through L2, 280 KB per tile and
// member.  Measured on 2^20 samples / 150001 with J: 2.73 / 2.31 ms with weights row by row, four waves of 64
// features and accumulators in AGPRs (two or three waves per SIMD, each value
// copied back before use); 2.39 / 1.49 ms with eight waves of 32 features (four
// waves per SIMD, no copies, weights one k step ahead); 1.39 / 1.03 ms with
// the weights in fragment order (row by row, a fragment is 16 half lines and
// the vector cache's line rate was the bound).
struct InferArgs {
  const float *X;
  int64_t n;
  int m0, mcount;
  const uint16_t *w1, *w2, *w3, *w4;
  const float *bias;
  const MlpNorm *nm;
  float *Y, *J, *spread;
};

// A wave's weight fragments of one k step: its 16 C features x 32 k.
template <int C>
struct WFrag {
  bf16x8 v[C];
};
template <int C, int KP>
__device__ __forceinline__ WFrag<C> load_w(const uint16_t *W, int kk, int w, int lane) {
  // uniform base (w is a scalar) plus one 32-bit lane offset for all blocks
  const uint32_t off = (uint32_t)lane * 16u;
  WFrag<C> f;
#pragma unroll
  for (int c = 0; c < C; ++c)
    f.v[c] = *reinterpret_cast<const bf16x8 *>(
        reinterpret_cast<const char *>(W + ((C * w + c) * (KP / 32) + kk) * 512) + off);
  return f;
}

// acc = W (16 C features of wave w) x act^T (16 P rows) over KS k steps.  `wf`
// holds the first step's weights (loaded before the barrier that published
// act); each later step's load while the one before is multiplied.
template <int P, int C, int KS, int LDA>
__device__ __forceinline__ void infer_layer(const uint16_t *act, const uint16_t *W, int w, int lane,
                                            WFrag<C> wf, f32x4 (&acc)[P][C]) {
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[p][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    WFrag<C> nx;
    if (kk + 1 < KS) nx = load_w<C, 32 * KS>(W, kk + 1, w, lane);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const bf16x8 x = ld8(act + (16 * p + (lane & 15)) * LDA + 32 * kk + (lane >> 4) * 8);
#pragma unroll
      for (int c = 0; c < C; ++c) acc[p][c] = mfma(wf.v[c], x, acc[p][c]);
    }
    // with all seven planes the loads of several steps at once would spill
    if (P > 4) __builtin_amdgcn_sched_barrier(0);
    if (kk + 1 < KS) wf = nx;
  }
}

template <int Q, int NPL, int C>
__device__ __forceinline__ void infer_hidden_epilogue(uint16_t *act, f32x4 (&acc)[Q * NPL][C],
                                                      const float4 (&bias)[C], int w, int lr,
                                                      int lq) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int f0 = 16 * (C * w + c) + lq;
    const float4 b = bias[c];
#pragma unroll
    for (int sb = 0; sb < Q; ++sb) {
      float h[4], d[4];
      h[0] = silu(acc[sb][c][0] + b.x, d[0]);
      h[1] = silu(acc[sb][c][1] + b.y, d[1]);
      h[2] = silu(acc[sb][c][2] + b.z, d[2]);
      h[3] = silu(acc[sb][c][3] + b.w, d[3]);
      *reinterpret_cast<uint2 *>(act + (16 * sb + lr) * kActLd + f0) =
          pack4(h[0], h[1], h[2], h[3]);
#pragma unroll
      for (int j = 1; j < NPL; ++j) {
        const int p = j * Q + sb;
        *reinterpret_cast<uint2 *>(act + (16 * p + lr) * kActLd + f0) =
            pack4(acc[p][c][0] * d[0], acc[p][c][1] * d[1], acc[p][c][2] * d[2],
                  acc[p][c][3] * d[3]);
      }
    }
  }
}

template <int C>
__device__ __forceinline__ void load_bias(const float *bias, int w, int lq, float4 (&b)[C]) {
#pragma unroll
  for (int c = 0; c < C; ++c)
    b[c] = *reinterpret_cast<const float4 *>(
        reinterpret_cast<const char *>(bias + 16 * (C * w + c)) + (uint32_t)lq * 4u);
}

constexpr int kInferWaves = 8;  // waves that evaluate one member of a tile
constexpr int kInLd = kInP + 8;  // LDS row stride (BF16) of the input tile
constexpr int kOutLd = 8;        // LDS row stride (FP32) of a member's outputs
// LDS of an inference workgroup of P row blocks and G members at a time: the
// input tile, each member's activations and (G > 1) its outputs.
constexpr size_t infer_lds(int P, int G) {
  return (size_t)P * 16 *
         ((kInLd + G * kActLd) * sizeof(uint16_t) + (G - 1) * kOutLd * sizeof(float));
}

template <int Q, int NT, int G>
__global__ __launch_bounds__(64 * kInferWaves * G, 4) void infer_kernel(InferArgs a) {
  constexpr int NW = kInferWaves, NPL = 1 + NT;
  constexpr int P = Q * NPL;
  constexpr int TS = 16 * Q;
  static_assert(P <= NW, "one output block per wave");
  constexpr int C = 16 / NW;  // 16-feature blocks per wave
  extern __shared__ uint16_t lds[];
  uint16_t *const xin = lds;
  const int tid = threadIdx.x;
  const int wg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = wg % NW, grp = wg / NW;  // wave of its member, member group
  uint16_t *const act = lds + P * 16 * (kInLd + grp * kActLd);
  float *const osh = reinterpret_cast<float *>(lds + P * 16 * (kInLd + G * kActLd));
  const int j0 = NT ? NT * blockIdx.y : 0;  // first tangent direction
  const int64_t s0 = (int64_t)blockIdx.x * TS;
  const MlpNorm *nm = a.nm;
  // inputs, the same for every member: plane 0 = normalised x (10 of 32
  // columns), plane j = e_j seed
  for (int e = tid; e < P * 16 * kInP; e += 64 * NW * G) {
    const int row = e / kInP, c = e % kInP;
    const int plane = row / TS, sr = row % TS;
    float v = 0.f;
    if (plane == 0) {
      const int64_t s = s0 + sr;
      if (c < kIn && s < a.n) v = (a.X[s * kIn + c] - nm->in_mean[c]) * nm->in_inv[c];
    } else if (c == j0 + plane - 1) {
      v = 1.f;
    }
    xin[row * kInLd + c] = bf(v);
  }
  f32x4 fsum = {0.f, 0.f, 0.f, 0.f}, fsq = fsum;
  f32x4 acc[P][C];
  const int last = a.m0 + a.mcount - 1;
  int mem = min(a.m0 + grp, last);
  WFrag<C> wf = load_w<C, kInP>(a.w1 + mem * kW1, 0, w, tid & 63);
  __syncthreads();
#pragma clang loop unroll(disable)
  for (int m = a.m0; m <= last; m += G) {
    // a group without a member of its own repeats the last one, unread
    mem = min(m + grp, last);
    // the lane's offsets are worked out anew: kept over the loop they spill
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int lr = lane & 15, lq = (lane >> 4) * 4;
    const float *bias = a.bias + mem * kBias;
    const uint16_t *W2 = a.w2 + mem * kW2, *W3 = a.w3 + mem * kW2, *W4 = a.w4 + mem * kW4;
    // before each epilogue the next product's first weights are requested:
    // they arrive while the activations are evaluated
    float4 b[C];
    load_bias<C>(bias, w, lq, b);
    infer_layer<P, C, 1, kInLd>(xin, a.w1 + mem * kW1, w, lane, wf, acc);
    wf = load_w<C, kHid>(W2, 0, w, lane);
    __syncthreads();  // the last member's output products have read act
    infer_hidden_epilogue<Q, NPL, C>(act, acc, b, w, lr, lq);
    __syncthreads();
    load_bias<C>(bias + kHid, w, lq, b);
    infer_layer<P, C, 8, kActLd>(act, W2, w, lane, wf, acc);
    wf = load_w<C, kHid>(W3, 0, w, lane);
    __syncthreads();
    infer_hidden_epilogue<Q, NPL, C>(act, acc, b, w, lr, lq);
    __syncthreads();
    load_bias<C>(bias + 2 * kHid, w, lq, b);
    infer_layer<P, C, 8, kActLd>(act, W3, w, lane, wf, acc);
    __syncthreads();
    infer_hidden_epilogue<Q, NPL, C>(act, acc, b, w, lr, lq);
    if (m + G <= last) wf = load_w<C, kInP>(a.w1 + min(m + G + grp, last) * kW1, 0, w, lane);
    const float4 b4 = *reinterpret_cast<const float4 *>(bias + 3 * kHid + lq);
    __syncthreads();
    // output layer: 16 (6 used) features x 16 rows, row block w by wave w
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (w < P) {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
        o = mfma(load_w<1, kHid>(W4, kk, 0, lane).v[0],
                 ld8(act + (16 * w + lr) * kActLd + 32 * kk + (lane >> 4) * 8), o);
      if (w < Q) o += f32x4{b4.x, b4.y, b4.z, b4.w};
    }
    if (G == 1) {
      if (w < Q) fsq += o * o;
      fsum += o;
    } else {  // group 0 adds the outputs in member order
      float4 *const row = reinterpret_cast<float4 *>(osh + (16 * w + lr) * kOutLd + lq);
      const bool mine = w < P && lq < kOutLd;
      if (grp == 1 && mine) *row = make_float4(o[0], o[1], o[2], o[3]);
      __syncthreads();
      if (grp == 0 && mine) {
        fsq += o * o;
        fsum += o;
        if (m < last) {
          const float4 r = *row;
          const f32x4 o1 = {r.x, r.y, r.z, r.w};
          fsq += o1 * o1;
          fsum += o1;
        }
      }
    }
  }
  if (grp > 0 || w >= P) return;
  const float inv_m = 1.0f / (float)a.mcount;
  const int plane = w / Q, lr = tid & 15, lq = ((tid & 63) >> 4) * 4;
  const int64_t s = s0 + 16 * (w % Q) + lr;
  if (s >= a.n || (plane == 0 && blockIdx.y > 0)) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = lq + q;
    if (i >= kOut) continue;
    const float mean = fsum[q] * inv_m;
    if (plane == 0) {
      a.Y[s * kOut + i] = mean * nm->out_std[i] + nm->out_mean[i];
      if (a.spread) {
        const float var = fmaxf(fsq[q] * inv_m - mean * mean, 0.f);
        a.spread[s * kOut + i] = sqrtf(var) * nm->out_std[i];
      }
    } else {
      const int j = j0 + plane - 1;
      a.J[s * 36 + 6 * i + j] = mean * nm->out_std[i] * nm->in_inv[j];
    }
  }
}

// ---------------------------------------------------------------------------
// Training.  One workgroup takes 16 Q samples of one member through the
// network and back, as in inference with the activations in LDS and a wave's
// 32 features in registers; silu' of a layer stays in the registers of the
// lanes that need it on the way back.  The operands of the weight gradients
// (k = the batch) are read from the LDS tile feature by feature and written
// as whole fragments.
//
// What bounds it, four members of 4096 samples: the chain of eight products
// with one workgroup per CU, and 50 MB of operands written (25 us at 2 TB/s).
// One product per launch, each in 32 x 32 tiles from and to memory in both
// layouts, this took ten launches and 103 us.
struct TrainArgs {
  const float *X, *Y;
  int64_t n_data;
  const int32_t *idx;
  int64_t idx_stride;
  int Bt;
  float gscale;  // 2 / (6 Bt)
  const uint16_t *w1, *w2, *w3, *w4, *w2t, *w3t, *w4t;
  const float *bias;
  const MlpNorm *nm;
  uint16_t *xt, *ht[3], *dt[3], *d4t;
  float *loss_v;
};

// Row blocks [0, NB) of the transposed tile (its columns) to T in fragment
// order: 32 samples x 16 columns per fragment, shared out over the waves.
template <int Q, int NB>
__device__ __forceinline__ void store_t(const uint16_t *tile, int ld, uint16_t *T, int Bt,
                                        int64_t b0, int w, int lane) {
  constexpr int KB = Q / 2;
#pragma unroll
  for (int i0 = 0; i0 < NB * KB; i0 += kInferWaves) {
    const int i = i0 + w;
    if (i >= NB * KB) break;
    const int rb = i / KB, kb = i % KB;
    const uint16_t *src = tile + (32 * kb + 8 * (lane >> 4)) * ld + 16 * rb + (lane & 15);
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = (uint32_t)src[2 * j * ld] | (uint32_t)src[(2 * j + 1) * ld] << 16;
    *reinterpret_cast<uint4 *>(T + frag(16 * rb, b0 + 32 * kb, Bt) + lane * 8) =
        make_uint4(v[0], v[1], v[2], v[3]);
  }
}

// act = silu(acc + bias), sd = silu' (BF16 pairs)
template <int P, int C>
__device__ __forceinline__ void train_epilogue(uint16_t *act, f32x4 (&acc)[P][C],
                                               const float4 (&bias)[C], int w, int lr, int lq,
                                               uint2 (&sd)[P][C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int f0 = 16 * (C * w + c) + lq;
    const float4 b = bias[c];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float h[4], d[4];
      h[0] = silu(acc[p][c][0] + b.x, d[0]);
      h[1] = silu(acc[p][c][1] + b.y, d[1]);
      h[2] = silu(acc[p][c][2] + b.z, d[2]);
      h[3] = silu(acc[p][c][3] + b.w, d[3]);
      *reinterpret_cast<uint2 *>(act + (16 * p + lr) * kActLd + f0) =
          pack4(h[0], h[1], h[2], h[3]);
      sd[p][c] = pack4(d[0], d[1], d[2], d[3]);
    }
  }
}

// act = acc * silu'
template <int P, int C>
__device__ __forceinline__ void back_epilogue(uint16_t *act, f32x4 (&acc)[P][C], int w, int lr,
                                              int lq, const uint2 (&sd)[P][C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int f0 = 16 * (C * w + c) + lq;
#pragma unroll
    for (int p = 0; p < P; ++p)
      *reinterpret_cast<uint2 *>(act + (16 * p + lr) * kActLd + f0) =
          pack4(acc[p][c][0] * unbf(sd[p][c].x & 0xffff),
                acc[p][c][1] * __uint_as_float(sd[p][c].x & 0xffff0000u),
                acc[p][c][2] * unbf(sd[p][c].y & 0xffff),
                acc[p][c][3] * __uint_as_float(sd[p][c].y & 0xffff0000u));
  }
}

constexpr size_t train_lds(int P) {
  return (size_t)P * 16 * (kActLd + 2 * kInLd) * sizeof(uint16_t);
}

template <int Q>
__global__ __launch_bounds__(64 * kInferWaves, 2) void train_kernel(TrainArgs a) {
  constexpr int P = Q, TS = 16 * Q, NW = kInferWaves, C = 16 / NW;
  static_assert(Q % 2 == 0 && Q <= NW, "whole fragments of 32 samples, one output block a wave");
  extern __shared__ uint16_t lds[];
  uint16_t *const xin = lds, *const d4 = lds + TS * kInLd, *const act = lds + 2 * TS * kInLd;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = (lane >> 4) * 4;
  const int64_t b0 = (int64_t)blockIdx.x * TS;
  const int mem = blockIdx.y;
  const MlpNorm *nm = a.nm;
  const int32_t *idx = a.idx ? a.idx + mem * a.idx_stride + b0 : nullptr;
  const auto row_of = [&](int b) {
    const int64_t r = idx ? idx[b] : b0 + b;
    return r < 0 ? 0 : (r >= a.n_data ? a.n_data - 1 : r);
  };
  for (int e = tid; e < TS * kInP; e += 64 * NW) {
    const int b = e / kInP, c = e % kInP;
    float v = 0.f;
    if (c < kIn) v = (a.X[row_of(b) * kIn + c] - nm->in_mean[c]) * nm->in_inv[c];
    xin[b * kInLd + c] = bf(v);
    d4[b * kInLd + c] = 0;
  }
  float yt[4] = {0.f, 0.f, 0.f, 0.f};  // this lane's normalised targets
  if (w < Q && lq < 8) {
    const float *y = a.Y + row_of(16 * w + lr) * kOut;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (lq + q < kOut) yt[q] = (y[lq + q] - nm->out_mean[lq + q]) * nm->out_inv[lq + q];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(yt[q]));  // rounded here
  const float *bias = a.bias + mem * kBias;
  const uint16_t *W2 = a.w2 + mem * kW2, *W3 = a.w3 + mem * kW2, *W4 = a.w4 + mem * kW4;
  const uint16_t *W2T = a.w2t + mem * kW2, *W3T = a.w3t + mem * kW2, *W4T = a.w4t + mem * kW4T;
  const int64_t sH = (int64_t)kTRows * a.Bt, sD = (int64_t)kHid * a.Bt;
  f32x4 acc[P][C];
  uint2 s1[P][C], s2[P][C], s3[P][C];
  float4 b[C];
  WFrag<C> wf = load_w<C, kInP>(a.w1 + mem * kW1, 0, w, lane);
  load_bias<C>(bias, w, lq, b);
  __syncthreads();
  // inputs, transposed, with the row of ones (kIn) of the bias gradient
  if (w < Q) {
    constexpr int KB = Q / 2;
    const int rb = w / KB, kb = w % KB, f = 16 * rb + lr;
    const uint16_t *src = xin + (32 * kb + 2 * lq) * kInLd + f;
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = (uint32_t)src[2 * j * kInLd] | (uint32_t)src[(2 * j + 1) * kInLd] << 16;
      if (f == kIn) v[j] = 0x3f803f80u;
    }
    *reinterpret_cast<uint4 *>(a.xt + (int64_t)mem * kInP * a.Bt +
                               frag(16 * rb, b0 + 32 * kb, a.Bt) + lane * 8) =
        make_uint4(v[0], v[1], v[2], v[3]);
  }
  infer_layer<P, C, 1, kInLd>(xin, a.w1 + mem * kW1, w, lane, wf, acc);
  wf = load_w<C, kHid>(W2, 0, w, lane);
  train_epilogue<P, C>(act, acc, b, w, lr, lq, s1);
  __syncthreads();
  load_bias<C>(bias + kHid, w, lq, b);
  infer_layer<P, C, 8, kActLd>(act, W2, w, lane, wf, acc);
  store_t<Q, 16>(act, kActLd, a.ht[0] + mem * sH, a.Bt, b0, w, lane);
  wf = load_w<C, kHid>(W3, 0, w, lane);
  __syncthreads();
  train_epilogue<P, C>(act, acc, b, w, lr, lq, s2);
  __syncthreads();
  load_bias<C>(bias + 2 * kHid, w, lq, b);
  infer_layer<P, C, 8, kActLd>(act, W3, w, lane, wf, acc);
  store_t<Q, 16>(act, kActLd, a.ht[1] + mem * sH, a.Bt, b0, w, lane);
  __syncthreads();
  train_epilogue<P, C>(act, acc, b, w, lr, lq, s3);
  wf = load_w<C, kInP>(W4T, 0, w, lane);
  __syncthreads();
  // outputs, squared errors (summed in output order) and dL/dY: 16 samples
  // per wave, outputs 0..3 in lanes 0..15 and 4, 5 in lanes 16..31
  if (w < Q) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
      o = mfma(load_w<1, kHid>(W4, kk, 0, lane).v[0],
               ld8(act + (16 * w + lr) * kActLd + 32 * kk + (lane >> 4) * 8), o);
    const float4 b4 = *reinterpret_cast<const float4 *>(bias + 3 * kHid + lq);
    const float r[4] = {o[0] + b4.x - yt[0], o[1] + b4.y - yt[1], o[2] + b4.z - yt[2],
                        o[3] + b4.w - yt[3]};
    float e = fmaf(r[0], r[0], r[1] * r[1]);
    e = fmaf(r[2], r[2], e);
    e = fmaf(r[3], r[3], e);
    e = __shfl(e, lr);  // outputs 0..3 of this sample
    e = fmaf(r[0], r[0], e);
    e = fmaf(r[1], r[1], e);
    if (lq == 4) a.loss_v[(int64_t)mem * a.Bt + b0 + 16 * w + lr] = e;
    if (lq < 8) {
      const bool six = lq == 0;  // outputs 6 and 7 are padding
      *reinterpret_cast<uint2 *>(d4 + (16 * w + lr) * kInLd + lq) =
          pack4(r[0] * a.gscale, r[1] * a.gscale, six ? r[2] * a.gscale : 0.f,
                six ? r[3] * a.gscale : 0.f);
    }
  }
  store_t<Q, 16>(act, kActLd, a.ht[2] + mem * sH, a.Bt, b0, w, lane);
  __syncthreads();
  store_t<Q, 1>(d4, kInLd, a.d4t + (int64_t)mem * kOutP * a.Bt, a.Bt, b0, w, lane);
  infer_layer<P, C, 1, kInLd>(d4, W4T, w, lane, wf, acc);
  wf = load_w<C, kHid>(W3T, 0, w, lane);
  back_epilogue<P, C>(act, acc, w, lr, lq, s3);
  __syncthreads();
  infer_layer<P, C, 8, kActLd>(act, W3T, w, lane, wf, acc);
  store_t<Q, 16>(act, kActLd, a.dt[2] + mem * sD, a.Bt, b0, w, lane);
  wf = load_w<C, kHid>(W2T, 0, w, lane);
  __syncthreads();
  back_epilogue<P, C>(act, acc, w, lr, lq, s2);
  __syncthreads();
  infer_layer<P, C, 8, kActLd>(act, W2T, w, lane, wf, acc);
  store_t<Q, 16>(act, kActLd, a.dt[1] + mem * sD, a.Bt, b0, w, lane);
  __syncthreads();
  back_epilogue<P, C>(act, acc, w, lr, lq, s1);
  __syncthreads();
  store_t<Q, 16>(act, kActLd, a.dt[0] + mem * sD, a.Bt, b0, w, lane);
}

// Weight gradients: part_L[split] = D_L^T [H_{L-1}^T; 1] over kSplitK rows of
// the batch.  Operands in fragment order; a wave takes R blocks of outputs o
// and N of inputs i and ends with four consecutive i of one o per lane.
// Bound by memory: 75 MB read and 36 MB written for four members of 4096
// samples, 24 us (4.6 TB/s); 60 us in 32 x 32 tiles from operands read row by
// row.  Two k steps in flight instead of four: 26 us.
struct DwArgs {
  const uint16_t *xt, *ht[3], *dt[3], *d4t;
  int Bt;
  float *part[4];
};
constexpr int kSplitK = 256;  // batch rows per K split of the weight gradients
constexpr int kLdp[4] = {kInP, kTRows, kTRows, kTRows};
constexpr int kPartM[4] = {kHid, kHid, kHid, kOutP};

template <int R, int N>
__device__ __forceinline__ void dw_tile(const uint16_t *D, const uint16_t *H, int kb, int ob,
                                        int ib, float *part, int ld, int lane) {
  constexpr int KS = kSplitK / 32;
  f32x4 acc[R][N];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int n = 0; n < N; ++n) acc[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint16_t *pd = D + (int64_t)ob * kb * 512 + lane * 8;
  const uint16_t *ph = H + (int64_t)ib * kb * 512 + lane * 8;
  constexpr int DEPTH = 4;  // k steps in flight
  bf16x8 d[DEPTH][R], h[DEPTH][N];
#pragma unroll
  for (int kk = 0; kk < KS + DEPTH - 1; ++kk) {
    if (kk < KS) {
#pragma unroll
      for (int r = 0; r < R; ++r) d[kk % DEPTH][r] = ld8(pd + ((int64_t)r * kb + kk) * 512);
#pragma unroll
      for (int n = 0; n < N; ++n) h[kk % DEPTH][n] = ld8(ph + ((int64_t)n * kb + kk) * 512);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int k = kk - (DEPTH - 1);
    if (k >= 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < N; ++n)
          acc[r][n] = mfma(h[k % DEPTH][n], d[k % DEPTH][r], acc[r][n]);
    }
  }
  const int lr = lane & 15, lq = (lane >> 4) * 4;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int n = 0; n < N; ++n)
      *reinterpret_cast<float4 *>(part + (int64_t)(16 * (ob + r) + lr) * ld + 16 * (ib + n) +
                                  lq) =
          make_float4(acc[r][n][0], acc[r][n][1], acc[r][n][2], acc[r][n][3]);
}

// Six units of eight waves per split: two halves of the outputs of layers 2
// and 3 (waves of 4 x 4 blocks, the last column of waves with the block of
// ones as a fifth), layer 1 and layer 4.
constexpr int kDwUnits = 6;
__global__ __launch_bounds__(512, 2) void dw_kernel(DwArgs a) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int unit = blockIdx.x % kDwUnits, split = blockIdx.x / kDwUnits, mem = blockIdx.y;
  const int kb = a.Bt / 32;
  const int64_t splits = a.Bt / kSplitK, k0 = (int64_t)split * (kSplitK / 32) * 512, B = a.Bt;
  if (unit < 4) {
    const int L = 1 + (unit >> 1);
    const uint16_t *D = a.dt[L] + mem * kHid * B + k0, *H = a.ht[L - 1] + mem * kTRows * B + k0;
    float *part = a.part[L] + (mem * splits + split) * (kHid * kTRows);
    const int ob = 8 * (unit & 1) + 4 * (w >> 2), ib = 4 * (w & 3);
    if ((w & 3) == 3)
      dw_tile<4, 5>(D, H, kb, ob, ib, part, kTRows, lane);
    else
      dw_tile<4, 4>(D, H, kb, ob, ib, part, kTRows, lane);
  } else if (unit == 4) {
    dw_tile<2, 2>(a.dt[0] + mem * kHid * B + k0, a.xt + mem * kInP * B + k0, kb, 2 * w, 0,
                  a.part[0] + (mem * splits + split) * (kHid * kInP), kInP, lane);
  } else {
    const uint16_t *D = a.d4t + mem * kOutP * B + k0, *H = a.ht[2] + mem * kTRows * B + k0;
    float *part = a.part[3] + (mem * splits + split) * (kOutP * kTRows);
    if (w == 7)
      dw_tile<1, 3>(D, H, kb, 0, 14, part, kTRows, lane);
    else
      dw_tile<1, 2>(D, H, kb, 0, 2 * w, part, kTRows, lane);
  }
}

// ---------------------------------------------------------------------------
// Surrogate path helpers.
__device__ inline const double *pick_F(const double *F, int nF, int r) {
  return F + 9 * (int64_t)(nF == 1 ? 0 : r);
}

__global__ void surrogate_inputs_kernel(const double *F, int nF, const float *desc, int n,
                                        float *X) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const double *f = pick_F(F, nF, r);
  float *x = X + (int64_t)r * kIn;
  x[0] = (float)(f[0] - 1.0);
  x[1] = (float)(f[4] - 1.0);
  x[2] = (float)(f[8] - 1.0);
  x[3] = (float)(f[5] + f[7]);
  x[4] = (float)(f[2] + f[6]);
  x[5] = (float)(f[1] + f[3]);
  for (int k = 0; k < 4; ++k) x[6 + k] = desc[4 * (int64_t)r + k];
}

__global__ void surrogate_flags_kernel(const float *X, const float *Y, const float *spread,
                                       int n, mf_estimator est, int32_t *flag) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int f = 0;
  for (int i = 0; i < kIn; ++i) {
    const float x = X[(int64_t)r * kIn + i];
    const float span = est.in_hi[i] - est.in_lo[i];
    const float pad = isfinite(span) ? est.margin * span : 0.f;  // open bounds stay open
    const float lo = est.in_lo[i] - pad, hi = est.in_hi[i] + pad;
    if (!(x >= lo && x <= hi)) f = 2;  // also catches NaN
  }
  if (f == 0) {
    float smax = 0.f, ymax = 0.f;
    for (int i = 0; i < kOut; ++i) {
      const float y = Y[(int64_t)r * kOut + i];
      ymax = fmaxf(ymax, fabsf(y));
      if (spread) smax = fmaxf(smax, spread[(int64_t)r * kOut + i]);
      if (!isfinite(y)) f = 1;
    }
    if (est.kappa * smax > est.tol * fmaxf(ymax, est.sigma_floor)) f = 1;
  }
  flag[r] = f;
}

// C[:, i] = J e(sym(E_i F)) + (W S - S W), W = skew(E_i F): the derivative
// of the stress along the perturbation F_i(h) F (dF_i/dh at 0 = E_i), with
// the rotation of the stress by the spin of the perturbation.
__global__ void surrogate_outputs_kernel(const double *F, int nF, const float *Y,
                                         const float *J, int n, double *sigma, double *C) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double s[6];
  for (int i = 0; i < 6; ++i) s[i] = Y[(int64_t)r * kOut + i];
  for (int i = 0; i < 6; ++i) sigma[(int64_t)r * 6 + i] = s[i];
  if (!C || !J) return;
  const double *f = pick_F(F, nF, r);
  const double S[3][3] = {{s[0], s[5], s[4]}, {s[5], s[1], s[3]}, {s[4], s[3], s[2]}};
  const int vi[6] = {0, 1, 2, 1, 0, 0}, vj[6] = {0, 1, 2, 2, 2, 1};
  for (int col = 0; col < 6; ++col) {
    double E[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    if (col < 3) {
      E[col][col] = 1.0;
    } else {
      E[vi[col]][vj[col]] = 0.5;
      E[vj[col]][vi[col]] = 0.5;
    }
    double G[3][3];
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b)
        G[a][b] = E[a][0] * f[b] + E[a][1] * f[3 + b] + E[a][2] * f[6 + b];
    const double de[6] = {G[0][0], G[1][1], G[2][2], G[1][2] + G[2][1], G[0][2] + G[2][0],
                          G[0][1] + G[1][0]};
    double Wm[3][3];
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) Wm[a][b] = 0.5 * (G[a][b] - G[b][a]);
    double R[3][3];  // W S - S W
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) {
        double v = 0;
        for (int k = 0; k < 3; ++k) v += Wm[a][k] * S[k][b] - S[a][k] * Wm[k][b];
        R[a][b] = v;
      }
    for (int row = 0; row < 6; ++row) {
      double v = 0;
      for (int k = 0; k < 6; ++k) v += (double)J[(int64_t)r * 36 + 6 * row + k] * de[k];
      v += R[vi[row]][vj[row]];
      C[(int64_t)r * 36 + 6 * row + col] = v;
    }
  }
}

}  // namespace mlpk
}  // namespace mf

using namespace mf;
using namespace mf::mlpk;

struct mf_mlp {
  int K = 1;
  int cus = device_cus();  // compute units of the device it lives on
  hipStream_t s = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  DevBuf<float> P, Mo, Ve, bias;
  DevBuf<uint16_t> w1, w2, w3, w4, w2t, w3t, w4t;
  DevBuf<MlpNorm> nm_dev;
  MlpNorm nm{};
  float in_std[kIn], out_std_user[kOut];
  int64_t adam_t = 0;
  // training workspace for mini-batches of Bt samples
  int Bt = 0;
  DevBuf<uint16_t> XT, HT[3], DT[3], D4T;  // operands of the weight gradients
  DevBuf<float> part[4], loss_v, loss_out, loss_acc, grad;
  DevBuf<int32_t> idx;
  mf_estimator est{};
  double last_ms = 0;
  ~mf_mlp() {
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (s) (void)hipStreamDestroy(s);
  }
};

namespace {

int upload_norm(mf_mlp *m) {
  MF_HIP(hipMemcpyAsync(m->nm_dev.p, &m->nm, sizeof(MlpNorm), hipMemcpyHostToDevice, m->s));
  return MF_OK;
}

int run_adam(mf_mlp *m, int mode, float lr, float b1, float b2, float eps, bool loss = false) {
  AdamArgs a;
  std::memset(&a, 0, sizeof(a));
  a.P = m->P.p;
  a.Mo = m->Mo.p;
  a.Ve = m->Ve.p;
  const int splits = m->Bt > 0 ? m->Bt / kSplitK : 0;
  for (int L = 0; L < 4; ++L) {
    a.part[L] = m->part[L].p;
    a.sSplit[L] = (int64_t)kPartM[L] * kLdp[L];
    a.sPart[L] = a.sSplit[L] * splits;
    a.ldp[L] = kLdp[L];
  }
  a.splits = splits;
  a.w1 = m->w1.p;
  a.w2 = m->w2.p;
  a.w3 = m->w3.p;
  a.w4 = m->w4.p;
  a.w2t = m->w2t.p;
  a.w3t = m->w3t.p;
  a.w4t = m->w4t.p;
  a.bias = m->bias.p;
  a.lr = lr;
  a.b1 = b1;
  a.b2 = b2;
  a.eps = eps;
  if (mode == 0) {
    a.bc1 = (float)(1.0 - std::pow((double)b1, (double)m->adam_t));
    a.bc2 = (float)(1.0 - std::pow((double)b2, (double)m->adam_t));
  }
  a.grad = m->grad.p;
  a.mode = mode;
  a.loss_v = m->loss_v.p;
  a.Bt = m->Bt;
  a.loss_inv = m->Bt > 0 ? 1.0f / (6.0f * (float)m->Bt) : 0.f;
  a.loss_out = m->loss_out.p;
  a.loss_acc = m->loss_acc.p;
  hipLaunchKernelGGL(adam_kernel, dim3(kAdamBlocks + (loss ? 1 : 0), m->K), dim3(256), 0, m->s,
                     a);
  MF_HIP(hipGetLastError());
  return MF_OK;
}

int ensure_workspace(mf_mlp *m, int Bt) {
  if (Bt == m->Bt) return MF_OK;
  m->Bt = 0;
  const size_t K = m->K, B = Bt;
  MF_HIP(m->XT.alloc(K * kInP * B));
  for (int l = 0; l < 3; ++l) {
    MF_HIP(m->HT[l].alloc(K * kTRows * B));
    MF_HIP(m->DT[l].alloc(K * kHid * B));
  }
  MF_HIP(m->D4T.alloc(K * kOutP * B));
  const size_t splits = B / kSplitK;
  for (int L = 0; L < 4; ++L) MF_HIP(m->part[L].alloc(K * splits * kPartM[L] * kLdp[L]));
  MF_HIP(m->loss_v.alloc(K * B));
  // rows 256..271 of the activations, which no tile writes: one row of ones
  for (int l = 0; l < 3; ++l) {
    MF_HIP(hipMemsetAsync(m->HT[l].p, 0, sizeof(uint16_t) * m->HT[l].n, m->s));
    hipLaunchKernelGGL(ones_row_kernel, dim3((Bt + 255) / 256, m->K), dim3(256), 0, m->s,
                       m->HT[l].p, (int64_t)kTRows * Bt, kHid, Bt);
    MF_HIP(hipGetLastError());
  }
  m->Bt = Bt;
  return MF_OK;
}

template <int Q>
void launch_train(const TrainArgs &a, int K, hipStream_t s) {
  hipLaunchKernelGGL(train_kernel<Q>, dim3((unsigned)(a.Bt / (16 * Q)), K),
                     dim3(64 * kInferWaves), train_lds(Q), s, a);
}

// Forward, loss and backward of one mini-batch for every member; leaves the
// weight-gradient partials in m->part and the squared errors in m->loss_v.
int forward_backward(mf_mlp *m, const float *X, const float *Y, int64_t n_data,
                     const int32_t *idx, int64_t idx_stride, int Bt) {
  int e = ensure_workspace(m, Bt);
  if (e != MF_OK) return e;
  const int K = m->K;
  TrainArgs a;
  a.X = X;
  a.Y = Y;
  a.n_data = n_data;
  a.idx = idx;
  a.idx_stride = idx_stride;
  a.Bt = Bt;
  a.gscale = 2.0f / (6.0f * (float)Bt);
  a.w1 = m->w1.p;
  a.w2 = m->w2.p;
  a.w3 = m->w3.p;
  a.w4 = m->w4.p;
  a.w2t = m->w2t.p;
  a.w3t = m->w3t.p;
  a.w4t = m->w4t.p;
  a.bias = m->bias.p;
  a.nm = m->nm_dev.p;
  a.xt = m->XT.p;
  a.d4t = m->D4T.p;
  a.loss_v = m->loss_v.p;
  DwArgs d;
  d.xt = a.xt;
  d.d4t = a.d4t;
  d.Bt = Bt;
  for (int l = 0; l < 3; ++l) {
    d.ht[l] = a.ht[l] = m->HT[l].p;
    d.dt[l] = a.dt[l] = m->DT[l].p;
  }
  for (int L = 0; L < 4; ++L) d.part[L] = m->part[L].p;
  // 64 samples per workgroup once that fills the chip
  if ((int64_t)Bt * K >= 64 * m->cus)
    launch_train<4>(a, K, m->s);
  else
    launch_train<2>(a, K, m->s);
  MF_HIP(hipGetLastError());
  hipLaunchKernelGGL(dw_kernel, dim3((unsigned)(Bt / kSplitK * kDwUnits), K), dim3(512), 0, m->s,
                     d);
  MF_HIP(hipGetLastError());
  return MF_OK;
}

// A grid dimension counts its threads in 32 bits and wraps silently, so calls of
// more than 2^21 tiles (at most 2^31 threads; 2^25 rows with a Jacobian, 2^27 without)
// take several launches, each of whole tiles.
template <int Q, int NT, int G>
void launch_infer(InferArgs a, hipStream_t s) {
  constexpr int64_t kRows = (int64_t)(1 << 21) * 16 * Q;
  static_assert(64 * kInferWaves * G * (kRows / (16 * Q)) <= (int64_t)UINT32_MAX, "threads");
  for (int64_t left = a.n; left > 0; left -= kRows) {
    a.n = std::min(left, kRows);
    hipLaunchKernelGGL((infer_kernel<Q, NT, G>),
                       dim3((unsigned)((a.n + 16 * Q - 1) / (16 * Q)), NT ? 6 / NT : 1),
                       dim3(64 * kInferWaves * G), infer_lds(Q * (1 + NT), G), s, a);
    a.X += kRows * kIn;
    a.Y += kRows * kOut;
    if (a.J) a.J += kRows * 36;
    if (a.spread) a.spread += kRows * kOut;
  }
}
template <int Q, int NT, int G>
hipError_t infer_attr() {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(&infer_kernel<Q, NT, G>),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)infer_lds(Q * (1 + NT), G));
}

// Row orders of epoch `ep`, one Fisher-Yates shuffle per member: a serial chain
// of 2.8 ns per row, so the members of a larger ensemble go to a thread each
// (four members of 131072 rows: 1.5 -> 0.5 ms; below some 10^5 rows in all
// starting the threads costs what they save).
void shuffle_members(int32_t *perm, int K, int64_t n, uint64_t seed, int64_t ep) {
  const auto one = [=](int k) {
    int32_t *p = perm + (size_t)k * n;
    for (int64_t i = 0; i < n; ++i) p[i] = (int32_t)i;
    SplitMix64 rng(seed, (uint64_t)ep * K + k);
    for (int64_t i = n - 1; i > 0; --i) {
      const int64_t j = (int64_t)(rng.next() % (uint64_t)(i + 1));
      std::swap(p[i], p[j]);
    }
  };
  std::vector<std::thread> ts;
  int k = 1;
  if (K > 1 && K * n >= 100000) {
    try {
      for (; k < K; ++k) ts.emplace_back(one, k);
    } catch (...) {  // no more threads: the rest here
    }
  }
  one(0);
  for (; k < K; ++k) one(k);
  for (auto &t : ts) t.join();
}

bool valid_batch(int64_t Bt) { return Bt > 0 && Bt % MF_MLP_BATCH_ALIGN == 0 && Bt <= (1 << 24); }

}  // namespace

namespace mf {

int mlp_members(const mf_mlp *m) { return m->K; }
const mf_estimator &mlp_estimator(const mf_mlp *m) { return m->est; }

int mlp_predict(mf_mlp *m, int member, const float *X, int64_t n, float *Y, float *J,
                float *spread, hipStream_t s) {
  if (n <= 0) return MF_OK;
  InferArgs a;
  a.X = X;
  a.n = n;
  a.m0 = member < 0 ? 0 : member;
  a.mcount = member < 0 ? m->K : 1;
  a.w1 = m->w1.p;
  a.w2 = m->w2.p;
  a.w3 = m->w3.p;
  a.w4 = m->w4.p;
  a.bias = m->bias.p;
  a.nm = m->nm_dev.p;
  a.Y = Y;
  a.J = J;
  a.spread = spread;
  // Up to one workgroup per CU the time is the chain of layers and members, so
  // the call is cut finer: two members at a time, 16 samples and (with J) two
  // of the six tangent planes per workgroup, each repeating plane 0.  Four
  // members, wide against fine: 777 points with J 47 -> 33 us (1361 points,
  // two workgroups on some CUs: 47 against 48), 4096 points without J
  // 42 -> 29.5 us (5600 points: 42 against 42).
  const int64_t t16 = (n + 15) / 16;
  if (J) {
    if (3 * t16 <= m->cus)
      launch_infer<1, 2, 2>(a, s);
    else
      launch_infer<1, 6, 1>(a, s);
  } else if (t16 <= m->cus) {
    launch_infer<1, 0, 2>(a, s);
  } else {
    launch_infer<4, 0, 1>(a, s);
  }
  MF_HIP(hipGetLastError());
  return MF_OK;
}

hipError_t launch_surrogate_inputs(const double *F, int nF, const float *desc, int n, float *X,
                                   hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(surrogate_inputs_kernel, dim3((n + 255) / 256), dim3(256), 0, s, F, nF,
                     desc, n, X);
  return hipGetLastError();
}

hipError_t launch_surrogate_flags(const float *X, const float *Y, const float *spread, int n,
                                  const mf_estimator &est, int32_t *flag, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(surrogate_flags_kernel, dim3((n + 255) / 256), dim3(256), 0, s, X, Y,
                     spread, n, est, flag);
  return hipGetLastError();
}

hipError_t launch_surrogate_outputs(const double *F, int nF, const float *Y, const float *J,
                                    int n, double *sigma, double *C, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(surrogate_outputs_kernel, dim3((n + 255) / 256), dim3(256), 0, s, F, nF,
                     Y, J, n, sigma, C);
  return hipGetLastError();
}

}  // namespace mf

extern "C" {

int32_t mf_mlp_num_params(void) { return kNumParams; }
int32_t mf_mlp_num_members(const mf_mlp *m) { return m ? m->K : 0; }

void mf_default_train_params(mf_train_params *tp) {
  if (!tp) return;
  tp->epochs = 20;
  tp->batch = 4096;
  tp->seed = 1;
  tp->lr = 2e-3f;
  tp->lr_final = 2e-5f;
  tp->beta1 = 0.9f;
  tp->beta2 = 0.999f;
  tp->eps = 1e-8f;
}

int mf_mlp_create(int32_t n_members, uint64_t seed, mf_mlp **out) {
  if (!out || n_members < 1 || n_members > MF_MLP_MAX_MEMBERS) {
    set_error("mf_mlp_create: n_members must be 1..MF_MLP_MAX_MEMBERS");
    return MF_ERR_INVALID;
  }
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
    set_error("mf_mlp_create: no HIP device");
    return MF_ERR_HIP;
  }
  mf_mlp *m = new mf_mlp;
  m->K = n_members;
  auto fail = [&](int e) {
    delete m;
    return e;
  };
  if (hipStreamCreateWithFlags(&m->s, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess) {
    set_error("mf_mlp_create: stream/event creation failed");
    return fail(MF_ERR_HIP);
  }
  // per device: the seven-plane tile needs 68 KB, above the 64 KB default
  if (infer_attr<4, 0, 1>() != hipSuccess || infer_attr<1, 0, 2>() != hipSuccess ||
      infer_attr<1, 6, 1>() != hipSuccess || infer_attr<1, 2, 2>() != hipSuccess) {
    set_error("mf_mlp_create: LDS attribute");
    return fail(MF_ERR_HIP);
  }
  const size_t K = n_members;
  std::vector<float> P(K * kNumParams);
  // U(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
  for (size_t k = 0; k < K; ++k) {
    SplitMix64 rng(seed, 1000 + k);
    float *w = P.data() + k * kNumParams;
    auto fill = [&](int off, int cnt, int fan_in) {
      const double b = 1.0 / std::sqrt((double)fan_in);
      for (int i = 0; i < cnt; ++i) w[off + i] = (float)((2.0 * rng.uniform() - 1.0) * b);
    };
    fill(kOffW1, kHid * kIn, kIn);
    fill(kOffB1, kHid, kIn);
    fill(kOffW2, kHid * kHid, kHid);
    fill(kOffB2, kHid, kHid);
    fill(kOffW3, kHid * kHid, kHid);
    fill(kOffB3, kHid, kHid);
    fill(kOffW4, kOut * kHid, kHid);
    fill(kOffB4, kOut, kHid);
  }
  int e = MF_OK;
  auto chk = [&](hipError_t h) {
    if (h != hipSuccess && e == MF_OK) {
      set_error(std::string("mf_mlp_create: ") + hipGetErrorString(h));
      e = MF_ERR_HIP;
    }
  };
  chk(m->P.upload(P, m->s));
  chk(m->Mo.alloc(P.size()));
  chk(m->Ve.alloc(P.size()));
  chk(m->bias.alloc(K * kBias));
  chk(m->w1.alloc(K * kW1));
  chk(m->w2.alloc(K * kW2));
  chk(m->w3.alloc(K * kW2));
  chk(m->w4.alloc(K * kW4));
  chk(m->w2t.alloc(K * kW2));
  chk(m->w3t.alloc(K * kW2));
  chk(m->w4t.alloc(K * kW4T));
  chk(m->nm_dev.alloc(1));
  chk(m->grad.alloc(K * kNumParams));
  chk(m->loss_out.alloc(K));
  chk(m->loss_acc.alloc(K));
  if (e != MF_OK) return fail(e);
  chk(hipMemsetAsync(m->Mo.p, 0, sizeof(float) * m->Mo.n, m->s));
  chk(hipMemsetAsync(m->Ve.p, 0, sizeof(float) * m->Ve.n, m->s));
  chk(hipMemsetAsync(m->bias.p, 0, sizeof(float) * m->bias.n, m->s));
  chk(hipMemsetAsync(m->w1.p, 0, sizeof(uint16_t) * m->w1.n, m->s));
  chk(hipMemsetAsync(m->w4.p, 0, sizeof(uint16_t) * m->w4.n, m->s));
  chk(hipMemsetAsync(m->w4t.p, 0, sizeof(uint16_t) * m->w4t.n, m->s));
  if (e != MF_OK) return fail(e);
  for (int i = 0; i < kIn; ++i) {
    m->nm.in_mean[i] = 0.f;
    m->nm.in_inv[i] = 1.f;
    m->in_std[i] = 1.f;
    m->est.in_lo[i] = -INFINITY;
    m->est.in_hi[i] = INFINITY;
  }
  for (int i = 0; i < 8; ++i) {
    m->nm.out_mean[i] = 0.f;
    m->nm.out_std[i] = 1.f;
    m->nm.out_inv[i] = 1.f;
  }
  for (int i = 0; i < kOut; ++i) m->out_std_user[i] = 1.f;
  m->est.margin = 0.f;
  m->est.kappa = 1.f;
  m->est.sigma_floor = 0.f;
  m->est.tol = INFINITY;
  if ((e = upload_norm(m)) != MF_OK) return fail(e);
  if ((e = run_adam(m, 2, 0, 0, 0, 0)) != MF_OK) return fail(e);
  if (hipStreamSynchronize(m->s) != hipSuccess) {
    set_error("mf_mlp_create: initialisation failed");
    return fail(MF_ERR_HIP);
  }
  *out = m;
  return MF_OK;
}

void mf_mlp_destroy(mf_mlp *m) { delete m; }

int mf_mlp_set_normalization(mf_mlp *m, const float *in_mean, const float *in_std,
                             const float *out_mean, const float *out_std) {
  if (!m || !in_mean || !in_std || !out_mean || !out_std) {
    set_error("mf_mlp_set_normalization: null argument");
    return MF_ERR_INVALID;
  }
  for (int i = 0; i < kIn; ++i) {
    const float sd = in_std[i] > 0.f ? in_std[i] : 1.f;
    m->nm.in_mean[i] = in_mean[i];
    m->in_std[i] = sd;
    m->nm.in_inv[i] = (float)(1.0 / (double)sd);
  }
  for (int i = 0; i < kOut; ++i) {
    const float sd = out_std[i] > 0.f ? out_std[i] : 1.f;
    m->nm.out_mean[i] = out_mean[i];
    m->nm.out_std[i] = sd;
    m->out_std_user[i] = sd;
    m->nm.out_inv[i] = (float)(1.0 / (double)sd);
  }
  int e = upload_norm(m);
  if (e != MF_OK) return e;
  MF_HIP(hipStreamSynchronize(m->s));
  return MF_OK;
}

int mf_mlp_get_normalization(const mf_mlp *m, float *in_mean, float *in_std, float *out_mean,
                             float *out_std) {
  if (!m) return MF_ERR_INVALID;
  for (int i = 0; i < kIn; ++i) {
    if (in_mean) in_mean[i] = m->nm.in_mean[i];
    if (in_std) in_std[i] = m->in_std[i];
  }
  for (int i = 0; i < kOut; ++i) {
    if (out_mean) out_mean[i] = m->nm.out_mean[i];
    if (out_std) out_std[i] = m->nm.out_std[i];
  }
  return MF_OK;
}

int mf_mlp_get_weights(mf_mlp *m, int32_t member, float *w) {
  if (!m || !w || member < 0 || member >= m->K) {
    set_error("mf_mlp_get_weights: bad member or buffer");
    return MF_ERR_INVALID;
  }
  MF_HIP(hipMemcpyAsync(w, m->P.p + (size_t)member * kNumParams, sizeof(float) * kNumParams,
                        hipMemcpyDeviceToHost, m->s));
  MF_HIP(hipStreamSynchronize(m->s));
  return MF_OK;
}

int mf_mlp_set_weights(mf_mlp *m, int32_t member, const float *w) {
  if (!m || !w || member < 0 || member >= m->K) {
    set_error("mf_mlp_set_weights: bad member or buffer");
    return MF_ERR_INVALID;
  }
  const size_t off = (size_t)member * kNumParams;
  MF_HIP(hipMemcpyAsync(m->P.p + off, w, sizeof(float) * kNumParams, hipMemcpyHostToDevice,
                        m->s));
  MF_HIP(hipMemsetAsync(m->Mo.p + off, 0, sizeof(float) * kNumParams, m->s));
  MF_HIP(hipMemsetAsync(m->Ve.p + off, 0, sizeof(float) * kNumParams, m->s));
  int e = run_adam(m, 2, 0, 0, 0, 0);
  if (e != MF_OK) return e;
  MF_HIP(hipStreamSynchronize(m->s));
  return MF_OK;
}

int mf_mlp_train_step_device(mf_mlp *m, const float *X_dev, const float *Y_dev,
                             int64_t n_data, const int32_t *idx_dev, int32_t batch, float lr,
                             float *loss) {
  if (!m || !X_dev || !Y_dev || n_data <= 0 || !valid_batch(batch) ||
      (!idx_dev && batch > n_data)) {
    set_error("mf_mlp_train_step_device: bad arguments (batch must be a positive multiple of "
              "MF_MLP_BATCH_ALIGN)");
    return MF_ERR_INVALID;
  }
  int e = forward_backward(m, X_dev, Y_dev, n_data, idx_dev, batch, batch);
  if (e != MF_OK) return e;
  m->adam_t += 1;
  if ((e = run_adam(m, 0, lr, 0.9f, 0.999f, 1e-8f, loss != nullptr)) != MF_OK) return e;
  if (loss) {
    std::vector<float> l(m->K);
    MF_HIP(hipMemcpyAsync(l.data(), m->loss_out.p, sizeof(float) * m->K,
                          hipMemcpyDeviceToHost, m->s));
    MF_HIP(hipStreamSynchronize(m->s));
    double sum = 0;
    for (float v : l) sum += v;
    *loss = (float)(sum / m->K);
  }
  return MF_OK;
}

int mf_mlp_fit_device(mf_mlp *m, const float *X_dev, const float *Y_dev, int64_t n,
                      const mf_train_params *tp, float *epoch_loss) {
  if (!m || !X_dev || !Y_dev || !tp || tp->epochs < 0 || !valid_batch(tp->batch) ||
      n < tp->batch || n > (int64_t)1 << 30) {
    set_error("mf_mlp_fit_device: bad arguments");
    return MF_ERR_INVALID;
  }
  const int K = m->K, Bt = tp->batch;
  const int64_t steps = n / Bt;
  const int64_t total = steps * tp->epochs;
  std::vector<int32_t> perm((size_t)K * n);
  MF_HIP(m->idx.ensure(perm.size()));
  int64_t it = 0;
  MF_HIP(hipStreamSynchronize(m->s));  // an earlier call is done with idx
  if (tp->epochs > 0) shuffle_members(perm.data(), K, n, tp->seed, 0);
  for (int ep = 0; ep < tp->epochs; ++ep) {
    MF_HIP(hipMemcpyAsync(m->idx.p, perm.data(), sizeof(int32_t) * perm.size(),
                          hipMemcpyHostToDevice, m->s));
    MF_HIP(hipEventRecord(m->ev0, m->s));
    MF_HIP(hipMemsetAsync(m->loss_acc.p, 0, sizeof(float) * K, m->s));
    for (int64_t st = 0; st < steps; ++st, ++it) {
      const double frac = total > 1 ? (double)it / (double)(total - 1) : 1.0;
      const float lr = (float)(tp->lr_final + 0.5 * (tp->lr - tp->lr_final) *
                                                  (1.0 + std::cos(3.14159265358979323846 * frac)));
      int e = forward_backward(m, X_dev, Y_dev, n, m->idx.p + st * Bt, n, Bt);
      if (e != MF_OK) return e;
      m->adam_t += 1;
      if ((e = run_adam(m, 0, lr, tp->beta1, tp->beta2, tp->eps, true)) != MF_OK) return e;
    }
    if (ep + 1 < tp->epochs) {  // the next epoch's orders, while this one runs
      MF_HIP(hipEventSynchronize(m->ev0));  // perm is uploaded
      shuffle_members(perm.data(), K, n, tp->seed, ep + 1);
    }
    if (epoch_loss) {
      std::vector<float> l(K);
      MF_HIP(hipMemcpyAsync(l.data(), m->loss_acc.p, sizeof(float) * K, hipMemcpyDeviceToHost,
                            m->s));
      MF_HIP(hipStreamSynchronize(m->s));
      for (int k = 0; k < K; ++k)
        epoch_loss[(size_t)ep * K + k] = steps > 0 ? l[k] / (float)steps : 0.f;
    }
  }
  MF_HIP(hipStreamSynchronize(m->s));
  return MF_OK;
}

int mf_mlp_gradient_device(mf_mlp *m, int32_t member, const float *X_dev, const float *Y_dev,
                           int32_t n, float *grad_host, float *loss) {
  if (!m || member < 0 || member >= m->K || !X_dev || !Y_dev || !grad_host ||
      !valid_batch(n)) {
    set_error("mf_mlp_gradient_device: bad arguments");
    return MF_ERR_INVALID;
  }
  int e = forward_backward(m, X_dev, Y_dev, n, nullptr, 0, n);
  if (e != MF_OK) return e;
  if ((e = run_adam(m, 1, 0, 0, 0, 0, true)) != MF_OK) return e;
  MF_HIP(hipMemcpyAsync(grad_host, m->grad.p + (size_t)member * kNumParams,
                        sizeof(float) * kNumParams, hipMemcpyDeviceToHost, m->s));
  float l = 0;
  MF_HIP(hipMemcpyAsync(&l, m->loss_out.p + member, sizeof(float), hipMemcpyDeviceToHost,
                        m->s));
  MF_HIP(hipStreamSynchronize(m->s));
  if (loss) *loss = l;
  return MF_OK;
}

int mf_mlp_predict_device(mf_mlp *m, int32_t member, const float *X_dev, int64_t n,
                          float *Y_dev, float *J_dev, float *spread_dev) {
  if (!m || member < -1 || member >= m->K || n < 0 || (n > 0 && (!X_dev || !Y_dev)) ||
      n > ((int64_t)1 << 31) * 16) {
    set_error("mf_mlp_predict_device: bad arguments");
    return MF_ERR_INVALID;
  }
  MF_HIP(hipEventRecord(m->ev0, m->s));
  int e = mlp_predict(m, member, X_dev, n, Y_dev, J_dev, spread_dev, m->s);
  if (e != MF_OK) return e;
  MF_HIP(hipEventRecord(m->ev1, m->s));
  MF_HIP(hipEventSynchronize(m->ev1));
  float ms = 0;
  MF_HIP(hipEventElapsedTime(&ms, m->ev0, m->ev1));
  m->last_ms = ms;
  return MF_OK;
}

int mf_mlp_last_predict_ms(const mf_mlp *m, double *ms) {
  if (!m || !ms) return MF_ERR_INVALID;
  *ms = m->last_ms;
  return MF_OK;
}

void *mf_mlp_stream(mf_mlp *m) { return m ? (void *)m->s : nullptr; }

int mf_mlp_set_estimator(mf_mlp *m, const mf_estimator *est) {
  if (!m || !est || !(est->margin >= 0.f) || !(est->kappa >= 0.f) ||
      !(est->sigma_floor >= 0.f) || !(est->tol >= 0.f)) {
    set_error("mf_mlp_set_estimator: bad arguments");
    return MF_ERR_INVALID;
  }
  m->est = *est;
  return MF_OK;
}

int mf_mlp_get_estimator(const mf_mlp *m, mf_estimator *est) {
  if (!m || !est) return MF_ERR_INVALID;
  *est = m->est;
  return MF_OK;
}

}  // extern "C"
