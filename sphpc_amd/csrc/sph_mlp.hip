// Lambda warm-start network: FP32 training kernels (forward, backward, Adam)
// and the BF16 MFMA inference path, behind the sph_mlp_* C ABI.
//
// The network has no counterpart in the reference; its inputs are reference
// quantities of the constraint solve (neighbour count, neighbors.h:27; density,
// particles.c:512; previous lambda, particles.c:664; |grad C|^2, particles.c:
// 654-661; SDF distance and gradient, obstacle_cuda.cu:33-53,88) plus the
// velocity divergence and first density moments.
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "sph_internal.h"
#include "sph_mlp_dev.h"

namespace sph {

constexpr int kGradGroup = 32;      // samples of a wave's pass through the network
constexpr int kGradWaves = 8;       // waves per block of the gradient kernel
constexpr int kMaxGradBlocks = 256; // one block per CU
constexpr int kMomentCols = 2 * (kMlpIn + 1);  // sums and squares of 12 features + target
constexpr int kMomentBlocks = 512;

// splitmix64 (Steele, Lea, Flood 2014) for counter-based batch sampling.
__host__ __device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ uint64_t batch_row(uint64_t k, uint64_t count, uint64_t seed,
                                              int random) {
  return random ? mix64(seed ^ mix64(k)) % count : k;
}

// ---------------------------------------------------------------------------
// FP32 network on the matrix cores
// ---------------------------------------------------------------------------
// All products of the training and of the FP32 forward pass are FP32 MFMA
// (v_mfma_f32_32x32x2_f32, FP32 inputs and accumulation).  A wave takes 32
// samples as the columns of Z^T = W^T X^T, hidden units as rows, so a lane
// holds one sample (lane % 32) and, in accumulator v of row block rb, hidden
// unit 32 rb + mfma_drow(v, lane / 32).  An MFMA's B operand wants k = lane / 32
// of column lane % 32, so accumulator (rb, v) is by itself a B operand whose
// two k are the units the two lane halves hold: the next layer takes it as its
// k chunk 16 rb + v without moving data, and the weights (its A operand) are
// laid out in LDS in that order of k.  Lane half h reads features 6 h .. 6 h + 5
// of its sample, chunk c of layer 1 being features (c, 6 + c).
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kHalfIn = kMlpIn / 2;
constexpr int kSA1 = 0;                         // W1 operands [rb][2][lane][4]: 6 chunks, 2 unused
constexpr int kSA2 = kSA1 + 2 * 2 * 64 * 4;     // W2^T operands [out block][8][lane][4]
constexpr int kSBias = kSA2 + 2 * 8 * 64 * 4;   // b1, b2, w3 by [rb][half][v]
constexpr int kSNorm = kSBias + 3 * kMlpH;      // feature means and reciprocal deviations
constexpr int kSForward = kSNorm + 2 * kMlpPad; // floats of the forward pass
constexpr int kSA3 = kSForward;                 // W2 operands [in block][8][lane][4]
constexpr int kSGrad = kSA3 + 2 * 8 * 64 * 4;   // floats of the gradient pass

// LDS word of the operand element (row `row`, k = hidden unit u) of a 64 x 64
// operand [row block][8][lane][4]: unit u is k chunk 16 rb + v of lane half hf
// where u = 32 rb + mfma_drow(v, hf).
__device__ __forceinline__ int mlp32_slot(int row, int u) {
  const int kc = 16 * (u >> 5) + 4 * ((u >> 3) & 3) + (u & 3);
  return (((row >> 5) * 8 + (kc >> 2)) * 64 + 32 * ((u >> 2) & 1) + (row & 31)) * 4 + (kc & 3);
}

// Lays the weights out in LDS as the operands above (all threads of a block).
template <bool GRAD>
__device__ __forceinline__ void mlp32_weights(const float *__restrict__ theta,
                                              const float *__restrict__ norm, float *sm) {
  static_assert(kNormMu == 0 && kNormIsd == kMlpPad, "means, then reciprocal deviations");
  if (threadIdx.x < 2 * kMlpPad) sm[kSNorm + threadIdx.x] = norm[threadIdx.x];
  for (int e = threadIdx.x; e < 2 * 2 * 64 * 4; e += blockDim.x) {
    const int rb = e >> 9, c = ((e >> 8) & 1) * 4 + (e & 3), l = (e >> 2) & 63;
    sm[kSA1 + e] = c < kHalfIn
                       ? theta[kMlpW1 + (c + kHalfIn * (l >> 5)) * kMlpH + 32 * rb + (l & 31)]
                       : 0.0f;
  }
  // W2 is read in its own order (coalesced) and scattered in LDS
  for (int e = threadIdx.x; e < kMlpH * kMlpH; e += blockDim.x) {
    const int r = e >> 6, c = e & 63;
    const float w = theta[kMlpW2 + e];
    sm[kSA2 + mlp32_slot(c, r)] = w;
    if (GRAD) sm[kSA3 + mlp32_slot(r, c)] = w;
  }
  if (threadIdx.x < kMlpH) {
    const int e = threadIdx.x, u = 32 * (e >> 5) + mfma_drow(e & 15, (e >> 4) & 1);
    sm[kSBias + e] = theta[kMlpB1 + u];
    sm[kSBias + kMlpH + e] = theta[kMlpB2 + u];
    sm[kSBias + 2 * kMlpH + e] = theta[kMlpW3 + u];
  }
}

// This lane's 16 values of a [rb][half][v] vector.
__device__ __forceinline__ void mlp32_vec(const float *v, int rb, int half, float (&out)[16]) {
  const float4 *q = reinterpret_cast<const float4 *>(v) + (rb * 2 + half) * 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 a = q[i];
    out[4 * i] = a.x; out[4 * i + 1] = a.y; out[4 * i + 2] = a.z; out[4 * i + 3] = a.w;
  }
}

__device__ __forceinline__ floatx16_t mlp32_bias(const float *v, int rb, int half) {
  float b[16];
  mlp32_vec(v, rb, half, b);
  floatx16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = b[i];
  return acc;
}

// Layer 1: z[rb] from this lane's six features.
__device__ __forceinline__ void mlp32_layer1(const float *sm, const float (&x)[kHalfIn], int lane,
                                             floatx16_t (&z)[2]) {
  const float4 *A = reinterpret_cast<const float4 *>(sm + kSA1);
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float4 a = A[(rb * 2) * 64 + lane], b = A[(rb * 2 + 1) * 64 + lane];
    const float w[kHalfIn] = {a.x, a.y, a.z, a.w, b.x, b.y};
    floatx16_t acc = mlp32_bias(sm + kSBias, rb, lane >> 5);
#pragma unroll
    for (int c = 0; c < kHalfIn; ++c)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(w[c], x[c], acc, 0, 0, 0);
    z[rb] = acc;
  }
}

// z[ob] += (64 x 64 operands at A) h, over the 32 k chunks that h's
// accumulators are.
__device__ __forceinline__ void mlp32_square(const float *ops, const floatx16_t (&h)[2], int lane,
                                             floatx16_t (&z)[2]) {
  const float4 *A = reinterpret_cast<const float4 *>(ops);
  float4 a = A[lane], b = A[8 * 64 + lane];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float wa[4] = {a.x, a.y, a.z, a.w}, wb[4] = {b.x, b.y, b.z, b.w};
    if (q < 7) {  // the next operands come in under this chunk's products
      a = A[(q + 1) * 64 + lane];
      b = A[(9 + q) * 64 + lane];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float k = h[q >> 2][(q & 3) * 4 + e];
      z[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[e], k, z[0], 0, 0, 0);
      z[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(wb[e], k, z[1], 0, 0, 0);
    }
    // without it the compiler loads all operands first and spills
    __builtin_amdgcn_sched_barrier(0);
  }
}

// 1 / (1 + e^-z) to about 1 ulp: e^-z as the hardware exp2 of -z log2(e) in two
// floats, and the hardware reciprocal with one Newton step (8 VALU and two
// transcendentals; expf and two IEEE divisions are about 40).  z is held to
// [-88.5, 100] for the exponential only: e^88.5 is still finite, and its reciprocal,
// below the normal range, is 0 from v_rcp_f32.  So z * sigmoid32(z) ends at 0 however
// large -z is; a bound with a normal reciprocal leaves 1.6e-38 z (-1.6 at -1e38).
__device__ __forceinline__ float sigmoid32(float z) {
  const float zc = __builtin_amdgcn_fmed3f(z, -88.5f, 100.0f);
  const float t = -1.44269504f * zc;  // log2(e) = 1.44269502 + 1.92596303e-8
  const float lo = fmaf(-1.92596303e-8f, zc, fmaf(-1.44269504f, zc, -t));
  const float p = __builtin_amdgcn_exp2f(t);
  const float d = 1.0f + fmaf(0.693147182f * p, lo, p);
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(r, fmaf(-d, r, 1.0f), r);
}

// The LDS writes of a wave before, its reads after: a lane reads what other
// lanes of its own wave wrote (LDS operations of a wave complete in order).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // and nothing of the next phase moves up into this one's registers
  __builtin_amdgcn_sched_barrier(0);
}

// Gradient sums leave a block in register order, slot x 64 lanes, and
// k_mlp_adam finds each parameter in it (grad_param): slots 0-63 dW2, 64-79 dW1
// with db1 as its thirteenth row, 80 dw3, 81 db2, 82 db3 and the loss.
constexpr int kSlotW2 = 0, kSlotW1 = 64, kSlotW3 = 80, kSlotB2 = 81, kSlotMisc = 82,
              kGradSlots = 83;
constexpr int kGradWords = kGradSlots * 64;

// Parameter of word (slot, lane), -1 for none, -2 for the loss.
__device__ __forceinline__ int grad_param(int slot, int lane) {
  if (slot < kSlotW1) {
    const int jb = slot >> 5, mb = (slot >> 4) & 1;
    return kMlpW2 + (32 * jb + mfma_drow(slot & 15, lane >> 5)) * kMlpH + 32 * mb + (lane & 31);
  }
  if (slot < kSlotW3) {
    const int q = slot - kSlotW1, i = lane & 15;
    const int j = 16 * (q >> 2) + 4 * (lane >> 4) + (q & 3);
    return i < kMlpIn ? kMlpW1 + i * kMlpH + j : (i == kMlpIn ? kMlpB1 + j : -1);
  }
  if (slot == kSlotW3) return kMlpW3 + lane;
  if (slot == kSlotB2) return kMlpB2 + lane;
  return lane == 0 ? kMlpB3 : (lane == 1 ? -2 : -1);
}

constexpr int kTLd = 68;  // LDS row of 64 units (16-byte aligned, rows 4 banks apart)
constexpr int kWaveLds = kGradGroup * kTLd + kGradGroup * 16;

constexpr size_t kGradLds = sizeof(float) * (kSGrad + kGradWaves * kWaveLds);
static_assert(4 * kGradWords * sizeof(float) <= kGradLds && kGradLds <= 160 * 1024,
              "four waves' sums fit in the LDS of the pass");

// Per-block partial gradient of L = 0.5/B sum (y - t_n)^2 over a batch, with
// x normalised by (x - mu) * inv_sigma and t_n = (t - y_shift) / y_scale.
//
// A wave takes 32 samples at a time through both passes in registers: 216 MFMA
// of 64 cycles and 32 of half the size, 14,800 matrix cycles, and about 1,800
// VALU.  FP32 MFMA runs in the vector units' time on this target (with two
// waves per SIMD the counters show the two one after the other, 47% MFMA busy),
// so their sum bounds it: 16 us for 65,536 samples.  The weight gradients sum
// over samples, so H1, dZ2 and dZ1 go through a 32 x 64 LDS tile of the wave's
// own to become operands with k = sample.  A block is a CU's worth of waves
// (two per SIMD, at 256 registers) and adds their sums in LDS, so that at most
// 256 partials leave the chip instead of one per 64 samples.  Measured with
// k_mlp_adam per step of 65,536 samples: 434 us with the products on the vector
// units, each reading its weight from LDS, to 44 us (39 of them here); of
// 1,000,003: 373 us.
__global__ __launch_bounds__(64 * kGradWaves) void k_mlp_grad(
    uint64_t batch, uint64_t count, const float *__restrict__ x, const float *__restrict__ t,
    uint64_t seed, int random, const float *__restrict__ theta, const float *__restrict__ norm,
    float inv_batch, float *__restrict__ partial) {
  extern __shared__ __align__(16) float sm[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31;
  const uint64_t groups = (batch + kGradGroup - 1) / kGradGroup;
  const uint64_t g0 = (uint64_t)wave * gridDim.x + blockIdx.x, gstep = (uint64_t)gridDim.x * kGradWaves;
  // a group's raw rows, loaded before the work that hides their latency: the
  // weights' way into LDS for the first group
  f2u raw[kHalfIn / 2];
  float traw = 0.0f;
  auto fetch = [&](uint64_t g) {
    const uint64_t k = g * kGradGroup + col;
#pragma unroll
    for (int c = 0; c < kHalfIn / 2; ++c) raw[c] = f2u{0.0f, 0.0f};
    if (k < batch) {
      const uint64_t row = batch_row(k, count, seed, random);
      const float *r = x + row * kMlpPad + kHalfIn * half;
#pragma unroll
      for (int c = 0; c < kHalfIn / 2; ++c) raw[c] = reinterpret_cast<const f2u *>(r)[c];
      traw = t[row];
    }
  };
  fetch(g0);
  mlp32_weights<true>(theta, norm, sm);
  float *T = sm + kSGrad + wave * kWaveLds;  // [sample][unit]
  float *X = T + kGradGroup * kTLd;          // [sample][feature], feature 12 = 1
  const float y_shift = norm[kNormYShift], inv_scale = 1.0f / norm[kNormYScale];
  const float b3 = theta[kMlpB3];
  __syncthreads();

  floatx16_t gW2[2][2] = {};  // [row block of W2's inputs][column block of its outputs]
  floatx4_t gW1[4] = {};
  float gw3 = 0.0f, gb2[2] = {0.0f, 0.0f}, gb3 = 0.0f, loss = 0.0f;
  for (uint64_t g = g0; g < groups; g += gstep) {
    // the operands are read again for each group: kept in registers over the
    // loop, as the compiler would, they cost 120 that the sums need
    int again = 0;
    asm volatile("" : "+s"(again));
    const float *W = sm + again;
    const uint64_t k = g * kGradGroup + col;
    const float tn = (traw - y_shift) * inv_scale;
    float xn[kHalfIn];
    const float *mu = W + kSNorm + kHalfIn * half, *isd = mu + kMlpPad;
#pragma unroll
    for (int c = 0; c < kHalfIn; ++c)  // a sample past the batch is zero after normalisation
      xn[c] = k < batch ? (raw[c / 2][c & 1] - mu[c]) * isd[c] : 0.0f;
#pragma unroll
    for (int c = 0; c < kHalfIn; ++c) X[col * 16 + kHalfIn * half + c] = xn[c];
    if (half) {
      X[col * 16 + 12] = 1.0f;
      X[col * 16 + 13] = X[col * 16 + 14] = X[col * 16 + 15] = 0.0f;
    }
    floatx16_t h1[2];
    mlp32_layer1(W, xn, lane, h1);
    if (g + gstep < groups) fetch(g + gstep);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float z = h1[rb][v];
        h1[rb][v] = z * sigmoid32(z);
      }
    __builtin_amdgcn_sched_barrier(0);
    floatx16_t d2[2];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) d2[ob] = mlp32_bias(W + kSBias + kMlpH, ob, half);
    mlp32_square(W + kSA2, h1, lane, d2);
    // H1 as dW2's A operand: unit lane % 32 of sample 2 c + half
    float4 *Tw = reinterpret_cast<float4 *>(T + col * kTLd + 4 * half);
    auto put = [&](const floatx16_t &m, int rb) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        Tw[8 * rb + 2 * q] = make_float4(m[4 * q], m[4 * q + 1], m[4 * q + 2], m[4 * q + 3]);
    };
    put(h1[0], 0);
    put(h1[1], 1);
    wave_lds_fence();
    float h1t[2][16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      h1t[0][c] = T[(2 * c + half) * kTLd + col];
      h1t[1][c] = T[(2 * c + half) * kTLd + 32 + col];
    }
    wave_lds_fence();
    float yp = 0.0f;
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
      float w3[16];
      mlp32_vec(W + kSBias + 2 * kMlpH, ob, half, w3);
      floatx16_t h2;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float z = d2[ob][v], s = sigmoid32(z);
        h2[v] = z * s;
        d2[ob][v] = s * fmaf(z, 1.0f - s, 1.0f) * w3[v];
        yp = fmaf(w3[v], h2[v], yp);
      }
      put(h2, ob);
      __builtin_amdgcn_sched_barrier(0);
    }
    yp += __shfl_xor(yp, 32, 64);
    float dy = 0.0f;
    if (k < batch) {
      const float r = yp + b3 - tn;
      if (!half) loss = fmaf(r, r, loss);
      dy = r * inv_batch;
    }
    if (!half) gb3 += dy;
    wave_lds_fence();
#pragma unroll
    for (int s = 0; s < kGradGroup; ++s)
      gw3 = fmaf(T[s * kTLd + lane],
                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dy), s)), gw3);
#pragma unroll
    for (int ob = 0; ob < 2; ++ob)
#pragma unroll
      for (int v = 0; v < 16; ++v) d2[ob][v] *= dy;  // dZ2
    wave_lds_fence();
    put(d2[0], 0);
    put(d2[1], 1);
    wave_lds_fence();
    // dW2 += H1^T dZ2, two samples a chunk
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const float z0 = T[(2 * c + half) * kTLd + col], z1 = T[(2 * c + half) * kTLd + 32 + col];
      gb2[0] += z0;
      gb2[1] += z1;
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        gW2[jb][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(h1t[jb][c], z0, gW2[jb][0], 0, 0, 0);
        gW2[jb][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(h1t[jb][c], z1, gW2[jb][1], 0, 0, 0);
      }
      if ((c & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
    // dZ1 = (W2 dZ2) * silu'(Z1), Z1 computed again: held since the forward
    // pass its derivative took 32 registers, and spilled
    floatx16_t a1[2] = {};
    mlp32_square(W + kSA3, d2, lane, a1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kHalfIn; ++c) xn[c] = X[col * 16 + kHalfIn * half + c];
    mlp32_layer1(W, xn, lane, d2);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float z = d2[rb][v], s = sigmoid32(z);
        a1[rb][v] *= s * fmaf(z, 1.0f - s, 1.0f);
      }
    wave_lds_fence();
    put(a1[0], 0);
    put(a1[1], 1);
    wave_lds_fence();
    // [dW1; db1]^T += dZ1^T [X 1], four samples a chunk
    const int r4 = lane >> 4, c16 = lane & 15;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float xv = X[(4 * c + r4) * 16 + c16];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        gW1[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(
            T[(4 * c + r4) * kTLd + 16 * jb + c16], xv, gW1[jb], 0, 0, 0);
      if (c & 1) __builtin_amdgcn_sched_barrier(0);
    }
    wave_lds_fence();
  }

  float sum[kGradSlots];
#pragma unroll
  for (int q = 0; q < 64; ++q) sum[kSlotW2 + q] = gW2[q >> 5][(q >> 4) & 1][q & 15];
#pragma unroll
  for (int q = 0; q < 16; ++q) sum[kSlotW1 + q] = gW1[q >> 2][q & 3];
  sum[kSlotW3] = gw3;
#pragma unroll
  for (int b = 0; b < 2; ++b) gb2[b] += __shfl_xor(gb2[b], 32, 64);
  sum[kSlotB2] = half ? gb2[1] : gb2[0];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    gb3 += __shfl_xor(gb3, o, 64);
    loss += __shfl_xor(loss, o, 64);
  }
  sum[kSlotMisc] = lane == 0 ? gb3 : (lane == 1 ? loss : 0.0f);
  // sums of the waves that had samples: the upper four onto the lower four,
  // then those by all threads (the weights' LDS is free by now)
  const int busy = (int)min((uint64_t)kGradWaves, (groups + gridDim.x - 1) / gridDim.x);
  __syncthreads();
  if (busy > 4) {
    if (wave >= 4 && wave < busy) {
#pragma unroll
      for (int q = 0; q < kGradSlots; ++q) sm[(wave - 4) * kGradWords + q * 64 + lane] = sum[q];
    }
    __syncthreads();
    if (wave + 4 < busy) {
#pragma unroll
      for (int q = 0; q < kGradSlots; ++q) sum[q] += sm[wave * kGradWords + q * 64 + lane];
    }
    __syncthreads();
  }
  const int left = min(busy, 4);
  if (wave < left) {
#pragma unroll
    for (int q = 0; q < kGradSlots; ++q) sm[wave * kGradWords + q * 64 + lane] = sum[q];
  }
  __syncthreads();
  float *P = partial + (size_t)blockIdx.x * kGradWords;
  for (int e = threadIdx.x; e < kGradWords; e += blockDim.x) {
    float a = sm[e];
    for (int w = 1; w < left; ++w) a += sm[w * kGradWords + e];
    P[e] = a;
  }
}

// Sums the block partials in a fixed order (deterministic) and optionally
// applies one Adam step (Kingma & Ba, beta1 0.9, beta2 0.999, eps 1e-8; bc =
// bias corrections).  One block per slot of 64 parameters, its eight waves
// taking every eighth partial: with one thread walking all partials of a
// parameter in turn (1024 of them, 21 blocks) this took 279 us, now 5.4 us
// (256 partials).  The padding inputs have no word here; their gradient stays
// the zero it was created as.
constexpr int kAdamWaves = 8;
__global__ __launch_bounds__(64 * kAdamWaves) void k_mlp_adam(
    int nblocks, const float *__restrict__ partial, float *__restrict__ theta,
    float *__restrict__ mom, float *__restrict__ vel, float *__restrict__ grad,
    float *__restrict__ loss_out, float inv_batch, float lr, float bc1, float bc2, int apply) {
  __shared__ float part[kAdamWaves][64];
  const int slot = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float g = 0.0f;
#pragma unroll 8
  for (int b = wave; b < nblocks; b += kAdamWaves)
    g += partial[(size_t)b * kGradWords + slot * 64 + lane];
  part[wave][lane] = g;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < kAdamWaves; ++w) g += part[w][lane];
  const int p = grad_param(slot, lane);
  if (p == -2) *loss_out = 0.5f * g * inv_batch;
  if (p < 0) return;
  grad[p] = g;
  if (apply) {
    const float m = 0.9f * mom[p] + 0.1f * g;
    const float v = 0.999f * vel[p] + 0.001f * g * g;
    mom[p] = m;
    vel[p] = v;
    theta[p] -= lr * (m / bc1) / (sqrtf(v / bc2) + 1e-8f);
  }
}

// FP32 forward pass on FP32 MFMA, 32 samples per wave and pass, the weights in
// LDS for all the passes of a block.  76 MFMA (4,900 cycles) and 64 sigmoids
// (4,400) bound it, 130 us for a million rows.  Measured at 1,000,003 rows: 311
// us with a thread per sample and its weights broadcast from LDS, to 138 us.
constexpr int kForwardBlocks = 1024;  // four per CU
__global__ __launch_bounds__(kBlock, 4) void k_mlp_forward(uint64_t count,
                                                           const float *__restrict__ x,
                                                           const float *__restrict__ theta,
                                                           const float *__restrict__ norm,
                                                           float *__restrict__ y) {
  __shared__ __align__(16) float sm[kSForward];
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  mlp32_weights<false>(theta, norm, sm);
  const float scale = norm[kNormYScale], shift = norm[kNormYShift], b3 = theta[kMlpB3];
  __syncthreads();
  const uint64_t groups = (count + kGradGroup - 1) / kGradGroup;
  for (uint64_t g = (uint64_t)blockIdx.x * (kBlock / kWave) + (threadIdx.x >> 6); g < groups;
       g += (uint64_t)gridDim.x * (kBlock / kWave)) {
    int again = 0;  // the operands stay in LDS, as in k_mlp_grad
    asm volatile("" : "+s"(again));
    const float *W = sm + again;
    const uint64_t k = g * kGradGroup + col;
    float xn[kHalfIn];
#pragma unroll
    for (int c = 0; c < kHalfIn; ++c) xn[c] = 0.0f;
    if (k < count) {
      const f2u *r = reinterpret_cast<const f2u *>(x + k * kMlpPad + kHalfIn * half);
      const float *mu = W + kSNorm + kHalfIn * half, *isd = mu + kMlpPad;
#pragma unroll
      for (int c = 0; c < kHalfIn; ++c) xn[c] = (r[c / 2][c & 1] - mu[c]) * isd[c];
    }
    floatx16_t h1[2], z2[2];
    mlp32_layer1(W, xn, lane, h1);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 16; ++v) h1[rb][v] *= sigmoid32(h1[rb][v]);
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) z2[ob] = mlp32_bias(W + kSBias + kMlpH, ob, half);
    mlp32_square(W + kSA2, h1, lane, z2);
    float out = 0.0f;
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
      float w3[16];
      mlp32_vec(W + kSBias + 2 * kMlpH, ob, half, w3);
#pragma unroll
      for (int v = 0; v < 16; ++v) out = fmaf(w3[v], z2[ob][v] * sigmoid32(z2[ob][v]), out);
    }
    out += __shfl_xor(out, 32, 64);
    if (!half && k < count) y[k] = (out + b3) * scale + shift;
  }
}

// BF16 MFMA inference of a standalone batch (the path fused into the solver).
template <bool AHEAD>
__global__ __launch_bounds__(kBlock) void k_mlp_infer(uint64_t count, const float *__restrict__ x,
                                                      const MlpPacked *__restrict__ M,
                                                      float *__restrict__ y) {
  const uint64_t s = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  float f[kMlpPad];
#pragma unroll
  for (int i = 0; i < kMlpPad; ++i) f[i] = 0.0f;
  if (s < count) {
    const float4 *r = reinterpret_cast<const float4 *>(x + s * kMlpPad);
    const float4 a = r[0], b = r[1], c = r[2];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    f[8] = c.x; f[9] = c.y; f[10] = c.z; f[11] = c.w;
  }
  const float out = mlp_wave<AHEAD>(f, M);  // whole wave, including lanes past the end
  if (s < count) y[s] = out;
}

// Rows up to which a wave has a SIMD to itself, or shares it with one more (us, without /
// with the operands loaded ahead): 4096 rows 7.0 / 5.8, 65,536 7.4 / 6.0, 131,072 8.3 /
// 8.2, 262,144 13.4 / 13.8, a million 42.7 / 47.2.
constexpr uint64_t kInferAhead = 1 << 17;

// Packs FP32 master weights into MFMA operand order (BF16) for inference.
__global__ __launch_bounds__(kBlock) void k_mlp_pack(const float *__restrict__ theta,
                                                     const float *__restrict__ norm,
                                                     MlpPacked *__restrict__ M) {
  const int tid = threadIdx.x;
  for (int e = tid; e < 2 * 64; e += kBlock) {  // a1[rb][lane]
    const int rb = e >> 6, l = e & 63, half = l >> 5, col = 32 * rb + (l & 31);
    uint32_t w[4];
    for (int q = 0; q < 4; ++q) {
      const int k0 = 8 * half + 2 * q;
      w[q] = pack_bf16x2(theta[kMlpW1 + k0 * kMlpH + col], theta[kMlpW1 + (k0 + 1) * kMlpH + col]);
    }
    M->a1[e] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  for (int e = tid; e < 2 * 4 * 64; e += kBlock) {  // a2[ob][kc][lane]
    const int ob = e >> 8, kc = (e >> 6) & 3, l = e & 63, half = l >> 5, col = 32 * ob + (l & 31);
    uint32_t w[4];
    for (int q = 0; q < 4; ++q) {
      const int r0 = mlp_l2_hidden(kc, half, 2 * q), r1 = mlp_l2_hidden(kc, half, 2 * q + 1);
      w[q] = pack_bf16x2(theta[kMlpW2 + r0 * kMlpH + col], theta[kMlpW2 + r1 * kMlpH + col]);
    }
    M->a2[e] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  if (tid < 64) {  // [rb][half][v]
    const int rb = tid >> 5, half = (tid >> 4) & 1, v = tid & 15;
    const int u = 32 * rb + mfma_drow(v, half);
    reinterpret_cast<float *>(M->b1)[tid] = theta[kMlpB1 + u];
    reinterpret_cast<float *>(M->b2)[tid] = theta[kMlpB2 + u];
    reinterpret_cast<float *>(M->w3)[tid] = bf16_round(theta[kMlpW3 + u]);
  }
  if (tid < kNormWords) M->norm[tid] = norm[tid];
  if (tid == 0) M->b3 = theta[kMlpB3];
}

// Per-block sums and squares (FP64) of the 12 features and the target.
__global__ __launch_bounds__(kBlock) void k_mlp_moments(uint64_t count, const float *__restrict__ x,
                                                        const float *__restrict__ t,
                                                        double *__restrict__ partial) {
  __shared__ double red[kBlock / 64][kMomentCols];
  double acc[kMomentCols];
#pragma unroll
  for (int c = 0; c < kMomentCols; ++c) acc[c] = 0.0;
  for (uint64_t s = (uint64_t)blockIdx.x * kBlock + threadIdx.x; s < count;
       s += (uint64_t)gridDim.x * kBlock) {
#pragma unroll
    for (int i = 0; i <= kMlpIn; ++i) {
      const double v = i < kMlpIn ? (double)x[s * kMlpPad + i] : (double)t[s];
      acc[2 * i] += v;
      acc[2 * i + 1] += v * v;
    }
  }
#pragma unroll
  for (int c = 0; c < kMomentCols; ++c) {
    double v = acc[c];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = v;
  }
  __syncthreads();
  if (threadIdx.x < kMomentCols) {
    double v = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) v += red[w][threadIdx.x];
    partial[(size_t)blockIdx.x * kMomentCols + threadIdx.x] = v;
  }
}

static int mlp_configure() {
  static int done = 0;
  if (done) return SPH_OK;
  SPH_HIP(hipFuncSetAttribute((const void *)k_mlp_grad,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kGradLds));
  done = 1;
  return SPH_OK;
}

}  // namespace sph

using namespace sph;

struct sph_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  float *theta = nullptr, *mom = nullptr, *vel = nullptr, *grad = nullptr;
  float *norm = nullptr;
  float *partial = nullptr, *loss = nullptr;
  double *moments = nullptr;
  MlpPacked *packed = nullptr;
  float host_norm[kNormWords] = {};
  long long step = 0;
};

static int mlp_arg(const char *msg) {
  set_error(msg);
  return SPH_ERR_ARG;
}

static int upload_norm(sph_mlp *m) {
  SPH_HIP(hipMemcpyAsync(m->norm, m->host_norm, sizeof(m->host_norm), hipMemcpyHostToDevice,
                         m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

static void mlp_free(sph_mlp *m) {
  void *bufs[] = {m->theta, m->mom, m->vel, m->grad, m->norm, m->partial,
                  m->loss, m->moments, m->packed};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  if (m->stream) (void)hipStreamDestroy(m->stream);
}

extern "C" int sph_mlp_create(sph_mlp **out) {
  if (!out) return mlp_arg("NULL argument");
  *out = nullptr;
  int rc = mlp_configure();
  if (rc) return rc;
  sph_mlp *m = new sph_mlp();
  hipError_t e = hipGetDevice(&m->device);
  if (e == hipSuccess) e = hipStreamCreate(&m->stream);
  struct { void **p; size_t bytes; } allocs[] = {
      {(void **)&m->theta, sizeof(float) * kMlpParams},
      {(void **)&m->mom, sizeof(float) * kMlpParams},
      {(void **)&m->vel, sizeof(float) * kMlpParams},
      {(void **)&m->grad, sizeof(float) * kMlpParams},
      {(void **)&m->norm, sizeof(float) * kNormWords},
      {(void **)&m->partial, sizeof(float) * kGradWords * kMaxGradBlocks},
      {(void **)&m->loss, sizeof(float)},
      {(void **)&m->moments, sizeof(double) * kMomentCols * kMomentBlocks},
      {(void **)&m->packed, sizeof(MlpPacked)},
  };
  for (auto &a : allocs)
    if (e == hipSuccess) e = hipMalloc(a.p, a.bytes);
  for (float *z : {m->theta, m->mom, m->vel, m->grad})
    if (e == hipSuccess) e = hipMemsetAsync(z, 0, sizeof(float) * kMlpParams, m->stream);
  if (e != hipSuccess) {
    mlp_free(m);
    delete m;
    return hip_fail(e, "sph_mlp_create");
  }
  for (int i = 0; i < kMlpIn; ++i) m->host_norm[kNormIsd + i] = 1.0f;
  m->host_norm[kNormYScale] = 1.0f;
  rc = upload_norm(m);
  if (rc) {
    mlp_free(m);
    delete m;
    return rc;
  }
  *out = m;
  return SPH_OK;
}

extern "C" int sph_mlp_destroy(sph_mlp *m) {
  if (!m) return SPH_OK;
  (void)hipStreamSynchronize(m->stream);
  mlp_free(m);
  delete m;
  return SPH_OK;
}

extern "C" int sph_mlp_set_weights(sph_mlp *m, const float *theta) {
  if (!m || !theta) return mlp_arg("NULL argument");
  SPH_HIP(hipMemcpyAsync(m->theta, theta, sizeof(float) * kMlpParams, hipMemcpyHostToDevice,
                         m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

extern "C" int sph_mlp_get_weights(sph_mlp *m, float *theta) {
  if (!m || !theta) return mlp_arg("NULL argument");
  SPH_HIP(hipMemcpyAsync(theta, m->theta, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost,
                         m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

// He-style uniform initialisation: W ~ U(-1, 1) * sqrt(3 / fan_in), zero biases,
// zero rows for the padding inputs.  Also resets the optimiser.
extern "C" int sph_mlp_init(sph_mlp *m, unsigned long long seed) {
  if (!m) return mlp_arg("NULL argument");
  std::vector<float> th(kMlpParams, 0.0f);
  uint64_t ctr = seed * 0x2545f4914f6cdd1dull;
  auto uni = [&]() { return (double)(mix64(ctr++) >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0; };
  for (int i = 0; i < kMlpIn; ++i)
    for (int j = 0; j < kMlpH; ++j) th[kMlpW1 + i * kMlpH + j] = (float)(uni() * sqrt(3.0 / kMlpIn));
  for (int i = 0; i < kMlpH * kMlpH; ++i) th[kMlpW2 + i] = (float)(uni() * sqrt(3.0 / kMlpH));
  for (int i = 0; i < kMlpH; ++i) th[kMlpW3 + i] = (float)(uni() * sqrt(3.0 / kMlpH));
  int rc = sph_mlp_set_weights(m, th.data());
  if (rc) return rc;
  SPH_HIP(hipMemsetAsync(m->mom, 0, sizeof(float) * kMlpParams, m->stream));
  SPH_HIP(hipMemsetAsync(m->vel, 0, sizeof(float) * kMlpParams, m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  m->step = 0;
  return SPH_OK;
}

extern "C" int sph_mlp_reset_optimizer(sph_mlp *m) {
  if (!m) return mlp_arg("NULL argument");
  SPH_HIP(hipMemsetAsync(m->mom, 0, sizeof(float) * kMlpParams, m->stream));
  SPH_HIP(hipMemsetAsync(m->vel, 0, sizeof(float) * kMlpParams, m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  m->step = 0;
  return SPH_OK;
}

extern "C" int sph_mlp_set_normalization(sph_mlp *m, const float *mean, const float *stddev,
                                         float target_mean, float target_std) {
  if (!m || !mean || !stddev) return mlp_arg("NULL argument");
  if (!(target_std > 0.0f)) return mlp_arg("target_std must be positive");
  for (int i = 0; i < kMlpIn; ++i) {
    if (!(stddev[i] >= 0.0f)) return mlp_arg("feature stddev must be >= 0");
    m->host_norm[kNormMu + i] = mean[i];
    m->host_norm[kNormIsd + i] = stddev[i] > 0.0f ? 1.0f / stddev[i] : 0.0f;
  }
  m->host_norm[kNormYShift] = target_mean;
  m->host_norm[kNormYScale] = target_std;
  return upload_norm(m);
}

extern "C" int sph_mlp_set_output_clip(sph_mlp *m, float max_target) {
  if (!m) return mlp_arg("NULL argument");
  if (!(max_target >= 0.0f)) return mlp_arg("max_target must be >= 0 (0: no clip)");
  m->host_norm[kNormYMax] = max_target;
  return upload_norm(m);
}

extern "C" float sph_mlp_get_output_clip(sph_mlp *m) { return m ? m->host_norm[kNormYMax] : 0.0f; }

extern "C" int sph_mlp_set_step_scale(sph_mlp *m, float scale) {
  if (!m) return mlp_arg("NULL argument");
  if (!(scale > 0.0f)) return mlp_arg("scale must be positive");
  m->host_norm[kNormStep] = scale;
  return upload_norm(m);
}

extern "C" float sph_mlp_get_step_scale(sph_mlp *m) {
  return (m && m->host_norm[kNormStep] > 0.0f) ? m->host_norm[kNormStep] : 1.0f;
}

extern "C" int sph_mlp_get_normalization(sph_mlp *m, float *mean, float *stddev,
                                         float *target_mean, float *target_std) {
  if (!m) return mlp_arg("NULL argument");
  for (int i = 0; i < kMlpIn; ++i) {
    if (mean) mean[i] = m->host_norm[kNormMu + i];
    const float isd = m->host_norm[kNormIsd + i];
    if (stddev) stddev[i] = isd > 0.0f ? 1.0f / isd : 0.0f;
  }
  if (target_mean) *target_mean = m->host_norm[kNormYShift];
  if (target_std) *target_std = m->host_norm[kNormYScale];
  return SPH_OK;
}

// Mean and standard deviation of the features and the target over a device
// dataset (FP64 sums), installed as the network's normalisation.
extern "C" int sph_mlp_fit_normalization(sph_mlp *m, const float *x, const float *t,
                                         size_t count) {
  if (!m || !x || !t) return mlp_arg("NULL argument");
  if (count < 2) return mlp_arg("need at least two samples");
  const int nb = (int)std::min<size_t>(kMomentBlocks, (count + kBlock - 1) / kBlock);
  k_mlp_moments<<<nb, kBlock, 0, m->stream>>>(count, x, t, m->moments);
  SPH_HIP(hipGetLastError());
  std::vector<double> part((size_t)nb * kMomentCols);
  SPH_HIP(hipMemcpyAsync(part.data(), m->moments, sizeof(double) * part.size(),
                         hipMemcpyDeviceToHost, m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  double sum[kMomentCols] = {};
  for (int b = 0; b < nb; ++b)
    for (int c = 0; c < kMomentCols; ++c) sum[c] += part[(size_t)b * kMomentCols + c];
  float mean[kMlpIn], sd[kMlpIn], tm = 0.0f, ts = 1.0f;
  for (int i = 0; i <= kMlpIn; ++i) {
    const double mu = sum[2 * i] / (double)count;
    const double var = std::max(0.0, sum[2 * i + 1] / (double)count - mu * mu);
    double s = sqrt(var);
    if (s < 1e-12 * std::max(1.0, fabs(mu))) s = 0.0;
    if (i < kMlpIn) {
      mean[i] = (float)mu;
      sd[i] = (float)s;
    } else {
      tm = (float)mu;
      ts = s > 0.0 ? (float)s : 1.0f;
    }
  }
  return sph_mlp_set_normalization(m, mean, sd, tm, ts);
}

static int grad_pass(sph_mlp *m, const float *x, const float *t, size_t count, size_t batch,
                     uint64_t seed, int random, float lr, int apply) {
  const uint64_t groups = (batch + kGradGroup - 1) / kGradGroup;
  const int nb = (int)std::min<uint64_t>(kMaxGradBlocks, groups);
  const float inv_batch = (float)(1.0 / (double)batch);
  k_mlp_grad<<<nb, 64 * kGradWaves, kGradLds, m->stream>>>(
      batch, count, x, t, seed, random, m->theta, m->norm, inv_batch, m->partial);
  SPH_HIP(hipGetLastError());
  float bc1 = 1.0f, bc2 = 1.0f;
  if (apply) {
    m->step += 1;
    bc1 = (float)(1.0 - pow(0.9, (double)m->step));
    bc2 = (float)(1.0 - pow(0.999, (double)m->step));
  }
  k_mlp_adam<<<kGradSlots, 64 * kAdamWaves, 0, m->stream>>>(
      nb, m->partial, m->theta, m->mom, m->vel, m->grad, m->loss, inv_batch, lr, bc1, bc2, apply);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

extern "C" int sph_mlp_gradient(sph_mlp *m, const float *x, const float *t, size_t count,
                                float *grad, float *loss) {
  if (!m || !x || !t) return mlp_arg("NULL argument");
  if (count == 0) return mlp_arg("empty batch");
  int rc = grad_pass(m, x, t, count, count, 0, 0, 0.0f, 0);
  if (rc) return rc;
  if (grad)
    SPH_HIP(hipMemcpyAsync(grad, m->grad, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost,
                           m->stream));
  if (loss)
    SPH_HIP(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

extern "C" int sph_mlp_train_step(sph_mlp *m, const float *x, const float *t, size_t count,
                                  size_t batch, float lr, unsigned long long seed, float *loss) {
  if (!m || !x || !t) return mlp_arg("NULL argument");
  if (count == 0) return mlp_arg("empty dataset");
  if (!(lr > 0.0f)) return mlp_arg("learning rate must be positive");
  const int random = batch != 0;
  if (!random) batch = count;
  int rc = grad_pass(m, x, t, count, batch, seed, random, lr, 1);
  if (rc) return rc;
  if (loss) {
    SPH_HIP(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
    SPH_HIP(hipStreamSynchronize(m->stream));
  }
  return SPH_OK;
}

extern "C" int sph_mlp_forward(sph_mlp *m, const float *x, size_t count, float *y) {
  if (!m || (count && (!x || !y))) return mlp_arg("NULL argument");
  if (!count) return SPH_OK;
  const uint64_t per_block = (uint64_t)kGradGroup * (kBlock / kWave);
  const uint64_t blocks = std::min<uint64_t>(kForwardBlocks, (count + per_block - 1) / per_block);
  k_mlp_forward<<<(unsigned)blocks, kBlock, 0, m->stream>>>(count, x, m->theta, m->norm, y);
  SPH_HIP(hipGetLastError());
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

namespace sph {
int mlp_pack(sph_mlp *m, MlpPacked *dst, hipStream_t s) {
  // the weights come from m's stream; work on that stream is ordered as it is
  if (s != m->stream) SPH_HIP(hipStreamSynchronize(m->stream));
  k_mlp_pack<<<1, kBlock, 0, s>>>(m->theta, m->norm, dst);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}
}  // namespace sph

extern "C" int sph_mlp_infer_bf16(sph_mlp *m, const float *x, size_t count, float *y) {
  if (!m || (count && (!x || !y))) return mlp_arg("NULL argument");
  if (((uintptr_t)x & 15u) != 0) return mlp_arg("features must be 16-byte aligned");
  int rc = mlp_pack(m, m->packed, m->stream);
  if (rc || !count) return rc;
  const auto infer = count <= kInferAhead ? k_mlp_infer<true> : k_mlp_infer<false>;
  infer<<<(unsigned)((count + kBlock - 1) / kBlock), kBlock, 0, m->stream>>>(count, x, m->packed,
                                                                             y);
  SPH_HIP(hipGetLastError());
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

extern "C" int sph_mlp_synchronize(sph_mlp *m) {
  if (!m) return mlp_arg("NULL argument");
  SPH_HIP(hipStreamSynchronize(m->stream));
  return SPH_OK;
}

// File format: 8-byte magic "SPHMLP01", int32 parameter count, int32 norm
// word count, FP32 parameters, FP32 normalisation words (little endian).
static const char kMagic[8] = {'S', 'P', 'H', 'M', 'L', 'P', '0', '1'};

extern "C" int sph_mlp_save(sph_mlp *m, const char *path) {
  if (!m || !path) return mlp_arg("NULL argument");
  std::vector<float> th(kMlpParams);
  int rc = sph_mlp_get_weights(m, th.data());
  if (rc) return rc;
  FILE *f = fopen(path, "wb");
  if (!f) return mlp_arg("cannot open file for writing");
  const int32_t hdr[2] = {kMlpParams, kNormWords};
  bool ok = fwrite(kMagic, 1, 8, f) == 8 && fwrite(hdr, 4, 2, f) == 2 &&
            fwrite(th.data(), 4, kMlpParams, f) == (size_t)kMlpParams &&
            fwrite(m->host_norm, 4, kNormWords, f) == (size_t)kNormWords;
  ok = (fclose(f) == 0) && ok;
  return ok ? SPH_OK : mlp_arg("write failed");
}

extern "C" int sph_mlp_load(sph_mlp *m, const char *path) {
  if (!m || !path) return mlp_arg("NULL argument");
  FILE *f = fopen(path, "rb");
  if (!f) return mlp_arg("cannot open network file");
  char magic[8];
  int32_t hdr[2];
  std::vector<float> th(kMlpParams);
  float nrm[kNormWords];
  bool ok = fread(magic, 1, 8, f) == 8 && memcmp(magic, kMagic, 8) == 0 &&
            fread(hdr, 4, 2, f) == 2 && hdr[0] == kMlpParams && hdr[1] == kNormWords &&
            fread(th.data(), 4, kMlpParams, f) == (size_t)kMlpParams &&
            fread(nrm, 4, kNormWords, f) == (size_t)kNormWords;
  fclose(f);
  if (!ok) return mlp_arg("not a network file of this layout");
  memcpy(m->host_norm, nrm, sizeof(nrm));
  int rc = upload_norm(m);
  if (rc) return rc;
  rc = sph_mlp_set_weights(m, th.data());
  if (rc) return rc;
  return sph_mlp_reset_optimizer(m);
}
