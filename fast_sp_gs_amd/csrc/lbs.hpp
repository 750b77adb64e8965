// Shared by the LBS blend forward and backward: the per-control-point table and the neighbour weights.
// Reference behaviour reproduced: fast_2d_gs/network.py:498-521 (calc_LBS_weight) and :545-573 (warp).
#pragma once
#include "common.hpp"

namespace fsgs {
namespace {

// Per control point (one lane each), kXf floats in 16-byte aligned rows, so that a point gathers a neighbour's transform and
// residuals as five 16-byte loads (as 18 separate words they were most of the blend's time: 15 us for 200k points):
//   [0,9)  rotation matrix of qhat = normalize(sp_rot + (0,0,0,1)) (identity without sp_rot)
//   [9,12) translation (re-centred about the control point for warp mode 2: t + c - R c)
//   [12,16) rotation residual     [16,20) scale residual (zeros behind the S columns)
//   [20]   1 / (2 exp(log_radius)^2)     [21] sigmoid(weight_logit) (1 without one)
//   [22,26) qhat     [26] 1 / |q| (floored at 1e-12)     [27] 1 if |q| <= 1e-12 (the projection term of the
//   normalisation's derivative then drops), else 0.
constexpr int kXf = 28, kXfRot = 12, kXfScale = 16, kXfI2 = 20, kXfSig = 21, kXfQ = 22, kXfInvLen = 26, kXfDegenerate = 27;
struct LbsTransform {  // what a point needs of a neighbour
  float4 a0, a1, a2, r, s;  // R row-major, then t
  __device__ __forceinline__ explicit LbsTransform(const float4* q) {
    a0 = q[0], a1 = q[1], a2 = q[2], r = q[3], s = q[4];
  }
  __device__ __forceinline__ float R(int k) const {
    const float v[9] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w, a2.x};
    return v[k];
  }
  __device__ __forceinline__ float t(int k) const { return k == 0 ? a2.y : k == 1 ? a2.z : a2.w; }
  __device__ __forceinline__ float rot(int k) const { return k == 0 ? r.x : k == 1 ? r.y : k == 2 ? r.z : r.w; }
  __device__ __forceinline__ float scale(int k) const { return k == 0 ? s.x : k == 1 ? s.y : k == 2 ? s.z : s.w; }
};
__global__ void __launch_bounds__(256) lbs_prepare_kernel(int M, int warp_mode, const float* __restrict__ sp_points,
    const float* __restrict__ sp_t, const float* __restrict__ sp_rot, const float* __restrict__ sp_r,
    const float* __restrict__ sp_s, int S, int sp_s_ld, const float* __restrict__ log_radius,
    const float* __restrict__ weight_logit, float* __restrict__ xf) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= M) return;
  float R[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  float t[3] = {sp_t[3 * j], sp_t[3 * j + 1], sp_t[3 * j + 2]};
  float qh[4] = {0, 0, 0, 1}, nq = 1.0f, degenerate = 0.0f;
  if (warp_mode != 0) {
    const float q[4] = {sp_rot[4 * j], sp_rot[4 * j + 1], sp_rot[4 * j + 2], sp_rot[4 * j + 3] + 1.0f};
    const float nrm  = sqrtf(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
    nq               = 1.0f / fmaxf(nrm, 1e-12f);
    degenerate       = nrm <= 1e-12f ? 1.0f : 0.0f;
    const float x = q[0] * nq, y = q[1] * nq, z = q[2] * nq, w = q[3] * nq;
    qh[0] = x, qh[1] = y, qh[2] = z, qh[3] = w;
    R[0] = 1 - 2 * (y * y + z * z), R[1] = 2 * (x * y - z * w), R[2] = 2 * (y * w + x * z);
    R[3] = 2 * (x * y + z * w), R[4] = 1 - 2 * (x * x + z * z), R[5] = 2 * (y * z - x * w);
    R[6] = 2 * (x * z - y * w), R[7] = 2 * (x * w + y * z), R[8] = 1 - 2 * (x * x + y * y);
    if (warp_mode == 2) {
      const float* c = sp_points + 3 * j;
#pragma unroll
      for (int a = 0; a < 3; ++a) t[a] = t[a] + c[a] - (R[a * 3] * c[0] + R[a * 3 + 1] * c[1] + R[a * 3 + 2] * c[2]);
    }
  }
  float* o = xf + (size_t) kXf * j;
#pragma unroll
  for (int k = 0; k < 9; ++k) o[k] = R[k];
#pragma unroll
  for (int k = 0; k < 3; ++k) o[9 + k] = t[k];
  const float r = log_radius ? expf(log_radius[j]) : 1.0f;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[kXfRot + k] = sp_r[4 * j + k], o[kXfScale + k] = k < S ? sp_s[(size_t) sp_s_ld * j + k] : 0.0f;
  o[kXfI2]  = 1.0f / (2.0f * r * r);
  o[kXfSig] = weight_logit ? 1.0f / (1.0f + expf(-weight_logit[j])) : 1.0f;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[kXfQ + k] = qh[k];
  o[kXfInvLen] = nq, o[kXfDegenerate] = degenerate;
}

// Unnormalised weights u[k] of a point's K neighbour slots and the inverse of their sum.
//   weight_mode 0: softmax(-d2 / temperature)                                              (network.py:517)
//               1: exp(-d2 / (2 r^2)) * sigmoid(omega) + 1e-7, divided by the sum          (network.py:507-513)
//               2: softmax(logits), the caller having gathered sp_W[n, index[n, k]]        (network.py:514-515)
//               3: the caller's weights as they are (inv_den = 1)                          (warp() called on its own)
// Slots whose index is outside [0, M) (the -1 padding of a K-NN with K > M) get 0 and take no part in the sum.
// kMaxK bounds K at compile time so that the per-slot arrays stay in registers (every loop over slots is unrolled).
// A point's neighbour slots in registers, all requested together (index -1: outside [0, M), or no slot).
template <int kMaxK>
struct LbsPairs {
  int j[kMaxK];
  float in[kMaxK];
  __device__ __forceinline__ LbsPairs(int K, int M, const float* __restrict__ pair_in, const int64_t* __restrict__ index) {
#pragma unroll
    for (int k = 0; k < kMaxK; ++k) {
      const int at = min(k, K - 1);
      const int64_t id = index[at];
      in[k] = pair_in[at];
      j[k]  = k < K && id >= 0 && id < M ? (int) id : -1;
    }
  }
};

template <int kMaxK>
__device__ __forceinline__ void lbs_weights(int weight_mode, float inv_t, const LbsPairs<kMaxK>& pair,
                                            const float* __restrict__ xf, float* u, float& inv_den) {
  float mx = -__builtin_inff();
  if (weight_mode == 0 || weight_mode == 2) {
#pragma unroll
    for (int k = 0; k < kMaxK; ++k)
      if (pair.j[k] >= 0) mx = fmaxf(mx, weight_mode == 0 ? -pair.in[k] * inv_t : pair.in[k]);
  }
  float den = 0.0f;
#pragma unroll
  for (int k = 0; k < kMaxK; ++k) {
    const int j = pair.j[k];
    float v = 0.0f;
    if (j >= 0) {
      if (weight_mode == 0) v = expf(-pair.in[k] * inv_t - mx);
      else if (weight_mode == 1) v = expf(-pair.in[k] * xf[(size_t) kXf * j + kXfI2]) * xf[(size_t) kXf * j + kXfSig] + 1e-7f;
      else if (weight_mode == 2) v = expf(pair.in[k] - mx);
      else v = pair.in[k];
    }
    u[k] = v, den += v;
  }
  inv_den = weight_mode == 3 ? 1.0f : (den > 0.0f ? 1.0f / den : 0.0f);
}

}  // namespace
}  // namespace fsgs
