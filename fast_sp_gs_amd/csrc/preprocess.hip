// 2D-Gaussian-surfel preprocess for gfx950: ray-splat transform, screen-space bound, tile rectangle, SH -> RGB,
// and the matching backward. One lane per surfel; pure HBM streaming.
//
// Reference behaviour reproduced: fast_2d_gs/_C/src/gaussian_splatting/gs_2d_preprocess.cu:24-329.
// The geometric part (transform, bound, radius, rectangle) is compiled with floating-point contraction off and in the
// reference's operation order, so radii / tiles_touched / means2D / trans_mat / depths are reproducible bit for bit
// against a plain IEEE evaluation of the same expressions.
#include "common.hpp"
#include "cull_bound.hpp"
#include "instance_slots.hpp"
#include "sh.hpp"
#include "sh_stage.hpp"
#include "surfel_geom.hpp"

namespace fsgs {
bool culling_enabled();  // host-side switch (api.hip)
namespace {

#pragma clang fp contract(off)

struct Mat4 {
  float m[16];
};

__device__ __forceinline__ void mat4_mul(const float* A, const float* B, float* C) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      C[i * 4 + j] = A[i * 4 + 0] * B[0 * 4 + j] + A[i * 4 + 1] * B[1 * 4 + j] + A[i * 4 + 2] * B[2 * 4 + j] +
                     A[i * 4 + 3] * B[3 * 4 + j];
}

__device__ __forceinline__ void ndc2pix(int W, int H, float* N) {
#pragma unroll
  for (int i = 0; i < 16; ++i) N[i] = 0.0f;
  N[0] = (float) (0.5 * W), N[3] = (float) (0.5 * (W - 1));
  N[5] = (float) (0.5 * H), N[7] = (float) (0.5 * (H - 1));
  N[11] = 1.0f, N[15] = 1.0f;
}

// Block-wide: Tw2c = Tv2c * Tw2v into shared memory (the reference does this product with a device matmul on the
// host side, gs_2d_preprocess.cu:381).
__device__ __forceinline__ void load_camera(const float* __restrict__ Tw2v, const float* __restrict__ Tv2c,
                                            float* s_Tw2v, float* s_Tw2c) {
  const int t = threadIdx.x;
  if (t < 16) {
    const int i = t >> 2, j = t & 3;
    s_Tw2v[t] = Tw2v[t];
    s_Tw2c[t] = Tv2c[i * 4 + 0] * Tw2v[0 * 4 + j] + Tv2c[i * 4 + 1] * Tw2v[1 * 4 + j] +
                Tv2c[i * 4 + 2] * Tw2v[2 * 4 + j] + Tv2c[i * 4 + 3] * Tw2v[3 * 4 + j];
  }
  __syncthreads();
}

__device__ __forceinline__ void transmat(int W, int H, const float* p, float sx, float sy, const float4 q,
                                         const float* Tw2c, const float* Tw2v, float* M, float* nrm) {
  float L[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) L[i] = 0.0f;
  const float x = q.x, y = q.y, z = q.z, w = q.w;
  L[0]  = (1 - 2 * (y * y + z * z)) * sx;
  L[1]  = 2 * (x * y - z * w) * sy;
  L[2]  = p[0];
  L[4]  = (2 * (x * y + z * w)) * sx;
  L[5]  = (1 - 2 * (x * x + z * z)) * sy;
  L[6]  = p[1];
  L[8]  = (2 * (x * z - y * w)) * sx;
  L[9]  = 2 * (x * w + y * z) * sy;
  L[10] = p[2];
  L[14] = 1.0f;
  const float t0 = 2 * (y * w + x * z), t1 = 2 * (y * z - x * w), t2 = 1 - 2 * (x * x + y * y);
  float N[16], A[16], B[16];
  ndc2pix(W, H, N);
  mat4_mul(Tw2c, L, A);
  mat4_mul(N, A, B);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) M[i * 3 + j] = B[i * 4 + j];
  nrm[0] = Tw2v[0] * t0 + Tw2v[1] * t1 + Tw2v[2] * t2;
  nrm[1] = Tw2v[4] * t0 + Tw2v[5] * t1 + Tw2v[6] * t2;
  nrm[2] = Tw2v[8] * t0 + Tw2v[9] * t1 + Tw2v[10] * t2;
}

// kRow: floats of a row that each wavefront moves on its own (sh_stage.hpp), 45 with the first coefficient apart; 0: none
// Bound by a chain of trips to memory for few surfels and by 440 bytes a surfel for many, both of which want more wavefronts in
// flight. The rows reach the lanes' registers through LDS for 32 of them (to_lanes), four blocks to a compute unit; with room for 64 it
// was three. Training, us: 3M 1352x1014 220 -> 207, 300k 800x800 36 -> 33, 200k 29 -> 22.5, 10k 256x256 12.0 -> 11.2; 400k 3840x2160
// without a backward 52 -> 47.
template <int kSh, int kRow>
__global__ void __launch_bounds__(256) preprocess_forward_kernel(
    int P, int W, int H, int sh_degree, int n_sh, const float* __restrict__ means3D, const float2* __restrict__ scales,
    const float4* __restrict__ rotations, const float* __restrict__ opacities, const float* __restrict__ shs,
    const float* __restrict__ sh_rest, const float* __restrict__ Tw2v_g, const float* __restrict__ Tv2c_g,
    const float* __restrict__ campos, const float* __restrict__ trans_precomp, const uint8_t* __restrict__ culling,
    int means2D_preserve, float2* __restrict__ means2D, float* __restrict__ colors, float* __restrict__ trans_mat,
    float4* __restrict__ normal_opacity, float* __restrict__ depths, int32_t* __restrict__ radii,
    int32_t* __restrict__ tiles_touched, float4* __restrict__ records, uint32_t* __restrict__ keep_masks,
    ViewOutputs view) {
  constexpr bool kWave = kRow != 0, kSplit = kRow == 45;
  constexpr int kStride = kWave ? kRow | 1 : kShStageStride;
  constexpr bool kStage = kSh == 16;  // degree <= 3: SH rows travel through LDS, read from HBM line by line
  constexpr int kWaveFloats = kWave ? ShWaveRows<kWave ? kRow : 48>::kHalfFloats : 64 * kStride;
  static_assert(!kWave || kWaveFloats >= 64 * 20, "a wavefront's records pass through the same LDS");
  __shared__ float s_Tw2v[16], s_Tw2c[16];
  __shared__ __align__(16) float s_rows[kStage ? 4 * kWaveFloats : 1];
  __shared__ unsigned char s_flag[kWave ? 1 : kShStageRows];
  __shared__ int s_wave_slots[4];
  __shared__ int s_block_slot;
  const int i      = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < P;
  // the surfel's own values are on their way while the block waits for the camera
  float p[3] = {0, 0, 0}, opac = 0.0f;
  float2 own_scale = make_float2(0.0f, 0.0f);
  float4 own_rot = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (valid) {
    p[0] = means3D[3 * (size_t) i], p[1] = means3D[3 * (size_t) i + 1], p[2] = means3D[3 * (size_t) i + 2];
    if (trans_precomp == nullptr) own_scale = scales[i], own_rot = rotations[i];
    opac = opacities[i];
  }
  load_camera(Tw2v_g, Tv2c_g, s_Tw2v, s_Tw2c);
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;

  bool ok = false;
  float M[9], nrm[3] = {0, 0, 0}, c2[2] = {0, 0}, rgb[3] = {0, 0, 0}, depth = 0, radius = 0;
  int area = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) M[k] = 0.0f;
  const int wave_base = blockIdx.x * blockDim.x + (threadIdx.x & ~63);
  float* s_wave_rows  = &s_rows[kWave ? (threadIdx.x >> 6) * kWaveFloats : 0];
  ShWaveRows<kWave ? kRow : 48> sh_regs;
  unsigned long long wanted = 0;
  float dc[3] = {0, 0, 0}, derivs[kColorDerivs] = {};
  if (kSplit && valid) dc[0] = shs[3 * (size_t) i], dc[1] = shs[3 * (size_t) i + 1], dc[2] = shs[3 * (size_t) i + 2];
  do {
    if (!valid || (culling && culling[i])) break;
    float Tw2v[16], Tw2c[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) Tw2v[k] = s_Tw2v[k], Tw2c[k] = s_Tw2c[k];
    const float pv[3] = {Tw2v[0] * p[0] + Tw2v[1] * p[1] + Tw2v[2] * p[2] + Tw2v[3],
                         Tw2v[4] * p[0] + Tw2v[5] * p[1] + Tw2v[6] * p[2] + Tw2v[7],
                         Tw2v[8] * p[0] + Tw2v[9] * p[1] + Tw2v[10] * p[2] + Tw2v[11]};
    if (pv[2] <= 0.2f) break;
    if (trans_precomp == nullptr) {
      transmat(W, H, p, own_scale.x, own_scale.y, own_rot, Tw2c, Tw2v, M, nrm);
    } else {
#pragma unroll
      for (int k = 0; k < 9; ++k) M[k] = trans_precomp[9 * (size_t) i + k];
      nrm[0] = 0.0f, nrm[1] = 0.0f, nrm[2] = 1.0f;
    }
    const float cosv = -(pv[0] * nrm[0] + pv[1] * nrm[1] + pv[2] * nrm[2]);
    if (cosv == 0.0f) break;
    const float mult = cosv > 0 ? 1.0f : -1.0f;
    nrm[0] = mult * nrm[0], nrm[1] = mult * nrm[1], nrm[2] = mult * nrm[2];
    float ext[2];
    if (!bound_3sigma(M, c2, ext)) break;
    radius = ceilf(fmaxf(fmaxf(ext[0], ext[1]), 3.0f * 0.707106f));
    const TileRect r = tile_rect(c2[0], c2[1], f2i_sat(radius), gx, gy);
    area = (r.y1 - r.y0) * (r.x1 - r.x0);
    if (area == 0) break;
    depth = pv[2];
    ok    = true;
  } while (false);
  if (kWave) {
    // Only the rows of surfels on the screen, and so not before that is known: requested ahead of the geometry for everything in
    // front of the camera the rows held 48 registers meanwhile. 3M surfels 1352x1014, 30 % of them beside the picture: 230 -> 209 us;
    // 300k, all on the screen: 35.9 -> 34.0.
    wanted = __ballot(ok);
    if (wanted) sh_regs.fetch(wanted, wave_base, P, kSplit ? sh_rest : shs, sh_regs.large(P));
  }

  // the block's record slots: the atomic is on its way while the colours are formed
  int slot = 0, total = 0;
  unsigned long long block_slot = 0;
  if (view.counters) {
    slot = slots_in_block(ok ? area : 0, s_wave_slots, total);
    if (threadIdx.x == 0) block_slot = add_slots(view, total);
  }
  if (sh_degree >= 0) {
    const int n = sh_count(sh_degree);
    float own[kWave ? kRow : 1];
    if constexpr (kWave) {
      if (wanted) sh_regs.to_lanes(own, s_wave_rows, wave_base, P);
    } else if (kStage) {
      s_flag[threadIdx.x] = ok;
      __syncthreads();
      stage_sh_rows(s_rows, s_flag, blockIdx.x * blockDim.x, P, n, n_sh, shs, sh_rest);
      __syncthreads();
    }
    if (ok) {
      float x, y, z;
      view_dir(p, campos, x, y, z);
      if constexpr (kWave) {
        sh_lane_colors(own, dc, sh_degree, x, y, z, view.color_derivs != nullptr, rgb, derivs);
      } else {
        float Y[kSh];
        sh_eval(sh_degree, x, y, z, Y);
        const float* row = &s_rows[kStage ? threadIdx.x * kStride : 0];  // coefficient l at 3 l
        const float* c0 = kStage ? row : shs + (size_t) i * (sh_rest ? 1 : n_sh) * 3;
        const float* cr = kStage ? row : (sh_rest ? sh_rest + (size_t) i * n_sh * 3 - 3 : c0);
        float r = c0[0] * Y[0], g = c0[1] * Y[0], b = c0[2] * Y[0];
        for (int l = 1; l < n; ++l) r += cr[3 * l] * Y[l], g += cr[3 * l + 1] * Y[l], b += cr[3 * l + 2] * Y[l];
        rgb[0] = fmaxf(0.0f, r + 0.5f), rgb[1] = fmaxf(0.0f, g + 0.5f), rgb[2] = fmaxf(0.0f, b + 0.5f);
      }
    }
  }
  SlotSums sums;
  if (view.counters && threadIdx.x == 0) sums.add(view, block_slot, total);
  if (view.slot_offsets) {
    if (threadIdx.x == 0) s_block_slot = (int) block_slot;
    __syncthreads();
    slot += s_block_slot;
  }
  if (sh_degree < 0 && valid) rgb[0] = shs[3 * (size_t) i], rgb[1] = shs[3 * (size_t) i + 1], rgb[2] = shs[3 * (size_t) i + 2];
  const float op = opac;
  // The rows of 80, 36 and 12 bytes leave through LDS (wave_rows_out): 3M surfels 279 -> 235 us, 300k 39 -> 33, with the
  // positions and shapes requested before the block waits for the camera.
  const bool rows = kWave && (((uintptr_t) trans_mat | (uintptr_t) colors) & 15) == 0;
  if (rows) {
    const int lane = threadIdx.x & 63;
    if (records) {
      float4* r = (float4*) s_wave_rows;
      wave_lds_sync();
      r[5 * lane]     = ok ? make_float4(M[0], M[1], M[2], M[3]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      r[5 * lane + 1] = ok ? make_float4(M[4], M[5], M[6], M[7]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      r[5 * lane + 2] = ok ? make_float4(M[8], c2[0], c2[1], op) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      r[5 * lane + 3] = ok ? make_float4(nrm[0], nrm[1], nrm[2], rgb[0]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      r[5 * lane + 4] = ok ? make_float4(rgb[1], rgb[2], __int_as_float(f2i_sat(radius)), __int_as_float(view.slot_offsets ? slot : -1))
                           : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      wave_lds_sync();
      wave_rows_out<20>(s_wave_rows, wave_base, P, (float*) records);
    }
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 9; ++k) s_wave_rows[9 * lane + k] = ok ? M[k] : 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) s_wave_rows[576 + 3 * lane + k] = rgb[k];
    wave_lds_sync();
    if (trans_precomp == nullptr) wave_rows_out<9>(s_wave_rows, wave_base, P, trans_mat);
    wave_rows_out<3>(s_wave_rows + 576, wave_base, P, colors);
  }
  if (kWave && view.color_derivs) wave_derivs_out(s_wave_rows, derivs, wave_base, P, view.color_derivs);
  if (threadIdx.x == 0) sums.publish(view);
  if (view.tile_rects)  // up to the last block's end
    view.tile_rects[i] = ok && f2i_sat(radius) > 0 ? tile_rect_word(tile_rect(c2[0], c2[1], f2i_sat(radius), gx, gy)) : kNoTiles;
  if (!valid) return;

  if (view.slot_offsets) view.slot_offsets[i] = slot;
  if (view.visible) view.visible[i] = ok && f2i_sat(radius) > 0;
  if (!rows && trans_precomp == nullptr) {
#pragma unroll
    for (int k = 0; k < 9; ++k) trans_mat[9 * (size_t) i + k] = ok ? M[k] : 0.0f;
  }
  if (!rows && sh_degree >= 0) {
    colors[3 * (size_t) i] = rgb[0], colors[3 * (size_t) i + 1] = rgb[1], colors[3 * (size_t) i + 2] = rgb[2];
  }
  depths[i]        = depth;
  radii[i]         = ok ? f2i_sat(radius) : 0;
  tiles_touched[i] = ok ? area : 0;
  if (ok || !means2D_preserve) means2D[i] = ok ? make_float2(c2[0], c2[1]) : make_float2(0.0f, 0.0f);
  normal_opacity[i] = ok ? make_float4(nrm[0], nrm[1], nrm[2], op) : make_float4(0, 0, 0, 0);
  if (records && !rows) {
    // The blend kernels' 80-byte record (layout of pack_records_kernel), written here while every field is in
    // registers. Surfels that are not rendered never enter a tile list; their records are zeros.
    float4* r = records + 5 * (size_t) i;
    if (ok) {
      r[0] = make_float4(M[0], M[1], M[2], M[3]);
      r[1] = make_float4(M[4], M[5], M[6], M[7]);
      r[2] = make_float4(M[8], c2[0], c2[1], op);
      r[3] = make_float4(nrm[0], nrm[1], nrm[2], rgb[0]);
      r[4] = make_float4(rgb[1], rgb[2], __int_as_float(f2i_sat(radius)), __int_as_float(view.slot_offsets ? slot : -1));  // -1: not known yet
    } else {
#pragma unroll
      for (int k = 0; k < 5; ++k) r[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
  }
  if (keep_masks) {
    // Which tiles of the surfel's rectangle some pixel of which can blend it (the culled binning's input): a bit per
    // tile, row-major, or for rectangles above kCullMaskTiles tiles a window of them. A backward sums
    // every position of a large rectangle, so where one may follow all bits are set. Evaluated here, where transform, centre and radius are
    // in registers and the vector units wait for memory anyway (in the flight of the rows instead: 3M 209 -> 204 us, but
    // 300k 34.0 -> 34.8, 400k at 3840x2160 53.7 -> 55.7).
    uint32_t keep = 0xffffffffu;
    if (ok) {
      const TileRect r = tile_rect(c2[0], c2[1], f2i_sat(radius), gx, gy);
      const int w = max(r.x1 - r.x0, 0), h = max(r.y1 - r.y0, 0);
      const bool small = w * h <= kCullMaskTiles;
      if (small || view.windows) {
        const CullBounds cb = cull_bounds(M, c2[0], c2[1], op);
        keep = 0u;
        int e = 0;
        if (small) {
          for (int y = 0; y < h; ++y)
            for (int x = 0; x < w; ++x, ++e)
              if (cull_keeps_tile(cb, c2[0], c2[1], r.x0 + x, r.y0 + y)) keep |= 1u << e;
        } else {
          keep = cull_window(cb, c2[0], c2[1], r);
        }
      }
    }
    keep_masks[i] = keep;
  }
}

__device__ __forceinline__ void transmat_backward(int W, int H, float sx, float sy, const float4 q, const float* Tw2c,
                                                  const float* Tw2v, const float* gM, const float* gN, float* gp,
                                                  float* gs, float* gq) {
  float N[16], G[16], GL[16], dR[16];
  ndc2pix(W, H, N);
#pragma unroll
  for (int i = 0; i < 16; ++i) G[i] = 0.0f, GL[i] = 0.0f, dR[i] = 0.0f;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) G[i * 4 + j] = gM[i * 3 + j];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) GL[i * 4 + j] += N[k * 4 + i] * G[k * 4 + j];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) dR[i * 4 + j] += Tw2c[k * 4 + i] * GL[k * 4 + j];
  gp[0] = dR[2], gp[1] = dR[6], gp[2] = dR[10];
  dR[2]  = gN[0] * Tw2v[0] + gN[1] * Tw2v[4] + gN[2] * Tw2v[8];
  dR[6]  = gN[0] * Tw2v[1] + gN[1] * Tw2v[5] + gN[2] * Tw2v[9];
  dR[10] = gN[0] * Tw2v[2] + gN[1] * Tw2v[6] + gN[2] * Tw2v[10];
  const float x = q.x, y = q.y, z = q.z, w = q.w;
  gs[0] = dR[0] * (1 - 2 * (y * y + z * z)) + dR[4] * (2 * (x * y + z * w)) + dR[8] * (2 * (x * z - y * w));
  gs[1] = dR[1] * (2 * (x * y - z * w)) + dR[5] * (1 - 2 * (x * x + z * z)) + dR[9] * (2 * (x * w + y * z));
  dR[0] *= sx, dR[1] *= sy, dR[4] *= sx, dR[5] *= sy, dR[8] *= sx, dR[9] *= sy;
  gq[0] = 2 * (-2 * x * (dR[5] + dR[10]) + y * (dR[1] + dR[4]) + z * (dR[2] + dR[8]) + w * (dR[9] - dR[6]));
  gq[1] = 2 * (x * (dR[1] + dR[4]) - 2 * y * (dR[0] + dR[10]) + z * (dR[6] + dR[9]) + w * (dR[2] - dR[8]));
  gq[2] = 2 * (x * (dR[2] + dR[8]) + y * (dR[6] + dR[9]) - 2 * z * (dR[0] + dR[5]) + w * (dR[4] - dR[1]));
  gq[3] = 2 * (x * (dR[9] - dR[6]) + y * (dR[2] - dR[8]) + z * (dR[4] - dR[1]));
}

// The records of a view: per-instance gradients in the order of the surfels (instance_slots.hpp), and which were written.
struct ViewRecords {
  SlotSource slots;
  const uint32_t* masks = nullptr;   // keep masks of culled lists, nullptr: every position was written
  const float* records = nullptr;    // [R][kGradFloats]
};
constexpr int kGradFloats = 18;  // 0-2 colours | 3-11 transform | 12-14 normal | 15 opacity | 16-17 centre
constexpr int kSumStride  = 19;

// Sums of the records of the wavefront's 64 surfels, in position order, to s_sums[64][kSumStride] (rows of surfels that
// were not rendered stay as they are), with kSumScratch floats of scratch behind them. `vis`: this lane's surfel was rendered.
// `first`, `count` and `mask` are its span and keep mask (any values where it was not).
// Spans that a mask word covers: nine lanes of a surfel read a record's 72 bytes; surfels are taken seven at
// a time and three such groups together, four kept positions of each surfel in flight, so the wavefront pays a handful of
// trips to memory for all of them.
// A longer span is complete, 72 bytes a position without gaps: the wavefront fetches 64 positions at a time, the next ones while it
// adds the present ones from LDS, a component per lane. Four positions a trip, a surfel near the camera with hundreds of tiles
// kept its wavefront, and with it the launch, for a hundred trips. Kernel, us: 300k surfels 800x800 64 -> 51, 3M 1352x1014
// 393 -> 370, 1M 1352x900 182 -> 131, 30k 1000x1000 33 -> 16.5, 10k 256x256 11.4 -> 11.0; six positions in flight 50, 367 and 11.6.
// 1000 surfels of 12 / 25 / 40 pixels 800x800 70 -> 51, 237 -> 150, 548 -> 287; 900 that all cover half of 480x288, in 15 wavefronts, 311
// -> 331: the wavefront drains between spans.
constexpr int kSumChunk = kWave, kSumScratch = kSumChunk * kGradFloats;
constexpr int kSumFloats = kWave * kSumStride + kSumScratch;  // of a wavefront

__device__ __forceinline__ void wave_record_sums(const ViewRecords& in, int first, int count, uint32_t mask, bool vis,
                                                 float* __restrict__ s_sums) {
  static_assert(kCullMaskTiles == 32, "a mask word holds a small rectangle's positions");
  constexpr int kLanes = kGradFloats / 2, kPerPass = 7, kGroups = 3, kDepth = 4;
  const int lane = (int) __lane_id(), sub = lane / kLanes, k = lane - sub * kLanes;
  const bool small = vis && count <= kCullMaskTiles;
  if (count < kCullMaskTiles) mask &= (1u << max(count, 0)) - 1u;
  const unsigned long long live_mask = wave_ballot(small);
  const int live = __popcll(live_mask);
  // lane r of the first `live` lanes learns which lane holds the r-th of them
  const int before = __popcll(live_mask & ((1ull << lane) - 1ull));
  const int holder = __builtin_amdgcn_ds_permute((small ? before : live + lane - before) * 4, lane);
  for (int r0 = 0; r0 < live; r0 += kGroups * kPerPass) {
    const float2* src[kGroups];
    int who[kGroups];
    uint32_t bits[kGroups];
    float2 acc[kGroups];
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
      const int r   = r0 + q * kPerPass + sub;
      const bool on = sub < kPerPass && r < live;
      who[q] = __shfl(holder, on ? r : 0, 64);
      const int e = __shfl(first, who[q], 64);
      bits[q] = __shfl(mask, who[q], 64);
      if (!on) who[q] = -1, bits[q] = 0u;
      src[q]  = (const float2*) in.records + (size_t) e * kLanes + k;
      acc[q]  = make_float2(0.0f, 0.0f);
    }
    while (wave_ballot((bits[0] | bits[1] | bits[2]) != 0u) != 0ull) {
      float2 v[kGroups][kDepth];
#pragma unroll
      for (int q = 0; q < kGroups; ++q)
#pragma unroll
        for (int j = 0; j < kDepth; ++j) {
          v[q][j] = make_float2(0.0f, 0.0f);
          if (bits[q]) v[q][j] = src[q][(size_t) __builtin_ctz(bits[q]) * kLanes];
          bits[q] &= bits[q] - 1u;
        }
#pragma unroll
      for (int q = 0; q < kGroups; ++q)
#pragma unroll
        for (int j = 0; j < kDepth; ++j) acc[q].x += v[q][j].x, acc[q].y += v[q][j].y;
    }
#pragma unroll
    for (int q = 0; q < kGroups; ++q)
      if (who[q] >= 0) s_sums[who[q] * kSumStride + 2 * k] = acc[q].x, s_sums[who[q] * kSumStride + 2 * k + 1] = acc[q].y;
  }
  float2* const s_chunk = (float2*) (s_sums + kWave * kSumStride);
  for (unsigned long long todo = wave_ballot(vis && !small); todo != 0ull; todo &= todo - 1ull) {
    const int holds = (int) __builtin_ctzll(todo);
    const int e = __builtin_amdgcn_readlane(first, holds), c = __builtin_amdgcn_readlane(count, holds);
    const float2* span = (const float2*) in.records + (size_t) e * kLanes;
    float2 v[kLanes];
    auto fetch = [&](int base) {
#pragma unroll
      for (int j = 0; j < kLanes; ++j) {
        const int at = j * kWave + lane;  // of the chunk's kSumChunk * kLanes pieces
        v[j] = at < (c - base) * kLanes ? span[(size_t) base * kLanes + at] : make_float2(0.0f, 0.0f);
      }
    };
    float acc = 0.0f;
    fetch(0);
    for (int base = 0; base < c; base += kSumChunk) {
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < kLanes; ++j) s_chunk[j * kWave + lane] = v[j];
      wave_lds_sync();
      if (base + kSumChunk < c) fetch(base + kSumChunk);
      if (lane < kGradFloats) {
        const float* s = (const float*) s_chunk + lane;
#pragma unroll 16
        for (int r = 0; r < kSumChunk; ++r) acc += s[r * kGradFloats];  // zeros behind the span's end
      }
    }
    if (lane < kGradFloats) s_sums[holds * kSumStride + lane] = acc;
  }
}

// kRecords: the upstream gradients are the sums of the view's records, taken here: summed by a kernel of its own they went
// through memory once more (72 bytes per surfel out and in), and that kernel waited for three dependent loads per seven
// surfels and wavefront. 3M surfels 1352x1014: sum 244 + preprocess 325 us -> 376 us; 300k 800x800: 34 + 36 -> 65 us.
// kDerivs: the forward left the colours' derivatives (36 bytes a surfel), and the rows of coefficients (192 bytes) are not read again. Bound
// by memory at 3M surfels (about 1.4 GB at 5.2 TB/s); with fewer, by the trips to the records. Kernel, us, 3M 1352x1014 / 300k 800x800 /
// 10k 256x256: 331 / 47 / 11.3 with the coefficients, 302 / 41 / 10.4 with the derivatives and LDS for 64 rows a wavefront (three of
// them per SIMD), 266 / 40 / 9.6 with half of the rows at a time (sh_products_to_global: four). For that the forward took 217, 36 and
// 10.5 instead of 198, 33 and 9.7, with room in LDS for 64 rows a wavefront on both sides.
template <int kSh, int kRow, bool kRecords, bool kDerivs>
__global__ void __launch_bounds__(256) preprocess_backward_kernel(
    int P, int W, int H, int sh_degree, int n_sh, const float* __restrict__ means3D, const float2* __restrict__ scales,
    const float4* __restrict__ rotations, const float* __restrict__ shs, const float* __restrict__ sh_rest,
    const float* __restrict__ Tw2v_g, const float* __restrict__ Tv2c_g, const float* __restrict__ campos,
    const float* __restrict__ trans_mat, const int32_t* __restrict__ radii, const float* __restrict__ colors,
    float2* __restrict__ grad_mean2D, const float* __restrict__ grad_trans, const float* __restrict__ grad_colors,
    const float4* __restrict__ grad_normal_opacity, float* __restrict__ g_means3D, float2* __restrict__ g_scales,
    float4* __restrict__ g_rot, float* __restrict__ g_opac, float* __restrict__ g_shs,
    float* __restrict__ g_sh_rest, ViewRecords view, const float* __restrict__ color_derivs) {
  static_assert(!kDerivs || kRow != 0);
  constexpr bool kWave = kRow != 0, kSplit = kRow == 45;
  constexpr int kStride = kWave ? kRow | 1 : kShStageStride;
  constexpr bool kStage = kSh == 16;
  __shared__ float s_Tw2v[16], s_Tw2c[16];
  constexpr int kWaveFloats = kDerivs ? kSumFloats : 64 * kStride;  // of LDS
  static_assert(!kDerivs || kSumFloats >= kShHalfRows * kStride);
  __shared__ __align__(16) float s_rows[kStage ? 4 * kWaveFloats : kRecords ? 4 * kSumFloats : 1];
  __shared__ unsigned char s_flag[kShStageRows];
  load_camera(Tw2v_g, Tv2c_g, s_Tw2v, s_Tw2c);
  const int i      = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < P;
  int first = 0, count = 0;
  uint32_t mask = 0xffffffffu;
  if (kRecords && valid) {  // beside the radius, not behind it
    int64_t e0;
    slot_span(view.slots, i, e0, count);
    first = (int) e0;  // the number of instances is below 2^31
    if (view.masks) mask = view.masks[i];
  }
  const bool vis   = valid && radii[i] > 0;
  const int n      = sh_degree >= 0 ? sh_count(sh_degree) : 0;
  const int m1     = sh_rest ? 1 : n_sh;
  float* my_row    = &s_rows[kStage && !kDerivs ? threadIdx.x * kStride : 0] - (kSplit ? 3 : 0);  // coefficient l at 3 l
  const int wave_base = blockIdx.x * blockDim.x + (threadIdx.x & ~63);
  float* s_wave_rows  = &s_rows[kWave ? (threadIdx.x >> 6) * kWaveFloats : 0];
  const unsigned long long wanted = kWave ? __ballot(vis) : 0ull;
  ShWaveRows<kWave ? kRow : 48> sh_regs;
  float up[kRecords ? kGradFloats : 1];
  if (kWave && !kDerivs && wanted) sh_regs.fetch(wanted, wave_base, P, kSplit ? sh_rest : shs, sh_regs.large(P));
  // what the geometry reads of the surfel
  float M[9], p[3] = {0, 0, 0}, col[3] = {0, 0, 0};
  float derivs[kColorDerivs] = {};
  float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float2 s = make_float2(0.0f, 0.0f);
#pragma unroll
  for (int k = 0; k < 9; ++k) M[k] = 0.0f;
  if (vis) {
#pragma unroll
    for (int k = 0; k < 9; ++k) M[k] = trans_mat[9 * (size_t) i + k];
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = means3D[3 * (size_t) i + k];
    q = rotations[i], s = scales[i];
    if (sh_degree >= 0)
#pragma unroll
      for (int k = 0; k < 3; ++k) col[k] = colors[3 * (size_t) i + k];
    if (kDerivs)
#pragma unroll
      for (int k = 0; k < kColorDerivs; ++k) derivs[k] = color_derivs[kColorDerivs * (size_t) i + k];
  }
  if (kRecords) {  // the rows of coefficients and the above are on their way meanwhile
    static_assert(!kStage || 64 * kStride >= kSumFloats, "the sums fit where the rows will be");
    float* s_sums = &s_rows[(threadIdx.x >> 6) * (kStage ? kWaveFloats : kSumFloats)];
    wave_record_sums(view, first, count, mask, vis, s_sums);
    wave_lds_sync();
    if (vis) {
#pragma unroll
      for (int c = 0; c < kGradFloats; ++c) up[kRecords ? c : 0] = s_sums[(threadIdx.x & 63) * kSumStride + c];
    } else if (valid) {
      grad_mean2D[i] = make_float2(0.0f, 0.0f);
    }
    wave_lds_sync();
  }
  if (kWave) {
    if (wanted == 0ull) {  // nothing of this wavefront was rendered: its gradient rows are zeros
      if (wave_base < P) {
        ShWaveRows<kWave ? kRow : 48>::zeros_to_global(wave_base, P, kSplit ? g_sh_rest : g_shs);
        if (kSplit && valid && g_shs)
          g_shs[3 * (size_t) i] = 0.0f, g_shs[3 * (size_t) i + 1] = 0.0f, g_shs[3 * (size_t) i + 2] = 0.0f;
      }
      if (valid) {
        g_opac[i] = 0.0f;
        g_means3D[3 * (size_t) i] = 0.0f, g_means3D[3 * (size_t) i + 1] = 0.0f, g_means3D[3 * (size_t) i + 2] = 0.0f;
        g_scales[i] = make_float2(0.0f, 0.0f);
        g_rot[i]    = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
      return;
    }
    if (!kDerivs) {
      sh_regs.to_lds(s_wave_rows, wave_base, P);
      wave_lds_sync();
    }
  } else if (kStage && sh_degree >= 0) {
    s_flag[threadIdx.x] = vis;
    __syncthreads();
    stage_sh_rows(s_rows, s_flag, blockIdx.x * blockDim.x, P, n, n_sh, shs, sh_rest);
    __syncthreads();
  }

  float g[3] = {}, Y[kSh];  // the colour's gradient and the basis: their products are the gradients of the coefficients
#pragma unroll
  for (int l = 0; l < (kDerivs ? kSh : 0); ++l) Y[l] = 0.0f;
  if (vis) {
    float Tw2v[16], Tw2c[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) Tw2v[k] = s_Tw2v[k], Tw2c[k] = s_Tw2c[k];

    constexpr int kUp = kRecords ? 1 : 0;  // indexes of `up` where it is there
    const float4 gno = kRecords ? make_float4(up[12 * kUp], up[13 * kUp], up[14 * kUp], up[15 * kUp]) : grad_normal_opacity[i];
    g_opac[i]        = gno.w;
    float gM[9], gM_in2, gM_in5;
#pragma unroll
    for (int k = 0; k < 9; ++k) gM[k] = kRecords ? up[(3 + k) * kUp] : grad_trans[9 * (size_t) i + k];
    gM_in2 = gM[2], gM_in5 = gM[5];
    const float2 g2 = kRecords ? make_float2(up[16 * kUp], up[17 * kUp]) : grad_mean2D[i];
    bound_backward(M, g2.x, g2.y, gM);

    const float t0 = 2 * (q.y * q.w + q.x * q.z), t1 = 2 * (q.y * q.z - q.x * q.w),
                t2 = 1 - 2 * (q.x * q.x + q.y * q.y);
    const float nrm[3] = {Tw2v[0] * t0 + Tw2v[1] * t1 + Tw2v[2] * t2, Tw2v[4] * t0 + Tw2v[5] * t1 + Tw2v[6] * t2,
                          Tw2v[8] * t0 + Tw2v[9] * t1 + Tw2v[10] * t2};
    const float pv[3] = {Tw2v[0] * p[0] + Tw2v[1] * p[1] + Tw2v[2] * p[2] + Tw2v[3],
                         Tw2v[4] * p[0] + Tw2v[5] * p[1] + Tw2v[6] * p[2] + Tw2v[7],
                         Tw2v[8] * p[0] + Tw2v[9] * p[1] + Tw2v[10] * p[2] + Tw2v[11]};
    const float cosv = -(pv[0] * nrm[0] + pv[1] * nrm[1] + pv[2] * nrm[2]);
    const float mult = cosv > 0 ? 1.0f : -1.0f;
    const float gN[3] = {mult * gno.x, mult * gno.y, mult * gno.z};
    float gp[3], gs[2], gq[4];
    transmat_backward(W, H, s.x, s.y, q, Tw2c, Tw2v, gM, gN, gp, gs, gq);

    if (sh_degree >= 0) {
      float x, y, z;
      const float nn = view_dir(p, campos, x, y, z);
      sh_eval(sh_degree, x, y, z, Y);
#pragma unroll
      for (int c = 0; c < 3; ++c) g[c] = (kRecords ? up[c * kUp] : grad_colors[3 * (size_t) i + c]) * (float) (col[c] > 0);
      // coefficient rows are read from LDS when staged, and each gradient row is written over the coefficients it
      // was computed from (a lane only ever touches its own row)
      const float* c0 = kStage ? my_row : shs + (size_t) i * m1 * 3;
      const float* cr = kStage ? my_row : (sh_rest ? sh_rest + (size_t) i * n_sh * 3 - 3 : c0);
      float* o0  = kDerivs && !kSplit ? nullptr : kStage && !kSplit ? my_row : (g_shs ? g_shs + (size_t) i * m1 * 3 : nullptr);
      float* orr = kDerivs ? nullptr : kStage ? my_row
                          : (sh_rest ? (g_sh_rest ? g_sh_rest + (size_t) i * n_sh * 3 - 3 : nullptr) : o0);
      if (o0) o0[0] = g[0] * Y[0], o0[1] = g[1] * Y[0], o0[2] = g[2] * Y[0];
      const float dir[3] = {x, y, z};
      float dx = 0, dy = 0, dz = 0;
      sh_direction_part<kSh, kDerivs>(sh_degree, dir, g, cr, derivs, dx, dy, dz);  // before the coefficients are written over
      for (int l = 1; l < n; ++l)
        if (orr) orr[3 * l] = g[0] * Y[l], orr[3 * l + 1] = g[1] * Y[l], orr[3 * l + 2] = g[2] * Y[l];
      if (!kStage && orr) {  // coefficients above the active degree
        for (int l = n; l < (sh_rest ? n_sh + 1 : n_sh); ++l)
          orr[3 * l] = 0.0f, orr[3 * l + 1] = 0.0f, orr[3 * l + 2] = 0.0f;
      }
      const float vx = p[0] - campos[0], vy = p[1] - campos[1], vz = p[2] - campos[2];
      const float tt = -(vx * dx + vy * dy + vz * dz) * nn * nn * nn;
      gp[0] = gp[0] + (dx * nn + tt * vx);
      gp[1] = gp[1] + (dy * nn + tt * vy);
      gp[2] = gp[2] + (dz * nn + tt * vz);
    }
    g_means3D[3 * (size_t) i] = gp[0], g_means3D[3 * (size_t) i + 1] = gp[1], g_means3D[3 * (size_t) i + 2] = gp[2];
    g_scales[i] = make_float2(gs[0], gs[1]);
    g_rot[i]    = make_float4(gq[0], gq[1], gq[2], gq[3]);
    // densification proxy written over the incoming screen-space gradient (gs_2d_preprocess.cu:325-328)
    const float depth = M[8];
    grad_mean2D[i] = make_float2(gM_in2 * depth * 0.5f * (float) W, gM_in5 * depth * 0.5f * (float) H);
  } else if (valid) {
    // rows of surfels that were not rendered get explicit zeros, so the outputs need no initialisation
    g_opac[i] = 0.0f;
    g_means3D[3 * (size_t) i] = 0.0f, g_means3D[3 * (size_t) i + 1] = 0.0f, g_means3D[3 * (size_t) i + 2] = 0.0f;
    g_scales[i] = make_float2(0.0f, 0.0f);
    g_rot[i]    = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (sh_degree >= 0) {
      if (kStage) {
        for (int c = kSplit ? 3 : 0; c < (kDerivs ? 0 : n * 3); ++c) my_row[c] = 0.0f;
        if (kSplit && g_shs)
          g_shs[3 * (size_t) i] = 0.0f, g_shs[3 * (size_t) i + 1] = 0.0f, g_shs[3 * (size_t) i + 2] = 0.0f;
      } else {
        if (g_shs)
          for (int c = 0; c < m1 * 3; ++c) g_shs[(size_t) i * m1 * 3 + c] = 0.0f;
        if (g_sh_rest)
          for (int c = 0; c < n_sh * 3; ++c) g_sh_rest[(size_t) i * n_sh * 3 + c] = 0.0f;
      }
    }
  }
  if constexpr (kDerivs) {
    sh_products_to_global<kRow>(s_wave_rows, g, Y, wave_base, P, kSplit ? g_sh_rest : g_shs);
  } else if (kWave) {
    wave_lds_sync();
    ShWaveRows<kWave ? kRow : 48>::to_global(s_wave_rows, wave_base, P, kSplit ? g_sh_rest : g_shs);
  } else if (kStage && sh_degree >= 0 && (g_shs || g_sh_rest)) {
    __syncthreads();
    unstage_sh_grads(s_rows, blockIdx.x * blockDim.x, P, n, n_sh, sh_rest != nullptr, g_shs, g_sh_rest);
  }
}

__global__ void __launch_bounds__(256) transmat_forward_kernel(int P, int W, int H, const float* __restrict__ means3D,
    const float2* __restrict__ scales, const float4* __restrict__ rotations, const float* __restrict__ Tw2v_g,
    const float* __restrict__ Tw2c_g, float* __restrict__ trans_mat, float* __restrict__ normals) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  float Tw2v[16], Tw2c[16], M[9], nrm[3];
#pragma unroll
  for (int k = 0; k < 16; ++k) Tw2v[k] = Tw2v_g[k], Tw2c[k] = Tw2c_g[k];
  const float p[3] = {means3D[3 * (size_t) i], means3D[3 * (size_t) i + 1], means3D[3 * (size_t) i + 2]};
  const float2 s = scales[i];
  transmat(W, H, p, s.x, s.y, rotations[i], Tw2c, Tw2v, M, nrm);
#pragma unroll
  for (int k = 0; k < 9; ++k) trans_mat[9 * (size_t) i + k] = M[k];
#pragma unroll
  for (int k = 0; k < 3; ++k) normals[3 * (size_t) i + k] = nrm[k];
}

__global__ void __launch_bounds__(256) transmat_backward_kernel(int P, int W, int H, const float2* __restrict__ scales,
    const float4* __restrict__ rotations, const float* __restrict__ Tw2v_g, const float* __restrict__ Tw2c_g,
    const float* __restrict__ g_mat, const float* __restrict__ g_normals, float* __restrict__ g_means3D,
    float2* __restrict__ g_scales, float4* __restrict__ g_rot) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  float Tw2v[16], Tw2c[16], gM[9], gN[3], gp[3], gs[2], gq[4];
#pragma unroll
  for (int k = 0; k < 16; ++k) Tw2v[k] = Tw2v_g[k], Tw2c[k] = Tw2c_g[k];
#pragma unroll
  for (int k = 0; k < 9; ++k) gM[k] = g_mat[9 * (size_t) i + k];
#pragma unroll
  for (int k = 0; k < 3; ++k) gN[k] = g_normals[3 * (size_t) i + k];
  const float2 s = scales[i];
  transmat_backward(W, H, s.x, s.y, rotations[i], Tw2c, Tw2v, gM, gN, gp, gs, gq);
#pragma unroll
  for (int k = 0; k < 3; ++k) g_means3D[3 * (size_t) i + k] = gp[k];
  g_scales[i] = make_float2(gs[0], gs[1]);
  g_rot[i]    = make_float4(gq[0], gq[1], gq[2], gq[3]);
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API int fsgs_view_keeps_color_derivs(int sh_degree, int n_sh, const float* shs, const float* sh_rest) {
  return wave_row_floats(sh_degree, n_sh, shs, sh_rest) != 0;
}

namespace {
int preprocess_forward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const float* trans_precomp, const uint8_t* culling,
    int means2D_preserve, float* means2D, float* colors, float* trans_mat, float* normal_opacity, float* depths,
    int32_t* radii, int32_t* tiles_touched, float* records, uint32_t* keep_masks, const ViewOutputs& view, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "gs_2d_preprocess_forward: bad sizes P=%d W=%d H=%d", P, W, H);
  FSGS_REQUIRE(((uintptr_t) records & 15) == 0, "gs_2d_preprocess_forward: records must be 16-byte aligned");
  FSGS_REQUIRE(sh_degree <= kMaxShDegree, "gs_2d_preprocess_forward: sh_degree %d > %d not supported", sh_degree,
               kMaxShDegree);
  if (sh_degree >= 0)
    FSGS_REQUIRE(n_sh + (sh_rest ? 1 : 0) >= (sh_degree + 1) * (sh_degree + 1),
                 "gs_2d_preprocess_forward: %d SH coefficients are too few for degree %d", n_sh, sh_degree);
  FSGS_REQUIRE(means3D && scales && rotations && opacities && shs && Tw2v && Tv2c && campos && means2D &&
                   normal_opacity && depths && radii && tiles_touched && (trans_mat || trans_precomp) &&
                   (colors || sh_degree < 0),
               "gs_2d_preprocess_forward: null pointer");
  if (P == 0) return kOk;
  const int rows = wave_row_floats(sh_degree, n_sh, shs, sh_rest);
  auto kernel = sh_degree > 3 ? preprocess_forward_kernel<64, 0>
                : rows == 48  ? preprocess_forward_kernel<16, 48>
                : rows == 45  ? preprocess_forward_kernel<16, 45>
                              : preprocess_forward_kernel<16, 0>;
  hipLaunchKernelGGL(kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, W, H, sh_degree, n_sh, means3D, (const float2*) scales, (const float4*) rotations, opacities, shs,
                     sh_rest, Tw2v, Tv2c, campos, trans_precomp, culling, means2D_preserve, (float2*) means2D, colors,
                     trans_mat, (float4*) normal_opacity, depths, radii, tiles_touched, (float4*) records, keep_masks, view);
  return check_launch("gs_2d_preprocess_forward");
}
}  // namespace

FSGS_API int fsgs_gs_2d_preprocess_forward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const float* trans_precomp, const uint8_t* culling,
    int means2D_preserve, float* means2D, float* colors, float* trans_mat, float* normal_opacity, float* depths,
    int32_t* radii, int32_t* tiles_touched, float* records, uint32_t* keep_masks, void* stream) {
  return preprocess_forward(P, W, H, sh_degree, n_sh, means3D, scales, rotations, opacities, shs, sh_rest, Tw2v, Tv2c,
                            campos, trans_precomp, culling, means2D_preserve, means2D, colors, trans_mat, normal_opacity,
                            depths, radii, tiles_touched, records, keep_masks, ViewOutputs{}, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess_derivs(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const uint8_t* culling, float* means2D, float* colors,
    float* trans_mat, float* normal_opacity, float* depths, int32_t* radii, uint8_t* visible, int32_t* tiles_touched,
    int32_t* slot_offsets, uint64_t* slot_counters, float* records, uint32_t* keep_masks, float* color_derivs, uint32_t* tile_rects,
    int64_t* num_rendered_host, void* stream) {
  FSGS_REQUIRE(slot_counters, "gs_2d_view_preprocess: slot_counters are required");
  if (num_rendered_host) __atomic_store_n(num_rendered_host, (int64_t) -1, __ATOMIC_RELEASE);
  FSGS_REQUIRE(!tile_rects || (W <= 127 * kTile && H <= 127 * kTile), "gs_2d_view_preprocess: %dx%d is too large for rectangles in a word", W, H);
  FSGS_REQUIRE(!color_derivs || wave_row_floats(sh_degree, n_sh, shs, sh_rest) != 0, "gs_2d_view_preprocess: no derivatives of these rows");
  return preprocess_forward(P, W, H, sh_degree, n_sh, means3D, scales, rotations, opacities, shs, sh_rest, Tw2v, Tv2c,
                            campos, nullptr, culling, 0, means2D, colors, trans_mat, normal_opacity, depths, radii,
                            tiles_touched, records, keep_masks,
                            ViewOutputs{(unsigned long long*) slot_counters, slot_offsets, visible, false, color_derivs, num_rendered_host, tile_rects}, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const uint8_t* culling, float* means2D, float* colors,
    float* trans_mat, float* normal_opacity, float* depths, int32_t* radii, uint8_t* visible, int32_t* tiles_touched,
    int32_t* slot_offsets, uint64_t* slot_counters, float* records, uint32_t* keep_masks, void* stream) {
  return fsgs_gs_2d_view_preprocess_derivs(P, W, H, sh_degree, n_sh, means3D, scales, rotations, opacities, shs, sh_rest, Tw2v, Tv2c,
                                           campos, culling, means2D, colors, trans_mat, normal_opacity, depths, radii, visible,
                                           tiles_touched, slot_offsets, slot_counters, records, keep_masks, nullptr, nullptr, nullptr, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess_no_backward_rects(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const uint8_t* culling, float* means2D, float* colors,
    float* trans_mat, float* normal_opacity, float* depths, int32_t* radii, uint8_t* visible, int32_t* tiles_touched,
    uint64_t* slot_counters, float* records, uint32_t* keep_masks, uint32_t* tile_rects, int64_t* num_rendered_host, void* stream) {
  FSGS_REQUIRE(slot_counters, "gs_2d_view_preprocess: slot_counters are required");
  if (num_rendered_host) __atomic_store_n(num_rendered_host, (int64_t) -1, __ATOMIC_RELEASE);
  FSGS_REQUIRE(!tile_rects || (W <= 127 * kTile && H <= 127 * kTile), "gs_2d_view_preprocess: %dx%d is too large for rectangles in a word", W, H);
  return preprocess_forward(P, W, H, sh_degree, n_sh, means3D, scales, rotations, opacities, shs, sh_rest, Tw2v, Tv2c,
                            campos, nullptr, culling, 0, means2D, colors, trans_mat, normal_opacity, depths, radii,
                            tiles_touched, records, keep_masks,
                            ViewOutputs{(unsigned long long*) slot_counters, nullptr, visible, true, nullptr, num_rendered_host, tile_rects}, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess_no_backward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* opacities, const float* shs, const float* sh_rest,
    const float* Tw2v, const float* Tv2c, const float* campos, const uint8_t* culling, float* means2D, float* colors,
    float* trans_mat, float* normal_opacity, float* depths, int32_t* radii, uint8_t* visible, int32_t* tiles_touched,
    uint64_t* slot_counters, float* records, uint32_t* keep_masks, void* stream) {
  return fsgs_gs_2d_view_preprocess_no_backward_rects(P, W, H, sh_degree, n_sh, means3D, scales, rotations, opacities, shs, sh_rest, Tw2v,
                                                      Tv2c, campos, culling, means2D, colors, trans_mat, normal_opacity, depths,
                                                      radii, visible, tiles_touched, slot_counters, records, keep_masks, nullptr,
                                                      nullptr, stream);
}

namespace {
template <bool kRecords>
int preprocess_backward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D, const float* scales,
    const float* rotations, const float* shs, const float* sh_rest, const float* Tw2v, const float* Tv2c,
    const float* campos, const float* trans_mat, const int32_t* radii, const float* colors, float* grad_mean2D,
    const float* grad_trans, const float* grad_colors, const float* grad_normal_opacity, float* g_means3D,
    float* g_scales, float* g_rot, float* g_opac, float* g_shs, float* g_sh_rest, const ViewRecords& view,
    const float* color_derivs, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "gs_2d_preprocess_backward: bad sizes");
  FSGS_REQUIRE(sh_degree <= kMaxShDegree, "gs_2d_preprocess_backward: sh_degree %d > %d not supported", sh_degree,
               kMaxShDegree);
  FSGS_REQUIRE(means3D && scales && rotations && Tw2v && Tv2c && campos && trans_mat && radii && grad_mean2D &&
                   (kRecords || (grad_trans && grad_normal_opacity)) && g_means3D && g_scales && g_rot && g_opac,
               "gs_2d_preprocess_backward: null pointer");
  if (sh_degree >= 0)
    FSGS_REQUIRE(shs && colors && (kRecords || grad_colors),
                 "gs_2d_preprocess_backward: SH path needs shs, colors and grad_colors");
  if (P == 0) return kOk;
  float* g_rows  = sh_rest ? g_sh_rest : g_shs;
  const int rows = g_rows ? wave_row_floats(sh_degree, n_sh, shs, sh_rest, g_rows) : 0;
  const bool derivs = kRecords && color_derivs;
  auto kernel = sh_degree > 3 ? preprocess_backward_kernel<64, 0, kRecords, false>
                : rows == 48  ? (derivs ? preprocess_backward_kernel<16, 48, kRecords, kRecords> : preprocess_backward_kernel<16, 48, kRecords, false>)
                : rows == 45  ? (derivs ? preprocess_backward_kernel<16, 45, kRecords, kRecords> : preprocess_backward_kernel<16, 45, kRecords, false>)
                              : preprocess_backward_kernel<16, 0, kRecords, false>;
  hipLaunchKernelGGL(kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, W, H, sh_degree, n_sh, means3D, (const float2*) scales, (const float4*) rotations, shs, sh_rest, Tw2v,
                     Tv2c, campos, trans_mat, radii, colors, (float2*) grad_mean2D, grad_trans, grad_colors,
                     (const float4*) grad_normal_opacity, g_means3D, (float2*) g_scales, (float4*) g_rot, g_opac,
                     g_shs, g_sh_rest, view, color_derivs);
  return check_launch("gs_2d_preprocess_backward");
}
}  // namespace

FSGS_API int fsgs_gs_2d_preprocess_backward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* shs, const float* sh_rest, const float* Tw2v,
    const float* Tv2c, const float* campos, const float* trans_mat, const int32_t* radii, const float* colors,
    float* grad_mean2D, const float* grad_trans, const float* grad_colors, const float* grad_normal_opacity,
    float* g_means3D, float* g_scales, float* g_rot, float* g_opac, float* g_shs, float* g_sh_rest, void* stream) {
  return preprocess_backward<false>(P, W, H, sh_degree, n_sh, means3D, scales, rotations, shs, sh_rest, Tw2v, Tv2c, campos,
                                    trans_mat, radii, colors, grad_mean2D, grad_trans, grad_colors, grad_normal_opacity,
                                    g_means3D, g_scales, g_rot, g_opac, g_shs, g_sh_rest, ViewRecords{}, nullptr, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess_backward_derivs(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* shs, const float* sh_rest, const float* Tw2v,
    const float* Tv2c, const float* campos, const float* trans_mat, const int32_t* radii, const float* colors,
    const int32_t* slot_offsets, const int32_t* slot_regions, const int32_t* tiles_touched, const uint32_t* keep_masks,
    const float* slot_grads, const float* color_derivs, float* g_means2D, float* g_means3D, float* g_scales, float* g_rot,
    float* g_opac, float* g_shs, float* g_sh_rest, void* stream) {
  FSGS_REQUIRE(P == 0 || (slot_offsets && slot_regions && tiles_touched && slot_grads),
               "gs_2d_view_preprocess_backward: record slots and records are required");
  ViewRecords view;
  view.slots   = SlotSource{nullptr, slot_offsets, slot_regions, tiles_touched};
  view.masks   = culling_enabled() ? keep_masks : nullptr;
  view.records = slot_grads;
  return preprocess_backward<true>(P, W, H, sh_degree, n_sh, means3D, scales, rotations, shs, sh_rest, Tw2v, Tv2c, campos,
                                   trans_mat, radii, colors, g_means2D, nullptr, nullptr, nullptr, g_means3D, g_scales,
                                   g_rot, g_opac, g_shs, g_sh_rest, view, color_derivs, stream);
}

FSGS_API int fsgs_gs_2d_view_preprocess_backward(int P, int W, int H, int sh_degree, int n_sh, const float* means3D,
    const float* scales, const float* rotations, const float* shs, const float* sh_rest, const float* Tw2v,
    const float* Tv2c, const float* campos, const float* trans_mat, const int32_t* radii, const float* colors,
    const int32_t* slot_offsets, const int32_t* slot_regions, const int32_t* tiles_touched, const uint32_t* keep_masks,
    const float* slot_grads, float* g_means2D, float* g_means3D, float* g_scales, float* g_rot, float* g_opac, float* g_shs,
    float* g_sh_rest, void* stream) {
  return fsgs_gs_2d_view_preprocess_backward_derivs(P, W, H, sh_degree, n_sh, means3D, scales, rotations, shs, sh_rest, Tw2v, Tv2c,
                                                    campos, trans_mat, radii, colors, slot_offsets, slot_regions, tiles_touched,
                                                    keep_masks, slot_grads, nullptr, g_means2D, g_means3D, g_scales, g_rot,
                                                    g_opac, g_shs, g_sh_rest, stream);
}

FSGS_API int fsgs_gs_2d_compute_transmat_forward(int P, int W, int H, const float* means3D, const float* scales,
    const float* rotations, const float* Tw2v, const float* Tw2c, float* trans_mat, float* normals, void* stream) {
  FSGS_REQUIRE(P >= 0 && means3D && scales && rotations && Tw2v && Tw2c && trans_mat && normals,
               "gs_2d_compute_transmat_forward: bad arguments");
  if (P == 0) return kOk;
  hipLaunchKernelGGL(transmat_forward_kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, W, H,
                     means3D, (const float2*) scales, (const float4*) rotations, Tw2v, Tw2c, trans_mat, normals);
  return check_launch("gs_2d_compute_transmat_forward");
}

FSGS_API int fsgs_gs_2d_compute_transmat_backward(int P, int W, int H, const float* means3D, const float* scales,
    const float* rotations, const float* Tw2v, const float* Tw2c, const float* g_mat, const float* g_normals,
    float* g_means3D, float* g_scales, float* g_rot, void* stream) {
  (void) means3D;
  FSGS_REQUIRE(P >= 0 && scales && rotations && Tw2v && Tw2c && g_mat && g_normals && g_means3D && g_scales && g_rot,
               "gs_2d_compute_transmat_backward: bad arguments");
  if (P == 0) return kOk;
  hipLaunchKernelGGL(transmat_backward_kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, W, H,
                     (const float2*) scales, (const float4*) rotations, Tw2v, Tw2c, g_mat, g_normals, g_means3D,
                     (float2*) g_scales, (float4*) g_rot);
  return check_launch("gs_2d_compute_transmat_backward");
}
