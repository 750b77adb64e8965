// The maps of a view that depend on one pixel's own sums alone (fast_2d_gs/renderer/gs_2d_render.py:608-615 and the composite of
// fast_2d_gs/network.py:725-726), written by the blend while it holds the sums: the per-pixel pass behind it (epilogue.hip) is left
// with the pseudo normal, which needs the neighbours' depths.
#pragma once

#include "common.hpp"

namespace fsgs {

// torch.nan_to_num(x, 0, 0): NaN and +inf become 0, -inf the lowest finite float.
__device__ __forceinline__ float nan0(float v) {
  if (v != v || v == __builtin_inff()) return 0.0f;
  return v == -__builtin_inff() ? -3.4028234663852886e38f : v;
}
__device__ __forceinline__ float mixed_depth(float depth, float median, float ratio) {
  return fmaf(ratio, nan0(median), nan0(depth) * (1.0f - ratio));  // written out: every kernel rounds alike, here and below
}

// Component j of the normal in world space: row vector times Tw2v[:3,:3].
__device__ __forceinline__ float world_normal(const float* Tw2v, int j, float n0, float n1, float n2) {
  return fmaf(n2, Tw2v[8 + j], fmaf(n1, Tw2v[4 + j], n0 * Tw2v[j]));
}

struct ViewMaps {
  const float* Tw2v;                       // [4, 4]
  const float* background;                 // [3] or nullptr: the picture is not composited
  float *normals, *depths, *surf_depth;    // normals == nullptr: no maps; depths may be
  float* distortion;                       // where it goes without the extra channels
  float ratio;

  __device__ __forceinline__ float colour(int c, float sum, float opacity) const {
    return background ? fmaf(1.0f - opacity, background[c], sum) : sum;
  }
  __device__ __forceinline__ void write(size_t HW, size_t p, float n0, float n1, float n2, float depth, float median,
                                        float dist) const {
#pragma unroll
    for (int j = 0; j < 3; ++j) normals[j * HW + p] = world_normal(Tw2v, j, n0, n1, n2);
    if (depths) depths[p] = nan0(median);
    surf_depth[p] = mixed_depth(depth, median, ratio);
    if (distortion) distortion[p] = dist;
  }
};

}  // namespace fsgs
