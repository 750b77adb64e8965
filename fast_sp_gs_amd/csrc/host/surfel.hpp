#pragma once
#include "torch_util.hpp"

namespace fsgs_host {

struct SurfelView {
  Tensor points, scales, rotations, opacities, shs;
  OptTensor sh_rest;
  Tensor means2D, Tw2v, Tv2c, campos;
  OptTensor background, trans_mat_t2, culling, accum_max_count, accum_weights_p, accum_weights_count;
  int W, H, sh_degree;
  double near_n, far_n, depth_ratio;
  bool epilogue;  // false: the blend's own maps (image, opacity, extras, flow)
  bool cull;      // tile lists without the instances no pixel of their tile can blend
};

struct SurfelResult {
  variable_list maps;
  Tensor n_contrib, radii, visible, ranges, point_list, normal_opacity, trans_mat;
};

SurfelResult surfel_render(const SurfelView& v);

}  // namespace fsgs_host
