#pragma once
#include "torch_util.hpp"

namespace fsgs_host {

struct FastSurfelView {
  Tensor points, scales, rotations, opacities, shs;
  OptTensor sh_rest;
  Tensor means2D, Tw2v, Tv2c, Tv2s, campos;
  OptTensor trans_mat_t2, culling, accum_max_count, accum_weights_p, accum_weights_count;
  int W, H, sh_degree;
  double near_n, far_n, depth_ratio;
  bool epilogue;  // false: the blend's own maps (image, opacity, extras, flow)
};

struct FastSurfelResult {
  variable_list maps;
  Tensor radii, visible;
};

FastSurfelResult fast_surfel_render(const FastSurfelView& v);

}  // namespace fsgs_host
