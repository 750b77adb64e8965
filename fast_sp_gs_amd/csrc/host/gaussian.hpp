#pragma once
#include "torch_util.hpp"

namespace fsgs_host {

struct GaussianView {
  Tensor points, scales, rotations, opacities, shs;
  OptTensor sh_rest, cov3D, cov2D;
  Tensor means2D;
  OptTensor extras;
  Tensor Tw2v, Tv2c, campos;
  OptTensor culling, accum_max_count, accum_weights_p, accum_weights_count;
  double tan_x, tan_y;
  int W, H, sh_degree;
  bool is_opengl;
  bool preserve;  // means2D keeps its values where a Gaussian is not rendered (otherwise: zeros)
  bool cull;      // tile lists without the instances no pixel of their tile can blend
};

struct GaussianResult {
  variable_list maps;  // image, opacity, screen positions, conics and opacities (, extras)
  Tensor n_contrib, radii, visible, ranges, point_list;
};

GaussianResult gaussian_render(const GaussianView& v);

}  // namespace fsgs_host
