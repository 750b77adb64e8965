#pragma once
#include "torch_util.hpp"

namespace fsgs_host {

// Squared distances [N,K] and indices [N,K] of the K nearest rows of y for every row of x.
std::tuple<Tensor, Tensor> knn_points(const Tensor& x, const Tensor& y, int64_t K);

struct SuperpointWarp {
  Tensor points, sp_points, sp_t, sp_r;
  OptTensor sp_s, sp_rot, sp_radius, sp_weight;
  int scale_columns;  // of sp_s that are scales (the rest is left alone)
  int64_t K;
  double temperature;
  int warp_mode, weight_mode;  // those of fsgs_lbs_blend; weight modes 0 and 1
};
// d_xyz, d_rotation, d_scale (undefined without sp_s), weights, indices
variable_list superpoint_warp(const SuperpointWarp& w);

// points + d_xyz, act(scales) + d_scale, normalize(rotations + d_rotation)
variable_list deform_apply(const Tensor& points, const Tensor& d_xyz, const Tensor& scales, const Tensor& d_scale,
                           const Tensor& rotations, const Tensor& d_rotation, bool log_scales);

struct DeformMlp {
  Tensor x, t;  // positions and time, encoded in the kernel; or
  OptTensor in;  // the encoded rows
  Tensor packed, bias;
  OptTensor packed_t, heads_w;
  int degree_x, degree_t, n_layers, skip;
  double scale_x, scale_t;
  std::vector<int> head_rows;
};
variable_list deform_mlp(const DeformMlp& m, const std::vector<Tensor>& params);

// packed, packed_t, bias, heads_w
std::tuple<Tensor, Tensor, Tensor, Tensor> mlp_pack(const std::vector<Tensor>& params, int n_layers, int skip);

std::tuple<Tensor, Tensor> image_loss(const Tensor& img, const Tensor& target, double C1, double C2, double lambda_dssim);

void adam_masked(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                 const std::vector<Tensor>& v, const Tensor& mask, const std::vector<double>& lr, double b1, double b2,
                 const std::vector<double>& eps, int64_t N);
// torch.optim.Adam's plain step; `steps` (one count per parameter) are advanced by it
// The same with step counts, which the call advances: the rates are lr * sqrt(1 - b2^t) / (1 - b1^t) on float32 tensors, as the
// reference forms them (sparse_gaussian_adam.py:42-46): the powers are torch's, every operation rounds to float32.
void adam_masked_step(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                      const std::vector<Tensor>& v, const std::vector<Tensor>& steps, const Tensor& mask,
                      const std::vector<double>& lr, double b1, double b2, const std::vector<double>& eps, int64_t N);
void adam_dense(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                const std::vector<Tensor>& v, const std::vector<Tensor>& steps, double lr, double b1, double b2, double eps);

}  // namespace fsgs_host
