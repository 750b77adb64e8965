// Python entry points of the native host layer (fast_sp_gs_amd._host).
#include <torch/csrc/utils/pybind.h>

#include "deform.hpp"
#include "encode.hpp"
#include "fast_surfel.hpp"
#include "gaussian.hpp"
#include "surfel.hpp"

namespace py = pybind11;
using namespace fsgs_host;

namespace {

template <typename Call>
auto without_gil(Call call) {
  py::gil_scoped_release released;
  return call();
}

py::tuple surfel_render_py(const Tensor& points, const Tensor& scales, const Tensor& rotations, const Tensor& opacities,
                           const Tensor& shs, const OptTensor& sh_rest, const Tensor& means2D, const Tensor& Tw2v,
                           const Tensor& Tv2c, const Tensor& campos, const OptTensor& background,
                           const OptTensor& trans_mat_t2, const OptTensor& culling, const OptTensor& accum_max_count,
                           const OptTensor& accum_weights_p, const OptTensor& accum_weights_count, int W, int H,
                           int sh_degree, double near_n, double far_n, double depth_ratio, bool epilogue, bool cull) {
  const SurfelView v{points, scales, rotations, opacities, shs, sh_rest, means2D, Tw2v, Tv2c, campos, background,
                     trans_mat_t2, culling, accum_max_count, accum_weights_p, accum_weights_count, W, H, sh_degree,
                     near_n, far_n, depth_ratio, epilogue, cull};
  const SurfelResult r = without_gil([&] { return surfel_render(v); });
  return py::make_tuple(r.maps, r.n_contrib, r.radii, r.visible, r.ranges, r.point_list, r.normal_opacity, r.trans_mat);
}

py::tuple fast_surfel_render_py(const Tensor& points, const Tensor& scales, const Tensor& rotations,
                                const Tensor& opacities, const Tensor& shs, const OptTensor& sh_rest,
                                const Tensor& means2D, const Tensor& Tw2v, const Tensor& Tv2c, const Tensor& Tv2s,
                                const Tensor& campos, const OptTensor& trans_mat_t2, const OptTensor& culling,
                                const OptTensor& accum_max_count, const OptTensor& accum_weights_p,
                                const OptTensor& accum_weights_count, int W, int H, int sh_degree, double near_n,
                                double far_n, double depth_ratio, bool epilogue) {
  const FastSurfelView v{points, scales, rotations, opacities, shs, sh_rest, means2D, Tw2v, Tv2c, Tv2s, campos, trans_mat_t2,
                         culling, accum_max_count, accum_weights_p, accum_weights_count, W, H, sh_degree, near_n, far_n,
                         depth_ratio, epilogue};
  const FastSurfelResult r = without_gil([&] { return fast_surfel_render(v); });
  return py::make_tuple(r.maps, r.radii, r.visible);
}

py::tuple gaussian_render_py(const Tensor& points, const Tensor& scales, const Tensor& rotations, const Tensor& opacities,
                             const Tensor& shs, const OptTensor& sh_rest, const OptTensor& cov3D, const OptTensor& cov2D,
                             const Tensor& means2D, const OptTensor& extras, const Tensor& Tw2v, const Tensor& Tv2c,
                             const Tensor& campos, const OptTensor& culling, const OptTensor& accum_max_count,
                             const OptTensor& accum_weights_p, const OptTensor& accum_weights_count, double tan_x,
                             double tan_y, int W, int H, int sh_degree, bool is_opengl, bool preserve, bool cull) {
  const GaussianView v{points, scales, rotations, opacities, shs, sh_rest, cov3D, cov2D, means2D, extras, Tw2v, Tv2c, campos,
                       culling, accum_max_count, accum_weights_p, accum_weights_count, tan_x, tan_y, W, H, sh_degree,
                       is_opengl, preserve, cull};
  const GaussianResult r = without_gil([&] { return gaussian_render(v); });
  return py::make_tuple(r.maps, r.n_contrib, r.radii, r.visible, r.ranges, r.point_list);
}

py::object or_none(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

py::tuple superpoint_warp_py(const Tensor& points, const Tensor& sp_points, const Tensor& sp_t, const Tensor& sp_r,
                             const OptTensor& sp_s, const OptTensor& sp_rot, const OptTensor& sp_radius,
                             const OptTensor& sp_weight, int scale_columns, int64_t K, double temperature, int warp_mode,
                             int weight_mode) {
  const SuperpointWarp w{points, sp_points, sp_t, sp_r, sp_s, sp_rot, sp_radius, sp_weight, scale_columns, K, temperature,
                         warp_mode, weight_mode};
  const variable_list r = without_gil([&] { return superpoint_warp(w); });
  return py::make_tuple(r[0], r[1], or_none(r[2]), r[3], r[4]);
}

variable_list deform_mlp_py(const Tensor& x, const Tensor& t, const OptTensor& in, const Tensor& packed, const Tensor& bias,
                            const OptTensor& packed_t, const OptTensor& heads_w, int degree_x, double scale_x, int degree_t,
                            double scale_t, int n_layers, int skip, const std::vector<int>& head_rows,
                            const std::vector<Tensor>& params) {
  const DeformMlp m{x, t, in, packed, bias, packed_t, heads_w, degree_x, degree_t, n_layers, skip, scale_x, scale_t, head_rows};
  return without_gil([&] { return deform_mlp(m, params); });
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("surfel_render", &surfel_render_py);
  m.def("fast_surfel_render", &fast_surfel_render_py);
  m.def("gaussian_render", &gaussian_render_py);
  m.def("superpoint_warp", &superpoint_warp_py);
  m.def("deform_mlp", &deform_mlp_py);
  const auto released = py::call_guard<py::gil_scoped_release>();
  m.def("knn_points", &knn_points, released);
  m.def("sh_encode", &sh_encode, released);
  m.def("sh_to_rgb", &sh_to_rgb, released);
  m.def("deform_apply", &deform_apply, released);
  m.def("mlp_pack", &mlp_pack, released);
  m.def("image_loss", &image_loss, released);
  m.def("adam_masked_step", &adam_masked_step, released);
  m.def("adam_dense", &adam_dense, released);
}
