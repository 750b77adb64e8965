// Python entry points of the native host layer (fast_sp_gs_amd._host).
#include <torch/csrc/utils/pybind.h>

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

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("surfel_render", &surfel_render_py);
  m.def("fast_surfel_render", &fast_surfel_render_py);
  m.def("gaussian_render", &gaussian_render_py);
}
