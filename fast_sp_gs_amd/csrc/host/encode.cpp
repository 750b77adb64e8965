// The spherical-harmonic operators. Forward and backward of both over 1M points are 137 us of kernels in four launches, for which the
// Python nodes needed 108 us of host time on the fastest core of a machine and 185 on others: the device waited. Both operators forward
// and backward, us, Python nodes -> these: 2k points 111 -> 60 and 188 -> 92; 400k 108 -> 61 and 185 -> 92; 1M 136 -> 134 and 189 -> 135
// (109 with the colours' derivatives kept, 113 us of kernels).
#include "encode.hpp"

#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>

#include <climits>

namespace fsgs_host {
namespace {

constexpr int64_t kMostDegree = 7;

// What asks for more than the values (forward-mode tangents, function transforms, a trace, a dispatch mode) gets the Python pair's answer.
bool plain_mode() {
  using c10::DispatchKey;
  const c10::DispatchKeySet modes{DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::Tracer, DispatchKey::Python,
                                  DispatchKey::PythonTLSSnapshot};
  return !torch::autograd::ForwardADLevel::try_get_by_idx(0) && !c10::impl::tls_local_dispatch_key_set().included_.has_any(modes);
}
bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided && t.is_contiguous() &&
         t.device().index() == c10::hip::current_device();
}
bool records(const Tensor& t) { return at::GradMode::is_enabled() && t.defined() && t.requires_grad(); }

Tensor encode_forward(const Tensor& dirs, int64_t degree) {
  Tensor basis = empty({dirs.size(0), (degree + 1) * (degree + 1)}, dirs);
  check(fsgs_sh_encode_forward((int) dirs.size(0), (int) dirs.size(1), (int) degree, f32(dirs), f32(basis), stream_of(dirs)),
        "sh_encode_forward");
  return basis;
}

struct Encode : public torch::autograd::Function<Encode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& dirs, int64_t degree) {
    ctx->save_for_backward({dirs});
    ctx->saved_data["degree"] = degree;
    return encode_forward(dirs, degree);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const Tensor& dirs = t[0];
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const char* what = "sh_encode_backward";
    const Tensor g_basis = contiguous(g[0]);
    require(what, "inputs", dirs, at::kFloat), require(what, "grad", g_basis, at::kFloat);
    // the operator writes the first three columns
    Tensor g_dirs = dirs.size(1) == 3 ? at::empty_like(dirs) : at::zeros_like(dirs);
    check(fsgs_sh_encode_backward((int) dirs.size(0), (int) dirs.size(1), (int) ctx->saved_data["degree"].toInt(), f32(g_basis),
                                  f32(dirs), f32(g_dirs), stream_of(dirs)),
          what);
    return first_order_only(g, {dirs}, {g_dirs, Tensor()});
  }
};

// derivs: where it is defined, it gets the colours' derivatives by the direction
Tensor rgb_forward(const Tensor& sh, const Tensor& dirs, const OptTensor& campos, int64_t degree, bool clamp, const Tensor& derivs) {
  Tensor rgb = empty({dirs.size(0), 3}, dirs);
  check(fsgs_sh_to_rgb_forward_derivs((int) dirs.size(0), (int) sh.size(1), (int) degree, clamp, f32(dirs), f32(opt(campos)), f32(sh),
                                      f32(rgb), f32(derivs), stream_of(dirs)),
        "SH_to_RGB_forward");
  return rgb;
}

struct Rgb : public torch::autograd::Function<Rgb> {
  static Tensor forward(AutogradContext* ctx, const Tensor& sh, const Tensor& dirs, const OptTensor& campos, int64_t degree, bool clamp) {
    Tensor derivs;  // for a gradient of the direction, where the rows of coefficients allow it
    if ((dirs.requires_grad() || (has(campos) && campos->requires_grad())) &&
        fsgs_view_keeps_color_derivs((int) degree, (int) sh.size(1), f32(sh), nullptr))
      derivs = empty({dirs.size(0), 9}, dirs);
    Tensor rgb = rgb_forward(sh, dirs, campos, degree, clamp, derivs);
    ctx->save_for_backward({sh, dirs, opt(campos), rgb, derivs});
    ctx->saved_data["degree"] = degree, ctx->saved_data["clamp"] = clamp;
    return rgb;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    at::AutoDispatchBelowADInplaceOrView no_graph;
    // handed back strided by a hook: as the Python pair, taken where no gradient in the same layout is asked for
    auto input = [&](size_t k) { return ctx->needs_input_grad(k) ? Tensor(t[k]) : contiguous(t[k]); };
    const Tensor sh = input(0), dirs = input(1);
    const Tensor &campos = t[2], &rgb = t[3], &derivs = t[4];
    const char* what = "SH_to_RGB_backward";
    const Tensor g_rgb = contiguous(g[0]);
    require(what, "sh_features", sh, at::kFloat), require(what, "dir_or_pos", dirs, at::kFloat);
    require(what, "rgb", rgb, at::kFloat), require(what, "grad_rgb", g_rgb, at::kFloat);
    if (derivs.defined()) require(what, "derivs", derivs, at::kFloat);
    const int64_t degree = ctx->saved_data["degree"].toInt();
    // the operator writes whole rows of the directions and the coefficients of its degree, and adds to the camera centre's
    const bool whole = sh.size(1) == (degree + 1) * (degree + 1);
    Tensor g_sh, g_dirs, g_campos;
    if (ctx->needs_input_grad(0)) g_sh = whole ? at::empty_like(sh) : at::zeros_like(sh);
    if (ctx->needs_input_grad(1)) g_dirs = at::empty_like(dirs);
    if (campos.defined() && ctx->needs_input_grad(2)) g_campos = at::zeros_like(campos);
    check(fsgs_sh_to_rgb_backward_derivs((int) dirs.size(0), (int) sh.size(1), (int) degree, ctx->saved_data["clamp"].toBool(),
                                         f32(dirs), f32(campos), f32(sh), f32(rgb), f32(g_rgb), f32(derivs), f32(g_dirs),
                                         f32(g_campos), f32(g_sh), stream_of(dirs)),
          what);
    return first_order_only(g, {t[0], t[1], campos}, {g_sh, g_dirs, g_campos, Tensor(), Tensor()});
  }
};

}  // namespace

OptTensor sh_encode(const Tensor& dirs, int64_t degree) {
  if (!plain_mode() || !plain(dirs) || dirs.dim() != 2 || dirs.size(0) < 1 || dirs.size(0) > INT_MAX || dirs.size(1) < 3 ||
      dirs.size(1) > INT_MAX || degree < 0 || degree > kMostDegree)
    return std::nullopt;
  return records(dirs) ? Encode::apply(dirs, degree) : encode_forward(dirs, degree);
}

OptTensor sh_to_rgb(const Tensor& sh, const Tensor& dirs, const OptTensor& campos, int64_t degree, bool clamp) {
  if (!plain_mode() || !plain(sh) || !plain(dirs) || (has(campos) && !plain(*campos))) return std::nullopt;
  const int64_t P = dirs.dim() == 2 ? dirs.size(0) : 0;
  if (P < 1 || P > INT_MAX || dirs.size(1) != 3 || sh.dim() != 3 || sh.size(0) != P || sh.size(2) != 3 || sh.size(1) > INT_MAX ||
      (has(campos) && (campos->dim() != 1 || campos->size(0) != 3)) || degree < 0 || degree > kMostDegree ||
      (degree + 1) * (degree + 1) > sh.size(1) || (int64_t) 1 << degree > sh.size(1))
    return std::nullopt;
  if (records(sh) || records(dirs) || (has(campos) && records(*campos))) return Rgb::apply(sh, dirs, campos, degree, clamp);
  return rgb_forward(sh, dirs, campos, degree, clamp, Tensor());
}

}  // namespace fsgs_host
