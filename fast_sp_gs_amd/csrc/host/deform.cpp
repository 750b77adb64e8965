// The superpoint deformation of a dynamic scene on the kernels: deformation network, K-NN + neighbour weights + warp,
// deformed parameters, photometric loss, optimiser steps, each one C++ call and one autograd node. Through Python a training
// iteration spent 1.2 ms of host time on a dozen autograd nodes and the two optimisers, more than the GPU needs for it.
#include "deform.hpp"

#include <climits>
#include <cmath>

namespace fsgs_host {
namespace {

Tensor byte_buffer(size_t bytes, const Tensor& like) { return empty({(int64_t) (bytes ? bytes : 1)}, like, at::kByte); }

bool wants(const OptTensor& t) { return has(t) && t->requires_grad(); }

void nearest(const Tensor& x, const Tensor& y, int64_t K, Tensor& d2, Tensor& index) {
  const char* what = "knn_topk";
  refuse_duals("knn_points", x, y);
  require(what, "x", x, at::kFloat), require(what, "y", y, at::kFloat);
  if (x.dim() != 2 || y.dim() != 2 || x.size(1) != y.size(1)) fail("knn_topk: feature dimensions differ");
  const int64_t N = x.size(0), M = y.size(0), D = x.size(1);
  d2 = empty({N, K}, x), index = empty({N, K}, x, at::kLong);
  const size_t bytes = fsgs_knn_topk_workspace_bytes((int) N, (int) M, (int) D, (int) K);
  const Tensor ws = bytes ? byte_buffer(bytes, x) : Tensor();
  check(fsgs_knn_topk_ws((int) N, (int) M, (int) D, (int) K, f32(x), f32(y), f32(d2), i64(index), data<void>(ws), bytes,
                         stream_of(x)),
        what);
}

// gradients of the squared distances; g_x only if asked for
void nearest_backward(const Tensor& x, const Tensor& y, const Tensor& index, const Tensor& g_d2, bool need_x, Tensor& g_x,
                      Tensor& g_y) {
  const int64_t N = x.size(0), M = y.size(0), D = x.size(1), K = index.size(1);
  if (need_x) g_x = at::empty_like(x);
  g_y = at::empty_like(y);
  const size_t bytes = fsgs_knn_topk_backward_workspace_bytes((int) N, (int) M, (int) D);
  const Tensor ws = byte_buffer(bytes, x);
  check(fsgs_knn_topk_backward((int) N, (int) M, (int) D, (int) K, f32(x), f32(y), i64(index), f32(g_d2), f32(g_x), f32(g_y),
                               ws.data_ptr(), bytes, stream_of(x)),
        "knn_topk_backward");
}

struct Nearest : public torch::autograd::Function<Nearest> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, int64_t K) {
    Tensor d2, index;
    nearest(x, y, K, d2, index);
    ctx->save_for_backward({x, y, index});
    ctx->mark_non_differentiable({index});
    ctx->set_materialize_grads(false);
    return {d2, index};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const auto t = ctx->get_saved_variables();
    at::AutoDispatchBelowADInplaceOrView no_graph;
    Tensor g_x, g_y;
    nearest_backward(t[0], t[1], t[2], contiguous(g[0]), ctx->needs_input_grad(0), g_x, g_y);
    return first_order_only(g, {t[0], t[1]}, {g_x, ctx->needs_input_grad(1) ? g_y : Tensor(), Tensor()});
  }
};

// The kernels take a table [M,C] whose rows are whole and lie one behind the other, with a stride between them.
int row_stride(const Tensor& t) { return (int) (t.size(0) > 1 ? t.stride(0) : t.size(1)); }
bool rows_of_floats(const Tensor& t) {
  return (t.size(1) <= 1 || t.stride(1) == 1) && (t.size(0) <= 1 || (t.stride(0) >= t.size(1) && t.stride(0) <= INT_MAX));
}

variable_list warp_forward(const SuperpointWarp& w, Tensor& d2, Tensor& table) {
  const char* what = "lbs_blend";
  refuse_duals("superpoint_deform", w.sp_t, w.sp_r, w.sp_s, w.sp_rot, w.sp_radius, w.sp_weight);
  Tensor index;
  nearest(w.points, w.sp_points, w.K, d2, index);
  require(what, "sp_t", w.sp_t, at::kFloat), require(what, "sp_r", w.sp_r, at::kFloat);
  const int64_t N = w.points.size(0), M = w.sp_points.size(0), K = w.K;
  require_shape(what, "sp_t", w.sp_t, {M, 3}), require_shape(what, "sp_r", w.sp_r, {M, 4});
  if (has(w.sp_rot)) require(what, "sp_rot", *w.sp_rot, at::kFloat), require_shape(what, "sp_rot", *w.sp_rot, {M, 4});
  if (w.points.size(1) < 3) fail("lbs_blend: positions [N,3] and [M,3] are expected");
  auto per_control = [&](const char* name, const OptTensor& t) {
    if (!has(t)) return;
    require(what, name, *t, at::kFloat);
    if (t->numel() < M) fail(std::string(what) + ": " + name + " must hold a value per control point");
  };
  per_control("sp_log_radius", w.sp_radius), per_control("sp_weight_logit", w.sp_weight);
  int S = 0, ld = 0;
  if (has(w.sp_s)) {
    const Tensor& s = *w.sp_s;
    if (!s.is_cuda() || s.scalar_type() != at::kFloat || s.dim() != 2 || s.size(0) != M || !rows_of_floats(s) ||
        s.size(1) < w.scale_columns)
      fail("lbs_blend: sp_s must be a float32 CUDA tensor [M,S]");
    S = w.scale_columns, ld = row_stride(s);
  }
  Tensor d_xyz = empty({N, 3}, w.points), d_rot = empty({N, 4}, w.points), d_scale, weights = empty({N, K}, w.points);
  if (S) d_scale = empty({N, S}, w.points);
  const size_t bytes = fsgs_lbs_blend_workspace_bytes((int) M);
  table = byte_buffer(bytes, w.points);
  check(fsgs_lbs_blend_strided((int) N, (int) M, (int) K, w.warp_mode, w.weight_mode, w.temperature, f32(w.points), f32(w.sp_points),
                       f32(w.sp_t), f32(opt(w.sp_rot)), f32(w.sp_r), f32(opt(w.sp_s)), S, ld, f32(d2), i64(index),
                       f32(opt(w.sp_radius)), f32(opt(w.sp_weight)), f32(weights), f32(d_xyz), f32(d_rot), f32(d_scale),
                       table.data_ptr(), bytes, stream_of(w.points)),
        what);
  variable_list out = {d_xyz, d_rot, weights, index};
  if (S) out.push_back(d_scale);
  return out;
}

struct WarpModes : torch::CustomClassHolder {
  int warp_mode, weight_mode, S;
  double temperature;
};

struct Warp : public torch::autograd::Function<Warp> {
  // the points are detached, as in the reference (network.py:577)
  static variable_list forward(AutogradContext* ctx, const Tensor& sp_points, const Tensor& sp_t, const Tensor& sp_r,
                               const OptTensor& sp_s, const OptTensor& sp_rot, const OptTensor& sp_radius,
                               const OptTensor& sp_weight, const SuperpointWarp* warp) {
    (void) sp_points, (void) sp_t, (void) sp_r, (void) sp_s, (void) sp_rot, (void) sp_radius, (void) sp_weight;
    const SuperpointWarp& w = *warp;
    Tensor d2, table;
    variable_list out = warp_forward(w, d2, table);
    ctx->save_for_backward({w.points, w.sp_points, w.sp_t, w.sp_r, opt(w.sp_s), opt(w.sp_rot), opt(w.sp_radius),
                            opt(w.sp_weight), d2, out[3], table});
    auto m = c10::make_intrusive<WarpModes>();
    m->warp_mode = w.warp_mode, m->weight_mode = w.weight_mode, m->temperature = w.temperature, m->S = w.scale_columns;
    ctx->saved_data["modes"] = c10::IValue::make_capsule(m);
    ctx->mark_non_differentiable({out[2], out[3]});
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const Tensor &points = t[0], &sp_points = t[1], &sp_t = t[2], &sp_r = t[3], &sp_s = t[4], &sp_rot = t[5],
                 &radius = t[6], &weight = t[7], &d2 = t[8], &index = t[9], &table = t[10];
    const auto capsule = ctx->saved_data["modes"].toCapsule();
    const WarpModes& m = *static_cast<const WarpModes*>(capsule.get());
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const int64_t N = points.size(0), M = sp_points.size(0), K = index.size(1);
    const int S = sp_s.defined() ? m.S : 0;
    const variable_list inputs = {sp_points, sp_t, sp_r, sp_s, sp_rot, radius, weight};
    auto given = [&](const Tensor& x, int64_t columns) {
      return x.defined() ? contiguous(x) : at::zeros({N, columns}, points.options());
    };
    const Tensor g_xyz = given(g[0], 3), g_rot = given(g[1], 4), g_scale = S ? given(g[4], S) : Tensor();
    Tensor g_c = empty({M, 3}, points), g_t = empty({M, 3}, points), g_r = empty({M, 4}, points);
    Tensor g_sp_rot, g_s, g_radius, g_weight;
    if (m.warp_mode) g_sp_rot = empty({M, 4}, points);
    if (S) g_s = empty({M, sp_s.size(1)}, points);
    if (m.weight_mode == 1) g_radius = at::empty_like(radius), g_weight = weight.defined() ? at::empty_like(weight) : Tensor();
    const size_t bytes = fsgs_lbs_blend_backward_workspace_bytes((int) N, (int) M, S);
    const Tensor ws = byte_buffer(bytes, points);
    const int ld = S ? row_stride(sp_s) : 0;
    auto pick = [&](size_t k, const Tensor& x) { return ctx->needs_input_grad(k) ? x : Tensor(); };
    if (fsgs_superpoint_backward_is_fused((int) M, (int) K, m.warp_mode, m.weight_mode, S)) {
      check(fsgs_superpoint_backward((int) N, (int) M, (int) K, m.warp_mode, m.weight_mode, m.temperature, f32(points),
                                     f32(sp_points), f32(sp_t), f32(sp_rot), f32(sp_r), f32(sp_s), S, ld, f32(d2), i64(index),
                                     f32(radius), f32(weight), table.data_ptr(), f32(g_xyz), f32(g_rot), f32(g_scale), f32(g_c),
                                     f32(g_t), f32(g_sp_rot), f32(g_r), f32(g_s), S ? (int) sp_s.size(1) : 0, f32(g_radius),
                                     f32(g_weight), ws.data_ptr(), bytes, stream_of(points)),
            "superpoint_backward");
      return first_order_only(g, inputs, {pick(0, g_c), g_t, g_r, g_s, g_sp_rot, g_radius, g_weight, Tensor()});
    }
    const Tensor g_pair = empty({N, K}, points);
    check(fsgs_lbs_blend_backward_strided((int) N, (int) M, (int) K, m.warp_mode, m.weight_mode, m.temperature, f32(points),
                                  f32(sp_points), f32(sp_t), f32(sp_rot), f32(sp_r), f32(sp_s), S, ld, f32(d2), i64(index),
                                  f32(radius), f32(weight), f32(g_xyz), f32(g_rot), f32(g_scale), nullptr, f32(g_pair),
                                  f32(g_c), f32(g_t), f32(g_sp_rot), f32(g_r), f32(g_s), S ? (int) sp_s.size(1) : 0,
                                  f32(g_radius), f32(g_weight), ws.data_ptr(), bytes, stream_of(points)),
          "lbs_blend_backward");
    if (ctx->needs_input_grad(0)) {
      Tensor none, g_y;
      nearest_backward(points, sp_points, index, g_pair, false, none, g_y);
      g_c = m.warp_mode == 2 ? g_c.add_(g_y) : g_y;  // the pivot's gradient exists in that mode only
    }
    return first_order_only(g, inputs, {pick(0, g_c), g_t, g_r, g_s, g_sp_rot, g_radius, g_weight, Tensor()});
  }
};

variable_list apply_forward(const Tensor& points, const Tensor& d_xyz, const Tensor& scales, const Tensor& d_scale,
                            const Tensor& rotations, const Tensor& d_rotation, bool log_scales) {
  const char* what = "deform_apply_forward";
  refuse_duals("deform_apply", points, d_xyz, scales, d_scale, rotations, d_rotation);
  require(what, "points", points, at::kFloat), require(what, "d_xyz", d_xyz, at::kFloat);
  require(what, "scales", scales, at::kFloat), require(what, "d_scale", d_scale, at::kFloat);
  require(what, "rotations", rotations, at::kFloat), require(what, "d_rotation", d_rotation, at::kFloat);
  if (scales.dim() != 2) fail("deform_apply_forward: scales must be [N,S]");
  const int64_t N = scales.size(0), S = scales.size(1);
  require_shape(what, "points", points, {N, 3}), require_shape(what, "d_xyz", d_xyz, {N, 3});
  require_shape(what, "d_scale", d_scale, {N, S}), require_shape(what, "rotations", rotations, {N, 4});
  require_shape(what, "d_rotation", d_rotation, {N, 4});
  const Tensor p = at::empty_like(points), s = at::empty_like(scales), r = at::empty_like(rotations);
  check(fsgs_deform_apply_forward((int) N, (int) S, log_scales, f32(points), f32(d_xyz), f32(scales), f32(d_scale),
                                  f32(rotations), f32(d_rotation), f32(p), f32(s), f32(r), stream_of(points)),
        what);
  return {p, s, r};
}

struct Apply : public torch::autograd::Function<Apply> {
  static variable_list forward(AutogradContext* ctx, const Tensor& points, const Tensor& d_xyz, const Tensor& scales,
                               const Tensor& d_scale, const Tensor& rotations, const Tensor& d_rotation, bool log_scales) {
    const variable_list out = apply_forward(points, d_xyz, scales, d_scale, rotations, d_rotation, log_scales);
    ctx->save_for_backward({scales, rotations, d_rotation});
    ctx->saved_data["log"] = log_scales;
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const bool log_scales = ctx->saved_data["log"].toBool();
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const variable_list upstream = g;
    for (auto& x : g) x = contiguous(x);
    const Tensor &scales = t[0], &rotations = t[1];
    const bool rot = g[2].defined(), logs = log_scales && g[1].defined();
    auto both = [&](size_t k) { return ctx->needs_input_grad(k) && ctx->needs_input_grad(k + 1); };
    // the sums hand their upstream gradient to both addends: a tensor each, or a leaf's accumulation copies it once more
    Tensor g_p = g[0], g_s = g[1], g_r, g_dr;
    if (g[0].defined() && both(0)) g_p = at::empty_like(g[0]);
    if (logs || (g[1].defined() && both(2))) g_s = at::empty_like(scales);
    if (rot || logs) g_r = at::empty_like(rotations);
    g_dr = rot && both(4) ? at::empty_like(rotations) : g_r;
    const bool copy_p = g[0].defined() && both(0), copy_s = !logs && g[1].defined() && both(2), copy_r = rot && both(4);
    if (rot || logs || copy_p || copy_s) {
      const Tensor up = rot || !logs ? g[2] : at::zeros_like(rotations);
      check(fsgs_deform_apply_backward_copies((int) scales.size(0), (int) scales.size(1), logs, f32(scales), f32(rotations),
                                              f32(t[2]), f32(g[0]), f32(g[1]), f32(up), logs ? f32(g_s) : nullptr, f32(g_r),
                                              copy_p ? f32(g_p) : nullptr, copy_s ? f32(g_s) : nullptr,
                                              copy_r ? f32(g_dr) : nullptr, stream_of(scales)),
            "deform_apply_backward");
    }
    if (!rot) g_r = g_dr = Tensor();
    auto pick = [&](size_t k, const Tensor& x) { return ctx->needs_input_grad(k) ? x : Tensor(); };
    return first_order_only(upstream, {t[0], t[1], t[2]}, {pick(0, g_p), pick(1, g[0]), pick(2, g_s), pick(3, g[1]), pick(4, g_r),
                                                           pick(5, g_dr), Tensor()});
  }
};

variable_list mlp_forward(const DeformMlp& m, bool train, Tensor& saved_in, Tensor& saved) {
  const char* what = "mlp_forward";
  const Tensor& rows = has(m.in) ? *m.in : m.x;
  require(what, "inputs", rows, at::kFloat), require(what, "bias", m.bias, at::kFloat);
  if (!has(m.in)) {
    require(what, "t", m.t, at::kFloat);
    if (m.x.dim() != 2 || m.x.size(1) != 3 || m.t.numel() != 1) fail("mlp_forward: positions [B,3] and one time are expected");
  }
  const int64_t B = rows.size(0), Din = has(m.in) ? m.in->size(1) : 3 * (1 + 2 * m.degree_x) + 1 + 2 * m.degree_t;
  int64_t n_out = 0;
  variable_list out;
  std::vector<float*> at;
  for (int r : m.head_rows) n_out += r, out.push_back(empty({B, r}, rows)), at.push_back(f32(out.back()));
  if (m.bias.numel() != m.n_layers * 256 + n_out) fail("mlp_forward: bias has the wrong size");
  if ((size_t) m.packed.numel() != fsgs_mlp_packed_elems((int) Din, m.n_layers, m.skip))
    fail("mlp_forward: packed weight buffer has the wrong size");
  if (train) {
    saved_in = empty({(int64_t) fsgs_mlp_saved_input_elems((int) B, (int) Din)}, rows, at::kShort);
    saved    = empty({(int64_t) fsgs_mlp_saved_elems((int) B, m.n_layers)}, rows, at::kShort);
  }
  check(fsgs_deform_mlp_forward((int) B, (int) Din, 256, m.n_layers, m.skip, (int) m.head_rows.size(), m.head_rows.data(),
                                has(m.in) ? f32(rows) : nullptr, has(m.in) ? nullptr : f32(m.x),
                                has(m.in) ? nullptr : f32(m.t), m.degree_x, m.scale_x, m.degree_t, m.scale_t,
                                data<uint16_t>(m.packed), f32(m.bias), at.data(), data<uint16_t>(saved_in),
                                data<uint16_t>(saved), stream_of(rows)),
        what);
  return out;
}

struct MlpShape : torch::CustomClassHolder {
  int64_t B, Din;
  int n_layers, skip;
  std::vector<int> head_rows;
};

struct Mlp : public torch::autograd::Function<Mlp> {
  static variable_list forward(AutogradContext* ctx, at::TensorList params, const DeformMlp* mlp) {
    (void) params;
    const DeformMlp& m = *mlp;
    Tensor saved_in, saved;
    const variable_list out = mlp_forward(m, true, saved_in, saved);
    ctx->save_for_backward({saved_in, saved, opt(m.packed_t), opt(m.heads_w)});
    auto s = c10::make_intrusive<MlpShape>();
    s->B = out[0].size(0), s->n_layers = m.n_layers, s->skip = m.skip, s->head_rows = m.head_rows;
    s->Din = has(m.in) ? m.in->size(1) : 3 * (1 + 2 * m.degree_x) + 1 + 2 * m.degree_t;
    ctx->saved_data["shape"] = c10::IValue::make_capsule(s);
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const auto capsule = ctx->saved_data["shape"].toCapsule();
    const MlpShape& s = *static_cast<const MlpShape*>(capsule.get());
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const variable_list upstream = g;
    const int64_t B = s.B, Din = s.Din, L = s.n_layers;
    int64_t n_out = 0;
    std::vector<const float*> up;
    for (size_t h = 0; h < s.head_rows.size(); ++h) n_out += s.head_rows[h], g[h] = contiguous(g[h]), up.push_back(f32(g[h]));
    const int64_t n_w = 256 * Din + (L - 1) * 65536 + 256 * Din + n_out * 256;
    const Tensor flat = empty({n_w + L * 256 + n_out}, t[3]);
    const size_t bytes = fsgs_deform_mlp_backward_workspace_bytes((int) B, (int) Din, (int) L);
    const Tensor ws = byte_buffer(bytes, t[3]);
    check(fsgs_deform_mlp_backward((int) B, (int) Din, 256, (int) L, s.skip, (int) s.head_rows.size(), s.head_rows.data(),
                                   nullptr, data<uint16_t>(t[0]), data<uint16_t>(t[2]), f32(t[3]), data<uint16_t>(t[1]),
                                   up.data(), f32(flat), f32(flat) + n_w, ws.data_ptr(), bytes, stream_of(t[3])),
          "mlp_backward");
    // views of one buffer, in parameter order: weight and bias per layer, then per head
    variable_list grads;
    int64_t w = 0, b = n_w;
    auto give = [&](int64_t rows, int64_t columns) {
      grads.push_back(flat.narrow(0, w, rows * columns).view({rows, columns}));
      grads.push_back(flat.narrow(0, b, rows));
      w += rows * columns, b += rows;
    };
    for (int64_t l = 0; l < L; ++l) give(256, l == 0 ? Din : l == s.skip + 1 ? Din + 256 : 256);
    for (int r : s.head_rows) give(r, 256);
    for (size_t k = 0; k < grads.size(); ++k)
      if (!ctx->needs_input_grad(k)) grads[k] = Tensor();
    grads.push_back(Tensor());
    return first_order_only(upstream, {}, std::move(grads));
  }
};

struct Loss : public torch::autograd::Function<Loss> {
  static variable_list forward(AutogradContext* ctx, const Tensor& img, const Tensor& target, double C1, double C2,
                               double lambda_dssim, bool train) {
    const char* what = "image_loss_forward";
    require(what, "img", img, at::kFloat), require(what, "target", target, at::kFloat);
    if (img.dim() != 4 || img.sizes() != target.sizes() || img.numel() == 0)
      fail("image_loss_forward: img and target must be non-empty [B,CH,H,W] tensors of the same shape");
    const int B = (int) img.size(0), CH = (int) img.size(1), H = (int) img.size(2), W = (int) img.size(3);
    const Tensor loss = empty({3}, img);
    Tensor maps;
    if (train) maps = empty({3, img.numel()}, img);
    const size_t bytes = fsgs_image_loss_workspace_bytes(B, H, W);
    const Tensor ws = byte_buffer(bytes, img);
    const int64_t n = img.numel();
    float* d = f32(maps);
    check(fsgs_image_loss_forward(B, CH, H, W, C1, C2, lambda_dssim, f32(img), f32(target), f32(loss), d, d ? d + n : nullptr,
                                  d ? d + 2 * n : nullptr, ws.data_ptr(), bytes, stream_of(img)),
          what);
    if (train) ctx->save_for_backward({img, target, maps});
    ctx->saved_data["lambda"] = lambda_dssim;
    const Tensor value = loss.select(0, 0), terms = loss.narrow(0, 1, 2);
    ctx->mark_non_differentiable({terms});
    ctx->set_materialize_grads(false);
    return {value, terms};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(6);
    const auto t = ctx->get_saved_variables();
    const Tensor &img = t[0], &target = t[1];
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const Tensor up = contiguous(g[0]), grad = at::empty_like(img);
    const int64_t n = img.numel();
    const float* d = f32(t[2]);
    check(fsgs_image_loss_backward((int) img.size(0), (int) img.size(1), (int) img.size(2), (int) img.size(3),
                                   ctx->saved_data["lambda"].toDouble(), f32(img), f32(target), f32(up), d, d + n, d + 2 * n,
                                   f32(grad), stream_of(img)),
          "image_loss_backward");
    return first_order_only(g, {img}, {grad, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()});
  }
};

}  // namespace

std::tuple<Tensor, Tensor> knn_points(const Tensor& x, const Tensor& y, int64_t K) {
  if (at::GradMode::is_enabled() && (x.requires_grad() || y.requires_grad())) {
    const variable_list out = Nearest::apply(x.contiguous(), y.contiguous(), K);
    return {out[0], out[1]};
  }
  Tensor d2, index;
  nearest(x.contiguous(), y.contiguous(), K, d2, index);
  return {d2, index};
}

variable_list superpoint_warp(const SuperpointWarp& given) {
  SuperpointWarp w = given;
  w.points = w.points.detach().contiguous(), w.sp_points = w.sp_points.contiguous();
  w.sp_t = w.sp_t.contiguous(), w.sp_r = w.sp_r.contiguous();
  auto whole = [](OptTensor& t) { if (has(t)) t = t->contiguous(); };
  whole(w.sp_rot), whole(w.sp_radius), whole(w.sp_weight);
  if (has(w.sp_s) && w.sp_s->dim() == 2 && !rows_of_floats(*w.sp_s)) w.sp_s = w.sp_s->contiguous();
  const bool train = at::GradMode::is_enabled() &&
                     (w.sp_points.requires_grad() || w.sp_t.requires_grad() || w.sp_r.requires_grad() || wants(w.sp_s) ||
                      wants(w.sp_rot) || wants(w.sp_radius) || wants(w.sp_weight));
  Tensor d2, table;
  const variable_list r = train ? Warp::apply(w.sp_points, w.sp_t, w.sp_r, w.sp_s, w.sp_rot, w.sp_radius, w.sp_weight, &w)
                                : warp_forward(w, d2, table);
  return {r[0], r[1], r.size() > 4 ? r[4] : Tensor(), r[2], r[3]};
}

variable_list deform_apply(const Tensor& points, const Tensor& d_xyz, const Tensor& scales, const Tensor& d_scale,
                           const Tensor& rotations, const Tensor& d_rotation, bool log_scales) {
  const Tensor a[6] = {points.contiguous(), d_xyz.contiguous(), scales.contiguous(), d_scale.contiguous(),
                       rotations.contiguous(), d_rotation.contiguous()};
  bool train = false;
  for (const Tensor& t : a) train = train || t.requires_grad();
  if (train && at::GradMode::is_enabled()) return Apply::apply(a[0], a[1], a[2], a[3], a[4], a[5], log_scales);
  return apply_forward(a[0], a[1], a[2], a[3], a[4], a[5], log_scales);
}

variable_list deform_mlp(const DeformMlp& m, const std::vector<Tensor>& params) {
  refuse_duals("DeformNetwork", m.x, m.t, m.in);
  for (const Tensor& p : params) refuse_duals("DeformNetwork", p);
  bool train = false;
  for (const Tensor& p : params) train = train || p.requires_grad();
  if (train && at::GradMode::is_enabled()) return Mlp::apply(at::TensorList(params), &m);
  Tensor saved_in, saved;
  return mlp_forward(m, false, saved_in, saved);
}

std::tuple<Tensor, Tensor, Tensor, Tensor> mlp_pack(const std::vector<Tensor>& params, int n_layers, int skip) {
  const char* what = "mlp_pack_all";
  if ((int) params.size() < 2 * n_layers || params.size() % 2) fail("mlp_pack_all: one bias per weight");
  const Tensor& first = params[0];
  const int64_t Din = first.dim() == 2 ? first.size(1) : 0;
  std::vector<const float*> w, b, hw, hb;
  std::vector<int> rows;
  int64_t n_out = 0;
  for (size_t k = 0; k < params.size() / 2; ++k) {
    const Tensor &weight = params[2 * k], &bias = params[2 * k + 1];
    require(what, "weight", weight, at::kFloat), require(what, "bias", bias, at::kFloat);
    const bool head = (int) k >= n_layers;
    const int64_t columns = head ? 256 : k == 0 ? Din : (int) k == skip + 1 ? Din + 256 : 256;
    if (weight.dim() != 2 || weight.size(1) != columns || (!head && weight.size(0) != 256) || bias.numel() != weight.size(0))
      fail("mlp_pack_all: parameter " + std::to_string(k) + " has weight " + shape_text(weight.sizes()) + " / bias " +
           shape_text(bias.sizes()));
    (head ? hw : w).push_back(f32(weight)), (head ? hb : b).push_back(f32(bias));
    if (head) rows.push_back((int) weight.size(0)), n_out += weight.size(0);
  }
  const Tensor packed = empty({(int64_t) fsgs_mlp_packed_elems((int) Din, n_layers, skip)}, first, at::kShort);
  const Tensor packed_t = empty({n_layers > 1 ? n_layers - 1 : 1, 256, 256}, first, at::kShort);
  const Tensor bias = empty({n_layers * 256 + n_out}, first), heads_w = empty({n_out, 256}, first);
  check(fsgs_mlp_pack_all((int) Din, n_layers, skip, w.data(), b.data(), (int) rows.size(), hw.data(), hb.data(), rows.data(),
                          data<uint16_t>(packed), n_layers > 1 ? data<uint16_t>(packed_t) : nullptr, f32(bias), f32(heads_w),
                          stream_of(first)),
        what);
  return {packed, packed_t, bias, heads_w};
}

std::tuple<Tensor, Tensor> image_loss(const Tensor& img, const Tensor& target, double C1, double C2, double lambda_dssim) {
  refuse_duals("image_loss", img, target);
  if (at::GradMode::is_enabled() && target.requires_grad()) fail("image_loss: differentiable in its first image only");
  const bool train = at::GradMode::is_enabled() && img.requires_grad();
  const variable_list out = Loss::apply(img.contiguous(), target.contiguous(), C1, C2, lambda_dssim, train);
  return {out[0], out[1]};
}

namespace {
struct AdamPointers {
  std::vector<float*> p, m, v;
  std::vector<const float*> g;
  std::vector<Tensor> alive;

  AdamPointers(const char* what, const std::vector<Tensor>& params, const std::vector<Tensor>& grads,
               const std::vector<Tensor>& first, const std::vector<Tensor>& second) {
    const size_t n = params.size();
    if (grads.size() != n || first.size() != n || second.size() != n)
      fail(std::string(what) + ": one gradient and two moments per parameter tensor");
    for (size_t k = 0; k < n; ++k) {
      alive.push_back(grads[k].contiguous());
      require(what, "param", params[k], at::kFloat), require(what, "grad", alive[k], at::kFloat);
      require(what, "exp_avg", first[k], at::kFloat), require(what, "exp_avg_sq", second[k], at::kFloat);
      const int64_t c = params[k].numel();
      if (alive[k].numel() != c || first[k].numel() != c || second[k].numel() != c)
        fail(std::string(what) + ": tensor " + std::to_string(k) + "'s gradient or moments differ from it in size");
      p.push_back(f32(params[k])), g.push_back(f32(alive[k])), m.push_back(f32(first[k])), v.push_back(f32(second[k]));
    }
  }
};
}  // namespace

void adam_masked(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                 const std::vector<Tensor>& v, const Tensor& mask, const std::vector<double>& lr, double b1, double b2,
                 const std::vector<double>& eps, int64_t N) {
  const char* what = "AdamMasksedUpdatedMulti";
  const AdamPointers t(what, params, grads, m, v);
  const size_t n = params.size();
  if (lr.size() != n || eps.size() != n) fail("AdamMasksedUpdatedMulti: a rate and an eps per parameter tensor");
  if (n == 0 || N == 0) return;
  const Tensor on = mask.contiguous();
  require(what, "tiles_touched", on, at::kBool);
  if (N < 0 || on.numel() < N) fail("AdamMasksedUpdatedMulti: the mask has fewer than N = " + std::to_string(N) + " entries");
  std::vector<int64_t> M;
  for (const Tensor& p : params) {
    if (p.numel() % N) fail("AdamMasksedUpdatedMulti: a tensor is not [N, M] with N = " + std::to_string(N));
    M.push_back(p.numel() / N);
  }
  const size_t most = (size_t) fsgs_adam_masked_update_max_tensors();
  for (size_t k = 0; k < n; k += most)
    check(fsgs_adam_masked_update_multi((int) std::min(most, n - k), N, M.data() + k, data<uint8_t>(on), lr.data() + k, b1, b2,
                                        eps.data() + k, t.p.data() + k, t.g.data() + k, t.m.data() + k, t.v.data() + k,
                                        stream_of(params[0])),
          what);
}

namespace {
// Advances a step count as torch keeps it (a float32 word on the host), or however a loaded state holds it.
double advanced(const char* what, const Tensor& step) {
  if (step.numel() != 1) fail(std::string(what) + ": a step count is one number");
  const bool plain = step.is_cpu() && step.scalar_type() == at::kFloat;
  return plain ? (double) (*step.data_ptr<float>() += 1.0f) : step.add_(1).item<double>();
}
}  // namespace

void adam_masked_step(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                      const std::vector<Tensor>& v, const std::vector<Tensor>& steps, const Tensor& mask,
                      const std::vector<double>& lr, double b1, double b2, const std::vector<double>& eps, int64_t N) {
  const char* what = "AdamMasksedUpdatedMulti";
  const size_t n = params.size();
  if (steps.size() != n || lr.size() != n) fail("AdamMasksedUpdatedMulti: a step count and a rate per parameter tensor");
  std::vector<double> rate;
  double at_count = -1.0;  // count of the corrections at hand: the tensors of a step share it
  float root_c2 = 0.0f, c1 = 0.0f;
  for (size_t k = 0; k < n; ++k) {
    const double taken = advanced(what, steps[k]);
    if (taken != at_count) {
      root_c2  = (float) at::pow(at::rsub(at::pow(b2, steps[k]), 1), 0.5).item<double>();
      c1       = (float) at::rsub(at::pow(b1, steps[k]), 1).item<double>();
      at_count = taken;
    }
    const float scaled = (float) lr[k] * root_c2;
    rate.push_back((double) (scaled / c1));
  }
  adam_masked(params, grads, m, v, mask, rate, b1, b2, eps, N);
}

void adam_dense(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& m,
                const std::vector<Tensor>& v, const std::vector<Tensor>& steps, double lr, double b1, double b2, double eps) {
  const AdamPointers t("adam_update", params, grads, m, v);
  const size_t n = params.size(), most = (size_t) fsgs_adam_update_max_tensors();
  if (steps.size() != n) fail("adam_update: a step count per parameter tensor");
  std::vector<int64_t> count;
  std::vector<double> step_size, root_c2;
  for (size_t k = 0; k < n; ++k) {
    const double taken = advanced("adam_update", steps[k]);
    count.push_back(params[k].numel());
    step_size.push_back(lr / (1 - std::pow(b1, taken))), root_c2.push_back(std::sqrt(1 - std::pow(b2, taken)));
  }
  for (size_t k = 0; k < n; k += most)
    check(fsgs_adam_update_multi((int) std::min(most, n - k), count.data() + k, step_size.data() + k, root_c2.data() + k, b1, b2,
                                 eps, t.p.data() + k, t.g.data() + k, t.m.data() + k, t.v.data() + k, stream_of(params[0])),
          "adam_update");
}

}  // namespace fsgs_host
