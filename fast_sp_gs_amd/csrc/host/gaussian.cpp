// One view of the 3D-Gaussian renderer, forward and backward, as one call and one autograd node: preprocess -> binning ->
// blend, the steps of fast_2d_gs/renderer/gaussian_render.py:226-274. Screen positions and conics are differentiable
// outputs, so that further tables can be blended with the view's weights afterwards.
#include "gaussian.hpp"

namespace fsgs_host {
namespace {

struct Saved : torch::CustomClassHolder {  // what the backward reads besides tensors
  int W, H, sh_degree, E;
  double tan_x, tan_y;
  bool is_opengl;
  size_t colors, cov3D, derivs;  // places in the slab
  bool has_derivs = false;
};

struct Buffers {
  Tensor radii, visible, ranges, point_list, n_contrib, conic_opacity;
  Tensor image, opacity, extras;
  Tensor hit_blocks;  // per list entry, for the backward
  Slab keep;
  c10::intrusive_ptr<Saved> saved;
};

Buffers forward_view(const GaussianView& v, bool train) {
  const char* what = "gs_preprocess_forward";
  refuse_duals("RasterizeGaussians", v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.cov3D, v.cov2D, v.means2D,
               v.extras, v.Tw2v, v.Tv2c, v.campos, v.accum_weights_p);
  require(what, "means3D", v.points, at::kFloat), require(what, "scales", v.scales, at::kFloat);
  require(what, "rotations", v.rotations, at::kFloat), require(what, "opacities", v.opacities, at::kFloat);
  require(what, "shs", v.shs, at::kFloat), require(what, "Tw2v", v.Tw2v, at::kFloat);
  require(what, "Tv2c", v.Tv2c, at::kFloat), require(what, "cam_pos", v.campos, at::kFloat);
  require(what, "means2D", v.means2D, at::kFloat);
  if (v.points.dim() != 2 || v.points.size(-1) != 3) fail("Error shape for means3D");
  const int64_t P = v.points.size(0);
  const int M = sh_coefficients(what, v.shs, v.sh_rest, v.sh_degree, P);
  require_shape(what, "means2D", v.means2D, {P, 2});
  require_point_mask(what, v.culling, P);
  require_shape(what, "scales", v.scales, {P, 3}), require_shape(what, "rotations", v.rotations, {P, 4});
  require_shape(what, "opacities", v.opacities, {P, 1});
  require_shape(what, "Tw2v", v.Tw2v, {4, 4}), require_shape(what, "Tv2c", v.Tv2c, {4, 4});
  require_shape(what, "cam_pos", v.campos, {3});
  if (has(v.cov3D)) require(what, "cov3D_precomp", *v.cov3D, at::kFloat), require_shape(what, "cov3D_precomp", *v.cov3D, {P, 6});
  if (has(v.cov2D)) require(what, "cov2D_precomp", *v.cov2D, at::kFloat), require_shape(what, "cov2D_precomp", *v.cov2D, {P, 3});
  const char* blend = "gaussian_rasterize_forward";
  int E = 0;
  if (has(v.extras)) {
    require(blend, "extras", *v.extras, at::kFloat);
    if (v.extras->dim() != 2 || v.extras->size(0) != P) fail(std::string(blend) + ": extras must be [P,E]");
    if (v.extras->size(1) > 4) fail("Only support NUM_EXTRA=0,1,2,3,4");
    E = (int) v.extras->size(1);
  }
  require_accumulators(blend, v.accum_max_count, v.accum_weights_p, v.accum_weights_count, P);
  const int W = v.W, H = v.H;
  if (W <= 0 || H <= 0) fail("gs_preprocess_forward: bad sizes");
  const int64_t T = (int64_t) ((W + kTile - 1) / kTile) * ((H + kTile - 1) / kTile);
  const Tensor& like = v.points;
  void* stream = stream_of(like);

  Buffers b;
  b.radii = empty({P}, like, at::kInt), b.visible = empty({P}, like, at::kBool);
  b.ranges = empty({T, 2}, like, at::kLong), b.conic_opacity = empty({P, 4}, like);
  b.saved = c10::make_intrusive<Saved>();
  Saved& s = *b.saved;
  s.W = W, s.H = H, s.sh_degree = v.sh_degree, s.E = E, s.tan_x = v.tan_x, s.tan_y = v.tan_y, s.is_opengl = v.is_opengl;
  s.colors = b.keep.reserve((size_t) P * 12);
  s.cov3D  = b.keep.reserve(train || !has(v.cov3D) ? (size_t) P * 24 : 0);
  const float* sh_rest = has(v.sh_rest) && v.sh_rest->numel() > 0 ? f32(*v.sh_rest) : nullptr;
  s.has_derivs = train && fsgs_view_keeps_color_derivs(v.sh_degree, M, f32(v.shs), sh_rest) != 0;
  if (s.has_derivs) s.derivs = b.keep.reserve((size_t) P * 36);
  b.keep.allocate(like);
  const ViewScratch scratch(P, W, H, like);

  const float* colors = v.sh_degree < 0 ? f32(v.shs) : b.keep.at<float>(s.colors);
  uint32_t* masks = v.cull ? scratch.at<uint32_t>(scratch.masks) : nullptr;
  auto blend_maps = [&] {
    b.image = empty({3, H, W}, like), b.opacity = empty({H, W}, like), b.n_contrib = empty({H, W}, like, at::kInt);
    if (has(v.extras)) b.extras = empty({E, H, W}, like);
  };
  if (P > 0) {
    SlotCounters counters(like);
    int64_t* count = pinned_count();
    check(fsgs_gs_view_preprocess_derivs((int) P, W, H, v.sh_degree, M, v.is_opengl, f32(v.points), f32(v.scales),
                                         f32(v.rotations), f32(v.opacities), f32(v.shs), sh_rest, f32(v.Tw2v), f32(v.Tv2c),
                                         f32(v.campos), v.tan_x, v.tan_y, data<uint8_t>(opt(v.culling)), f32(opt(v.cov3D)),
                                         f32(opt(v.cov2D)), v.preserve, f32(v.means2D), scratch.at<float>(scratch.depths),
                                         v.sh_degree < 0 ? nullptr : b.keep.at<float>(s.colors), i32(b.radii),
                                         data<uint8_t>(b.visible), counters.data(),
                                         has(v.cov3D) ? nullptr : b.keep.at<float>(s.cov3D), f32(b.conic_opacity), masks,
                                         s.has_derivs ? b.keep.at<float>(s.derivs) : nullptr, scratch.small_rects(),
                                         scratch.small ? count : nullptr, stream),
          what);
    if (scratch.small) {
      b.point_list = small_view_lists(scratch, P, W, H, masks, counters, nullptr, b.ranges, count, stream, blend_maps);
    } else {
      check(fsgs_gs_view_count((int) P, W, H, f32(v.means2D), nullptr, nullptr, i32(b.radii), masks, counters.data(),
                               nullptr, count, i64(b.ranges), scratch.at<void>(scratch.bins), scratch.bins_bytes, stream),
            "GS_prepare");
      PendingCount pending(count, stream);
      counters.give_back();
      const Instances in = scatter_instances("GS_prepare", pending, instances_to_guess(P, T), like, [&](const Instances& to) {
        check(fsgs_gs_view_scatter((int) P, W, H, f32(v.means2D), nullptr, scratch.at<float>(scratch.depths), nullptr, i32(b.radii),
                                   masks, to.room, i64(b.ranges), scratch.at<void>(scratch.bins), scratch.bins_bytes, to.space.data_ptr(),
                                   to.space.numel(), stream),
              "GS_prepare");
      }, blend_maps);
      b.point_list = empty({in.count}, like, at::kInt);
      check(fsgs_gs_view_sort((int) P, W, H, f32(v.means2D), nullptr, scratch.at<float>(scratch.depths), nullptr, i32(b.radii), masks,
                              in.count, in.room, i64(b.ranges), i32(b.point_list), scratch.at<void>(scratch.bins), scratch.bins_bytes,
                              data<void>(in.space), in.room > 0 ? in.space.numel() : 0, stream),
            "GS_prepare");
    }
  } else {
    blend_maps();
    b.point_list = empty({0}, like, at::kInt);
    check(fsgs_gs_prepare_count(0, W, H, nullptr, nullptr, i64(b.ranges), scratch.at<void>(scratch.bins), scratch.bins_bytes, stream),
          "GS_prepare");
  }
  if (train) b.hit_blocks = empty({b.point_list.numel()}, like, at::kInt);
  check(fsgs_gaussian_view_forward((int) P, W, H, E, f32(v.means2D), f32(b.conic_opacity), colors,
                                   E ? f32(*v.extras) : nullptr, i32(b.point_list), i64(b.ranges),
                                   i32(opt(v.accum_max_count)), f32(opt(v.accum_weights_p)),
                                   i32(opt(v.accum_weights_count)), f32(b.image), f32(b.opacity),
                                   E ? f32(b.extras) : nullptr, i32(b.n_contrib), (uint32_t*) i32(b.hit_blocks), stream),
        blend);
  return b;
}

variable_list outputs_of(const GaussianView& v, const Buffers& b) {
  Tensor screen;
  {
    at::AutoDispatchBelowADInplaceOrView plain;  // shares the leaf's storage, no view in the graph's sense
    screen = sharing_edits(v.means2D, at::alias(v.means2D));
  }
  variable_list out = {b.image, b.opacity, screen, b.conic_opacity};
  if (b.extras.defined()) out.push_back(b.extras);
  return out;
}

struct GaussianRender : public torch::autograd::Function<GaussianRender> {
  // all but the last two are what the node has edges to
  static variable_list forward(AutogradContext* ctx, const Tensor& points, const Tensor& scales, const Tensor& rotations,
                               const Tensor& opacities, const Tensor& shs, const OptTensor& sh_rest,
                               const OptTensor& cov3D, const OptTensor& cov2D, const Tensor& means2D,
                               const OptTensor& extras, const GaussianView* view, Buffers* out) {
    (void) points, (void) scales, (void) rotations, (void) opacities, (void) shs, (void) sh_rest, (void) cov3D,
        (void) cov2D, (void) means2D, (void) extras;
    const GaussianView& v = *view;
    *out = forward_view(v, true);
    const Buffers& b = *out;
    ctx->save_for_backward({v.points, v.scales, v.rotations, v.opacities, v.shs, opt(v.sh_rest), opt(v.cov3D), opt(v.cov2D),
                            v.means2D, opt(v.extras), v.Tw2v, v.Tv2c, v.campos, b.radii, b.ranges, b.point_list,
                            b.n_contrib, b.conic_opacity, b.opacity, b.keep.memory(), b.hit_blocks});
    ctx->saved_data["view"] = c10::IValue::make_capsule(b.saved);
    ctx->set_materialize_grads(false);
    return outputs_of(v, b);
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const Tensor &points = t[0], &scales = t[1], &rotations = t[2], &opacities = t[3], &shs = t[4], &sh_rest = t[5],
                 &cov3D = t[6], &cov2D = t[7], &means2D = t[8], &extras = t[9], &Tw2v = t[10], &Tv2c = t[11],
                 &campos = t[12], &radii = t[13], &ranges = t[14], &point_list = t[15], &n_contrib = t[16],
                 &conic_opacity = t[17], &opacity = t[18];
    const auto capsule = ctx->saved_data["view"].toCapsule();
    const Saved& s = *static_cast<const Saved*>(capsule.get());
    auto keep = [&](size_t at) { return (float*) ((char*) t[19].data_ptr() + at); };
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const int W = s.W, H = s.H;
    const int64_t P = points.size(0);
    void* stream = stream_of(points);
    const variable_list upstream = g;
    for (auto& x : g) x = contiguous(x);
    auto given = [&](const Tensor& x, at::IntArrayRef shape) { return x.defined() ? x : at::zeros(shape, points.options()); };
    const Tensor g_image = given(g[0], {3, H, W}), g_opacity = given(g[1], {H, W});
    const Tensor g_maps = s.E ? given(g[4], {s.E, H, W}) : Tensor();

    // the context numbers the node's edges, and an optional input that was left out has none
    size_t edge = 0;
    auto wanted = [&](const Tensor& x) { return x.defined() && ctx->needs_input_grad(edge++); };
    wanted(points);
    const bool want_scales = wanted(scales), want_rot = wanted(rotations);
    wanted(opacities);
    const bool want_sh = wanted(shs), want_rest = wanted(sh_rest), want_cov3D = wanted(cov3D), want_cov2D = wanted(cov2D);
    auto like_if = [](bool want, const Tensor& x) { return want ? at::empty_like(x) : Tensor(); };
    // the blend adds its sums to these: screen positions 2 | conic and opacity 4 | colours 3 | extras E
    const Tensor sums = at::zeros({P * (9 + s.E)}, points.options());
    Tensor g_means2D = sums.narrow(0, 0, 2 * P).view({P, 2}), g_conic = sums.narrow(0, 2 * P, 4 * P).view({P, 4}),
           g_colors = sums.narrow(0, 6 * P, 3 * P).view({P, 3}), g_extras;
    if (extras.defined()) g_extras = sums.narrow(0, 9 * P, s.E * P).view({P, s.E});
    const bool sh = s.sh_degree >= 0, rest_used = sh_rest.defined() && sh_rest.numel() > 0;
    Tensor g_points = at::empty_like(points), g_opac = at::empty_like(opacities), g_scales, g_rot, g_cov3D, g_cov2D, g_sh,
           g_rest;
    // which covariance was given decides where its gradient goes
    if (cov2D.defined()) g_cov2D = like_if(want_cov2D, cov2D);
    else if (cov3D.defined()) g_cov3D = like_if(want_cov3D, cov3D);
    else g_scales = like_if(want_scales, scales), g_rot = like_if(want_rot, rotations);
    if (sh) g_sh = like_if(want_sh, shs), g_rest = like_if(want_rest, sh_rest);
    if (P > 0) {
      const float* colors = sh ? keep(s.colors) : f32(shs);
      const int M = rest_used ? (int) sh_rest.size(1) : shs.dim() == 3 ? (int) shs.size(1) : 0;
      check(fsgs_gaussian_view_backward((int) P, W, H, s.E, f32(means2D), f32(conic_opacity), colors,
                                             s.E ? f32(extras) : nullptr, f32(opacity), i32(n_contrib), f32(g_image),
                                             f32(g_maps), f32(g_opacity), i32(point_list), i64(ranges), f32(g_means2D),
                                             f32(g_conic), f32(g_colors), s.E ? f32(g_extras) : nullptr,
                                             (const uint32_t*) i32(t[20]), stream),
            "gaussian_rasterize_backward");
      if (g[2].defined()) g_means2D.add_(g[2]);
      if (g[3].defined()) g_conic.add_(g[3]);
      check(fsgs_gs_view_preprocess_backward_derivs((int) P, W, H, s.sh_degree, M, s.is_opengl, f32(points), f32(scales),
                                                    f32(rotations), f32(shs), rest_used ? f32(sh_rest) : nullptr, f32(Tw2v),
                                                    f32(Tv2c), f32(campos), s.tan_x, s.tan_y, i32(radii), colors,
                                                    cov3D.defined() ? f32(cov3D) : keep(s.cov3D), f32(cov2D),
                                                    s.has_derivs ? keep(s.derivs) : nullptr, f32(g_means2D), f32(g_colors),
                                                    f32(g_conic), f32(g_points), f32(g_scales), f32(g_rot), f32(g_opac),
                                                    f32(g_sh), rest_used ? f32(g_rest) : nullptr,
                                                    f32(cov2D.defined() ? g_cov2D : g_cov3D), nullptr, nullptr, stream),
            "gs_preprocess_backward");
    }
    if (!sh && want_sh) g_sh = g_colors;  // pre-computed colours: the blend's sums are their gradient
    return first_order_only(upstream, {points, scales, rotations, opacities, shs, sh_rest, cov3D, cov2D, means2D, extras},
                            {g_points, g_scales, g_rot, g_opac, g_sh, g_rest, g_cov3D, g_cov2D, g_means2D, g_extras, Tensor(),
                             Tensor()});
  }
};

}  // namespace

GaussianResult gaussian_render(const GaussianView& v) {
  GaussianResult r;
  Buffers b;
  auto wants = [](const OptTensor& t) { return has(t) && t->requires_grad(); };
  const bool train = at::GradMode::is_enabled() &&
                     (v.points.requires_grad() || v.scales.requires_grad() || v.rotations.requires_grad() ||
                      v.opacities.requires_grad() || v.shs.requires_grad() || v.means2D.requires_grad() || wants(v.sh_rest) ||
                      wants(v.cov3D) || wants(v.cov2D) || wants(v.extras));
  if (train) {
    r.maps = GaussianRender::apply(v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.cov3D, v.cov2D,
                                   v.means2D, v.extras, &v, &b);
  } else {
    b      = forward_view(v, false);
    r.maps = outputs_of(v, b);
  }
  r.n_contrib = b.n_contrib, r.radii = b.radii, r.visible = b.visible, r.ranges = b.ranges, r.point_list = b.point_list;
  return r;
}

}  // namespace fsgs_host
