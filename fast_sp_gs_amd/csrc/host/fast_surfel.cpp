// One view of the "fast" 2D-Gaussian-surfel renderer (adjugate transforms, corner-tested tile lists), forward and
// backward, as one call and one autograd node: the steps of fast_2d_gs/renderer/gs_2d_fast_render.py:592-754, the
// per-pixel tail (:733-743) as the fused epilogue kernel. In torch that tail and its backward were 75 launches with two
// LU factorisations and three copies to the host among them: 0.75 of the 1.24 ms of a training pass over 150k surfels at
// 1001x667.
#include "fast_surfel.hpp"

namespace fsgs_host {
namespace {

struct Saved : torch::CustomClassHolder {  // what the backward reads besides tensors
  int W, H, sh_degree;
  double near_n, far_n, depth_ratio;
  bool epilogue;
  int64_t R = 0;
  size_t colors, trans_mat, inverse_m, normal_opacity, masks, offsets, regions, tiles, derivs;  // places in the slab
  bool has_derivs = false;
};

struct Buffers {
  Tensor radii, visible, ranges, point_list, n_contrib;
  Tensor image, opacity, extras, flow;        // what the blend writes
  Tensor normals, surf_depth, surf_normal;    // the epilogue's maps
  Tensor distortion;                          // instead of the extras, when nothing is kept for a backward
  Tensor hit_blocks;                          // per list entry, for the backward
  Slab keep;                                  // per-surfel intermediates, read again by the backward
  c10::intrusive_ptr<Saved> saved;
};

Buffers forward_view(const FastSurfelView& v, bool train) {
  const char* what = "gs_2d_fast_preprocess_forward";
  refuse_duals("GS_2D_fast_render", v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.means2D, v.Tw2v, v.Tv2c,
               v.Tv2s, v.campos, v.trans_mat_t2, v.accum_weights_p);
  require(what, "means3D", v.points, at::kFloat), require(what, "scales", v.scales, at::kFloat);
  require(what, "rotations", v.rotations, at::kFloat), require(what, "opacities", v.opacities, at::kFloat);
  require(what, "shs", v.shs, at::kFloat), require(what, "Tw2v", v.Tw2v, at::kFloat);
  require(what, "Tv2c", v.Tv2c, at::kFloat), require(what, "Tv2s", v.Tv2s, at::kFloat);
  require(what, "cam_pos", v.campos, at::kFloat);
  if (v.points.dim() != 2 || v.points.size(-1) != 3) fail("Error shape for means3D");
  const int64_t P = v.points.size(0);
  const int M = sh_coefficients(what, v.shs, v.sh_rest, v.sh_degree, P);
  require_point_mask(what, v.culling, P);
  require_shape(what, "scales", v.scales, {P, 2}), require_shape(what, "rotations", v.rotations, {P, 4});
  require_shape(what, "opacities", v.opacities, {P, 1});
  require_shape(what, "Tw2v", v.Tw2v, {4, 4}), require_shape(what, "Tv2c", v.Tv2c, {4, 4});
  require_shape(what, "Tv2s", v.Tv2s, {3, 3}), require_shape(what, "cam_pos", v.campos, {3});
  const char* blend = "GS_2D_fast_render_forward";
  const bool flow = has(v.trans_mat_t2);
  if (flow) {
    require(blend, "trans_mat_t2", *v.trans_mat_t2, at::kFloat);
    require_shape(blend, "trans_mat_t2", *v.trans_mat_t2, {P, 3, 3});
  }
  require_accumulators(blend, v.accum_max_count, v.accum_weights_p, v.accum_weights_count, P);
  const int W = v.W, H = v.H;
  if (W <= 0 || H <= 0) fail("gs_2d_fast_preprocess_forward: bad sizes");
  const int64_t T = (int64_t) ((W + kTile - 1) / kTile) * ((H + kTile - 1) / kTile);
  const Tensor& like = v.points;
  void* stream = stream_of(like);

  Buffers b;
  b.radii = empty({P}, like, at::kInt), b.visible = empty({P}, like, at::kBool);
  b.ranges = empty({T, 2}, like, at::kLong);
  b.saved = c10::make_intrusive<Saved>();
  Saved& s = *b.saved;
  s.W = W, s.H = H, s.sh_degree = v.sh_degree, s.near_n = v.near_n, s.far_n = v.far_n;
  s.depth_ratio = v.depth_ratio, s.epilogue = v.epilogue;
  s.normal_opacity = b.keep.reserve((size_t) P * 16);
  s.colors    = b.keep.reserve((size_t) P * 12);
  s.trans_mat = b.keep.reserve((size_t) P * 36);
  s.inverse_m = b.keep.reserve((size_t) P * 36);
  s.masks     = b.keep.reserve((size_t) P * 4);
  s.tiles     = b.keep.reserve((size_t) P * 4);
  const float* sh_rest = has(v.sh_rest) && v.sh_rest->numel() > 0 ? f32(*v.sh_rest) : nullptr;
  if (train) s.offsets = b.keep.reserve((size_t) P * 4), s.regions = b.keep.reserve(kSlotRegions * 4);
  s.has_derivs = train && fsgs_view_keeps_color_derivs(v.sh_degree, M, f32(v.shs), sh_rest) != 0;
  if (s.has_derivs) s.derivs = b.keep.reserve((size_t) P * 36);
  b.keep.allocate(like);
  Slab scratch;
  const size_t depths = scratch.reserve((size_t) P * 4);
  const size_t bins_bytes = fsgs_gs_prepare_bins_bytes((int) P, W, H);
  const size_t bins = scratch.reserve(bins_bytes);
  scratch.allocate(like);

  const float* colors = v.sh_degree < 0 ? f32(v.shs) : b.keep.at<float>(s.colors);
  float *trans_mat = b.keep.at<float>(s.trans_mat), *inverse_m = b.keep.at<float>(s.inverse_m),
        *normal_opacity = b.keep.at<float>(s.normal_opacity);
  uint32_t* masks = b.keep.at<uint32_t>(s.masks);
  auto blend_maps = [&] {
    b.image = empty({3, H, W}, like), b.opacity = empty({H, W}, like);
    if (train || !v.epilogue) b.extras = empty({8, H, W}, like);
    else b.distortion = empty({1, H, W}, like);
    b.n_contrib = empty({2, H, W}, like, at::kInt);
    if (flow) b.flow = empty({H, W, 2}, like);
    // the blend writes the maps that need no neighbour, and the extra channels only where a backward will read them
    if (v.epilogue)
      b.normals = empty({3, H, W}, like), b.surf_depth = empty({1, H, W}, like), b.surf_normal = empty({3, H, W}, like);
  };
  if (P > 0) {
    SlotCounters counters(like);
    int64_t* count = pinned_count();
    check(fsgs_gs_2d_fast_view_preprocess_derivs(
              (int) P, W, H, v.sh_degree, M, f32(v.points), f32(v.scales), f32(v.rotations), f32(v.opacities), f32(v.shs), sh_rest,
              f32(v.Tw2v), f32(v.Tv2s), f32(v.campos), data<uint8_t>(opt(v.culling)), f32(v.means2D),
              v.sh_degree < 0 ? nullptr : b.keep.at<float>(s.colors), trans_mat, inverse_m, normal_opacity,
              scratch.at<float>(depths), i32(b.radii), data<uint8_t>(b.visible), b.keep.at<int32_t>(s.tiles),
              train ? b.keep.at<int32_t>(s.offsets) : nullptr, counters.data(), masks,
              s.has_derivs ? b.keep.at<float>(s.derivs) : nullptr, stream),
          what);
    check(fsgs_gs_view_count((int) P, W, H, f32(v.means2D), inverse_m, f32(v.opacities), i32(b.radii), masks, counters.data(),
                             train ? b.keep.at<int32_t>(s.regions) : nullptr, count, i64(b.ranges), scratch.at<void>(bins),
                             bins_bytes, stream),
          what);
    PendingCount pending(count, stream);
    counters.give_back();
    const Instances in = scatter_instances(what, pending, instances_to_guess(P, T), like, [&](const Instances& to) {
      check(fsgs_gs_view_scatter((int) P, W, H, f32(v.means2D), inverse_m, scratch.at<float>(depths), f32(v.opacities), i32(b.radii),
                                 masks, to.room, i64(b.ranges), scratch.at<void>(bins), bins_bytes, to.space.data_ptr(),
                                 to.space.numel(), stream),
            what);
    }, blend_maps);
    s.R = in.count;
    b.point_list = empty({in.count}, like, at::kInt);
    check(fsgs_gs_view_sort((int) P, W, H, f32(v.means2D), inverse_m, scratch.at<float>(depths), f32(v.opacities), i32(b.radii), masks,
                            in.count, in.room, i64(b.ranges), i32(b.point_list), scratch.at<void>(bins), bins_bytes,
                            data<void>(in.space), in.room > 0 ? in.space.numel() : 0, stream),
          what);
  } else {
    blend_maps();
    b.point_list = empty({0}, like, at::kInt);
    check(fsgs_gs_prepare_count(0, W, H, nullptr, nullptr, i64(b.ranges), scratch.at<void>(bins), bins_bytes, stream), what);
  }
  if (train) b.hit_blocks = empty({b.point_list.numel()}, like, at::kInt);
  check(fsgs_gs_2d_fast_view_forward((int) P, W, H, v.near_n, v.far_n, f32(v.means2D), colors, normal_opacity, trans_mat,
                                     inverse_m, i32(b.point_list), i64(b.ranges), f32(opt(v.trans_mat_t2)),
                                     i32(opt(v.accum_max_count)), f32(opt(v.accum_weights_p)),
                                     i32(opt(v.accum_weights_count)), f32(b.image), f32(b.opacity), f32(b.extras),
                                     f32(b.flow), i32(b.n_contrib), (uint32_t*) i32(b.hit_blocks), v.depth_ratio,
                                     f32(v.Tw2v), f32(b.normals), f32(b.surf_depth), f32(b.distortion), stream),
        blend);
  if (v.epilogue)
    check(fsgs_gs_2d_view_surf_normal(W, H, f32(v.Tw2v), f32(v.Tv2c), f32(b.surf_depth), f32(b.opacity), f32(b.surf_normal),
                                      stream),
          "gs_2d_epilogue_forward");
  return b;
}

// Output order of a view, with and without the epilogue; the flow comes last, when there is one.
variable_list outputs_of(const Buffers& b) {
  variable_list out;
  if (!b.saved->epilogue) {
    out = {b.image, b.opacity, b.extras};
  } else {
    Tensor distortion = b.distortion;
    if (b.extras.defined()) {
      at::AutoDispatchBelowADInplaceOrView plain;  // shares extras' storage, no view in the graph's sense
      distortion = sharing_edits(b.extras, b.extras.narrow(0, 5, 1));
    }
    out = {b.image, b.opacity, b.normals, b.surf_depth, b.surf_normal, distortion};
  }
  if (b.flow.defined()) out.push_back(b.flow);
  return out;
}

struct FastSurfelRender : public torch::autograd::Function<FastSurfelRender> {
  // points, scales, rotations, opacities, shs, sh_rest and means2D are what the node has edges to
  static variable_list forward(AutogradContext* ctx, const Tensor& points, const Tensor& scales, const Tensor& rotations,
                               const Tensor& opacities, const Tensor& shs, const OptTensor& sh_rest,
                               const Tensor& means2D, const FastSurfelView* view, Buffers* out) {
    (void) points, (void) scales, (void) rotations, (void) opacities, (void) shs, (void) sh_rest, (void) means2D;
    const FastSurfelView& v = *view;
    *out = forward_view(v, true);
    const Buffers& b = *out;
    ctx->save_for_backward({v.points, v.scales, v.rotations, v.opacities, v.shs, opt(v.sh_rest), v.means2D, v.Tw2v, v.Tv2c,
                            v.Tv2s, v.campos, opt(v.trans_mat_t2), b.radii, b.ranges, b.point_list, b.n_contrib,
                            b.opacity, b.extras, b.flow, b.keep.memory(), b.hit_blocks});
    ctx->saved_data["view"] = c10::IValue::make_capsule(b.saved);
    ctx->set_materialize_grads(false);
    return outputs_of(b);
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const Tensor &points = t[0], &scales = t[1], &rotations = t[2], &opacities = t[3], &shs = t[4], &sh_rest = t[5],
                 &means2D = t[6], &Tw2v = t[7], &Tv2c = t[8], &Tv2s = t[9], &campos = t[10], &t2 = t[11], &radii = t[12],
                 &ranges = t[13], &point_list = t[14], &n_contrib = t[15], &opacity = t[16], &extras = t[17],
                 &flow = t[18];
    const auto capsule = ctx->saved_data["view"].toCapsule();
    const Saved& s = *static_cast<const Saved*>(capsule.get());
    auto keep = [&](size_t at) { return (float*) ((char*) t[19].data_ptr() + at); };
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const int W = s.W, H = s.H;
    const int64_t P = points.size(0);
    void* stream = stream_of(points);
    const variable_list upstream = g;
    for (auto& x : g) x = contiguous(x);

    Tensor g_image = g[0], g_opacity = g[1], g_extras, g_flow;
    if (s.epilogue) {
      if (g.size() > 6) g_flow = g[6];
      if (g[2].defined() || g[3].defined() || g[4].defined() || g[5].defined()) {
        g_extras = empty({6, H, W}, points);  // the channels that the blend has a gradient for
        check(fsgs_gs_2d_view_epilogue_backward(W, H, 6, s.depth_ratio, f32(Tw2v), f32(Tv2c), f32(extras), f32(opacity),
                                                nullptr, f32(g[2]), nullptr, f32(g[3]), f32(g[4]), f32(g[5]), nullptr,
                                                nullptr, f32(g_extras), nullptr, stream),
              "gs_2d_epilogue_backward");
      }
    } else {
      g_extras = g[2];
      if (g.size() > 3) g_flow = g[3];
    }
    if (!g_extras.defined()) g_flow = Tensor();
    if (!g_image.defined()) g_image = at::zeros({3, H, W}, points.options());
    if (!g_opacity.defined() && s.R == 0) g_opacity = at::zeros({H, W}, points.options());  // without notes it has to be there

    const bool want_sh = ctx->needs_input_grad(4), has_rest = sh_rest.defined(), rest_used = has_rest && sh_rest.numel() > 0;
    Tensor g_means2D = empty({P, 2}, points);
    Tensor g_points = at::empty_like(points), g_scales = at::empty_like(scales), g_rot = at::empty_like(rotations),
           g_opac = at::empty_like(opacities), g_sh, g_rest;
    if (want_sh) g_sh = at::empty_like(shs);  // pre-computed colours: the blend's sums are their gradient
    if (has_rest && ctx->needs_input_grad(5)) g_rest = at::empty_like(sh_rest);
    if (P > 0) {
      const bool sh = s.sh_degree >= 0, aux = g_extras.defined();
      Slab scratch;
      const size_t g_no = scratch.reserve((size_t) P * 16), g_trans = scratch.reserve((size_t) P * 36),
                   g_inv = scratch.reserve((size_t) P * 36), g_col = scratch.reserve(sh || !want_sh ? (size_t) P * 12 : 0);
      const size_t ws_bytes = fsgs_gs_2d_fast_render_backward_workspace_bytes(s.R);
      const size_t ws = scratch.reserve(ws_bytes);
      scratch.allocate(points);
      float* g_colors = sh || !want_sh ? scratch.at<float>(g_col) : f32(g_sh);
      const float* colors = sh ? keep(s.colors) : f32(shs);
      const int M = rest_used ? (int) sh_rest.size(1) : shs.dim() == 3 ? (int) shs.size(1) : 0;
      check(fsgs_gs_2d_fast_view_backward_hits((int) P, W, H, s.near_n, s.far_n, f32(means2D), keep(s.normal_opacity), colors,
                                          keep(s.trans_mat), keep(s.inverse_m), f32(t2), f32(opacity),
                                          aux ? f32(extras) : nullptr, g_flow.defined() ? f32(flow) : nullptr, f32(g_image),
                                          f32(g_opacity), f32(g_extras), f32(g_flow), i64(ranges), i32(point_list),
                                          i32(n_contrib), g_colors, f32(g_means2D), scratch.at<float>(g_trans),
                                          scratch.at<float>(g_inv), scratch.at<float>(g_no), s.R,
                                          (const int32_t*) keep(s.offsets), (const int32_t*) keep(s.regions),
                                          (const int32_t*) keep(s.tiles), i32(radii), scratch.at<void>(ws), ws_bytes,
                                          (const uint32_t*) keep(s.masks), (const uint32_t*) i32(t[20]), stream),
            "GS_2D_fast_render_backward");
      check(fsgs_gs_2d_fast_view_preprocess_backward_derivs(
                (int) P, W, H, s.sh_degree, M, f32(points), f32(scales), f32(rotations), f32(shs),
                rest_used ? f32(sh_rest) : nullptr, f32(Tw2v), f32(Tv2s), f32(campos), keep(s.trans_mat), i32(radii), colors,
                s.has_derivs ? keep(s.derivs) : nullptr, f32(g_means2D), scratch.at<float>(g_trans), scratch.at<float>(g_inv),
                g_colors, scratch.at<float>(g_no), f32(g_points), f32(g_scales), f32(g_rot), f32(g_opac),
                sh ? f32(g_sh) : nullptr, rest_used ? f32(g_rest) : nullptr, stream),
            "gs_2d_fast_preprocess_backward");
    }
    return first_order_only(upstream, {points, scales, rotations, opacities, shs, sh_rest, means2D},
                            {g_points, g_scales, g_rot, g_opac, g_sh, g_rest, g_means2D, Tensor(), Tensor()});
  }
};

}  // namespace

FastSurfelResult fast_surfel_render(const FastSurfelView& v) {
  FastSurfelResult r;
  Buffers b;
  const bool train = at::GradMode::is_enabled() &&
                     (v.points.requires_grad() || v.scales.requires_grad() || v.rotations.requires_grad() ||
                      v.opacities.requires_grad() || v.shs.requires_grad() || (has(v.sh_rest) && v.sh_rest->requires_grad()) ||
                      v.means2D.requires_grad());
  if (train) {
    r.maps = FastSurfelRender::apply(v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.means2D, &v, &b);
  } else {
    b      = forward_view(v, false);
    r.maps = outputs_of(b);
  }
  r.radii = b.radii, r.visible = b.visible;
  return r;
}

}  // namespace fsgs_host
