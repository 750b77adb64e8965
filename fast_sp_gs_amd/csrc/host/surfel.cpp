// One view of the 2D-Gaussian-surfel renderer, forward and backward, as one call and one autograd node: preprocess ->
// binning -> blend (-> per-pixel epilogue), the steps of fast_2d_gs/renderer/gs_2d_render.py:480-633.
#include "surfel.hpp"

namespace fsgs_host {
namespace {

struct Saved {  // what the backward reads besides tensors
  int W, H, sh_degree;
  double near_n, far_n, depth_ratio;
  bool epilogue;
  int64_t R;
  size_t colors, records, masks, offsets, regions, tiles, derivs;  // places in the slab
  bool has_derivs;
};

struct Buffers {
  Tensor trans_mat, normal_opacity, radii, visible, ranges, point_list, n_contrib;
  Tensor image, opacity, extras, flow;                       // what the blend writes
  Tensor normals, depths, surf_depth, surf_normal;  // the epilogue's maps; the image is composited then, given a background
  Tensor distortion;                                          // instead of the extras, when nothing is kept for a backward
  Tensor hit_blocks;                                          // per list entry, for the backward
  Slab keep;                                                  // what only the backward reads
  Saved saved;
};

Buffers forward_view(const SurfelView& v, bool train) {
  const char* what = "gs_2d_preprocess_forward";
  refuse_duals("GS_2D_render", v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.means2D, v.Tw2v, v.Tv2c,
               v.campos, v.background, v.trans_mat_t2, v.accum_weights_p);
  require(what, "means3D", v.points, at::kFloat), require(what, "scales", v.scales, at::kFloat);
  require(what, "rotations", v.rotations, at::kFloat), require(what, "opacities", v.opacities, at::kFloat);
  require(what, "shs", v.shs, at::kFloat), require(what, "Tw2v", v.Tw2v, at::kFloat);
  require(what, "Tv2c", v.Tv2c, at::kFloat), require(what, "cam_pos", v.campos, at::kFloat);
  if (v.points.dim() != 2 || v.points.size(-1) != 3) fail("Error shape for means3D");
  const int64_t P = v.points.size(0);
  const int M = sh_coefficients(what, v.shs, v.sh_rest, v.sh_degree, P);
  require_point_mask(what, v.culling, P);
  require_shape(what, "scales", v.scales, {P, 2}), require_shape(what, "rotations", v.rotations, {P, 4});
  require_shape(what, "opacities", v.opacities, {P, 1});
  require_shape(what, "Tw2v", v.Tw2v, {4, 4}), require_shape(what, "Tv2c", v.Tv2c, {4, 4});
  require_shape(what, "cam_pos", v.campos, {3});
  const char* blend = "GS_2D_render_forward";
  const bool flow = has(v.trans_mat_t2);
  if (flow) {
    require(blend, "trans_mat_t2", *v.trans_mat_t2, at::kFloat);
    require_shape(blend, "trans_mat_t2", *v.trans_mat_t2, {P, 3, 3});
  }
  require_accumulators(blend, v.accum_max_count, v.accum_weights_p, v.accum_weights_count, P);
  if (has(v.background)) {
    require("gs_2d_epilogue_forward", "background", *v.background, at::kFloat);
    if (v.background->numel() != 3) fail("gs_2d_epilogue_forward: background must have 3 elements");
  }
  const int W = v.W, H = v.H, gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  if (W <= 0 || H <= 0)
    fail("gs_2d_preprocess_forward: bad sizes P=" + std::to_string(P) + " W=" + std::to_string(W) + " H=" + std::to_string(H));
  const int64_t T = (int64_t) gx * gy;
  const Tensor& like = v.points;
  void* stream = stream_of(like);

  Buffers b;
  b.trans_mat = empty({P, 3, 3}, like), b.normal_opacity = empty({P, 4}, like);
  b.radii = empty({P}, like, at::kInt), b.visible = empty({P}, like, at::kBool);
  b.ranges = empty({T, 2}, like, at::kLong);
  Saved& s = b.saved;
  s = Saved{W, H, v.sh_degree, v.near_n, v.far_n, v.depth_ratio, v.epilogue, 0, 0, 0, 0, 0, 0, 0, 0, false};
  s.records = b.keep.reserve((size_t) P * 80);
  s.colors  = b.keep.reserve((size_t) P * 12);
  s.masks   = b.keep.reserve((size_t) P * 4);
  s.tiles   = b.keep.reserve((size_t) P * 4);
  const float* sh_rest = has(v.sh_rest) && v.sh_rest->numel() > 0 ? f32(*v.sh_rest) : nullptr;
  if (train) {
    s.offsets = b.keep.reserve((size_t) P * 4), s.regions = b.keep.reserve(kSlotRegions * 4);
    s.has_derivs = fsgs_view_keeps_color_derivs(v.sh_degree, M, f32(v.shs), sh_rest) != 0;
    if (s.has_derivs) s.derivs = b.keep.reserve((size_t) P * 36);
  }
  b.keep.allocate(like);
  const ViewScratch scratch(P, W, H, like);

  const float* colors = v.sh_degree < 0 ? f32(v.shs) : b.keep.at<float>(s.colors);
  uint32_t* masks = v.cull ? b.keep.at<uint32_t>(s.masks) : nullptr;
  float* records  = b.keep.at<float>(s.records);
  auto blend_maps = [&] {
    b.image = empty({3, H, W}, like), b.opacity = empty({H, W}, like), b.n_contrib = empty({2, H, W}, like, at::kInt);
    if (train || !v.epilogue) b.extras = empty({9, H, W}, like);
    else b.distortion = empty({1, H, W}, like);
    if (flow) b.flow = empty({H, W, 2}, like);
    // the blend writes the maps that need no neighbour, and the extra channels only where a backward will read them
    if (v.epilogue) {
      b.normals = empty({3, H, W}, like), b.depths = empty({1, H, W}, like), b.surf_depth = empty({1, H, W}, like);
      b.surf_normal = empty({3, H, W}, like);
    }
  };
  if (P > 0) {
    SlotCounters counters(like);
    int64_t* count = pinned_count();
    int64_t* count_of_small = scratch.small ? count : nullptr;
    auto preprocess = [&](auto entry, auto... outputs) {
      check(entry((int) P, W, H, v.sh_degree, M, f32(v.points), f32(v.scales), f32(v.rotations), f32(v.opacities), f32(v.shs),
                  sh_rest, f32(v.Tw2v), f32(v.Tv2c), f32(v.campos), data<uint8_t>(opt(v.culling)), f32(v.means2D),
                  v.sh_degree < 0 ? nullptr : b.keep.at<float>(s.colors), f32(b.trans_mat), f32(b.normal_opacity),
                  scratch.at<float>(scratch.depths), i32(b.radii), data<uint8_t>(b.visible), b.keep.at<int32_t>(s.tiles), outputs...,
                  stream),
            what);
    };
    if (train)
      preprocess(fsgs_gs_2d_view_preprocess_derivs, b.keep.at<int32_t>(s.offsets), counters.data(), records, masks,
                 s.has_derivs ? b.keep.at<float>(s.derivs) : nullptr, scratch.small_rects(), count_of_small);
    else preprocess(fsgs_gs_2d_view_preprocess_no_backward_rects, counters.data(), records, masks, scratch.small_rects(), count_of_small);
    int32_t* regions = train ? b.keep.at<int32_t>(s.regions) : nullptr;
    if (scratch.small) {
      b.point_list = small_view_lists(scratch, P, W, H, masks, counters, regions, b.ranges, count, stream, blend_maps);
      s.R = b.point_list.numel();
    } else {
      check(fsgs_gs_view_count((int) P, W, H, f32(v.means2D), nullptr, nullptr, i32(b.radii), masks, counters.data(),
                               regions, count, i64(b.ranges), scratch.at<void>(scratch.bins), scratch.bins_bytes, stream),
            "GS_prepare");
      PendingCount pending(count, stream);
      counters.give_back();
      const Instances in = scatter_instances("GS_prepare", pending, instances_to_guess(P, T), like, [&](const Instances& to) {
        check(fsgs_gs_view_scatter((int) P, W, H, f32(v.means2D), nullptr, scratch.at<float>(scratch.depths), nullptr, i32(b.radii),
                                   masks, to.room, i64(b.ranges), scratch.at<void>(scratch.bins), scratch.bins_bytes, to.space.data_ptr(),
                                   to.space.numel(), stream),
              "GS_prepare");
      }, blend_maps);
      s.R = in.count;
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
  const bool composite = v.epilogue && has(v.background);
  check(fsgs_gs_2d_view_forward((int) P, W, H, v.near_n, v.far_n, f32(v.means2D), colors, f32(b.normal_opacity),
                                  f32(b.trans_mat), i32(b.point_list), i64(b.ranges), f32(opt(v.trans_mat_t2)),
                                  i32(opt(v.accum_max_count)), f32(opt(v.accum_weights_p)),
                                  i32(opt(v.accum_weights_count)), f32(b.image), f32(b.opacity), f32(b.extras),
                                  f32(b.flow), i32(b.n_contrib), records, (uint32_t*) i32(b.hit_blocks), v.depth_ratio,
                                  f32(v.Tw2v), composite ? f32(*v.background) : nullptr, f32(b.normals), f32(b.depths),
                                  f32(b.surf_depth), f32(b.distortion), stream),
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
  if (!b.saved.epilogue) {
    out = {b.image, b.opacity, b.extras};
    if (b.flow.defined()) out.push_back(b.flow);
    return out;
  }
  Tensor distortion = b.distortion;
  if (b.extras.defined()) {
    at::AutoDispatchBelowADInplaceOrView plain;  // shares extras' storage, no view in the graph's sense
    distortion = sharing_edits(b.extras, b.extras.narrow(0, 5, 1));
  }
  out = {b.image, b.opacity, b.normals, b.depths, b.surf_depth, b.surf_normal,
         distortion};
  if (b.flow.defined()) out.push_back(b.flow);
  return out;
}

struct SurfelRender : public torch::autograd::Function<SurfelRender> {
  // points, scales, rotations, opacities, shs, sh_rest and means2D are what the node has edges to
  static variable_list forward(AutogradContext* ctx, const Tensor& points, const Tensor& scales, const Tensor& rotations,
                               const Tensor& opacities, const Tensor& shs, const OptTensor& sh_rest,
                               const Tensor& means2D, const SurfelView* view, Buffers* out) {
    (void) points, (void) scales, (void) rotations, (void) opacities, (void) shs, (void) sh_rest, (void) means2D;
    const SurfelView& v = *view;
    *out = forward_view(v, true);
    const Buffers& b = *out;
    ctx->save_for_backward({v.points, v.scales, v.rotations, v.opacities, v.shs, opt(v.sh_rest), v.means2D, v.Tw2v,
                            v.Tv2c, v.campos, opt(v.background), opt(v.trans_mat_t2), b.trans_mat, b.normal_opacity,
                            b.radii, b.ranges, b.point_list, b.n_contrib, b.opacity, b.extras, b.flow, b.keep.memory(),
                            b.hit_blocks});
    ctx->saved_data["view"] = c10::IValue::make_capsule(c10::make_intrusive<SavedHolder>(b.saved, v.cull));
    ctx->set_materialize_grads(false);
    return outputs_of(b);
  }

  struct SavedHolder : torch::CustomClassHolder {
    SavedHolder(const Saved& s, bool c) : saved(s), cull(c) {}
    Saved saved;
    bool cull;
  };

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto t = ctx->get_saved_variables();
    const Tensor &points = t[0], &scales = t[1], &rotations = t[2], &opacities = t[3], &shs = t[4], &sh_rest = t[5],
                 &means2D = t[6], &Tw2v = t[7], &Tv2c = t[8], &campos = t[9], &background = t[10], &t2 = t[11],
                 &trans_mat = t[12], &normal_opacity = t[13], &radii = t[14], &ranges = t[15], &point_list = t[16],
                 &n_contrib = t[17], &opacity = t[18], &extras = t[19], &flow = t[20];
    const auto capsule = ctx->saved_data["view"].toCapsule();
    const auto* holder = static_cast<const SavedHolder*>(capsule.get());
    const Saved& s = holder->saved;
    auto keep = [&](size_t at) { return (char*) t[21].data_ptr() + at; };
    at::AutoDispatchBelowADInplaceOrView no_graph;
    const int W = s.W, H = s.H;
    const int64_t P = points.size(0);
    void* stream = stream_of(points);
    const variable_list upstream = g;
    for (auto& x : g) x = contiguous(x);

    Tensor g_image = g[0], g_opacity = g[1], g_extras, g_flow;
    if (s.epilogue) {
      const Tensor &g_normals = g[2], &g_depths = g[3], &g_surf_depth = g[4], &g_surf_normal = g[5], &g_dist = g[6];
      if (g.size() > 7) g_flow = g[7];
      const bool composite = background.defined() && g_image.defined();
      if (composite || g_normals.defined() || g_depths.defined() || g_surf_depth.defined() || g_surf_normal.defined() ||
          g_dist.defined()) {
        g_extras = empty({6, H, W}, points);  // the channels that the blend has a gradient for
        Tensor g_total = composite || !g_opacity.defined() ? empty({H, W}, points) : Tensor();
        check(fsgs_gs_2d_view_epilogue_backward(W, H, 6, s.depth_ratio, f32(Tw2v), f32(Tv2c), f32(extras), f32(opacity),
                                                f32(background), f32(g_normals), f32(g_depths), f32(g_surf_depth),
                                                f32(g_surf_normal), f32(g_dist), composite ? f32(g_image) : nullptr,
                                                f32(g_opacity), f32(g_extras), f32(g_total), stream),
              "gs_2d_epilogue_backward");
        if (g_total.defined()) g_opacity = g_total;
      }
    } else {
      g_extras = g[2];
      if (g.size() > 3) g_flow = g[3];
    }
    if (!g_image.defined()) g_image = at::zeros({3, H, W}, points.options());
    if (!g_opacity.defined()) g_opacity = at::zeros({H, W}, points.options());

    const bool want_sh = ctx->needs_input_grad(4), has_rest = sh_rest.defined();
    const bool want_rest = has_rest && ctx->needs_input_grad(5);
    Tensor g_means2D = empty({P, 2}, points);
    Tensor g_points = at::empty_like(points), g_scales = at::empty_like(scales), g_rot = at::empty_like(rotations),
           g_opac = at::empty_like(opacities), g_sh, g_rest;
    // pre-computed colours (sh_degree < 0) receive no gradient, as in the reference
    if (want_sh) g_sh = s.sh_degree >= 0 ? at::empty_like(shs) : at::zeros_like(shs);
    if (want_rest) g_rest = at::empty_like(sh_rest);
    if (P > 0) {
      Slab scratch;
      const size_t ws_bytes = fsgs_gs_2d_render_backward_workspace_bytes(s.R);
      const size_t ws = scratch.reserve(ws_bytes);
      scratch.allocate(points);
      const bool aux = g_extras.defined();
      const float* colors = s.sh_degree < 0 ? f32(shs) : (const float*) keep(s.colors);
      const int M = has_rest && sh_rest.numel() > 0 ? (int) sh_rest.size(1) : shs.dim() == 3 ? (int) shs.size(1) : 0;
      check(fsgs_gs_2d_view_backward_hits((int) P, W, H, s.near_n, s.far_n, f32(means2D), f32(normal_opacity), colors,
                                     f32(trans_mat), f32(t2), f32(opacity), aux ? f32(extras) : nullptr,
                                     g_flow.defined() ? f32(flow) : nullptr, f32(g_image), f32(g_opacity),
                                     f32(g_extras), f32(g_flow), i64(ranges), i32(point_list), i32(n_contrib),
                                     s.R, (const int32_t*) keep(s.offsets), (const int32_t*) keep(s.regions),
                                     (const int32_t*) keep(s.tiles), i32(radii), scratch.at<void>(ws), ws_bytes,
                                     (const float*) keep(s.records), (const uint32_t*) i32(t[22]), stream),
            "GS_2D_render_backward");
      check(fsgs_gs_2d_view_preprocess_backward_derivs(
                (int) P, W, H, s.sh_degree, M, f32(points), f32(scales), f32(rotations), f32(shs),
                has_rest && sh_rest.numel() > 0 ? f32(sh_rest) : nullptr, f32(Tw2v), f32(Tv2c), f32(campos),
                f32(trans_mat), i32(radii), colors, (const int32_t*) keep(s.offsets), (const int32_t*) keep(s.regions),
                (const int32_t*) keep(s.tiles), holder->cull ? (const uint32_t*) keep(s.masks) : nullptr,
                scratch.at<const float>(ws), s.has_derivs ? (const float*) keep(s.derivs) : nullptr, f32(g_means2D), f32(g_points), f32(g_scales), f32(g_rot), f32(g_opac),
                s.sh_degree >= 0 ? f32(g_sh) : nullptr, has_rest && sh_rest.numel() > 0 ? f32(g_rest) : nullptr, stream),
            "gs_2d_preprocess_backward");
    }
    return first_order_only(upstream, {points, scales, rotations, opacities, shs, sh_rest, means2D},
                            {g_points, g_scales, g_rot, g_opac, g_sh, g_rest, g_means2D, Tensor(), Tensor()});
  }
};

}  // namespace

SurfelResult surfel_render(const SurfelView& v) {
  SurfelResult r;
  Buffers b;
  const bool train = at::GradMode::is_enabled() &&
                     (v.points.requires_grad() || v.scales.requires_grad() || v.rotations.requires_grad() ||
                      v.opacities.requires_grad() || v.shs.requires_grad() || (has(v.sh_rest) && v.sh_rest->requires_grad()) ||
                      v.means2D.requires_grad());
  if (train) {
    r.maps = SurfelRender::apply(v.points, v.scales, v.rotations, v.opacities, v.shs, v.sh_rest, v.means2D, &v, &b);
  } else {
    b      = forward_view(v, false);
    r.maps = outputs_of(b);
  }
  r.n_contrib = b.n_contrib, r.radii = b.radii, r.visible = b.visible, r.ranges = b.ranges;
  r.point_list = b.point_list, r.normal_opacity = b.normal_opacity, r.trans_mat = b.trans_mat;
  return r;
}

}  // namespace fsgs_host
