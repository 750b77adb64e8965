// Per-tile front-to-back alpha blend of 2D Gaussian surfels for gfx950.
//
// Reference behaviour reproduced: fast_2d_gs/_C/src/gaussian_splatting/gs_2d_redner.cu:28-236 (kernel) and :541-629
// (host entry GS_2D_render_forward): colour, opacity, the 9 auxiliary maps (depth, normal xyz, median depth,
// distortion, M1, M2, weight sum), optional flow, n_contrib = (last contributor, median contributor), and the optional
// accum_max_count / accum_weights_p / accum_weights_count side outputs with their quirks (the arg-max flag is never
// reset once set, :180-197). The side outputs are sums over (pixel, surfel) pairs; the kernel forms them per wavefront
// or per pixel first and issues few atomics (see ArgmaxRun and the weight staging below) instead of up to three per
// pair.
//
// Layout: one 256-lane block per 16x16 tile; wavefront w owns an 8x8 pixel quadrant, eight lanes at a time a 2x4 block of
// it with a work list of its own (block_lists.hpp). Surfels of the tile's sorted range are gathered 192 at a time (one per
// lane of the first three wavefronts, colours included so the blend never goes back to HBM) into LDS as 80-byte records; the
// next batch's gather is issued before the current batch is blended so its HBM latency overlaps the arithmetic.
// Bound by vector issue (60 instructions a step, three of them transcendental). 300k surfels 800x800: 147 us with one list
// per quadrant, 107 with lists per 4x4 block, 94 per 2x4 block; 3M 1352x1014: 506, 333, 282; 400k 3840x2160: 930, 845, 849;
// 10k 256x256: 28, 19, 18. With flow the second transforms are loaded when a batch is staged (requested ahead they hold nine
// registers) and the quotient takes a reciprocal instead of two divisions: 300k 164 -> 142 us, 2000 surfels with deviations of
// 128 pixels 592 -> 501. Batches of 64 / 128 / 192 surfels (a list's length varies less over a long batch), 2x4: 113 / 97 /
// 94 us at 300k, 346 / 297 / 282 at 3M. An entry is intersected beside the blend of the one before (walk_block_list_ahead).
#include "block_lists.hpp"
#include "view_maps.hpp"

namespace fsgs {
namespace {

constexpr int kFwdLanes = 8;    // lanes (pixels) that share a work list
constexpr int kFwdBatch = 192;  // surfels staged per round (<= block size)

// kAccum: 0 = no side outputs, 1 = accum_max_count only (what the reference's training loop passes on every step),
// 2 = accum_weights_p and / or accum_weights_count as well.
// kHits: notes which blocks blended an entry (hit_blocks), for the backward.
template <bool kAux, bool kFlow, int kAccum, bool kHits>
__global__ void __launch_bounds__(kBlendThreads) __attribute__((amdgpu_waves_per_eu(!kFlow && kAccum < 2 ? 5 : 1)))
blend_forward_kernel(
    int ordered, const int* __restrict__ tile_order, int W, int H, float near_n, float far_n, const int64_t* __restrict__ ranges, const int32_t* __restrict__ point_list,
    const float2* __restrict__ means2D, const float* __restrict__ colors, const float* __restrict__ trans_mat,
    const float4* __restrict__ normal_opacity, const float4* __restrict__ records,
    const float* __restrict__ trans_mat_t2, int32_t* __restrict__ n_contrib,
    float* __restrict__ out_color, float* __restrict__ out_opacity, float* __restrict__ out_extras,
    float2* __restrict__ out_flow, int32_t* __restrict__ accum_max_count, float* __restrict__ accum_weights_p,
    int32_t* __restrict__ accum_weights_count, uint32_t* __restrict__ hit_blocks, ViewMaps maps) {
  using Shape = BlockShape<kFwdLanes>;
  static_assert(!kHits || kFwdLanes == kHitLanes);
  __shared__ Splat s_splat[kFwdBatch + 1];  // the last one is what padding names: no pixel blends it
  __shared__ float s_t2[kFlow ? kFwdBatch * 9 : 1];
  __shared__ unsigned s_mask[kFwdBatch];  // which blocks of the tile each staged surfel can reach
  __shared__ __attribute__((aligned(16))) unsigned char s_list[Shape::kPerTile * kFwdBatch + 16];
  // accum_weights_*: the weights of the tile's pixels per staged surfel, summed over a row in registers, over the tile's
  // rows here; one global atomic per staged surfel and output
  __shared__ float s_accw[kAccum == 2 ? kFwdBatch : 1];
  __shared__ int s_accn[kAccum == 2 ? kFwdBatch : 1];
  __shared__ uint4 s_hit[kHits ? kFwdBatch : 1][2];  // which blocks blended each staged surfel, a byte per block (hit_bits)

  const int gx = (W + kTile - 1) / kTile;
  const int tile = scheduled_tile(ordered, tile_order), tile_x = tile % gx, tile_y = tile / gx;
  int px, py;
  Shape::lane_pixel(tile_x, tile_y, px, py);
  const bool inside = px < W && py < H;
  const size_t HW   = (size_t) H * W;
  const size_t pix  = (size_t) W * py + px;
  const float pxf = (float) px, pyf = (float) py;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;

  const int64_t r0 = ranges[2 * (size_t) tile], r1 = ranges[2 * (size_t) tile + 1];
  const int n_todo = (int) (r1 - r0);
  const int rounds = (n_todo + kFwdBatch - 1) / kFwdBatch;

  // The pixels still blending (their transmittance has not fallen below 1e-4), as a lane mask in scalar registers: neither
  // keeping it nor asking "is anybody left" costs vector work.
  unsigned long long live_lanes = wave_ballot(inside);
  const float far_scale = far_n / (far_n - near_n), far_near = far_scale * near_n;
  float T = 1.0f, C0 = 0, C1 = 0, C2 = 0;
  float N0 = 0, N1 = 0, N2 = 0, D = 0, M1 = 0, M2 = 0, dist = 0, median = 0, wsum = 0, f0 = 0, f1 = 0;
  int last = 0, median_c = -1;
  ArgmaxRun argmax;
  // this thread's staged surfel: its sums of the batch before go out, its places are cleared for the next
  auto flush_weights = [&]() {
    const int t = (int) threadIdx.x;
    if (t >= kFwdBatch || s_accn[t] == 0) return;
    const int id = s_splat[t].cold.id;
    if (accum_weights_p) atomicAdd(&accum_weights_p[id], s_accw[t]);
    if (accum_weights_count) atomicAdd(&accum_weights_count[id], s_accn[t]);
    s_accw[t] = 0.0f, s_accn[t] = 0;
  };
  uint32_t* const tile_hits = hit_blocks + (kHits ? r0 : 0);
  // the same for the blocks that blended it; `b` is the batch
  auto flush_hits = [&](int b) {
    const int t = (int) threadIdx.x;
    if (t >= kFwdBatch) return;
    if (b * kFwdBatch + t < n_todo) tile_hits[keep_local(b * kFwdBatch + t)] = hit_bits(s_hit[t][0], s_hit[t][1]);
    s_hit[t][0] = s_hit[t][1] = make_uint4(0u, 0u, 0u, 0u);
  };
  if (kHits && threadIdx.x < kFwdBatch) s_hit[threadIdx.x][0] = s_hit[threadIdx.x][1] = make_uint4(0u, 0u, 0u, 0u);
  unsigned char* const my_hit = (unsigned char*) &s_hit[0][0] + ((Shape::kPerWave * wave + lane / kFwdLanes) ^ 3);
  if (threadIdx.x == 0) s_splat[kFwdBatch] = Splat{};  // all zero: p_z == 0 everywhere
  if (threadIdx.x < 4) ((unsigned*) &s_list[Shape::kPerTile * kFwdBatch])[threadIdx.x] = 0u;
  if (kAccum == 2 && threadIdx.x < kFwdBatch) s_accw[threadIdx.x] = 0.0f, s_accn[threadIdx.x] = 0;

  Splat next;
  if ((int) threadIdx.x < min(n_todo, kFwdBatch))
    next = gather_splat(point_list[r0 + threadIdx.x], means2D, colors, normal_opacity, trans_mat, records);

  int b = 0;
  for (; b < rounds; ++b) {
    // everyone has finished reading the previous batch; leave as soon as no pixel of the tile is still blending
    if (__syncthreads_and(live_lanes == 0ull)) break;
    const int n_here = min(kFwdBatch, n_todo - b * kFwdBatch);
    if (kAccum == 2) flush_weights();
    if (kHits && b > 0) flush_hits(b - 1);
    if ((int) threadIdx.x < kFwdBatch) {
      unsigned mask = 0u;
      if ((int) threadIdx.x < n_here) {
        s_splat[threadIdx.x] = next;
        mask = surfel_blocks<kFwdLanes>(next.hot, keep_local(tile_x) * kTile, keep_local(tile_y) * kTile, ordered);
        if (kFlow)
#pragma unroll
          for (int k = 0; k < 9; ++k) s_t2[threadIdx.x * 9 + k] = trans_mat_t2[9 * (size_t) next.cold.id + k];
      }
      s_mask[threadIdx.x] = mask;
    }
    __syncthreads();
    const int nxt = (b + 1) * kFwdBatch + threadIdx.x;
    if ((int) threadIdx.x < kFwdBatch && nxt < n_todo)
      next = gather_splat(point_list[r0 + nxt], means2D, colors, normal_opacity, trans_mat, records);

    // One list entry per block of the wavefront. The intersection runs without early exits and yields one predicate; what the
    // pixel's sums take of the entry is one divergent region.
    unsigned char* const lists = &s_list[Shape::kPerWave * wave * kFwdBatch];
    unsigned masks[kFwdBatch / kWave];
#pragma unroll
    for (int c = 0; c < kFwdBatch / kWave; ++c) masks[c] = s_mask[c * kWave + lane];
    const int steps = build_block_lists<kFwdLanes, kFwdBatch>(lists, masks, wave, live_lanes);
    struct Eval {
      float alpha, depth, sx, sy;
      unsigned long long pass;
    };
    auto eval_entry = [&](const SplatHot& hot) {
      Hit h;
      Eval e;
      intersect_flat(hot, pxf, pyf, near_n, h, &e.pass);
      e.alpha = h.alpha, e.depth = h.depth, e.sx = h.sx, e.sy = h.sy;
      return e;
    };
    auto cold_of = [&](int j) {  // used only if a pixel blends the surfel, but then without waiting
      const SplatCold cold = s_splat[j].cold;
      __builtin_amdgcn_sched_barrier(0);
      return cold;
    };
    auto blend_entry = [&](const Eval& e, const SplatCold& cold, int j, int) {
#pragma clang fp contract(off)  // several copies of this body exist (alternating registers): they must round alike
        const unsigned long long pass = e.pass & live_lanes;
        const float test_T = T * (1.0f - e.alpha);
        const unsigned long long sat = pass & wave_ballot(test_T < 0.0001f);
        live_lanes &= ~sat;
        const unsigned long long blends = pass & ~sat;
        const float w = e.alpha * T;
        // by all lanes, beside the next entry's intersection; where a lane does not blend, nothing of it is kept (the asm keeps it here)
        float m  = fmaf(-far_near, __builtin_amdgcn_rcpf(e.depth), far_scale);
        float mm = m * m;
        float spread = fmaf(-2.0f * m, M1, fmaf(mm, 1.0f - T, M2));
        if (kAux) asm volatile("" : "+v"(m), "+v"(mm), "+v"(spread));
        if (blends == 0ull) return;
        const bool blend = __builtin_amdgcn_inverse_ballot_w64(blends);
        if (kAccum == 2) {
          const int n = (int) __popcll(blends >> (lane & -kFwdLanes) & ((1ull << kFwdLanes) - 1ull));
          const float sum = block_sum_to_last<kFwdLanes>(blend ? w : 0.0f);
          if ((lane & (kFwdLanes - 1)) == kFwdLanes - 1 && n > 0) atomicAdd(&s_accw[j], sum), atomicAdd(&s_accn[j], n);
        }
        if (blend) {
          if (kHits) my_hit[j * 32] = 1;
          const int contributor = b * kFwdBatch + j + 1;
          if (kAux) {
            dist = fmaf(spread, w, dist);
            D    = fmaf(e.depth, w, D);
            M1   = fmaf(m, w, M1);
            M2   = fmaf(mm, w, M2);
            if (T > 0.5f) median = e.depth, median_c = contributor;
            N0 = fmaf(cold.nx, w, N0), N1 = fmaf(cold.ny, w, N1), N2 = fmaf(cold.nz, w, N2);
            if (kAccum != 0) argmax_run_step(argmax, w, cold.id, accum_max_count);
            if (kFlow) {
              const float* Q = &s_t2[j * 9];
              const float u2 = fmaf(Q[0], e.sx, fmaf(Q[1], e.sy, Q[2]));
              const float v2 = fmaf(Q[3], e.sx, fmaf(Q[4], e.sy, Q[5]));
              float w2       = fmaf(Q[6], e.sx, fmaf(Q[7], e.sy, Q[8]));
              w2             = fabsf(w2) < 1e-5f ? 1e-5f : w2;
              const float rw = newton_rcp(w2);
              f0 = fmaf(fmaf(-pxf, w2, u2) * rw, w, f0);  // u2 / w2 - x: one rounding in the difference
              f1 = fmaf(fmaf(-pyf, w2, v2) * rw, w, f1);
            }
            wsum += w;
          }
          C0 = fmaf(cold.r, w, C0), C1 = fmaf(cold.g, w, C1), C2 = fmaf(cold.b, w, C2);
          T    = test_T;
          last = contributor;
        }
      };
    walk_block_list_ahead(lists + lane / kFwdLanes * kFwdBatch, steps, [&](int j) { return s_splat[j].hot; }, cold_of, eval_entry,
                          blend_entry,
                          [&]() { return live_lanes != 0ull; });
  }

  if (kAccum != 0) argmax_run_flush(argmax, accum_max_count);
  if (kAccum == 2 || kHits) __syncthreads();
  if (kAccum == 2) flush_weights();
  if (kHits && b > 0) flush_hits(b - 1);  // entries behind it are behind every pixel's last one
  if (inside) {
    const float opacity   = 1.0f - T;
    out_opacity[pix]      = opacity;
    n_contrib[pix]        = last;
    n_contrib[pix + HW]   = kAux ? median_c : 0;
    out_color[pix]        = kAux ? maps.colour(0, C0, opacity) : C0;
    out_color[pix + HW]   = kAux ? maps.colour(1, C1, opacity) : C1;
    out_color[pix + 2 * HW] = kAux ? maps.colour(2, C2, opacity) : C2;
    if (kAux) {
      if (maps.normals) maps.write(HW, pix, N0, N1, N2, D, median, dist);
      if (out_extras) {
        out_extras[pix + 0 * HW] = D;
        out_extras[pix + 1 * HW] = N0;
        out_extras[pix + 2 * HW] = N1;
        out_extras[pix + 3 * HW] = N2;
        out_extras[pix + 4 * HW] = median;
        out_extras[pix + 5 * HW] = dist;
        out_extras[pix + 6 * HW] = M1;
        out_extras[pix + 7 * HW] = M2;
        out_extras[pix + 8 * HW] = wsum;
      }
      if (kFlow) {
        const float ws = wsum == 0.0f ? 1e-7f : wsum;
        out_flow[pix]  = make_float2(f0 / ws, f1 / ws);
      }
    }
  }
}

__global__ void __launch_bounds__(256) pack_records_kernel(int P, const float2* __restrict__ means2D,
    const float* __restrict__ colors, const float4* __restrict__ normal_opacity, const float* __restrict__ trans_mat,
    const int32_t* __restrict__ radii, const int64_t* __restrict__ point_offsets, float4* __restrict__ records) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  const float* M  = trans_mat + 9 * (size_t) i;
  const float2 c  = means2D[i];
  const float4 no = normal_opacity[i];
  const float* rgb = colors + 3 * (size_t) i;
  const int radius  = radii ? radii[i] : -1;  // -1: not known, the backward then reads its radii argument
  const int offset  = point_offsets ? (i == 0 ? 0 : (int) point_offsets[i - 1]) : -1;  // -1: not known
  float4* r = records + 5 * (size_t) i;
  r[0] = make_float4(M[0], M[1], M[2], M[3]);
  r[1] = make_float4(M[4], M[5], M[6], M[7]);
  r[2] = make_float4(M[8], c.x, c.y, no.w);
  r[3] = make_float4(no.x, no.y, no.z, rgb[0]);
  r[4] = make_float4(rgb[1], rgb[2], __int_as_float(radius), __int_as_float(offset));
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API int fsgs_gs_2d_pack_records(int P, const float* means2D, const float* colors, const float* normal_opacity,
    const float* trans_mat, const int32_t* radii, const int64_t* point_offsets, float* records, void* stream) {
  FSGS_REQUIRE(P >= 0, "gs_2d_pack_records: bad size");
  if (P == 0) return kOk;
  FSGS_REQUIRE(means2D && colors && normal_opacity && trans_mat && records && ((uintptr_t) records & 15) == 0,
               "gs_2d_pack_records: null or misaligned pointer");
  hipLaunchKernelGGL(pack_records_kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P,
                     (const float2*) means2D, colors, (const float4*) normal_opacity, trans_mat, radii, point_offsets,
                     (float4*) records);
  return check_launch("gs_2d_pack_records");
}

namespace {
// hit_blocks[R], if given: per list entry the 2x4 blocks of its tile with a pixel that blended it
int render_forward(int P, int W, int H, double near_n, double far_n, int only_image,
    const float* means2D, const float* colors, const float* normal_opacity, const float* trans_mat,
    const int32_t* point_list, const int64_t* ranges, const float* trans_mat_t2, int32_t* accum_max_count,
    float* accum_weights_p, int32_t* accum_weights_count, float* out_color, float* out_opacity, float* out_extras,
    float* out_flow, int32_t* n_contrib, const float* records, uint32_t* hit_blocks, const ViewMaps& maps, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "GS_2D_render_forward: bad sizes");
  FSGS_REQUIRE(ranges && out_color && out_opacity && n_contrib, "GS_2D_render_forward: null pointer");
  FSGS_REQUIRE(P == 0 || records || (means2D && colors && normal_opacity && trans_mat),
               "GS_2D_render_forward: null surfel tensor");
  FSGS_REQUIRE(((uintptr_t) records & 15) == 0, "GS_2D_render_forward: records must be 16-byte aligned");
  FSGS_REQUIRE(only_image || out_extras || (maps.normals && maps.distortion),
               "GS_2D_render_forward: out_extras is required unless only_image");
  FSGS_REQUIRE(!maps.normals || (maps.Tw2v && maps.surf_depth), "GS_2D_render_forward: null map");
  const bool aux   = !only_image;
  const bool flow  = aux && trans_mat_t2 != nullptr;
  const int accum = !aux ? 0 : (accum_weights_p || accum_weights_count) ? 2 : accum_max_count ? 1 : 0;
  FSGS_REQUIRE(!flow || out_flow, "GS_2D_render_forward: out_flow is required with trans_mat_t2");
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const dim3 grid(gx * gy), block(kBlendThreads);
  hipStream_t s = (hipStream_t) stream;
  const int* tile_order = nullptr;
  const int ordered = launch_tile_order(gx, gy, ranges, s, &tile_order);
#define FSGS_LAUNCH_FWD(AUX, FLOW, ACC, HITS)                                                                        \
  hipLaunchKernelGGL((blend_forward_kernel<AUX, FLOW, ACC, HITS>), grid, block, 0, s, ordered, tile_order, W, H, (float) near_n, \
                     (float) far_n, ranges, point_list, (const float2*) means2D, colors, trans_mat,                  \
                     (const float4*) normal_opacity, (const float4*) records, trans_mat_t2, n_contrib, out_color, out_opacity, \
                     out_extras, (float2*) out_flow, accum_max_count, accum_weights_p, accum_weights_count, hit_blocks, maps)
#define FSGS_LAUNCH_FWD_HITS(FLOW, ACC)              \
  if (hit_blocks) FSGS_LAUNCH_FWD(true, FLOW, ACC, true); \
  else FSGS_LAUNCH_FWD(true, FLOW, ACC, false)
  if (!aux) FSGS_LAUNCH_FWD(false, false, 0, false);
  else if (flow && accum == 2) { FSGS_LAUNCH_FWD_HITS(true, 2); }
  else if (flow && accum == 1) { FSGS_LAUNCH_FWD_HITS(true, 1); }
  else if (flow) { FSGS_LAUNCH_FWD_HITS(true, 0); }
  else if (accum == 2) { FSGS_LAUNCH_FWD_HITS(false, 2); }
  else if (accum == 1) { FSGS_LAUNCH_FWD_HITS(false, 1); }
  else { FSGS_LAUNCH_FWD_HITS(false, 0); }
#undef FSGS_LAUNCH_FWD_HITS
#undef FSGS_LAUNCH_FWD
  return check_launch("GS_2D_render_forward");
}

}  // namespace

FSGS_API int fsgs_gs_2d_render_forward(int P, int W, int H, double near_n, double far_n, int only_image,
    const float* means2D, const float* colors, const float* normal_opacity, const float* trans_mat,
    const int32_t* point_list, const int64_t* ranges, const float* trans_mat_t2, int32_t* accum_max_count,
    float* accum_weights_p, int32_t* accum_weights_count, float* out_color, float* out_opacity, float* out_extras,
    float* out_flow, int32_t* n_contrib, const float* records, void* stream) {
  return render_forward(P, W, H, near_n, far_n, only_image, means2D, colors, normal_opacity, trans_mat, point_list, ranges,
                        trans_mat_t2, accum_max_count, accum_weights_p, accum_weights_count, out_color, out_opacity, out_extras,
                        out_flow, n_contrib, records, nullptr, ViewMaps{}, stream);
}

FSGS_API int fsgs_gs_2d_view_forward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* colors, const float* normal_opacity, const float* trans_mat, const int32_t* point_list,
    const int64_t* ranges, const float* trans_mat_t2, int32_t* accum_max_count, float* accum_weights_p,
    int32_t* accum_weights_count, float* out_color, float* out_opacity, float* out_extras, float* out_flow,
    int32_t* n_contrib, const float* records, uint32_t* hit_blocks, double depth_ratio, const float* Tw2v,
    const float* background, float* normals, float* depths, float* surf_depth, float* distortion, void* stream) {
  return render_forward(P, W, H, near_n, far_n, 0, means2D, colors, normal_opacity, trans_mat, point_list, ranges, trans_mat_t2,
                        accum_max_count, accum_weights_p, accum_weights_count, out_color, out_opacity, out_extras, out_flow,
                        n_contrib, records, hit_blocks,
                        ViewMaps{Tw2v, background, normals, depths, surf_depth, distortion, (float) depth_ratio}, stream);
}

FSGS_API int fsgs_debug_tile_order(int gx, int gy, const int64_t* ranges, int32_t* table, void* stream) {
  using namespace fsgs;
  FSGS_REQUIRE(gx > 0 && gy > 0 && (int64_t) gx * gy <= kMaxOrderedTiles && ranges && table,
               "debug_tile_order: bad arguments (at most %d tiles)", kMaxOrderedTiles);
  hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, (hipStream_t) stream, gx, gy, ranges, table,
                     (int*) nullptr);
  return check_launch("debug_tile_order");
}

