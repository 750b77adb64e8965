// Per-tile alpha blend of the "fast" 2D-Gaussian-surfel path for gfx950: the ray-splat intersection is three dot
// products with the adjugate of the transform (p = adj(M) (x, y, 1), s = p.xy / p.z) instead of a cross product of two
// planes, 8 auxiliary maps, optional snapshots of the running state every 32 list entries, and two backward channel
// sets.
//
// Reference behaviour reproduced: fast_2d_gs/_C/src/gaussian_splatting/gs_2d_fast_redner.cu:22-271 (forward),
// :273-561 (backward, per-pixel form), :563-837 (backward, per-splat form), :839-1074 (host entries).
// The per-splat form of the reference re-walks 32-entry buckets from the forward snapshots with one warp per bucket;
// its result is the same derivative with a different set of live channels (no distortion gradient, M1/M2 maps as
// plain weighted sums with the M1 depth term overwritten, :751-757). Here both forms run the same tile-per-block
// back-to-front kernel by default and differ only in that channel set; the per-splat decomposition itself is
// fast_bucket_backward_kernel below, which consumes the forward's snapshots (slower on this chip). Optical flow (a second set of transforms, :247-255): the forward divides the weighted sum of
// displacements by the final opacity (:259-263); both backward forms take dL/dflow as the gradient of the UNDIVIDED sum
// (:366, :704), and the per-splat form subtracts the DIVIDED final flow from its partial sums (:706), which amounts to
// an opacity-map gradient lowered by (final flow . dL/dflow) -- reproduced here in that algebraic form.
//
// Layout as in the standard blend: one 256-lane block per tile, surfels staged in LDS as 96-byte records with the adjugate, a
// work list per 2x4 (forward) or 4x4 (backward) block of pixels (block_lists.hpp).
#include "binning.hpp"
#include "block_lists.hpp"
#include "instance_slots.hpp"
#include "ordered_sums.hpp"
#include "view_maps.hpp"

namespace fsgs {
namespace {

struct __attribute__((aligned(16))) FastHot {
  float a[9];           // adjugate of the ray-splat transform
  float tw0, tw1, tw2;  // third row of the transform (depth along the ray)
  float cx, cy, opacity, pad;
};

struct FastRecord {
  FastHot hot;
  SplatCold cold;
};
struct FastSplat : FastRecord {
  float m[6];  // first two rows of the transform, only used for the footprint's bound while staging
};

__device__ __forceinline__ FastSplat gather_fast(int id, const float2* __restrict__ means2D,
                                                 const float* __restrict__ colors,
                                                 const float4* __restrict__ normal_opacity,
                                                 const float* __restrict__ trans_mat,
                                                 const float* __restrict__ inverse_m) {
  FastSplat s;
  const float* A = inverse_m + 9 * (size_t) id;
  const float* M = trans_mat + 9 * (size_t) id;
#pragma unroll
  for (int k = 0; k < 9; ++k) s.hot.a[k] = A[k];
#pragma unroll
  for (int k = 0; k < 6; ++k) s.m[k] = M[k];
  s.hot.tw0 = M[6], s.hot.tw1 = M[7], s.hot.tw2 = M[8];
  const float2 c  = means2D[id];
  const float4 no = normal_opacity[id];
  s.hot.cx = c.x, s.hot.cy = c.y, s.hot.opacity = no.w, s.hot.pad = 0.0f;
  s.cold.nx = no.x, s.cold.ny = no.y, s.cold.nz = no.z;
  s.cold.r = colors[3 * (size_t) id], s.cold.g = colors[3 * (size_t) id + 1], s.cold.b = colors[3 * (size_t) id + 2];
  s.cold.id = id, s.cold.pad = 0;
  return s;
}

template <int kLanes>
__device__ __forceinline__ unsigned fast_blocks(const FastSplat& s, int tile_px, int tile_py, int flags) {
  SplatHot h;
#pragma unroll
  for (int k = 0; k < 6; ++k) h.m[k] = s.m[k];
  h.m[6] = s.hot.tw0, h.m[7] = s.hot.tw1, h.m[8] = s.hot.tw2;
  h.cx = s.hot.cx, h.cy = s.hot.cy, h.opacity = s.hot.opacity;
  return surfel_blocks<kLanes>(h, tile_px, tile_py, flags);
}

struct FastHit {
  float pz, sx, sy, dx, dy, rho3d, rho2d, depth, G, alpha;
};

// gs_2d_fast_redner.cu:150-186. Returns false when the reference would `continue`.
// Written without early exits: every lane runs the whole sequence and the rejections (behind the camera plane, nearer
// than `near`, positive exponent, alpha < 1/255) are combined into one predicate at the end, so the callers have one
// divergent region instead of a nest of them on their per-entry critical path.
// `lanes`, if given: mask of the lanes that pass, from the four comparisons' own lane masks (scalar registers).
__device__ __forceinline__ bool fast_intersect_flat(const FastHot& h, float pxf, float pyf, float near_n, FastHit& o,
                                                    unsigned long long* lanes = nullptr) {
  // Every fused multiply-add is written out and contraction is off: the kernels inline this more than once (two copies
  // of a loop body that alternate their registers), and which copy evaluates an entry depends on the work list, so the
  // copies must round alike. Exponent in base 2 (one v_exp_f32, the factor folded into the scale of rho); the
  // reference's `power > 0` rejection cannot fire for a sum of squares and is not evaluated.
#pragma clang fp contract(off)
  const float p0 = fmaf(h.a[0], pxf, fmaf(h.a[1], pyf, h.a[2]));
  const float p1 = fmaf(h.a[3], pxf, fmaf(h.a[4], pyf, h.a[5]));
  o.pz           = fmaf(h.a[6], pxf, fmaf(h.a[7], pyf, h.a[8]));
  const float rz = __builtin_amdgcn_rcpf(o.pz);
  o.sx = p0 * rz, o.sy = p1 * rz;
  o.rho3d = fmaf(o.sx, o.sx, o.sy * o.sy);
  o.dx = h.cx - pxf, o.dy = h.cy - pyf;
  const float d2 = fmaf(o.dx, o.dx, o.dy * o.dy);
  o.rho2d = 2.0f * d2;
  o.depth = fmaf(o.sx, h.tw0, fmaf(o.sy, h.tw1, h.tw2));
  const float power2 = fmaxf(o.rho3d * -0.72134752044448170368f, d2 * -1.44269504088896340736f);
  o.G     = __builtin_amdgcn_exp2f(power2);
  o.alpha = fminf(0.99f, h.opacity * o.G);
  const bool c0 = o.pz != 0.0f, c1 = !(o.depth < near_n), c3 = !(o.alpha < (1.0f / 255.0f));
  if (lanes) *lanes = wave_ballot(c0) & wave_ballot(c1) & wave_ballot(c3);
  return c0 & c1 & c3;
}

// Five per-lane values summed over each 16-lane row, as row_sum16_transposed does: a lane with bit 1 returns the row's total of
// v[4], another that of v[(l >> 2 & 1) * 2 + (l >> 3)]. 12 instructions.
__device__ __forceinline__ float row_sum5_transposed(const float (&v)[5]) {
#pragma clang fp contract(off)  // an input that is a product must not be formed a second time inside a fused add
  const int lane = __lane_id();
  float w0 = v[0] + dpp_shift_zero<0x128, 0xf, 0xf>(v[0]), w1 = v[2] + dpp_shift_zero<0x128, 0xf, 0xf>(v[2]);  // row_ror:8
  float w2 = v[4] + dpp_shift_zero<0x128, 0xf, 0xf>(v[4]);
  asm volatile("s_nop 1\n\t"
               "v_add_f32_dpp %0, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
               "v_add_f32_dpp %1, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
               "s_nop 1"
               : "+v"(w0), "+v"(w1)
               : "v"(v[1]), "v"(v[3]));
  float x = w0 + dpp_shift_zero<0x104, 0xf, 0xf>(w0);              // row_shl:4
  const float y = w2 + dpp_shift_zero<0x124, 0xf, 0xf>(w2);        // row_ror:4, of halves that are alike
  asm volatile("s_nop 1\n\t"
               "v_add_f32_dpp %0, %1, %1 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
               "s_nop 1"
               : "+v"(x)
               : "v"(w1));
  const float a = y + dpp_shift_zero<0x112, 0xf, 0xf>(y);  // row_shr:2, kept by lanes with bit 1
  const float b = x + dpp_shift_zero<0x102, 0xf, 0xf>(x);  // row_shl:2
  const float z = (lane & 2) ? a : b;
  return z + dpp_shift_zero<0xb1, 0xf, 0xf>(z);  // quad_perm [1,0,3,2]
}

// Bound by vector issue. 150k surfels 1001x667: 62 -> 57 us with lists per 2x4 block instead of 8x8 quadrant,
// noting the blocks (batches of 192 surfels instead of 128: 58; held to five wavefronts per SIMD, which spills: 62).
// With flow or weights held to four, with flow as in the other forward (transforms loaded at the staging, a reciprocal): 300k
// 800x800 88 -> 75 us, with snapshots 129 -> 94; 2000 surfels with deviations of 128 pixels 530 -> 436 and 555 -> 436.
// kHits: notes which blocks blended an entry (hit_blocks), for the backward.
template <bool kAux, bool kSnap, bool kAccum, bool kFlow, bool kHits>
__global__ void __launch_bounds__(kBlendThreads) __attribute__((amdgpu_waves_per_eu(kFlow || kAccum ? 4 : 1)))
fast_blend_forward_kernel(
    int ordered, const int* __restrict__ tile_order, int W, int H, float near_n, float far_n, const int64_t* __restrict__ ranges, const int32_t* __restrict__ point_list,
    const float2* __restrict__ means2D, const float* __restrict__ colors, const float* __restrict__ trans_mat,
    const float* __restrict__ inverse_m, const float4* __restrict__ normal_opacity,
    const float* __restrict__ trans_mat_t2, const int64_t* __restrict__ bucket_offset, int32_t* __restrict__ n_contrib,
    float* __restrict__ out_color, float* __restrict__ out_opacity, float* __restrict__ out_extras,
    float2* __restrict__ out_flow, int32_t* __restrict__ max_contrib,
    int32_t* __restrict__ bucket_to_tile, float* __restrict__ sampled_T, float* __restrict__ sampled_acc,
    float* __restrict__ sampled_aux, int32_t* __restrict__ accum_max_count, float* __restrict__ accum_weights_p,
    int32_t* __restrict__ accum_weights_count, uint32_t* __restrict__ hit_blocks, ViewMaps maps) {
  // With snapshots the lists end at the buckets of 32 entries, two of which are staged at a time.
  constexpr int kLanes = 8, kB = kSnap ? 64 : 128;
  using Shape = BlockShape<kLanes>;
  static_assert(!kHits || kLanes == kHitLanes);
  __shared__ FastRecord s_splat[kB + 1];      // the last one is what padding names: no pixel blends it
  __shared__ float s_t2[kFlow ? kB * 9 : 1];  // second-time-step transforms of the staged surfels
  __shared__ unsigned s_mask[kB];             // which blocks of the tile each staged surfel can reach
  __shared__ __attribute__((aligned(16))) unsigned char s_list[Shape::kPerTile * kB + 16];
  __shared__ float s_accw[kAccum ? kB : 1];  // accum_weights_*: sums over the tile per staged surfel
  __shared__ int s_accn[kAccum ? kB : 1];
  __shared__ uint4 s_hit[kHits ? kB : 1][2];  // which blocks blended each staged surfel, a byte per block (hit_bits)
  __shared__ int s_max_contrib;
  constexpr int kNum = kFlow ? 10 : 8;  // channels of a snapshot

  const int gx = (W + kTile - 1) / kTile;
  const int tile = scheduled_tile(ordered, tile_order), tile_x = tile % gx, tile_y = tile / gx;
  int px, py;
  Shape::lane_pixel(tile_x, tile_y, px, py);
  const bool inside = px < W && py < H;
  const size_t HW   = (size_t) H * W;
  const size_t pix  = (size_t) W * py + px;
  const float pxf = (float) px, pyf = (float) py;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rank = (py - tile_y * kTile) * kTile + (px - tile_x * kTile);  // row-major position inside the tile

  const int64_t r0 = ranges[2 * (size_t) tile], r1 = ranges[2 * (size_t) tile + 1];
  const int n_todo = (int) (r1 - r0);
  const int rounds = (n_todo + kB - 1) / kB;

  int64_t bucket0 = 0;
  if (kSnap) {
    bucket0 = tile == 0 ? 0 : bucket_offset[tile - 1];
    const int nb = (n_todo + 31) / 32;
    for (int k = threadIdx.x; k < nb; k += kBlendThreads) bucket_to_tile[bucket0 + k] = tile;
    if (threadIdx.x == 0) s_max_contrib = 0;
  }

  // the pixels still blending, as a lane mask in scalar registers
  unsigned long long live_lanes = wave_ballot(inside);
  const float far_scale = far_n / (far_n - near_n);
  float T = 1.0f, C0 = 0, C1 = 0, C2 = 0;
  float N0 = 0, N1 = 0, N2 = 0, D = 0, M1 = 0, M2 = 0, dist = 0, median = 0, f0 = 0, f1 = 0;
  int last = 0, median_c = -1;
  ArgmaxRun argmax;

  const bool weights = kAccum && (accum_weights_p || accum_weights_count);
  uint32_t* const tile_hits = hit_blocks + (kHits ? r0 : 0);
  // this thread's staged surfel: its sums of the batch before go out, its places are cleared for the next
  auto flush = [&](int b) {
    const int t = (int) threadIdx.x;
    if (t >= kB) return;
    if (weights && s_accn[t] != 0) {
      const int id = s_splat[t].cold.id;
      if (accum_weights_p) atomicAdd(&accum_weights_p[id], s_accw[t]);
      if (accum_weights_count) atomicAdd(&accum_weights_count[id], s_accn[t]);
      s_accw[t] = 0.0f, s_accn[t] = 0;
    }
    if (kHits) {
      if (b * kB + t < n_todo) tile_hits[keep_local(b * kB + t)] = hit_bits(s_hit[t][0], s_hit[t][1]);
      s_hit[t][0] = s_hit[t][1] = make_uint4(0u, 0u, 0u, 0u);
    }
  };
  if (threadIdx.x == 0) s_splat[kB] = FastRecord{};  // all zero: p_z == 0 everywhere
  if (threadIdx.x < 4) ((unsigned*) &s_list[Shape::kPerTile * kB])[threadIdx.x] = 0u;
  if (kAccum && threadIdx.x < kB) s_accw[threadIdx.x] = 0.0f, s_accn[threadIdx.x] = 0;
  if (kHits && threadIdx.x < kB) s_hit[threadIdx.x][0] = s_hit[threadIdx.x][1] = make_uint4(0u, 0u, 0u, 0u);
  unsigned char* const my_hit = (unsigned char*) &s_hit[0][0] + ((Shape::kPerWave * wave + lane / kLanes) ^ 3);
  unsigned char* const lists  = &s_list[Shape::kPerWave * wave * kB];

  FastSplat next;
  auto gather = [&](int at) {
    if ((int) threadIdx.x >= kB || at >= n_todo) return;
    const int id = point_list[r0 + at];
    next = gather_fast(id, means2D, colors, normal_opacity, trans_mat, inverse_m);
  };
  gather((int) threadIdx.x);

  int b = 0;
  for (; b < rounds; ++b) {
    if (__syncthreads_and(live_lanes == 0ull)) break;
    const int n_here = min(kB, n_todo - b * kB);
    if ((kAccum || kHits) && b > 0) flush(b - 1);
    if ((int) threadIdx.x < kB) {
      unsigned mask = 0u;
      if ((int) threadIdx.x < n_here) {
        s_splat[threadIdx.x] = next;
        mask = fast_blocks<kLanes>(next, keep_local(tile_x) * kTile, keep_local(tile_y) * kTile, ordered);
        if (kFlow) {
#pragma unroll
          for (int k = 0; k < 9; ++k) s_t2[threadIdx.x * 9 + k] = trans_mat_t2[9 * (size_t) next.cold.id + k];
        }
      }
      s_mask[threadIdx.x] = mask;
    }
    __syncthreads();
    gather((b + 1) * kB + (int) threadIdx.x);

    auto blend_entry = [&](const FastHot& hot, int j, int) {
#pragma clang fp contract(off)  // several copies of this body exist (alternating registers): they must round alike
      const SplatCold cold = s_splat[j].cold;  // used only if a pixel blends the surfel, but then without waiting
      __builtin_amdgcn_sched_barrier(0);
      FastHit h;
      unsigned long long pass;
      fast_intersect_flat(hot, pxf, pyf, near_n, h, &pass);
      pass &= live_lanes;
      if (pass == 0ull) return;
      const float test_T = T * (1.0f - h.alpha);
      const unsigned long long sat = pass & wave_ballot(test_T < 0.0001f);
      live_lanes &= ~sat;
      const unsigned long long blends = pass & ~sat;
      const bool blend = __builtin_amdgcn_inverse_ballot_w64(blends);
      const float w    = h.alpha * T;
      if (weights) {
        const int n = (int) __popcll(blends >> (lane & -kLanes) & ((1ull << kLanes) - 1ull));
        const float sum = block_sum_to_last<kLanes>(blend ? w : 0.0f);
        if ((lane & (kLanes - 1)) == kLanes - 1 && n > 0) atomicAdd(&s_accw[j], sum), atomicAdd(&s_accn[j], n);
      }
      if (blend) {
        if (kHits) my_hit[j * 32] = 1;
        const int contributor = b * kB + j + 1;
        if (kAux) {
          const float A = 1.0f - T;
          const float m = far_scale * (1.0f - near_n * __builtin_amdgcn_rcpf(h.depth));
          const float mm = m * m;
          dist = fmaf(fmaf(mm, A, fmaf(-2.0f * m, M1, M2)), w, dist);
          D    = fmaf(h.depth, w, D);
          M1   = fmaf(m, w, M1);
          M2   = fmaf(mm, w, M2);
          if (T > 0.5f) median = h.depth, median_c = contributor;
          N0 = fmaf(cold.nx, w, N0), N1 = fmaf(cold.ny, w, N1), N2 = fmaf(cold.nz, w, N2);
          if (kAccum) argmax_run_step(argmax, w, cold.id, accum_max_count);
          if (kFlow) {
            const float* Q = &s_t2[j * 9];
            const float u2 = fmaf(Q[0], h.sx, fmaf(Q[1], h.sy, Q[2]));
            const float v2 = fmaf(Q[3], h.sx, fmaf(Q[4], h.sy, Q[5]));
            float w2       = fmaf(Q[6], h.sx, fmaf(Q[7], h.sy, Q[8]));
            w2             = fabsf(w2) < 1e-5f ? 1e-5f : w2;
            const float rw = newton_rcp(w2);
            f0 = fmaf(fmaf(-pxf, w2, u2) * rw, w, f0);  // u2 / w2 - x: one rounding in the difference
            f1 = fmaf(fmaf(-pyf, w2, v2) * rw, w, f1);
          }
        }
        C0 = fmaf(cold.r, w, C0), C1 = fmaf(cold.g, w, C1), C2 = fmaf(cold.b, w, C2);
        T    = test_T;
        last = contributor;
      }
    };
    unsigned masks[kB / kWave];
    auto walk = [&]() {
      const int steps = build_block_lists<kLanes, kB>(lists, masks, wave, live_lanes);
      walk_block_list(lists + lane / kLanes * kB, steps, [&](int j) { return s_splat[j].hot; }, blend_entry,
                      [&]() { return live_lanes != 0ull; });
    };
    if (kSnap) {
      for (int half = 0; half < 2 && half * 32 < n_here; ++half) {
        if (__builtin_amdgcn_inverse_ballot_w64(live_lanes)) {
          // state before a list entry that starts a bucket of 32 (gs_2d_fast_redner.cu:126-147)
          const size_t bk = (size_t) (bucket0 + (b * kB + half * 32) / 32);
          sampled_T[bk * 256 + rank]             = T;
          sampled_acc[(bk * 3 + 0) * 256 + rank] = C0;
          sampled_acc[(bk * 3 + 1) * 256 + rank] = C1;
          sampled_acc[(bk * 3 + 2) * 256 + rank] = C2;
          if (kAux) {
            sampled_aux[(bk * kNum + 0) * 256 + rank] = D;
            sampled_aux[(bk * kNum + 1) * 256 + rank] = N0;
            sampled_aux[(bk * kNum + 2) * 256 + rank] = N1;
            sampled_aux[(bk * kNum + 3) * 256 + rank] = N2;
            sampled_aux[(bk * kNum + 5) * 256 + rank] = dist;
            sampled_aux[(bk * kNum + 6) * 256 + rank] = M1;
            sampled_aux[(bk * kNum + 7) * 256 + rank] = M2;
            if (kFlow) {
              sampled_aux[(bk * kNum + 8) * 256 + rank] = f0;
              sampled_aux[(bk * kNum + 9) * 256 + rank] = f1;
            }
          }
        }
        masks[0] = lane >> 5 == half ? s_mask[lane] : 0u;
        walk();
      }
    } else {
#pragma unroll
      for (int c = 0; c < kB / kWave; ++c) masks[c] = s_mask[c * kWave + lane];
      walk();
    }
  }

  if (kAccum || kHits) {
    __syncthreads();
    if (b > 0) flush(b - 1);  // entries behind it are behind every pixel's last one
  }
  if (kAccum) argmax_run_flush(argmax, accum_max_count);
  if (inside) {
    out_opacity[pix]        = 1.0f - T;
    n_contrib[pix]          = last;
    n_contrib[pix + HW]     = kAux ? median_c : 0;
    out_color[pix]          = C0;
    out_color[pix + HW]     = C1;
    out_color[pix + 2 * HW] = C2;
    if (kAux) {
      if (!kSnap && maps.normals) maps.write(HW, pix, N0, N1, N2, D, median, dist);
      if (kSnap || out_extras) {
        out_extras[pix + 0 * HW] = D;
        out_extras[pix + 1 * HW] = N0;
        out_extras[pix + 2 * HW] = N1;
        out_extras[pix + 3 * HW] = N2;
        out_extras[pix + 4 * HW] = median;
        out_extras[pix + 5 * HW] = dist;
        out_extras[pix + 6 * HW] = M1;
        out_extras[pix + 7 * HW] = M2;
      }
      if (kFlow) {
        const float A = 1.0f - T;
        out_flow[pix] = A > 0.0f ? make_float2(f0 / A, f1 / A) : make_float2(0.0f, 0.0f);
      }
    }
  }
  if (kSnap) {
    int wave_max = last;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) wave_max = max(wave_max, __shfl_xor(wave_max, d, kWave));
    __syncthreads();  // s_max_contrib was cleared before the first barrier of the loop only if the loop ran
    if (lane == 0) atomicMax(&s_max_contrib, wave_max);
    __syncthreads();
    if (threadIdx.x == 0) max_contrib[tile] = s_max_contrib;
  }
}

// Per-surfel gradient slots: 0-2 colours | 3-11 adjugate | 12-14 normal | 15 opacity | 16-18 transform row 2 |
// 19-20 means2D.
constexpr int kFastGradSlots  = 21;
constexpr int kFastRecordSlots = 22;  // a record of the ordered-sum path: the 21 slots + one float of padding

// Where the sums of a surfel go: 0-2 colours | 3-11 inverse transform | 12-15 normal, opacity |
// 16-18 third row of the transform (the other two rows get no gradient from the blend: zeros) | 19-20 means2D.
struct FastScatter {
  float *g_means2D, *g_normal_opacity, *g_colors, *g_trans, *g_inv;
  // Rows of n surfels from i0 on, by a wavefront: consecutive lanes write consecutive addresses.
  template <int kSurfels, int kStride>
  __device__ __forceinline__ void rows(const float* __restrict__ s_sums, int i0, int n) const {
    auto table = [&](auto width, float* g, auto value) {
      constexpr int kWidth = decltype(width)::value;
#pragma unroll
      for (int t0 = 0; t0 < kSurfels * kWidth; t0 += kWave) {
        const int t = t0 + (int) __lane_id(), r = t / kWidth, c = t - r * kWidth;
        if (t < n * kWidth) g[(size_t) kWidth * i0 + t] = value(s_sums + r * kStride, c);
      }
    };
    table(std::integral_constant<int, 3>(), g_colors, [](const float* s, int c) { return s[c]; });
    table(std::integral_constant<int, 9>(), g_inv, [](const float* s, int c) { return s[3 + c]; });
    table(std::integral_constant<int, 4>(), g_normal_opacity, [](const float* s, int c) { return s[12 + c]; });
    table(std::integral_constant<int, 9>(), g_trans, [](const float* s, int c) { return c < 6 ? 0.0f : s[10 + c]; });
    table(std::integral_constant<int, 2>(), g_means2D, [](const float* s, int c) { return s[19 + c]; });
  }
};

// Sum of a surfel's records on the fast path. Its key span holds one position per tile of its rectangle, x-major, but
// only the tiles that pass the binning's corner test are in a tile list, and only those positions were written by the
// blend (a list entry's record by the flush of its batch, or zeros by its tile's block if the entry lies behind the
// deepest contributor). The test is repeated here, with the binning's own arithmetic, so the other positions are
// neither cleared nor read. `keep_masks` (optional, what the preprocess kernel left): the verdicts for rectangles of at most
// 32 tiles, bit = position in the span.
// A wavefront takes 20 surfels. Spans of up to 32 positions: 11 lanes of a surfel read a record's 88 bytes, five surfels beside each
// other and four such groups together, four written positions of each surfel in flight. Longer ones by the whole wavefront, 64
// positions tested and their records requested while the last ones are added from LDS, a component per lane. (With five surfels a
// wavefront, and 11 positions of every span a step, nearly all of the launch was a row of trips to memory, and as many steps as the
// largest surfel asked for; each component was stored on its own.) 150k surfels 1001x667 24 -> 16.7 us, 300k 1000x700 44 -> 32,
// 30k 1000x1000 12.3 -> 8.2, 10k 256x256 4.3 -> 4.5.
constexpr int kFastSumSurfels = 20;

__global__ void __launch_bounds__(256) fast_slot_sum_kernel(int P, int gx, int gy,
    const SlotSource slots, const int32_t* __restrict__ radii, const float2* __restrict__ means2D,
    const float* __restrict__ inverse_m, const float4* __restrict__ normal_opacity,
    const uint32_t* __restrict__ keep_masks, const float* __restrict__ records, FastScatter out) {
  constexpr int kLanes = kFastRecordSlots / 2, kPerPass = 64 / kLanes, kGroups = 4, kDepth = 4;
  static_assert(kFastSumSurfels == kPerPass * kGroups);
  __shared__ float2 s_records[4][kWave * kLanes];
  __shared__ int s_positions[4][kWave];
  __shared__ float2 s_sums[4][kFastSumSurfels * kLanes];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane / kLanes, k = lane - sub * kLanes;
  const int i0 = ((int) blockIdx.x * 4 + wave) * kFastSumSurfels, i = i0 + lane;
  const float2* const src = (const float2*) records;
  // lanes 0 to 19: a surfel's span and what was written of it
  int count = 0, h = 1, x0 = 0, y0 = 0, first = 0;
  uint32_t bits = 0u;
  const int radius = lane < kFastSumSurfels && i < P ? radii[i] : 0;
  if (radius > 0) {
    const float2 c = means2D[i];
    if (keep_masks) bits = keep_masks[i];
    first = (int) slot_first(slots, i);  // the number of instances is below 2^31
    const TileRect r = tile_rect(c.x, c.y, radius, gx, gy);
    h = max(r.y1 - r.y0, 1), count = max(r.x1 - r.x0, 0) * max(r.y1 - r.y0, 0), x0 = r.x0, y0 = r.y0;
  }
  auto corner_test = [&](int id) {
    float IM[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) IM[q] = inverse_m[9 * (size_t) id + q];
    return CornerTest(IM, normal_opacity[id].w);
  };
  const bool large = count > 32;
  if (large) bits = 0u;
  else if (keep_masks) bits &= count == 32 ? 0xffffffffu : (1u << count) - 1u;
  else if (count > 0) {
    const CornerTest ct = corner_test(i);
    for (int p = 0; p < count; ++p) {
      const int x = p / h;
      if (ct.tile(x0 + x, y0 + (p - x * h))) bits |= 1u << p;
    }
  }
  {
    uint32_t left[kGroups];
    int at[kGroups];
    float2 acc[kGroups];
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
      const int holds = min(q * kPerPass + sub, kFastSumSurfels - 1);
      left[q] = (uint32_t) __shfl((int) bits, holds, kWave), at[q] = __shfl(first, holds, kWave);
      if (sub >= kPerPass) left[q] = 0u;
      acc[q] = make_float2(0.0f, 0.0f);
    }
    while (wave_ballot((left[0] | left[1] | left[2] | left[3]) != 0u) != 0ull) {
      float2 v[kGroups][kDepth];
#pragma unroll
      for (int q = 0; q < kGroups; ++q)
#pragma unroll
        for (int j = 0; j < kDepth; ++j) {
          v[q][j] = make_float2(0.0f, 0.0f);
          if (left[q]) v[q][j] = src[(size_t) (at[q] + __builtin_ctz(left[q])) * kLanes + k];
          left[q] &= left[q] - 1u;
        }
#pragma unroll
      for (int q = 0; q < kGroups; ++q)
#pragma unroll
        for (int j = 0; j < kDepth; ++j) acc[q].x += v[q][j].x, acc[q].y += v[q][j].y;
    }
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
      const int holds = q * kPerPass + sub;
      if (sub < kPerPass) s_sums[wave][holds * kLanes + k] = acc[q];
    }
  }
  wave_lds_sync();
  for (unsigned long long todo = wave_ballot(large); todo != 0ull; todo &= todo - 1ull) {
    const int holds = (int) __builtin_ctzll(todo), id = i0 + holds;
    const int s_first = __builtin_amdgcn_readlane(first, holds), s_count = __builtin_amdgcn_readlane(count, holds);
    const int s_h = __builtin_amdgcn_readlane(h, holds), s_x0 = __builtin_amdgcn_readlane(x0, holds), s_y0 = __builtin_amdgcn_readlane(y0, holds);
    const CornerTest ct = corner_test(id);
    float2 v[kLanes];
    auto fetch = [&](int base) {  // how many of the 64 positions from `base` on were written
      const int p = base + lane, x = p / s_h;
      const bool on = p < s_count && ct.tile(s_x0 + x, s_y0 + (p - x * s_h));
      const unsigned long long who = wave_ballot(on);
      const int n = (int) __popcll(who);
      wave_lds_sync();
      if (on) s_positions[wave][__builtin_amdgcn_mbcnt_hi((unsigned) (who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned) who, 0))] = p;
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < kLanes; ++j) {
        const int t = j * kWave + lane, r = t / kLanes;
        v[j] = make_float2(0.0f, 0.0f);
        if (r < n) v[j] = src[(size_t) (s_first + s_positions[wave][r]) * kLanes + (t - r * kLanes)];
      }
      return n;
    };
    float acc = 0.0f;
    int n = fetch(0);
    for (int base = 0; base < s_count; base += kWave) {
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < kLanes; ++j) s_records[wave][j * kWave + lane] = v[j];
      wave_lds_sync();
      const int here = n;
      if (base + kWave < s_count) n = fetch(base + kWave);
      if (lane < kFastRecordSlots) {
        const float* f = (const float*) s_records[wave] + lane;
#pragma unroll 4
        for (int r = 0; r < here; ++r) acc += f[r * kFastRecordSlots];
      }
    }
    if (lane < kFastRecordSlots) ((float*) s_sums[wave])[holds * kFastRecordSlots + lane] = acc;
  }
  wave_lds_sync();
  out.rows<kFastSumSurfels, kFastRecordSlots>((const float*) s_sums[wave], i0, min(kFastSumSurfels, P - i0));
}

// Bound by vector issue and, like every launch here, by its longest tile; four blocks per compute unit. 150k surfels 1001x667:
// 165 -> 132 us with a row of lanes per 4x4 block, over the blocks that the forward noted, instead of a wavefront per 8x8 quadrant
// that queued its blended pairs; 130 with several batches per staging.
// kSlots: the per-surfel sums go through per-instance records (ordered_sums.hpp) instead of device-scope atomics.
template <bool kAux, bool kPerSplat, bool kFlow, bool kSlots>
__global__ void __launch_bounds__(kBlendThreads)
    __attribute__((amdgpu_waves_per_eu(kSlots && !kFlow ? 4 : 1, kSlots && !kFlow ? 4 : 8))) fast_blend_backward_kernel(
    int ordered, const int* __restrict__ tile_order, int W, int H, float near_n, float far_n, const int64_t* __restrict__ ranges, const int32_t* __restrict__ point_list,
    const int32_t* __restrict__ n_contrib, const float2* __restrict__ means2D,
    const float4* __restrict__ normal_opacity, const float* __restrict__ colors, const float* __restrict__ trans_mat,
    const float* __restrict__ inverse_m, const float* __restrict__ trans_mat_t2, const float* __restrict__ out_opacity,
    const float* __restrict__ out_extras, const float2* __restrict__ out_flow,
    const float* __restrict__ dL_dpix, const float* __restrict__ dL_dextras, const float* __restrict__ dL_dopacity,
    const float2* __restrict__ dL_dflow,
    float* __restrict__ g_means2D, float* __restrict__ g_normal_opacity, float* __restrict__ g_colors,
    float* __restrict__ g_trans, float* __restrict__ g_inv, const SlotSource slots,
    const int32_t* __restrict__ radii, float* __restrict__ slot_records, const uint32_t* __restrict__ hit_blocks) {
  constexpr int kB = kRowBatch, kRowPlaces = 224;  // 40 KB of LDS with records' stride
  using Shape = BlockShape<16>;
  __shared__ FastRecord s_splat[kB + 1];  // the last one is what padding names: no pixel blends it
  __shared__ float s_t2[kFlow ? kB * 9 : 1];
  __shared__ __attribute__((aligned(16))) unsigned char s_list[16 * kB + 16];
  __shared__ float s_sum[kRowPlaces + 1][kFastGradSlots];
  // What the flush of a batch reads is kept twice, by batch parity: the next batch is staged while others still flush.
  __shared__ uint4 s_place[2][kB];  // where each of the 16 rows stores its sums of each staged surfel
  __shared__ int s_slot[2][kB];     // where they go from there: the instance's record (kSlots) or the surfel's number
  __shared__ unsigned s_mask[kB];   // which 4x4 blocks of the tile it can reach
  __shared__ int s_max_contrib;

  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const int tile = scheduled_tile(ordered, tile_order), tile_x = tile % gx, tile_y = tile / gx;
  int px, py;
  Shape::lane_pixel(tile_x, tile_y, px, py);
  const bool inside = px < W && py < H;
  const size_t HW   = (size_t) H * W;
  const size_t pix  = (size_t) W * py + px;
  const float pxf = (float) px, pyf = (float) py;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;

  const int64_t r0 = ranges[2 * (size_t) tile], r1 = ranges[2 * (size_t) tile + 1];
  const int last_contrib   = inside ? n_contrib[pix] : 0;
  const int median_contrib = (kAux && inside) ? n_contrib[pix + HW] : 0;

  if (threadIdx.x == 0) s_max_contrib = 0;
  __syncthreads();
  int row_max = last_contrib;  // deepest position blended in this lane's 4x4 block
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) row_max = max(row_max, __shfl_xor(row_max, d, kWave));
  int row_last[4];  // the same of the wavefront's four blocks
#pragma unroll
  for (int r = 0; r < 4; ++r) row_last[r] = __builtin_amdgcn_readlane(row_max, 16 * r);
  if (lane == 0) atomicMax(&s_max_contrib, max(max(row_last[0], row_last[1]), max(row_last[2], row_last[3])));
  if (threadIdx.x == 0) s_splat[kB] = FastRecord{};  // all zero: p_z == 0 everywhere
  if (threadIdx.x < kFastGradSlots) s_sum[kRowPlaces][threadIdx.x] = 0.0f;
  if (threadIdx.x < 4) ((unsigned*) &s_list[16 * kB])[threadIdx.x] = 0u;
  __syncthreads();
  const int n_todo = __builtin_amdgcn_readfirstlane(min(s_max_contrib, (int) (r1 - r0)));
  // No zero fill of the record buffer: every staged instance writes its record at the flush, zeros included, and the
  // instances behind the tile's deepest contributor, which are never staged, are cleared here.
  if (kSlots) {
    for (int e = n_todo + (int) threadIdx.x; e < (int) (r1 - r0); e += kBlendThreads) {
      const int id = point_list[r0 + e];
      const float2 c = means2D[id];
      const TileRect r = tile_rect(c.x, c.y, radii[id], gx, gy);
      const int64_t at = slot_first(slots, id) + (int64_t) (tile_x - r.x0) * (r.y1 - r.y0) + (tile_y - r.y0);
      float2* dst = (float2*) (slot_records + (size_t) at * kFastRecordSlots);
#pragma unroll
      for (int c2 = 0; c2 < kFastRecordSlots / 2; ++c2) dst[c2] = make_float2(0.0f, 0.0f);
    }
  }

  const float T_final = inside ? 1.0f - out_opacity[pix] : 0.0f;
  float T = T_final;
  float dLp0 = 0, dLp1 = 0, dLp2 = 0;
  float dL_dreg = 0, dL_ddepth = 0, dL_daccum = 0, dLn0 = 0, dLn1 = 0, dLn2 = 0, dL_dmedian = 0, dL_dM1 = 0, dL_dM2 = 0;
  float final_D = 0, final_D2 = 0, dLf0 = 0, dLf1 = 0;
  if (inside) {
    dLp0 = dL_dpix[pix], dLp1 = dL_dpix[pix + HW], dLp2 = dL_dpix[pix + 2 * HW];
    if (kAux) {
      dL_daccum  = dL_dopacity ? dL_dopacity[pix] : 0.0f;
      dL_ddepth  = dL_dextras[pix + 0 * HW];
      dLn0       = dL_dextras[pix + 1 * HW];
      dLn1       = dL_dextras[pix + 2 * HW];
      dLn2       = dL_dextras[pix + 3 * HW];
      dL_dmedian = dL_dextras[pix + 4 * HW];
      if (kPerSplat) dL_dM1 = dL_dextras[pix + 6 * HW], dL_dM2 = dL_dextras[pix + 7 * HW];
      else dL_dreg = dL_dextras[pix + 5 * HW];
      final_D  = out_extras[pix + 6 * HW];
      final_D2 = out_extras[pix + 7 * HW];
    } else if (kPerSplat) {
      dL_daccum = dL_dopacity ? dL_dopacity[pix] : 0.0f;
    }
    if (kFlow) {
      const float2 gf = dL_dflow[pix];
      dLf0 = gf.x, dLf1 = gf.y;
      if (kPerSplat) {
        // partial sum - DIVIDED final flow  ==  -(sum over later entries) - final flow * T_final: the second part acts
        // like the opacity map's gradient (both carry T_final / (1 - alpha) per entry)
        const float2 ff = out_flow[pix];
        dL_daccum -= ff.x * gf.x + ff.y * gf.y;
      }
    }
  }
  const float far_scale = far_n / (far_n - near_n), far_near = far_scale * near_n;
  // the distortion term's per-pixel constants, folded once: with m the normalised depth of a pair,
  //   dL/dweight = (D2 + m^2 A - 2 m D) dL/dreg = reg_D2 + m (m reg_A - reg_2D),  dL/dm = w (m reg_2A - reg_2D)
  const float reg_A = (1.0f - T_final) * dL_dreg, reg_2A = 2.0f * reg_A, reg_2D = 2.0f * final_D * dL_dreg,
              reg_D2 = final_D2 * dL_dreg;

  float acc_lin = 0;  // what the pairs behind the current one accumulated: alpha_j c_j weighted by the transmittance between

  FastSplat next;
  unsigned next_hits = 0u;
  int next_radius = 0;
  int64_t next_off = 0;
  // entry e of the 128 staged behind `done` entries, counted from the back of the list
  auto gather = [&](int done) {
    const int e = (int) threadIdx.x;
    if (e >= min(kB, n_todo - done)) return;
    const int64_t at = r0 + (n_todo - 1 - done - e);
    if (hit_blocks) next_hits = hit_blocks[at];
    const int id = point_list[at];
    next = gather_fast(id, means2D, colors, normal_opacity, trans_mat, inverse_m);
    if (kSlots) next_radius = radii[id], next_off = slot_first(slots, id);
  };
  gather(0);

  const BlockPriority<4> priority(ordered, tile_order);
  for (int done = 0, parity = 0; done < n_todo; parity ^= 1) {
    priority.set(n_todo - done);
    const int n_staged = min(kB, n_todo - done);
    if ((int) threadIdx.x < kB) {
      const int e = (int) threadIdx.x;
      unsigned mask = 0u;
      if (e < n_staged) {
        s_splat[e] = next;
        mask = hit_blocks ? pair_blocks(next_hits)
                          : fast_blocks<16>(next, keep_local(tile_x) * kTile, keep_local(tile_y) * kTile, ordered);
        if (kFlow) {
#pragma unroll
          for (int k = 0; k < 9; ++k) s_t2[e * 9 + k] = trans_mat_t2[9 * (size_t) next.cold.id + k];
        }
        if (kSlots) {
          // The fused binning reserves one key position per tile of the surfel's rectangle, from its prefix-scan offset
          // on (the tiles that pass its corner test are packed to the front of that span, the rest is padding). Any
          // position of the span that no other tile of the surfel uses will do for the record: x-major over the rectangle.
          const TileRect r = tile_rect(next.hot.cx, next.hot.cy, next_radius, gx, gy);
          s_slot[parity][e] = (int) (next_off + (int64_t) (tile_x - r.x0) * (r.y1 - r.y0) + (tile_y - r.y0));
        } else {
          s_slot[parity][e] = next.cold.id;
        }
        s_place[parity][e] = no_places(kRowPlaces);
      }
      s_mask[e] = mask;
    }
    __syncthreads();
    unsigned masks[2] = {s_mask[lane], s_mask[kWave + lane]};
    const RowCounts counts(masks, wave);
    int base = 0;  // staged entries of the batches before
    for (bool more = true; more;) {
      int start, before[4];
      const int end = row_batch<kRowPlaces>(counts, base, n_staged, start);
      masks[0] = s_mask[lane], masks[1] = s_mask[kWave + lane];  // read again rather than kept through the walk
      more = end - base < kRewalkBelow && end < n_staged;
      if (!more) gather(done + end);
      // Entry j of the batch is position n_todo - 1 - done - j of the list; a pixel takes part from its deepest contributor on.
      const int behind = n_todo - done;
      int first[4] = {behind - row_last[0], behind - row_last[1], behind - row_last[2], behind - row_last[3]};
      for (int& f : first) f = max(f, base);
      const int steps = build_row_lists(&s_list[4 * kB * wave], (unsigned char*) s_place[parity], masks, wave, first, start, before,
                                        end);
      const int my_first = behind - last_contrib, my_median = behind - median_contrib;

      // The part of a pair that is bound to the list's order: advances the pixel's back-to-front state and leaves the
      // pair's weight, dL/dalpha (times the transmittance in front of the pair), dL/d(depth along the ray) and, with a
      // second set of transforms, dL/d(intersection) through it. Only entered by lanes whose pixel blends the entry.
      auto advance_pixel = [&](const SplatCold& cold, int j, const FastHit& h, float& w, float& dL_dalpha,
                               float& dL_dz, float& fsx, float& fsy) {
        T = T * __builtin_amdgcn_rcpf(1.0f - h.alpha);
        w = h.alpha * T;
        // one back-to-front recurrence for every channel that enters the image linearly: c = <upstream gradient,
        // channel values of this surfel> replaces the reference's per-channel accumulators
        float c_lin = cold.r * dLp0 + cold.g * dLp1 + cold.b * dLp2;
        if (kAux) {
          const float rd     = __builtin_amdgcn_rcpf(h.depth);
          const float m_d    = far_scale - far_near * rd;
          const float dmd_dd = far_near * rd * rd;
          if (j == my_median) dL_dz += dL_dmedian;
          if (!kPerSplat) {
            // dL/dweight of the distortion enters dL/dalpha as a linear channel does (its value minus what the pairs
            // behind it accumulated, with the same weights): it rides on the shared recurrence
            c_lin += reg_D2 + m_d * (m_d * reg_A - reg_2D);
            dL_dz += w * (m_d * reg_2A - reg_2D) * dmd_dd;
          } else {
            c_lin += m_d * dL_dM1 + (m_d * m_d) * dL_dM2;
            dL_dz += dmd_dd * (2.0f * m_d * w * dL_dM2);
          }
          c_lin += h.depth * dL_ddepth + cold.nx * dLn0 + cold.ny * dLn1 + cold.nz * dLn2;
          dL_dz += w * dL_ddepth;
        }
        if (kAux || kPerSplat) c_lin += dL_daccum;
        if (kFlow) {
          const float* Q = &s_t2[j * 9];
          const float u2 = Q[0] * h.sx + Q[1] * h.sy + Q[2];
          const float v2 = Q[3] * h.sx + Q[4] * h.sy + Q[5];
          float w2       = Q[6] * h.sx + Q[7] * h.sy + Q[8];
          w2             = fabsf(w2) < 1e-5f ? 1e-5f : w2;
          const float rw = newton_rcp(w2);
          const float fu = fmaf(-pxf, w2, u2) * rw, fv = fmaf(-pyf, w2, v2) * rw;  // u2 / w2 - x: one rounding in the difference
          c_lin = fmaf(fu, dLf0, fmaf(fv, dLf1, c_lin));
          const float wr = w * rw, gu = wr * dLf0, gv = wr * dLf1, gw = -wr * fmaf(fu + pxf, dLf0, (fv + pyf) * dLf1);
          fsx = Q[0] * gu + Q[3] * gv + Q[6] * gw;
          fsy = Q[1] * gu + Q[4] * gv + Q[7] * gw;
        }
        dL_dalpha = c_lin - acc_lin;
        acc_lin   = fmaf(1.0f - h.alpha, acc_lin, h.alpha * c_lin);
        dL_dalpha *= T;
      };

      const int row = lane >> 4, place = row == 0 ? before[0] : row == 1 ? before[1] : row == 2 ? before[2] : before[3];
      float* const sums  = &s_sum[place][lane & 15];  // component lane & 15 of the row's first place
      float* const sums2 = &s_sum[place][16 + ((lane & 2) ? 4 : (lane >> 2 & 1) * 2 + (lane >> 3 & 1))];
      auto blend_entry = [&](const FastHot& hot, int j, int i) {
          const SplatCold cold = s_splat[j].cold;  // used only if a pixel blends the surfel, but then without waiting
          __builtin_amdgcn_sched_barrier(0);
          FastHit h;
          unsigned long long pass;
          fast_intersect_flat(hot, pxf, pyf, near_n, h, &pass);
          pass &= wave_ballot(j >= my_first);
          if (pass == 0ull) {
            if (j != kB) {  // not a padding step; zeros, too, have their place
              sums[i * kFastGradSlots] = 0.0f;
              if ((lane & 1) == 0) sums2[i * kFastGradSlots] = 0.0f;
            }
            return;
          }
          const bool hit = __builtin_amdgcn_inverse_ballot_w64(pass);
          float w = 0.0f, dL_dalpha = 0.0f, dL_dz = 0.0f, fsx = 0.0f, fsy = 0.0f;
          // The part under `hit` leaves a few factors (zero in a lane whose pixel does not blend the entry); the components are
          // products of those factors with quantities that are finite in every lane, formed by all lanes alike: no
          // component needs a zero of its own, and the projected-centre case is the intersection case with a zero in
          // place of 1 / p_z.
          float g[16], g5[5];
          float GdA = 0.0f, oG = 0.0f, dsx = 0.0f, dsy = 0.0f, s_ds = 0.0f, z_sx = 0.0f, z_sy = 0.0f;
          if (hit) {
            advance_pixel(cold, j, h, w, dL_dalpha, dL_dz, fsx, fsy);
            // d/ds of the intersection case (times 1 / p_z below); s is not finite in a lane whose p_z is 0, and such a
            // lane never blends: every use of s sits on this side
            GdA  = dL_dalpha * h.G;
            oG   = hot.opacity * GdA;
            dsx  = fsx - oG * h.sx, dsy = fsy - oG * h.sy;
            if (kAux) dsx += dL_dz * hot.tw0, dsy += dL_dz * hot.tw1;
            s_ds = dsx * h.sx + dsy * h.sy;
            z_sx = dL_dz * h.sx, z_sy = dL_dz * h.sy;
          }
          const bool by_ray   = h.rho3d <= h.rho2d;
          const bool filtered = hit && !by_ray;
          const float rz = (hit && by_ray) ? __builtin_amdgcn_rcpf(h.pz) : 0.0f;
          const float da = dsx * rz, db = dsy * rz, dc = -(s_ds * rz);
          g[0] = w * dLp0, g[1] = w * dLp1, g[2] = w * dLp2;
          g[3] = da * pxf, g[4] = da * pyf, g[5] = da;
          g[6] = db * pxf, g[7] = db * pyf, g[8] = db;
          g[9] = dc * pxf, g[10] = dc * pyf, g[11] = dc;
          if (kAux) g[12] = w * dLn0, g[13] = w * dLn1, g[14] = w * dLn2;
          else      g[12] = g[13] = g[14] = 0.0f;
          g[15] = GdA;
          const float to_centre = filtered ? -2.0f * oG : 0.0f;
          g5[0] = z_sx, g5[1] = z_sy, g5[2] = dL_dz;
          g5[3] = to_centre * h.dx, g5[4] = to_centre * h.dy;
          const float tot = row_sum16_transposed(g), tot5 = row_sum5_transposed(g5);
          if (j != kB) {
            sums[i * kFastGradSlots] = tot;
            if ((lane & 1) == 0) sums2[i * kFastGradSlots] = tot5;
          }
      };
      if (base > 0) __syncthreads();  // the sums of the batch before have been read
      walk_block_list(&s_list[(4 * wave + row) * kB], steps, [&](int j) { return s_splat[j].hot; }, blend_entry,
                      [] { return true; });
      __syncthreads();
      // Flush the batch: add the sums of the rows that hold an entry, in a fixed order.
      if (kSlots) {
        // two lanes per entry, eleven of the record's floats each (component 10 is summed by both)
        static_assert(kBlendThreads == 2 * kB && kFastGradSlots == 21 && kFastRecordSlots == 22);
        if (const int e = base + ((int) threadIdx.x >> 1); e < end) {
          const int h = (int) threadIdx.x & 1;
          float a[11];
          sum_places<kFastGradSlots>(&s_sum[0][0], s_place[parity][e], 10 * h, a);
          float* dst = slot_records + (size_t) s_slot[parity][e] * kFastRecordSlots + 11 * h;
#pragma unroll
          for (int c = 0; c < 11; ++c) dst[c] = h == 0 ? a[c] : c < 10 ? a[c < 10 ? c + 1 : 0] : 0.0f;
        }
      } else {
        // one global atomic per surfel and component for this tile, a lane per component
        for (int t = (int) threadIdx.x; t < (end - base) * kFastGradSlots; t += kBlendThreads) {
          const int q = t / kFastGradSlots, c = t - q * kFastGradSlots, e = base + q, id = s_slot[parity][e];
          float a[1];
          sum_places<kFastGradSlots>(&s_sum[0][0], s_place[parity][e], c, a);
          float* const out = c < 3    ? g_colors + 3 * (size_t) id + c
                             : c < 12 ? g_inv + 9 * (size_t) id + (c - 3)
                             : c < 16 ? g_normal_opacity + 4 * (size_t) id + (c - 12)
                             : c < 19 ? g_trans + 9 * (size_t) id + 6 + (c - 16)
                                      : g_means2D + 2 * (size_t) id + (c - 19);
          if (a[0] != 0.0f) atomicAdd(out, a[0]);
        }
      }
      base = end;
    }
    done += base;
    // No barrier needed here: until the barrier behind the next batch's staging, a wavefront that has flushed touches the
    // records, which nobody reads before, and the other copy of what the flush reads.
  }
}

// The reference's second backward (gs_2d_fast_redner.cu:563-837), the per-splat decomposition itself: a lane owns ONE
// list entry of a tile and keeps that surfel's 21 gradient sums in registers, the tile's pixels pass through the lanes
// one lane per step, front to back, each carrying its blending state from the forward's snapshot in front of the
// bucket on. Where the reference hands 27 values from lane to lane (transmittance, three colour and eight auxiliary
// partial sums, the upstream gradients and counters of the pixel), here two travel: the transmittance T and
//   S = <dL/d(outputs), partial sums - final outputs> + T_final dL/dopacity,
// because dL/dalpha = T c + S / (1 - alpha) with c = <dL/d(outputs), this pair's channel values> only needs the partial
// sums through that one product (S += w c per blended pair); the per-pixel constants are staged in LDS once and read
// by pixel number. Laid out for a 64-lane wavefront as the 3D-Gaussian form of this decomposition: one wavefront takes
// 64 consecutive entries = two of the forward's 32-entry buckets (the wavefront of the odd bucket leaves at once), the
// state moves with one whole-wavefront DPP shift per value, and only the pixels that still blend at the group's first
// entry are fed in. Channel set of the reference's kernel: image, opacity, depth, normal, median depth, M1, M2 (no
// distortion; the depth gradient through M1 is dropped as there, :751-757).
template <bool kAux, bool kSlots>
__global__ void __launch_bounds__(64) fast_bucket_backward_kernel(int W, int H, float near_n, float far_n,
    const int64_t* __restrict__ ranges, const int32_t* __restrict__ point_list, const float2* __restrict__ means2D,
    const float4* __restrict__ normal_opacity, const float* __restrict__ colors, const float* __restrict__ trans_mat,
    const float* __restrict__ inverse_m, const float* __restrict__ images, const float* __restrict__ out_opacity,
    const float* __restrict__ out_extras, const int32_t* __restrict__ n_contrib,
    const int32_t* __restrict__ max_contrib, const int64_t* __restrict__ bucket_offset,
    const int32_t* __restrict__ bucket_to_tile, const float* __restrict__ sampled_T,
    const float* __restrict__ sampled_acc, const float* __restrict__ sampled_aux, const float* __restrict__ dL_dpix,
    const float* __restrict__ dL_dextras, const float* __restrict__ dL_dopacity, float* __restrict__ g_means2D,
    float* __restrict__ g_normal_opacity, float* __restrict__ g_colors, float* __restrict__ g_trans,
    float* __restrict__ g_inv, const SlotSource slots, const int32_t* __restrict__ radii,
    float* __restrict__ slot_records) {
  __shared__ float4 s_up[256];                // dL/d(r, g, b) | dL/ddepth
  __shared__ float4 s_up2[kAux ? 256 : 1];    // dL/dnormal | dL/dM1
  __shared__ float4 s_up3[kAux ? 256 : 1];    // dL/dM2 | dL/d(median depth) | median contributor (int bits) | -
  __shared__ float4 s_pixel[256];             // x | y | last contributor (int bits) | -
  __shared__ float2 s_state[256];             // snapshot: T | S
  const int bucket = blockIdx.x, lane = threadIdx.x;
  const int tile = bucket_to_tile[bucket];
  const int in_tile = bucket - (int) (tile == 0 ? 0 : bucket_offset[tile - 1]);
  if (in_tile & 1) return;
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const int tile_x = tile % gx, tile_y = tile / gx;
  const int64_t r0 = ranges[2 * (size_t) tile], r1 = ranges[2 * (size_t) tile + 1];
  const int first = in_tile * 32, entry = first + lane;
  const bool valid = entry < (int) (r1 - r0);
  const size_t HW = (size_t) H * W;
  const float far_scale = far_n / (far_n - near_n), far_near = far_scale * near_n;

  FastHot hot{};
  SplatCold cold{};
  size_t slot = 0;
  if (valid) {
    const FastSplat g = gather_fast(point_list[r0 + entry], means2D, colors, normal_opacity, trans_mat, inverse_m);
    hot = g.hot, cold = g.cold;
    if (kSlots) {
      const TileRect r = tile_rect(hot.cx, hot.cy, radii[cold.id], gx, gy);
      slot = (size_t) (slot_first(slots, cold.id) + (int64_t) (tile_x - r.x0) * (r.y1 - r.y0) +
                       (tile_y - r.y0));
    }
  }

  // the pixels that still blend at this group's first entry, in row-major order of the tile
  int n_live = 0;
  if (first < max_contrib[tile]) {
#pragma unroll
    for (int part = 0; part < 4; ++part) {
      const int rank = part * 64 + lane;
      const int px = tile_x * kTile + (rank & 15), py = tile_y * kTile + (rank >> 4);
      const bool inside = px < W && py < H;
      const size_t pix = (size_t) W * py + px;
      const int last = inside ? n_contrib[pix] : 0;
      const bool live = last > first;
      const unsigned long long live_lanes = wave_ballot(live);
      if (live) {
        const int at = n_live + __builtin_amdgcn_mbcnt_hi((unsigned) (live_lanes >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((unsigned) live_lanes, 0u));
        const size_t snap = (size_t) bucket * 256 + rank;
        const float up0 = dL_dpix[pix], up1 = dL_dpix[HW + pix], up2 = dL_dpix[2 * HW + pix];
        float S = (1.0f - out_opacity[pix]) * dL_dopacity[pix];
        S += up0 * (sampled_acc[((size_t) bucket * 3 + 0) * 256 + rank] - images[pix]);
        S += up1 * (sampled_acc[((size_t) bucket * 3 + 1) * 256 + rank] - images[HW + pix]);
        S += up2 * (sampled_acc[((size_t) bucket * 3 + 2) * 256 + rank] - images[2 * HW + pix]);
        float up_depth = 0.0f;
        if (kAux) {
          auto behind = [&](int c) { return sampled_aux[((size_t) bucket * 8 + c) * 256 + rank] - out_extras[c * HW + pix]; };
          up_depth = dL_dextras[pix];
          const float n0 = dL_dextras[1 * HW + pix], n1 = dL_dextras[2 * HW + pix], n2 = dL_dextras[3 * HW + pix];
          const float m1 = dL_dextras[6 * HW + pix], m2 = dL_dextras[7 * HW + pix];
          S += up_depth * behind(0) + n0 * behind(1) + n1 * behind(2) + n2 * behind(3) + m1 * behind(6) + m2 * behind(7);
          s_up2[at] = make_float4(n0, n1, n2, m1);
          s_up3[at] = make_float4(m2, dL_dextras[4 * HW + pix], __int_as_float(n_contrib[HW + pix]), 0.0f);
        }
        s_up[at]    = make_float4(up0, up1, up2, up_depth);
        s_state[at] = make_float2(sampled_T[snap], S);
        s_pixel[at] = make_float4((float) px, (float) py, __int_as_float(last), 0.0f);
      }
      n_live += __builtin_popcountll(live_lanes);
    }
  }
  __syncthreads();

  float g[kFastGradSlots];
#pragma unroll
  for (int c = 0; c < kFastGradSlots; ++c) g[c] = 0.0f;
  float T = 0.0f, S = 0.0f;
  // whole-wavefront shift by one lane (DPP wave_shr:1); lane 0 keeps `fresh`
  auto pass_on = [](float fresh, float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fresh),
                                                                 __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, false));
  };
  const int steps = n_live > 0 ? n_live + 63 : 0;
  float2 next_state = s_state[0];
  for (int i = 0; i < steps; ++i) {
    const float2 fresh = next_state;
    next_state = s_state[min(i + 1, n_live - 1)];  // requested a step ahead of its use (nothing new once all have entered)
    T = pass_on(fresh.x, T);
    S = pass_on(fresh.y, S);
    const int q = i - lane;
    if (q < 0 || q >= n_live) continue;
    const float4 pixel = s_pixel[q];
    FastHit h;
    const bool hit = fast_intersect_flat(hot, pixel.x, pixel.y, near_n, h) && valid && entry < __float_as_int(pixel.z);
    if (!hit) continue;
    const float4 up = s_up[q];
    const float w = h.alpha * T, inv = __builtin_amdgcn_rcpf(1.0f - h.alpha);
    float c_lin = cold.r * up.x + cold.g * up.y + cold.b * up.z;
    float dL_dz = 0.0f;
    if (kAux) {
      const float4 upn = s_up2[q], upm = s_up3[q];
      const float rd     = __builtin_amdgcn_rcpf(h.depth);
      const float m_d    = far_scale - far_near * rd;
      const float dmd_dd = far_near * rd * rd;
      c_lin += h.depth * up.w + cold.nx * upn.x + cold.ny * upn.y + cold.nz * upn.z + m_d * upn.w + (m_d * m_d) * upm.x;
      dL_dz = w * up.w + dmd_dd * (2.0f * m_d * w * upm.x);
      if (entry == __float_as_int(upm.z) - 1) dL_dz += upm.y;
      g[12] += w * upn.x, g[13] += w * upn.y, g[14] += w * upn.z;
    }
    S += w * c_lin;  // the partial sums up to and including this pair, minus the final outputs
    const float dL_dalpha = T * c_lin + inv * S;
    T *= 1.0f - h.alpha;
    const float GdA = h.G * dL_dalpha, oG = hot.opacity * GdA;
    const bool by_ray = h.rho3d <= h.rho2d;
    const float rz = by_ray ? __builtin_amdgcn_rcpf(h.pz) : 0.0f;
    const float dsx = dL_dz * hot.tw0 - oG * h.sx, dsy = dL_dz * hot.tw1 - oG * h.sy;
    const float da = dsx * rz, db = dsy * rz, dc = -(da * h.sx + db * h.sy);
    g[0] += w * up.x, g[1] += w * up.y, g[2] += w * up.z;
    g[3] += da * pixel.x, g[4] += da * pixel.y, g[5] += da;
    g[6] += db * pixel.x, g[7] += db * pixel.y, g[8] += db;
    g[9] += dc * pixel.x, g[10] += dc * pixel.y, g[11] += dc;
    g[15] += GdA;
    g[16] += dL_dz * h.sx, g[17] += dL_dz * h.sy, g[18] += dL_dz;
    const float to_centre = by_ray ? 0.0f : -2.0f * oG;
    g[19] += to_centre * h.dx, g[20] += to_centre * h.dy;
  }
  if (!valid) return;
  if (kSlots) {  // every list entry has a lane in some wavefront of this launch: all records are written, zeros included
    float2* dst = (float2*) (slot_records + slot * kFastRecordSlots);
#pragma unroll
    for (int c = 0; c < kFastRecordSlots / 2; ++c)
      dst[c] = make_float2(g[2 * c], 2 * c + 1 < kFastGradSlots ? g[2 * c + 1] : 0.0f);
  } else {
    const int id = cold.id;
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (g[c] != 0.0f) atomicAdd(&g_colors[3 * (size_t) id + c], g[c]);
#pragma unroll
    for (int c = 0; c < 9; ++c)
      if (g[3 + c] != 0.0f) atomicAdd(&g_inv[9 * (size_t) id + c], g[3 + c]);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (g[12 + c] != 0.0f) atomicAdd(&g_normal_opacity[4 * (size_t) id + c], g[12 + c]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (g[16 + c] != 0.0f) atomicAdd(&g_trans[9 * (size_t) id + 6 + c], g[16 + c]);
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (g[19 + c] != 0.0f) atomicAdd(&g_means2D[2 * (size_t) id + c], g[19 + c]);
  }
}

void launch_fast_slot_sum(int P, int gx, int gy, const SlotSource& slots, const int32_t* radii,
                          const float* means2D, const float* inverse_m, const float* normal_opacity,
                          const uint32_t* keep_masks, const SlotWorkspace& ws, FastScatter out, hipStream_t s) {
  hipLaunchKernelGGL(fast_slot_sum_kernel, dim3((unsigned) div_up(P, 4 * kFastSumSurfels)), dim3(256), 0, s, P, gx, gy,
                     slots, radii, (const float2*) means2D, inverse_m, (const float4*) normal_opacity,
                     keep_masks, ws.records, out);
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

namespace {
// hit_blocks[R], if given (without snapshots): per list entry the 2x4 blocks of its tile with a pixel that blended it
int fast_render_forward(int P, int W, int H, double near_n, double far_n, int only_image,
    const float* means2D, const float* colors, const float* normal_opacity, const float* trans_mat,
    const float* inverse_m, const int32_t* point_list, const int64_t* ranges, const float* trans_mat_t2,
    int32_t* accum_max_count, float* accum_weights_p, int32_t* accum_weights_count, const int64_t* bucket_offset,
    float* out_color, float* out_opacity, float* out_extras, float* out_flow, int32_t* n_contrib,
    int32_t* max_contrib, int32_t* bucket_to_tile, float* sampled_T, float* sampled_acc, float* sampled_aux,
    uint32_t* hit_blocks, const ViewMaps& maps, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "GS_2D_fast_render_forward: bad sizes");
  FSGS_REQUIRE(ranges && out_color && out_opacity && n_contrib, "GS_2D_fast_render_forward: null pointer");
  FSGS_REQUIRE(P == 0 || (means2D && colors && normal_opacity && trans_mat && inverse_m),
               "GS_2D_fast_render_forward: null surfel tensor");
  FSGS_REQUIRE(only_image || out_extras || (maps.normals && maps.distortion),
               "GS_2D_fast_render_forward: out_extras is required unless only_image");
  FSGS_REQUIRE(!maps.normals || (maps.Tw2v && maps.surf_depth), "GS_2D_fast_render_forward: null map");
  const bool aux   = !only_image;
  const bool snap  = aux && bucket_offset != nullptr;
  const bool accum = aux && (accum_max_count || accum_weights_p || accum_weights_count);
  const bool flow  = aux && trans_mat_t2 != nullptr;
  FSGS_REQUIRE(!flow || out_flow, "GS_2D_fast_render_forward: out_flow is required with trans_mat_t2");
  FSGS_REQUIRE(!snap || (max_contrib && bucket_to_tile && sampled_T && sampled_acc && sampled_aux),
               "GS_2D_fast_render_forward: snapshot outputs are required with per_tile_bucket_offset");
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const dim3 grid(gx * gy), block(kBlendThreads);
  hipStream_t s = (hipStream_t) stream;
  const int* tile_order = nullptr;
  const int ordered = launch_tile_order(gx, gy, ranges, s, &tile_order);
#define FSGS_LAUNCH_FWD(AUX, SNAP, ACC, FLOW, HITS)                                                                  \
  hipLaunchKernelGGL((fast_blend_forward_kernel<AUX, SNAP, ACC, FLOW, HITS>), grid, block, 0, s, ordered, tile_order, W, H,      \
                     (float) near_n, (float) far_n, ranges, point_list, (const float2*) means2D, colors, trans_mat,  \
                     inverse_m, (const float4*) normal_opacity, trans_mat_t2, bucket_offset, n_contrib, out_color,   \
                     out_opacity, out_extras, (float2*) out_flow, max_contrib, bucket_to_tile, sampled_T,            \
                     sampled_acc, sampled_aux, accum_max_count, accum_weights_p, accum_weights_count, hit_blocks, maps)
#define FSGS_LAUNCH_FWD_F(AUX, SNAP, ACC, HITS) \
  do { if (flow) FSGS_LAUNCH_FWD(AUX, SNAP, ACC, true, HITS); else FSGS_LAUNCH_FWD(AUX, SNAP, ACC, false, HITS); } while (0)
  if (!aux) FSGS_LAUNCH_FWD(false, false, false, false, false);
  else if (snap && accum) FSGS_LAUNCH_FWD_F(true, true, true, false);
  else if (snap) FSGS_LAUNCH_FWD_F(true, true, false, false);
  else if (accum && hit_blocks) FSGS_LAUNCH_FWD_F(true, false, true, true);
  else if (accum) FSGS_LAUNCH_FWD_F(true, false, true, false);
  else if (hit_blocks) FSGS_LAUNCH_FWD_F(true, false, false, true);
  else FSGS_LAUNCH_FWD_F(true, false, false, false);
#undef FSGS_LAUNCH_FWD_F
#undef FSGS_LAUNCH_FWD
  return check_launch("GS_2D_fast_render_forward");
}
}  // namespace

FSGS_API int fsgs_gs_2d_fast_render_forward(int P, int W, int H, double near_n, double far_n, int only_image,
    const float* means2D, const float* colors, const float* normal_opacity, const float* trans_mat,
    const float* inverse_m, const int32_t* point_list, const int64_t* ranges, const float* trans_mat_t2,
    int32_t* accum_max_count, float* accum_weights_p, int32_t* accum_weights_count, const int64_t* bucket_offset,
    float* out_color, float* out_opacity, float* out_extras, float* out_flow, int32_t* n_contrib,
    int32_t* max_contrib, int32_t* bucket_to_tile, float* sampled_T, float* sampled_acc, float* sampled_aux,
    void* stream) {
  return fast_render_forward(P, W, H, near_n, far_n, only_image, means2D, colors, normal_opacity, trans_mat, inverse_m,
                             point_list, ranges, trans_mat_t2, accum_max_count, accum_weights_p, accum_weights_count,
                             bucket_offset, out_color, out_opacity, out_extras, out_flow, n_contrib, max_contrib,
                             bucket_to_tile, sampled_T, sampled_acc, sampled_aux, nullptr, ViewMaps{}, stream);
}

FSGS_API int fsgs_gs_2d_fast_view_forward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* colors, const float* normal_opacity, const float* trans_mat, const float* inverse_m,
    const int32_t* point_list, const int64_t* ranges, const float* trans_mat_t2, int32_t* accum_max_count,
    float* accum_weights_p, int32_t* accum_weights_count, float* out_color, float* out_opacity, float* out_extras,
    float* out_flow, int32_t* n_contrib, uint32_t* hit_blocks, double depth_ratio, const float* Tw2v, float* normals,
    float* surf_depth, float* distortion, void* stream) {
  return fast_render_forward(P, W, H, near_n, far_n, 0, means2D, colors, normal_opacity, trans_mat, inverse_m, point_list,
                             ranges, trans_mat_t2, accum_max_count, accum_weights_p, accum_weights_count, nullptr, out_color,
                             out_opacity, out_extras, out_flow, n_contrib, nullptr, nullptr, nullptr, nullptr, nullptr,
                             hit_blocks,
                             ViewMaps{Tw2v, nullptr, normals, nullptr, surf_depth, distortion, (float) depth_ratio}, stream);
}

FSGS_API size_t fsgs_gs_2d_fast_render_backward_workspace_bytes(int64_t R) {
  return slot_workspace_bytes(R, kFastRecordSlots);
}

namespace {
int fast_render_backward(int P, int W, int H, double near_n, double far_n, int per_splat_form,
    const float* means2D, const float* normal_opacity, const float* colors, const float* trans_mat,
    const float* inverse_m, const float* trans_mat_t2, const float* out_opacity, const float* out_extras,
    const float* out_flow, const float* dL_dpix, const float* dL_dopacity, const float* dL_dextras,
    const float* dL_dflow, const int64_t* ranges, const int32_t* point_list, const int32_t* n_contrib,
    float* g_colors, float* g_means2D, float* g_trans, float* g_inv, float* g_normal_opacity, int64_t R,
    const SlotSource& source, const int32_t* radii, void* workspace, size_t workspace_bytes,
    const uint32_t* keep_masks, const uint32_t* hit_blocks, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "GS_2D_fast_render_backward: bad sizes");
  if (P == 0) return kOk;
  FSGS_REQUIRE(means2D && normal_opacity && colors && trans_mat && inverse_m && out_opacity && dL_dpix && (dL_dopacity || hit_blocks) &&
                   ranges && n_contrib && g_colors && g_means2D && g_trans && g_inv && g_normal_opacity,
               "GS_2D_fast_render_backward: null pointer");
  const bool aux  = out_extras && dL_dextras;
  const bool flow = dL_dflow != nullptr;
  FSGS_REQUIRE(!flow || (aux && trans_mat_t2 && out_flow),
               "GS_2D_fast_render_backward: flow gradients need trans_mat2, out_flows and the auxiliary maps");
  const bool slots = source.scan || source.region;
  SlotWorkspace ws{nullptr};
  if (slots) {
    FSGS_REQUIRE(radii && workspace && R >= 0 && R < (int64_t) 0x7fffffff,
                 "GS_2D_fast_render_backward: the ordered-sum path needs radii, a workspace and the instance count R");
    if (workspace_bytes < slot_workspace_bytes(R, kFastRecordSlots))
      return fail(kWorkspaceSmall, "GS_2D_fast_render_backward: workspace %zu < %zu bytes", workspace_bytes,
                  slot_workspace_bytes(R, kFastRecordSlots));
    FSGS_REQUIRE(((uintptr_t) workspace & 15) == 0, "GS_2D_fast_render_backward: workspace must be 16-byte aligned");
    ws = slot_workspace(workspace, R, kFastRecordSlots);
  }
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const dim3 grid(gx * gy), block(kBlendThreads);
  hipStream_t s = (hipStream_t) stream;
  const int* tile_order = nullptr;
  const int ordered = launch_tile_order(gx, gy, ranges, s, &tile_order);
#define FSGS_LAUNCH_BWD_S(AUX, SPLAT, FLOW, SL)                                                                      \
  hipLaunchKernelGGL((fast_blend_backward_kernel<AUX, SPLAT, FLOW, SL>), grid, block, 0, s, ordered, tile_order, W, H, \
                     (float) near_n, (float) far_n, ranges, point_list, n_contrib, (const float2*) means2D,          \
                     (const float4*) normal_opacity, colors, trans_mat, inverse_m, trans_mat_t2, out_opacity,        \
                     out_extras, (const float2*) out_flow, dL_dpix, dL_dextras, dL_dopacity,                         \
                     (const float2*) dL_dflow, g_means2D, g_normal_opacity, g_colors, g_trans, g_inv, source,        \
                     radii, ws.records, hit_blocks)
#define FSGS_LAUNCH_BWD(AUX, SPLAT, FLOW) \
  do { if (slots) FSGS_LAUNCH_BWD_S(AUX, SPLAT, FLOW, true); else FSGS_LAUNCH_BWD_S(AUX, SPLAT, FLOW, false); } while (0)
  if (aux && per_splat_form && flow) FSGS_LAUNCH_BWD(true, true, true);
  else if (aux && flow) FSGS_LAUNCH_BWD(true, false, true);
  else if (aux && per_splat_form) FSGS_LAUNCH_BWD(true, true, false);
  else if (aux) FSGS_LAUNCH_BWD(true, false, false);
  else if (per_splat_form) FSGS_LAUNCH_BWD(false, true, false);
  else FSGS_LAUNCH_BWD(false, false, false);
#undef FSGS_LAUNCH_BWD
#undef FSGS_LAUNCH_BWD_S
  if (slots)
    launch_fast_slot_sum(P, gx, gy, source, radii, means2D, inverse_m, normal_opacity, keep_masks, ws,
                         FastScatter{g_means2D, g_normal_opacity, g_colors, g_trans, g_inv}, s);
  return check_launch("GS_2D_fast_render_backward");
}
}  // namespace

FSGS_API int fsgs_gs_2d_fast_render_backward(int P, int W, int H, double near_n, double far_n, int per_splat_form,
    const float* means2D, const float* normal_opacity, const float* colors, const float* trans_mat,
    const float* inverse_m, const float* trans_mat_t2, const float* out_opacity, const float* out_extras,
    const float* out_flow, const float* dL_dpix, const float* dL_dopacity, const float* dL_dextras,
    const float* dL_dflow, const int64_t* ranges, const int32_t* point_list, const int32_t* n_contrib,
    float* g_colors, float* g_means2D, float* g_trans, float* g_inv, float* g_normal_opacity, int64_t R,
    const int64_t* point_offsets, const int32_t* radii, void* workspace, size_t workspace_bytes,
    const uint32_t* keep_masks, void* stream) {
  return fast_render_backward(P, W, H, near_n, far_n, per_splat_form, means2D, normal_opacity, colors, trans_mat, inverse_m,
                              trans_mat_t2, out_opacity, out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow,
                              ranges, point_list, n_contrib, g_colors, g_means2D, g_trans, g_inv, g_normal_opacity, R,
                              SlotSource{point_offsets}, radii, workspace, workspace_bytes, keep_masks, nullptr, stream);
}

// The same for views whose preprocess handed out the record slots by regions (instance_slots.hpp), over the blocks that blended an
// entry as the forward noted them (nullptr: bounded here).
FSGS_API int fsgs_gs_2d_fast_view_backward_hits(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* inverse_m,
    const float* trans_mat_t2, const float* out_opacity, const float* out_extras, const float* out_flow,
    const float* dL_dpix, const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow,
    const int64_t* ranges, const int32_t* point_list, const int32_t* n_contrib, float* g_colors, float* g_means2D,
    float* g_trans, float* g_inv, float* g_normal_opacity, int64_t R, const int32_t* slot_offsets,
    const int32_t* slot_regions, const int32_t* tiles_touched, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const uint32_t* keep_masks, const uint32_t* hit_blocks, void* stream) {
  FSGS_REQUIRE(P == 0 || (slot_offsets && slot_regions && tiles_touched),
               "gs_2d_fast_view_backward: record slots are required");
  return fast_render_backward(P, W, H, near_n, far_n, 0, means2D, normal_opacity, colors, trans_mat, inverse_m,
                              trans_mat_t2, out_opacity, out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow,
                              ranges, point_list, n_contrib, g_colors, g_means2D, g_trans, g_inv, g_normal_opacity, R,
                              SlotSource{nullptr, slot_offsets, slot_regions, tiles_touched}, radii, workspace,
                              workspace_bytes, keep_masks, hit_blocks, stream);
}

FSGS_API int fsgs_gs_2d_fast_view_backward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* inverse_m,
    const float* trans_mat_t2, const float* out_opacity, const float* out_extras, const float* out_flow,
    const float* dL_dpix, const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow,
    const int64_t* ranges, const int32_t* point_list, const int32_t* n_contrib, float* g_colors, float* g_means2D,
    float* g_trans, float* g_inv, float* g_normal_opacity, int64_t R, const int32_t* slot_offsets,
    const int32_t* slot_regions, const int32_t* tiles_touched, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const uint32_t* keep_masks, void* stream) {
  return fsgs_gs_2d_fast_view_backward_hits(P, W, H, near_n, far_n, means2D, normal_opacity, colors, trans_mat, inverse_m,
                                            trans_mat_t2, out_opacity, out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras,
                                            dL_dflow, ranges, point_list, n_contrib, g_colors, g_means2D, g_trans, g_inv,
                                            g_normal_opacity, R, slot_offsets, slot_regions, tiles_touched, radii, workspace,
                                            workspace_bytes, keep_masks, nullptr, stream);
}

// The per-splat decomposition itself (fast_bucket_backward_kernel), for callers that want the reference's second
// algorithm rather than its result: B = the number of 32-entry buckets the forward announced (bucket_to_tile's length).
FSGS_API int fsgs_gs_2d_fast_render_bucket_backward(int P, int W, int H, double near_n, double far_n, int B,
    const float* means2D, const float* normal_opacity, const float* colors, const float* trans_mat,
    const float* inverse_m, const float* images, const float* out_opacity, const float* out_extras,
    const int32_t* n_contrib, const int32_t* max_contrib, const int64_t* bucket_offset,
    const int32_t* bucket_to_tile, const float* sampled_T, const float* sampled_acc, const float* sampled_aux,
    const float* dL_dpix, const float* dL_dopacity, const float* dL_dextras, const int64_t* ranges,
    const int32_t* point_list, float* g_colors, float* g_means2D, float* g_trans, float* g_inv,
    float* g_normal_opacity, int64_t R, const int64_t* point_offsets, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const uint32_t* keep_masks, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && B >= 0, "GS_2D_fast_render_bucket_backward: bad sizes");
  if (P == 0) return kOk;
  FSGS_REQUIRE(means2D && normal_opacity && colors && trans_mat && inverse_m && images && out_opacity && n_contrib &&
                   max_contrib && bucket_offset && dL_dpix && dL_dopacity && ranges && g_colors && g_means2D &&
                   g_trans && g_inv && g_normal_opacity &&
                   (B == 0 || (bucket_to_tile && point_list && sampled_T && sampled_acc)),
               "GS_2D_fast_render_bucket_backward: null pointer");
  const bool aux = out_extras && dL_dextras;
  FSGS_REQUIRE(!aux || B == 0 || sampled_aux,
               "GS_2D_fast_render_bucket_backward: the auxiliary maps need their snapshots");
  const bool slots = point_offsets != nullptr;
  SlotWorkspace ws{nullptr};
  if (slots) {
    FSGS_REQUIRE(radii && workspace && R >= 0 && R < (int64_t) 0x7fffffff,
                 "GS_2D_fast_render_bucket_backward: the ordered-sum path needs radii, a workspace and the instance count R");
    if (workspace_bytes < slot_workspace_bytes(R, kFastRecordSlots))
      return fail(kWorkspaceSmall, "GS_2D_fast_render_bucket_backward: workspace %zu < %zu bytes", workspace_bytes,
                  slot_workspace_bytes(R, kFastRecordSlots));
    FSGS_REQUIRE(((uintptr_t) workspace & 15) == 0, "GS_2D_fast_render_bucket_backward: workspace must be 16-byte aligned");
    ws = slot_workspace(workspace, R, kFastRecordSlots);
  }
  hipStream_t s = (hipStream_t) stream;
#define FSGS_FAST_BKT(AUX, SL)                                                                                        \
  hipLaunchKernelGGL((fast_bucket_backward_kernel<AUX, SL>), dim3(B), dim3(64), 0, s, W, H, (float) near_n,           \
                     (float) far_n, ranges, point_list, (const float2*) means2D, (const float4*) normal_opacity,      \
                     colors, trans_mat, inverse_m, images, out_opacity, out_extras, n_contrib, max_contrib,           \
                     bucket_offset, bucket_to_tile, sampled_T, sampled_acc, sampled_aux, dL_dpix, dL_dextras,         \
                     dL_dopacity, g_means2D, g_normal_opacity, g_colors, g_trans, g_inv, SlotSource{point_offsets}, radii, \
                     ws.records)
  if (B > 0) {
    if (aux && slots) FSGS_FAST_BKT(true, true);
    else if (aux) FSGS_FAST_BKT(true, false);
    else if (slots) FSGS_FAST_BKT(false, true);
    else FSGS_FAST_BKT(false, false);
  }
#undef FSGS_FAST_BKT
  if (slots)
    launch_fast_slot_sum(P, (W + kTile - 1) / kTile, (H + kTile - 1) / kTile, SlotSource{point_offsets}, radii, means2D, inverse_m,
                         normal_opacity, keep_masks, ws,
                         FastScatter{g_means2D, g_normal_opacity, g_colors, g_trans, g_inv}, s);
  return check_launch("GS_2D_fast_render_bucket_backward");
}
