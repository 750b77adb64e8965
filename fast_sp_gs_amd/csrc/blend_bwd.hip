// Per-tile back-to-front backward pass of the 2D-Gaussian-surfel alpha blend for gfx950.
//
// Reference behaviour reproduced: fast_2d_gs/_C/src/gaussian_splatting/gs_2d_redner.cu:238-539 (kernel) and :631-717
// (host entry GS_2D_render_backward). The transmittance is rebuilt by division T <- T / (1 - alpha) while walking the
// tile's list backwards, gradient channels consumed are image, opacity, aux 0-5 (depth, normal, median depth,
// distortion) and optional flow; the 0.99 alpha clamp is not masked in the gradient, as in the reference.
//
// Where the reference issues 18-21 global float atomics per (pixel, surfel) pair, a 16-lane row of a wavefront owns a 4x4
// block of pixels, walks its own list of the staged surfels that reach it (block_lists.hpp) and sums an entry's components
// over its pixels with DPP row shifts; per staged batch the sums of a tile's 16 rows are added in a fixed order, and every staged
// (surfel, tile) instance writes one record at its position in surfel order; slot_reduce_kernel or the preprocess backward
// sums a surfel's records in a fixed order. (Without scan offsets: one global atomic per surfel, component and tile.)
// With flow the step is 50 instructions longer. Its channels, and the sum of weights that it is divided by, ride on the recurrence
// that the image's share, its three quotients take one reciprocal, and the second transforms are loaded when a batch is staged:
// in 128 registers, four wavefronts per SIMD instead of three. Backward with flow, 300k surfels 800x800:
// 485 -> 340 us; 5000 surfels with deviations of about 43 pixels 784 -> 627, 2000 of about 128 pixels 1468 -> 1149 (with a work
// list per 8x8 quadrant they took 530, 715 and 1280).
// Bound by vector issue (152 instructions a step) and by the waits between batches. Against a work list per 8x8 quadrant with
// the blended pairs queued and their components formed 64 pairs at a time: 300k surfels 800x800 311 -> 289 us, 3M 1352x1014
// 1170 -> 950, 10k 256x256 58 -> 40; with the forward's hit_blocks in place of a bound per footprint (a tenth fewer steps, 260
// instructions less per staged wavefront, for 7 us more in the forward) 245, 805 and 36; with batches of up to 128 entries
// whose rows share out one pool of places, instead of 96 with 24 places a row, and a flush that waits for no entry's rows one by
// one, 230, 782 and 37; with priorities (BlockPriority) 206 at 300k. One tile of 1800 entries alone, which the launch cannot be
// shorter than: 179 -> 127.
#include <algorithm>

#include "block_lists.hpp"
#include "instance_slots.hpp"

namespace fsgs {
namespace {

// Per-surfel gradient slots: 0-2 colours | 3-11 trans_mat | 12-14 normal | 15 opacity | 16-17 means2D.
// The first 16 go through one transposed row reduction; the means2D pair is only non-zero for pixels where the
// screen-space low-pass filter wins (rho2d < rho3d) and is reduced separately when any lane took that branch.
constexpr int kGradSlots = 18;

template <bool kAux, bool kFlow, bool kSlots>
__global__ void __launch_bounds__(kBlendThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
blend_backward_kernel(
    int ordered, const int* __restrict__ tile_order, int W, int H, float near_n, float far_n, const int64_t* __restrict__ ranges, const int32_t* __restrict__ point_list,
    const int32_t* __restrict__ n_contrib, const float2* __restrict__ means2D,
    const float4* __restrict__ normal_opacity, const float* __restrict__ colors, const float* __restrict__ trans_mat,
    const float* __restrict__ trans_mat_t2, const float* __restrict__ out_opacity, const float* __restrict__ out_extras,
    const float2* __restrict__ out_flow, const float* __restrict__ dL_dpix, const float* __restrict__ dL_dextras,
    const float* __restrict__ dL_dopacity, const float2* __restrict__ dL_dflow, float* __restrict__ g_means2D,
    float* __restrict__ g_normal_opacity, float* __restrict__ g_colors, float* __restrict__ g_trans,
    SlotSource slots, const int32_t* __restrict__ radii, float* __restrict__ slot_grads,
    const float4* __restrict__ records, const uint32_t* __restrict__ hit_blocks) {
  // First record slot of a surfel; `stored` is what its packed record says (-1: packed before the offsets were known).
  auto first_slot = [&](int id, int64_t stored) -> int64_t {
    if (slots.region) return (stored >= 0 ? stored : (int64_t) slots.offset[id]) + slots.region[slot_region(id)];
    return stored >= 0 ? stored : (id == 0 ? 0 : slots.scan[id - 1]);
  };
  constexpr bool kRewalk = kFlow || !kSlots;  // several batches per staging (kRewalkBelow); a view's entries come as notes and
                                              // rarely fill their tile: with it 781 -> 787 us at 3M surfels
  constexpr int kRowPlaces = kFlow ? 248 : 255;  // of a batch: with 36.5 KB (flow: 40 KB) of LDS four blocks share a compute unit
  using Shape = BlockShape<16>;
  __shared__ Splat s_splat[kRowBatch + 1];  // the last one is what padding names: no pixel blends it
  __shared__ float s_t2[kFlow ? kRowBatch * 9 : 1];
  __shared__ __attribute__((aligned(16))) unsigned char s_list[16 * kRowBatch + 16];
  __shared__ float s_sum[kRowPlaces + 1][kGradSlots];
  // What the flush of a batch reads is kept twice, by batch parity: the next batch is staged while others still flush.
  __shared__ uint4 s_place[2][kRowBatch];  // where each of the 16 rows stores its sums of each staged surfel
  __shared__ int s_slot[2][kRowBatch];     // where they go from there: its position in surfel order (kSlots) or the surfel's id
  __shared__ unsigned s_mask[kRowBatch];   // which 4x4 blocks of the tile it can reach
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

  // deepest list position any pixel of the tile blended: nothing behind it needs to be gathered
  if (threadIdx.x == 0) s_max_contrib = 0;
  __syncthreads();
  int row_max = last_contrib;  // deepest position blended in this lane's 4x4 block
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) row_max = max(row_max, __shfl_xor(row_max, d, kWave));
  int row_last[4];  // the same of the wavefront's four blocks
#pragma unroll
  for (int r = 0; r < 4; ++r) row_last[r] = __builtin_amdgcn_readlane(row_max, 16 * r);
  if (lane == 0) atomicMax(&s_max_contrib, max(max(row_last[0], row_last[1]), max(row_last[2], row_last[3])));
  if (threadIdx.x == 0) s_splat[kRowBatch] = Splat{};  // all zero: p_z == 0 everywhere
  if (threadIdx.x < kGradSlots) s_sum[kRowPlaces][threadIdx.x] = 0.0f;
  if (threadIdx.x < 4) ((unsigned*) &s_list[16 * kRowBatch])[threadIdx.x] = 0u;
  __syncthreads();
  const int n_todo = __builtin_amdgcn_readfirstlane(min(s_max_contrib, (int) (r1 - r0)));  // positions [0, n_todo) of the tile's list, walked from n_todo-1 down to 0
  // No zero fill of the records: the instances behind the tile's deepest contributor are never staged, their records
  // are cleared here; every staged instance writes its record at the flush, zeros included
  if (kSlots) {
    for (int e = n_todo + (int) threadIdx.x; e < (int) (r1 - r0); e += kBlendThreads) {
      const int id = point_list[r0 + e];
      float cx, cy;
      int rad;
      int64_t off;
      if (records) {
        const float4 q2 = records[5 * (size_t) id + 2], q4 = records[5 * (size_t) id + 4];
        cx = q2.y, cy = q2.z, rad = __float_as_int(q4.z), off = first_slot(id, (int64_t) __float_as_int(q4.w));
        if (rad < 0) rad = radii[id];  // a record packed without radii holds -1 there
      } else {
        const float2 c = means2D[id];
        cx = c.x, cy = c.y, rad = radii[id], off = first_slot(id, -1);
      }
      const TileRect r = tile_rect(cx, cy, rad, gx, gy);
      const int64_t slot = off + (int64_t) (tile_y - r.y0) * (r.x1 - r.x0) + (tile_x - r.x0);
      float2* dst = (float2*) (slot_grads + (size_t) slot * kGradSlots);
#pragma unroll
      for (int c = 0; c < kGradSlots / 2; ++c) dst[c] = make_float2(0.0f, 0.0f);
    }
  }

  const float T_final = inside ? 1.0f - out_opacity[pix] : 0.0f;
  float T = T_final;
  float dLp0 = 0, dLp1 = 0, dLp2 = 0;
  float dL_dreg = 0, dL_ddepth = 0, dL_daccum = 0, dLn0 = 0, dLn1 = 0, dLn2 = 0, dL_dmedian = 0;
  float final_D = 0, final_D2 = 0, sum_w = 0;
  if (inside) {
    dLp0 = dL_dpix[pix], dLp1 = dL_dpix[pix + HW], dLp2 = dL_dpix[pix + 2 * HW];
    if (kAux) {
      dL_daccum  = dL_dopacity[pix];
      dL_ddepth  = dL_dextras[pix + 0 * HW];
      dLn0       = dL_dextras[pix + 1 * HW];
      dLn1       = dL_dextras[pix + 2 * HW];
      dLn2       = dL_dextras[pix + 3 * HW];
      dL_dmedian = dL_dextras[pix + 4 * HW];
      dL_dreg    = dL_dextras[pix + 5 * HW];
      final_D    = out_extras[pix + 6 * HW];
      final_D2   = out_extras[pix + 7 * HW];
      sum_w      = out_extras[pix + 8 * HW];
    }
  }
  const float far_scale = far_n / (far_n - near_n), far_near = far_scale * near_n;
  // The distortion term's per-pixel constants, folded once: with m the normalised depth of a pair,
  //   dL/dweight = (D2 + m^2 A - 2 m D) dL/dreg = D2 dL/dreg + m (m reg_A - reg_2D),
  //   dL/dm      = 2 w (m A - D) dL/dreg        = w (m reg_2A - reg_2D).
  const float reg_A = (1.0f - T_final) * dL_dreg, reg_2A = 2.0f * reg_A, reg_2D = 2.0f * final_D * dL_dreg;
  float lin_const = final_D2 * dL_dreg + dL_daccum;  // dL/dweight's constant and the opacity map's gradient
  float dLf0 = 0, dLf1 = 0;
  if (kFlow && inside) {
    const float2 g = dL_dflow[pix], o = out_flow[pix];
    dLf0 = g.x / sum_w, dLf1 = g.y / sum_w;
    lin_const -= (g.x * o.x + g.y * o.y) / (sum_w * sum_w);  // the sum of weights is a channel whose value is 1
  }

  float acc_lin = 0;

  Splat next;
  int next_radius = 0;
  unsigned next_hits = 0u;
  int64_t next_off = 0;
  // entry e of the 128 staged behind `done` entries, counted from the back of the list
  auto gather = [&](int done) {
    const int e = (int) threadIdx.x;
    if (e >= min(kRowBatch, n_todo - done)) return;
    SplatExtra ex;
    if (hit_blocks) next_hits = hit_blocks[r0 + (n_todo - 1 - done - e)];
    next = gather_splat(point_list[r0 + (n_todo - 1 - done - e)], means2D, colors, normal_opacity, trans_mat, records, &ex);
    if (kSlots) {
      // a record carries the surfel's radius (-1 if it was packed without radii) and, once the binning's scan has
      // stored it, its offset (-1 until then)
      next_radius = records && ex.radius >= 0 ? ex.radius : radii[next.cold.id];
      next_off    = first_slot(next.cold.id, records ? ex.offset : -1);
    }
  };
  gather(0);

  const BlockPriority<4> priority(ordered, tile_order);
  for (int done = 0, parity = 0; done < n_todo; parity ^= 1) {
    priority.set(n_todo - done);
    const int n_staged = min(kRowBatch, n_todo - done);
    if ((int) threadIdx.x < kRowBatch) {
      const int e = (int) threadIdx.x;
      unsigned mask = 0u;
      if (e < n_staged) {
        s_splat[e] = next;
        mask = hit_blocks ? pair_blocks(next_hits) : surfel_blocks<16>(next.hot, keep_local(tile_x) * kTile, keep_local(tile_y) * kTile, ordered);
        if (kFlow)  // not requested ahead: nine registers more would be spilled, and the spill would wait for them
#pragma unroll
          for (int k = 0; k < 9; ++k) s_t2[e * 9 + k] = trans_mat_t2[9 * (size_t) next.cold.id + k];
        if (kSlots) {
          // position of this instance in the surfel-ordered key list: the binning emits a surfel's tiles row-major
          // over its rectangle, starting at the surfel's prefix-scan offset (gaussian_prepare.cu:47-83)
          const TileRect r = tile_rect(next.hot.cx, next.hot.cy, next_radius, gx, gy);
          s_slot[parity][e] = (int) (next_off + (int64_t) (tile_y - r.y0) * (r.x1 - r.x0) + (tile_x - r.x0));
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
      if (kRewalk) masks[0] = s_mask[lane], masks[1] = s_mask[kWave + lane];  // read again rather than kept through the walk
      more = kRewalk && end - base < kRewalkBelow && end < n_staged;
      if (!more) gather(done + end);
      // Entry j of the batch is position n_todo - 1 - done - j of the list; a pixel takes part from its deepest contributor on.
      const int behind = n_todo - done;
      int first[4] = {behind - row_last[0], behind - row_last[1], behind - row_last[2], behind - row_last[3]};
      if (kRewalk) for (int& f : first) f = max(f, base);
      const int steps = build_row_lists(&s_list[4 * kRowBatch * wave], (unsigned char*) s_place[parity], masks, wave, first, start,
                                        before, end);
      const int my_first = behind - last_contrib, my_median = behind - median_contrib;
      // ---- order-bound part of one (pixel, entry) pair: advances the pixel's back-to-front state -------------------------
      // All channels that enter the image linearly (colour, depth, opacity, normal, flow) share one recurrence: with
      // c = <upstream gradient, channel values of this surfel>, the reference's per-channel accumulators
      // acc_x = last_alpha * last_x + (1 - last_alpha) * acc_x contract to a single scalar, updated at the end of the
      // pair that supplies alpha and x. Leaves the blend weight w, dL/dalpha and dL/ddepth of the pair, and the flow's part of
      // dL/d(intersection); call under `hit` only.
      auto advance_pixel = [&](const SplatCold& cold, int j, const Hit& h, float& w, float& dL_dalpha, float& dL_dz, float& fsx,
                               float& fsy) {
        const float keep = 1.0f - h.alpha;
        T = T * __builtin_amdgcn_rcpf(keep);
        w = h.alpha * T;
        // one chain of fused multiply-adds; the per-pixel constant of the distortion term sits in lin_const
        float c_lin;
        if (kAux) {
          const float rd     = __builtin_amdgcn_rcpf(h.depth);
          const float m_d    = fmaf(-far_near, rd, far_scale);
          const float dmd_dd = far_near * rd * rd;
          // dL/dweight of the distortion enters dL/dalpha exactly as a linear channel does (its own value minus what the
          // pairs behind it accumulated, with the same weights), so it rides on the shared recurrence
          c_lin = fmaf(h.depth, dL_ddepth, lin_const);
          c_lin = fmaf(m_d, fmaf(m_d, reg_A, -reg_2D), c_lin);
          c_lin = fmaf(cold.nx, dLn0, fmaf(cold.ny, dLn1, fmaf(cold.nz, dLn2, c_lin)));
          // dL/ddepth: through the distortion's normalised depth, the depth map, and the median depth
          const float per_w = fmaf(fmaf(m_d, reg_2A, -reg_2D), dmd_dd, dL_ddepth);
          dL_dz = fmaf(w, per_w, j == my_median ? dL_dmedian : 0.0f);
        } else {
          c_lin = 0.0f;
        }
        c_lin = fmaf(cold.r, dLp0, fmaf(cold.g, dLp1, fmaf(cold.b, dLp2, c_lin)));
        if (kFlow) {
          const float* Q = &s_t2[j * 9];
          const float u2 = Q[0] * h.sx + Q[1] * h.sy + Q[2];
          const float v2 = Q[3] * h.sx + Q[4] * h.sy + Q[5];
          float w2       = Q[6] * h.sx + Q[7] * h.sy + Q[8];
          w2             = fabsf(w2) < 1e-5f ? 1e-5f : w2;
          const float rw = newton_rcp(w2);
          // flow u2 / w2 - x as (u2 - x w2) / w2: one rounding in the difference of two nearly equal numbers
          const float fu = fmaf(-pxf, w2, u2) * rw, fv = fmaf(-pyf, w2, v2) * rw;
          c_lin = fmaf(fu, dLf0, fmaf(fv, dLf1, c_lin));
          const float wr = w * rw, gu = wr * dLf0, gv = wr * dLf1, gw = -wr * fmaf(fu + pxf, dLf0, (fv + pyf) * dLf1);
          fsx = Q[0] * gu + Q[3] * gv + Q[6] * gw;
          fsy = Q[1] * gu + Q[4] * gv + Q[7] * gw;
        }
        // acc_lin: what the pairs behind this one accumulated, alpha_j c_j weighted by the transmittance between
        dL_dalpha = c_lin - acc_lin;
        acc_lin   = fmaf(keep, acc_lin, h.alpha * c_lin);
      };
       // Gradient terms of one (pixel, entry) pair. The part under `hit` leaves
       // a few factors (zero for a lane whose pixel does not blend the entry); the 16 + 2 per-surfel components are
       // products of those factors with quantities that are finite in every lane, formed by all lanes alike, so no
       // component needs a zero of its own and the two ways a surfel is met (ray-splat intersection / projected centre)
       // share one instruction stream.
       auto pair_gradients = [&](const SplatHot& hot, const SplatCold& cold, int j, const Hit& h, bool hit,
                                 float (&g)[16], float& g2x, float& g2y, unsigned long long& filtered_lanes) {
         float w = 0.0f, dL_dalpha = 0.0f, dL_dz = 0.0f, GdA = 0.0f, oG = 0.0f, dsx = 0.0f, dsy = 0.0f, sx = 0.0f, sy = 0.0f;
         if (hit) {
           advance_pixel(cold, j, h, w, dL_dalpha, dL_dz, dsx, dsy);
           if (kFlow) dsx += dL_dz * hot.m[6], dsy += dL_dz * hot.m[7];
           else if (kAux) dsx = dL_dz * hot.m[6], dsy = dL_dz * hot.m[7];
           GdA = dL_dalpha * T * h.G;
           // the Gaussian's own part of d/ds: only the intersection case uses it (times 1 / p_z below)
           oG = hot.opacity * GdA;
           dsx -= oG * h.sx, dsy -= oG * h.sy;
           // s is not finite in a lane whose plane pair degenerates (p_z == 0), and such a lane never blends: what is used of
           // it is zero there
           sx = h.sx, sy = h.sy;
         }
         const bool by_ray   = h.rho3d <= h.rho2d;
         const bool filtered = hit && !by_ray;
         filtered_lanes      = ~wave_ballot(by_ray);  // taken where the comparison is made: its own lane mask, no instruction
         // s = (s, 1) solves k s = l s = 0, so with dk_z and dl_z from the 2x2 system of its first two components (whose
         // determinant is p_z) the gradients of the planes are dk = dk_z (s, 1) and dl = dl_z (s, 1), those of the
         // transform's rows -dk, -dl and, with the depth <row 2, (s, 1)>, x dk + y dl + dL/dz (s, 1). As l x dp and dp x k, dp the
         // gradient of p = k x l, they were 14 instructions more: 300k 215 -> 205 us, 3M 843 -> 805, and less exact.
         const float rz  = (hit && by_ray) ? __builtin_amdgcn_rcpf(h.pz) : 0.0f;
         const float ax = dsx * rz, ay = dsy * rz;
         const float nk = h.ly * ax - h.lx * ay, nl = h.kx * ay - h.ky * ax, nw = dL_dz - (pxf * nk + pyf * nl);
         g[0] = w * dLp0, g[1] = w * dLp1, g[2] = w * dLp2;
         g[3] = nk * sx, g[4] = nk * sy, g[5] = nk;
         g[6] = nl * sx, g[7] = nl * sy, g[8] = nl;
         g[9] = nw * sx, g[10] = nw * sy, g[11] = nw;
         if (kAux) g[12] = w * dLn0, g[13] = w * dLn1, g[14] = w * dLn2;
         else      g[12] = g[13] = g[14] = 0.0f;
         g[15] = GdA;
         const float to_centre = filtered ? -2.0f * oG : 0.0f;
         g2x = to_centre * h.dx, g2y = to_centre * h.dy;
       };
       const int row = lane >> 4, place = row == 0 ? before[0] : row == 1 ? before[1] : row == 2 ? before[2] : before[3];
       float* const sums   = &s_sum[place][lane & 15];               // component lane & 15 of the row's first place
       float* const centre = &s_sum[place][16 + (lane >> 3 & 1)];  // the row's lanes 0 and 8: means2D
       auto backward_entry = [&](const SplatHot& hot, int j, int i) {
        const SplatCold cold = s_splat[j].cold;  // used only if a pixel blends the surfel, but then without waiting
        __builtin_amdgcn_sched_barrier(0);
        Hit h;
        unsigned long long pass, filtered = 0ull;
        intersect_flat(hot, pxf, pyf, near_n, h, &pass);
        pass &= wave_ballot(j >= my_first);
        float tot = 0.0f, mid = 0.0f;
        if (pass != 0ull) {
          float g[16], g2x, g2y;
          pair_gradients(hot, cold, j, h, __builtin_amdgcn_inverse_ballot_w64(pass), g, g2x, g2y, filtered);
          tot = row_sum16_transposed(g);
          if ((pass & filtered) != 0ull) {  // some lane met the surfel by its projected centre
            g2x += dpp_shift_zero<0x128, 0xf, 0xf>(g2x), g2y += dpp_shift_zero<0x128, 0xf, 0xf>(g2y);  // row_ror:8
            mid = (lane & 8) ? g2y : g2x;
            mid += dpp_shift_zero<0x104, 0xf, 0xf>(mid);  // row_shl:4, 2, 1: totals in lanes 0 and 8
            mid += dpp_shift_zero<0x102, 0xf, 0xf>(mid);
            mid += dpp_shift_zero<0x101, 0xf, 0xf>(mid);
          }
        }
        if (j != kRowBatch) {  // not a padding step; zeros, too, have their place
          sums[i * kGradSlots] = tot;
          if ((lane & 7) == 0) centre[i * kGradSlots] = mid;
        }
       };
      if (kRewalk && base > 0) __syncthreads();  // the sums of the batch before have been read
       walk_block_list(&s_list[(4 * wave + row) * kRowBatch], steps, [&](int j) { return s_splat[j].hot; }, backward_entry,
                       [] { return true; });
      __syncthreads();
      // Flush the batch: add the sums of the rows that hold an entry, in a fixed order.
      if (kSlots) {
        // One 72-byte record per (surfel, tile) instance at the instance's position in surfel order, nine components per lane; the
        // per-surfel sums are taken afterwards. Every staged instance writes its record, zeros included (the instances that
        // are never staged were cleared at the start), so nobody has to clear the buffer beforehand.
        static_assert(kBlendThreads == 2 * kRowBatch);
        if (const int e = base + ((int) threadIdx.x >> 1); e < end) {
          constexpr int kHalf = kGradSlots / 2;
          const int h = (int) threadIdx.x & 1;
          float a[kHalf];
          sum_places<kGradSlots>(&s_sum[0][0], s_place[parity][e], h * kHalf, a);
          float* dst = slot_grads + (size_t) s_slot[parity][e] * kGradSlots + h * kHalf;
#pragma unroll
          for (int k = 0; k < kHalf; ++k) dst[k] = a[k];
        }
      } else {
        // one global atomic per surfel and component for this tile, a lane per component: a surfel's are a few requests
        for (int t = (int) threadIdx.x; t < (end - base) * kGradSlots; t += kBlendThreads) {
          const int q = t / kGradSlots, c = t - q * kGradSlots, e = base + q, id = s_slot[parity][e];
          float a[1];
          sum_places<kGradSlots>(&s_sum[0][0], s_place[parity][e], c, a);
          float* const out = c < 3    ? g_colors + 3 * (size_t) id + c
                             : c < 12 ? g_trans + 9 * (size_t) id + (c - 3)
                             : c < 16 ? g_normal_opacity + 4 * (size_t) id + (c - 12)
                                      : g_means2D + 2 * (size_t) id + (c - 16);
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

// Per-surfel sums of the instance records. Nine lanes per surfel, each owning one float2 of the 18-float record, so
// the lanes of a surfel read 72 contiguous bytes per record and neighbouring surfels continue where the previous one
// ends. A surfel's records are fetched eight at a time (past its last record the last one is read again and not added),
// so most surfels need one round trip to memory; the sum itself runs in instance order. Every row of the four outputs
// is written (zeros for surfels without instances): no initialisation, no atomics, and the sum order is fixed.
__global__ void __launch_bounds__(256) slot_reduce_kernel(int P, SlotSource slots,
    const float* __restrict__ slot_grads, float* __restrict__ g_colors, float* __restrict__ g_means2D,
    float* __restrict__ g_trans, float* __restrict__ g_normal_opacity) {
  constexpr int kPerWave = 7, kLanes = 9;  // 63 of 64 lanes busy
  constexpr int kDepth   = 8;              // records of one surfel in flight together
  const int lane = threadIdx.x & 63;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int sub = lane / kLanes, k = lane - sub * kLanes;
  const int i = wave * kPerWave + sub;
  if (sub >= kPerWave || i >= P) return;
  // A surfel without instances (not rendered) has an empty span, so the visibility need not be read.
  int64_t e0;
  int count;
  slot_span(slots, i, e0, count);
  const int64_t e1 = e0 + count;
  const float2* src = (const float2*) slot_grads + k;
  float2 acc = make_float2(0.0f, 0.0f);
  for (int64_t base = e0; base < e1; base += kDepth) {
    float2 v[kDepth];
#pragma unroll
    for (int j = 0; j < kDepth; ++j) v[j] = src[(size_t) (base + j < e1 ? base + j : e1 - 1) * kLanes];
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      const bool on = base + j < e1;
      acc.x += on ? v[j].x : 0.0f, acc.y += on ? v[j].y : 0.0f;
    }
  }
  // record layout: 0-2 colours | 3-11 trans_mat | 12-14 normal | 15 opacity | 16-17 means2D
  const float vals[2] = {acc.x, acc.y};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = 2 * k + h;
    if (c < 3) g_colors[3 * (size_t) i + c] = vals[h];
    else if (c < 12) g_trans[9 * (size_t) i + (c - 3)] = vals[h];
    else if (c < 16) g_normal_opacity[4 * (size_t) i + (c - 12)] = vals[h];
    else g_means2D[2 * (size_t) i + (c - 16)] = vals[h];
  }
}

// The same sum over lists built by the culled binning (fsgs_gs_prepare_*_culled): the positions of a surfel's span
// whose bit is clear in its keep mask belong to no list, were never written and are not read. Nine positions of the
// span per step, row-major over the surfel's rectangle, the records of the kept ones requested together.
__global__ void __launch_bounds__(256) slot_reduce_culled_kernel(int P, SlotSource slots,
    const uint32_t* __restrict__ masks, const float* __restrict__ slot_grads, float* __restrict__ g_colors,
    float* __restrict__ g_means2D, float* __restrict__ g_trans, float* __restrict__ g_normal_opacity) {
  constexpr int kPerWave = 7, kLanes = 9;
  const int lane = threadIdx.x & 63;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int sub = lane / kLanes, k = lane - sub * kLanes;
  const int i = wave * kPerWave + sub;
  if (sub >= kPerWave || i >= P) return;
  int64_t e0;
  int count;
  slot_span(slots, i, e0, count);
  // rectangles above kCullMaskTiles tiles are kept whole
  const uint32_t mask = count > kCullMaskTiles ? 0xffffffffu : masks[i];
  const float2* src = (const float2*) slot_grads + (size_t) e0 * kLanes + k;
  float2 acc = make_float2(0.0f, 0.0f);
  for (int base = 0; base < count; base += kLanes) {
    const uint32_t bits = count > kCullMaskTiles ? 0xffffffffu : (mask >> base);
    float2 v[kLanes];
#pragma unroll
    for (int j = 0; j < kLanes; ++j)
      v[j] = (base + j < count && ((bits >> j) & 1u)) ? src[(size_t) (base + j) * kLanes] : make_float2(0.0f, 0.0f);
#pragma unroll
    for (int j = 0; j < kLanes; ++j) acc.x += v[j].x, acc.y += v[j].y;
  }
  const float vals[2] = {acc.x, acc.y};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = 2 * k + h;
    if (c < 3) g_colors[3 * (size_t) i + c] = vals[h];
    else if (c < 12) g_trans[9 * (size_t) i + (c - 3)] = vals[h];
    else if (c < 16) g_normal_opacity[4 * (size_t) i + (c - 12)] = vals[h];
    else g_means2D[2 * (size_t) i + (c - 16)] = vals[h];
  }
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API size_t fsgs_gs_2d_render_backward_workspace_bytes(int64_t R) {
  return align_up((size_t) (R > 0 ? R : 0) * kGradSlots * 4 + 16, 256);
}

namespace {
// keep_masks: the lists come from fsgs_gs_prepare_*_culled, so the record sum has to skip the positions the binning left out
int render_backward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* trans_mat_t2,
    const float* out_opacity, const float* out_extras, const float* out_flow, const float* dL_dpix,
    const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow, const int64_t* ranges,
    const int32_t* point_list, const int32_t* n_contrib, float* g_colors, float* g_means2D, float* g_trans,
    float* g_normal_opacity, int64_t R, const SlotSource& source, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const float* records, const uint32_t* keep_masks, const uint32_t* hit_blocks, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "GS_2D_render_backward: bad sizes");
  if (P == 0) return kOk;
  FSGS_REQUIRE(means2D && normal_opacity && colors && trans_mat && out_opacity && dL_dpix && dL_dopacity && ranges &&
                   n_contrib && (source.region || (g_colors && g_means2D && g_trans && g_normal_opacity)),
               "GS_2D_render_backward: null pointer");
  const bool aux  = out_extras && dL_dextras;
  const bool flow = dL_dflow != nullptr;
  FSGS_REQUIRE(!flow || (trans_mat_t2 && out_flow && aux),
               "GS_2D_render_backward: flow gradients need trans_mat_t2, out_flow and the auxiliary maps");
  FSGS_REQUIRE(((uintptr_t) records & 15) == 0, "GS_2D_render_backward: records must be 16-byte aligned");
  const bool slots = source.scan || source.region;
  if (slots) {
    FSGS_REQUIRE(radii && workspace && R >= 0 && R < (int64_t) 0x7fffffff,
                 "GS_2D_render_backward: the ordered-sum path needs radii, a workspace and the instance count R");
    if (workspace_bytes < fsgs_gs_2d_render_backward_workspace_bytes(R))
      return fail(kWorkspaceSmall, "GS_2D_render_backward: workspace %zu < %zu bytes", workspace_bytes,
                  fsgs_gs_2d_render_backward_workspace_bytes(R));
  }
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const dim3 grid(gx * gy), block(kBlendThreads);
  hipStream_t s = (hipStream_t) stream;
  float* slot_grads = slots ? (float*) workspace : nullptr;
  const int* tile_order = nullptr;
  const int ordered = launch_tile_order(gx, gy, ranges, s, &tile_order);
#define FSGS_LAUNCH_BWD(AUX, FLOW, SLOTS)                                                                            \
  hipLaunchKernelGGL((blend_backward_kernel<AUX, FLOW, SLOTS>), grid, block, 0, s, ordered, tile_order, W, H, (float) near_n,    \
                     (float) far_n, ranges, point_list, n_contrib, (const float2*) means2D,                          \
                     (const float4*) normal_opacity, colors, trans_mat, trans_mat_t2, out_opacity, out_extras,       \
                     (const float2*) out_flow, dL_dpix, dL_dextras, dL_dopacity, (const float2*) dL_dflow,           \
                     g_means2D, g_normal_opacity, g_colors, g_trans, source, radii, slot_grads,               \
                     (const float4*) records, hit_blocks)
  if (slots) {
    if (aux && flow) FSGS_LAUNCH_BWD(true, true, true);
    else if (aux) FSGS_LAUNCH_BWD(true, false, true);
    else FSGS_LAUNCH_BWD(false, false, true);
    const dim3 sums(div_up((int64_t) div_up(P, 7) * 64, 256));  // kPerWave surfels per wavefront
    if (source.region) return check_launch("GS_2D_render_backward");  // summed by the preprocess backward
    if (keep_masks && culling_enabled())
      hipLaunchKernelGGL(slot_reduce_culled_kernel, sums, dim3(256), 0, s, P, source, keep_masks, slot_grads, g_colors,
                         g_means2D, g_trans, g_normal_opacity);
    else
      hipLaunchKernelGGL(slot_reduce_kernel, sums, dim3(256), 0, s, P, source, slot_grads, g_colors, g_means2D, g_trans,
                         g_normal_opacity);
  } else {
    if (aux && flow) FSGS_LAUNCH_BWD(true, true, false);
    else if (aux) FSGS_LAUNCH_BWD(true, false, false);
    else FSGS_LAUNCH_BWD(false, false, false);
  }
#undef FSGS_LAUNCH_BWD
  return check_launch("GS_2D_render_backward");
}
}  // namespace

FSGS_API int fsgs_gs_2d_render_backward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* trans_mat_t2,
    const float* out_opacity, const float* out_extras, const float* out_flow, const float* dL_dpix,
    const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow, const int64_t* ranges,
    const int32_t* point_list, const int32_t* n_contrib, float* g_colors, float* g_means2D, float* g_trans,
    float* g_normal_opacity, int64_t R, const int64_t* point_offsets, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const float* records, void* stream) {
  return render_backward(P, W, H, near_n, far_n, means2D, normal_opacity, colors, trans_mat, trans_mat_t2, out_opacity,
                         out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow, ranges, point_list, n_contrib,
                         g_colors, g_means2D, g_trans, g_normal_opacity, R, SlotSource{point_offsets}, radii, workspace,
                         workspace_bytes, records, nullptr, nullptr, stream);
}

FSGS_API int fsgs_gs_2d_render_backward_culled(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* trans_mat_t2,
    const float* out_opacity, const float* out_extras, const float* out_flow, const float* dL_dpix,
    const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow, const int64_t* ranges,
    const int32_t* point_list, const int32_t* n_contrib, float* g_colors, float* g_means2D, float* g_trans,
    float* g_normal_opacity, int64_t R, const int64_t* point_offsets, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const float* records, const uint32_t* keep_masks, void* stream) {
  FSGS_REQUIRE(P == 0 || !point_offsets || keep_masks,
               "GS_2D_render_backward_culled: the ordered-sum path over culled lists needs the keep masks");
  return render_backward(P, W, H, near_n, far_n, means2D, normal_opacity, colors, trans_mat, trans_mat_t2, out_opacity,
                         out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow, ranges, point_list, n_contrib,
                         g_colors, g_means2D, g_trans, g_normal_opacity, R, SlotSource{point_offsets}, radii, workspace,
                         workspace_bytes, records, keep_masks, nullptr, stream);
}

// The same for views whose preprocess handed out the record slots by regions (instance_slots.hpp), over the blocks that blended an
// entry as the forward noted them (nullptr: bounded here): the records stay in the workspace, the preprocess backward sums them.
FSGS_API int fsgs_gs_2d_view_backward_hits(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* trans_mat_t2,
    const float* out_opacity, const float* out_extras, const float* out_flow, const float* dL_dpix,
    const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow, const int64_t* ranges,
    const int32_t* point_list, const int32_t* n_contrib, int64_t R, const int32_t* slot_offsets,
    const int32_t* slot_regions, const int32_t* tiles_touched, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const float* records, const uint32_t* hit_blocks, void* stream) {
  FSGS_REQUIRE(P == 0 || (slot_offsets && slot_regions && tiles_touched && records),
               "gs_2d_view_backward: record slots and packed records are required");
  return render_backward(P, W, H, near_n, far_n, means2D, normal_opacity, colors, trans_mat, trans_mat_t2, out_opacity,
                         out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow, ranges, point_list, n_contrib,
                         nullptr, nullptr, nullptr, nullptr, R,
                         SlotSource{nullptr, slot_offsets, slot_regions, tiles_touched}, radii, workspace,
                         workspace_bytes, records, nullptr, hit_blocks, stream);
}

FSGS_API int fsgs_gs_2d_view_backward(int P, int W, int H, double near_n, double far_n, const float* means2D,
    const float* normal_opacity, const float* colors, const float* trans_mat, const float* trans_mat_t2,
    const float* out_opacity, const float* out_extras, const float* out_flow, const float* dL_dpix,
    const float* dL_dopacity, const float* dL_dextras, const float* dL_dflow, const int64_t* ranges,
    const int32_t* point_list, const int32_t* n_contrib, int64_t R, const int32_t* slot_offsets,
    const int32_t* slot_regions, const int32_t* tiles_touched, const int32_t* radii, void* workspace,
    size_t workspace_bytes, const float* records, void* stream) {
  return fsgs_gs_2d_view_backward_hits(P, W, H, near_n, far_n, means2D, normal_opacity, colors, trans_mat, trans_mat_t2,
                                       out_opacity, out_extras, out_flow, dL_dpix, dL_dopacity, dL_dextras, dL_dflow, ranges,
                                       point_list, n_contrib, R, slot_offsets, slot_regions, tiles_touched, radii, workspace,
                                       workspace_bytes, records, nullptr, stream);
}
