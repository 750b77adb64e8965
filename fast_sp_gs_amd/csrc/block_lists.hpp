// Work lists per small block of pixels: the bound that fills them and the lists themselves, shared by the blend kernels.
//
// The blend kernels are bound by the vector instructions of a (wavefront, entry) pass. A wavefront owns an 8x8 quadrant of a
// tile; with one list for all of it, an entry that reaches any of its pixels costs a pass of 64 lanes, few of which have something to
// blend where surfels are small. Here every group of 16 (or 8) lanes owns a block of 4x4 (2x4) pixels and walks a list of its own,
// the staged entries that can reach the block, in list order: all groups run one instruction stream on different entries. A pass
// then lasts as long as the longest of the wavefront's lists, per staged batch. Forward blend of 300k surfels 800x800: 78 M vector
// instructions and 147 us with a list per quadrant, 107 us per 4x4 block, 51 M and 94 us per 2x4; 3M 1352x1014: 506, 333, 282 us;
// 400k 3840x2160: 930, 845, 849. Blocks of 2x2 would double the lists to build and the records to fetch.
#pragma once
#include "blend.hpp"

namespace fsgs {

// Lanes of a block: 16 (4x4 pixels) or 8 (2 wide, 4 tall). Bit q * kPerWave + g of a block mask: block g of quadrant q.
template <int kLanes>
struct BlockShape {
  static_assert(kLanes == 16 || kLanes == 8);
  static constexpr int kWide = kLanes / 4, kColumns = kTile / kWide, kPerWave = kWave / kLanes, kPerTile = 4 * kPerWave;
  // pixel of this lane: its wavefront's quadrant, its block (kPerWave / 2 beside each other, two rows of them), row-major inside
  static __device__ __forceinline__ void lane_pixel(int tile_x, int tile_y, int& px, int& py) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane / kLanes, in = lane % kLanes;
    px = tile_x * kTile + (wave & 1) * 8 + g % (kPerWave / 2) * kWide + in % kWide;
    py = tile_y * kTile + (wave >> 1) * 8 + g / (kPerWave / 2) * 4 + in / kWide;
  }
};

// Where an entry can reach alpha >= 1/255, relative to a centre (ox, oy): the ellipse around (cx, cy) with half extents
// (ex, ey) along the axes whose boundary at height y is cx + slope (y - cy) -+ wide sqrt(1 - (y - cy)^2 / ey^2), and the
// disc of radius disc around the centre (0: none).
struct Footprint {
  float ox, oy;
  float cx, cy, ex, ey;
  float slope, wide, inv_hy, top;  // top: height (relative to cy) of the ellipse's rightmost point; its leftmost is at -top
  float disc;
  int state;  // 0: reaches no pixel; 1: no finite bound, every block is kept; 2: test
};

// hx, hy, hxy: the ellipse { d : d^T [[hx, hxy], [hxy, hy]]^-1 d <= 1 }. One so thin that hxy^2 is within rounding of
// hx hy (a surfel seen edge-on, its intersections no more accurate than that) is replaced by its bounding box.
__device__ __forceinline__ void footprint_ellipse(Footprint& f, float hx, float hy, float hxy) {
#pragma clang fp contract(off)
  hx = fmaxf(hx, 1e-4f), hy = fmaxf(hy, 1e-4f);
  f.ex = __builtin_amdgcn_sqrtf(hx), f.ey = __builtin_amdgcn_sqrtf(hy);
  f.inv_hy = __builtin_amdgcn_rcpf(hy);
  f.slope  = hxy * f.inv_hy;
  const float wide2 = hx - hxy * f.slope;
  f.wide = __builtin_amdgcn_sqrtf(fmaxf(wide2, 0.0f));
  f.top  = hxy * __builtin_amdgcn_rcpf(f.ex);
  if (!(wide2 > 1e-5f * hx)) f.slope = 0.0f, f.wide = f.ex, f.inv_hy = 0.0f;
}

// The blocks of the tile whose pixel centres' hull meets the footprint. Per row of blocks (a slab of heights) the
// ellipse's extent along x is exact: its right (left) boundary is highest at `top` (-top), or at the slab's nearer edge.
// Against rounding the footprint is grown by 1/8 pixel and 0.5 % of its extent, as the other bounds are.
template <int kLanes, bool kDisc>
__device__ __forceinline__ unsigned footprint_blocks(const Footprint& f, int tile_px, int tile_py) {
#pragma clang fp contract(off)
  using Shape = BlockShape<kLanes>;
  constexpr unsigned kAll = (unsigned) ((1ull << Shape::kPerTile) - 1ull);
  constexpr float kWidth = (float) Shape::kWide, kCols = (float) Shape::kColumns;
  if (f.state != 2) return f.state == 1 ? kAll : 0u;
  const float padx = kCullPad + 0.01f * f.ex, pady = kCullPad + 0.01f * f.ey, r2 = kDisc ? f.disc * f.disc : 0.0f;
  const float qx = (float) tile_px - f.ox, qy = (float) tile_py - f.oy;  // first pixel of the tile
  unsigned m = 0u;
#pragma unroll
  for (int by = 0; by < 4; ++by) {
    const float y0 = qy + (float) (4 * by), y1 = y0 + 3.0f;
    const float lo = y0 - f.cy - pady, hi = y1 - f.cy + pady;
    const float yr = __builtin_amdgcn_fmed3f(f.top, lo, hi), yl = __builtin_amdgcn_fmed3f(-f.top, lo, hi);
    const float sr = __builtin_amdgcn_sqrtf(fmaxf(1.0f - yr * yr * f.inv_hy, 0.0f));
    const float sl = __builtin_amdgcn_sqrtf(fmaxf(1.0f - yl * yl * f.inv_hy, 0.0f));
    float right = f.cx + (f.slope * yr + f.wide * sr) + padx, left = f.cx + (f.slope * yl - f.wide * sl) - padx;
    const bool in_ellipse = lo <= f.ey && hi >= -f.ey;
    right = in_ellipse ? right : -1e30f, left = in_ellipse ? left : 1e30f;
    if (kDisc) {
      const float yd = __builtin_amdgcn_fmed3f(0.0f, y0 - kCullPad, y1 + kCullPad), t = r2 - yd * yd;
      const float half = __builtin_amdgcn_sqrtf(fmaxf(t, 0.0f)) + kCullPad;
      right = fmaxf(right, t >= 0.0f ? half : -1e30f), left = fminf(left, t >= 0.0f ? -half : 1e30f);
    }
    // columns [first, last) whose pixels meet [left, right]
    const int last  = (int) __builtin_amdgcn_fmed3f(floorf((right - qx) / kWidth) + 1.0f, 0.0f, kCols);
    const int first = (int) __builtin_amdgcn_fmed3f(ceilf((left - qx - (kWidth - 1.0f)) / kWidth), 0.0f, kCols);
    const unsigned cols = ((1u << last) - 1u) & (0xffu << first);
    constexpr int kHalf = Shape::kColumns / 2;  // a quadrant's columns, and its two rows of blocks
    const int shift = (by >> 1) * 2 * Shape::kPerWave + (by & 1) * kHalf;
    m |= (cols & ((1u << kHalf) - 1u)) << shift | (cols >> kHalf) << (shift + Shape::kPerWave);
  }
  return m;
}

// A surfel: the perspective image of its tangent plane's ellipse u^2 + v^2 <= tau and the low-pass disc (cull_bounds
// explains both). `m`: its ray-splat matrix, (ox, oy): its projected centre.
__device__ __forceinline__ Footprint surfel_footprint(const float* m, float ox, float oy, float opacity) {
#pragma clang fp contract(off)
  Footprint f;
  f.ox = ox, f.oy = oy, f.state = 0;
  const float oa = 255.0f * opacity;
  if (!(oa >= 1.0f)) return f;
  f.state = 1;
  const float tau = 2.0f * __logf(oa) * 1.0001f + 1e-3f;
  f.disc = __builtin_amdgcn_sqrtf(0.5f * tau);
  const float u0 = m[0] - ox * m[6], u1 = m[1] - ox * m[7], u2 = m[2] - ox * m[8];
  const float v0 = m[3] - oy * m[6], v1 = m[4] - oy * m[7], v2 = m[5] - oy * m[8];
  const float d  = tau * (m[6] * m[6] + m[7] * m[7]) - m[8] * m[8];
  if (!((m[8] > 0.0f) && (d < -1e-6f * m[8] * m[8]))) return f;  // reaches the camera plane
  const float inv = __builtin_amdgcn_rcpf(d), f0 = tau * inv, f2 = -inv;
  f.cx = f0 * (u0 * m[6] + u1 * m[7]) + f2 * (u2 * m[8]);
  f.cy = f0 * (v0 * m[6] + v1 * m[7]) + f2 * (v2 * m[8]);
  const float hx  = f.cx * f.cx - (f0 * (u0 * u0 + u1 * u1) + f2 * (u2 * u2));
  const float hy  = f.cy * f.cy - (f0 * (v0 * v0 + v1 * v1) + f2 * (v2 * v2));
  const float hxy = f.cx * f.cy - (f0 * (u0 * v0 + u1 * v1) + f2 * (u2 * v2));
  if (!(hx < 1e30f) || !(hy < 1e30f) || !(fabsf(hxy) < 1e30f) || !(fabsf(f.cx) < 1e15f) || !(fabsf(f.cy) < 1e15f)) return f;
  f.state = 2;
  footprint_ellipse(f, hx, hy, hxy);
  return f;
}

template <int kLanes>
__device__ __forceinline__ unsigned surfel_blocks(const SplatHot& h, int tile_px, int tile_py, int flags) {
  if (flags & kFlagNoCull) return (unsigned) ((1ull << BlockShape<kLanes>::kPerTile) - 1ull);
  return footprint_blocks<kLanes, true>(surfel_footprint(h.m, h.cx, h.cy, h.opacity), tile_px, tile_py);
}

// A 3D Gaussian's conic Q = [[a, b], [b, c]] around (x, y): the ellipse d^T Q d <= 2 ln(255 o). One that is not positive definite
// has no finite bound.
__device__ __forceinline__ Footprint conic_footprint(float x, float y, float a, float b, float c, float opacity) {
#pragma clang fp contract(off)
  Footprint f;
  f.ox = x, f.oy = y, f.cx = f.cy = f.disc = 0.0f, f.state = 0;
  const float oa = 255.0f * opacity;
  if (!(oa >= 1.0f)) return f;
  f.state = 1;
  const float det = a * c - b * b;
  if (!(det > 0.0f) || !(a > 0.0f)) return f;
  const float s = 2.0f * (__logf(oa) * 1.0001f + 1e-3f) * __builtin_amdgcn_rcpf(det);
  if (!(s * a < 1e30f) || !(s * c < 1e30f) || !(fabsf(x) < 1e15f) || !(fabsf(y) < 1e15f)) return f;
  f.state = 2;
  footprint_ellipse(f, s * c, s * a, -(s * b));
  return f;
}

template <int kLanes>
__device__ __forceinline__ unsigned conic_blocks(float x, float y, float a, float b, float c, float opacity, int tile_px,
                                                 int tile_py, int flags) {
  if (flags & kFlagNoCull) return (unsigned) ((1ull << BlockShape<kLanes>::kPerTile) - 1ull);
  return footprint_blocks<kLanes, false>(conic_footprint(x, y, a, b, c, opacity), tile_px, tile_py);
}

// Fills the lists of one wavefront from the masks of the batch's staged entries (lane l holds those of entries
// l, 64 + l, ...; zero past the last one): list g at
// lists + g * kEntries, a byte per entry, padded with `kEntries` -- the number of a record that no pixel blends -- to its
// full length. Blocks without a lane in `lanes` get an empty list. Returns the longest list's length. One wavefront writes and
// reads its lists: wave_lds_sync() orders its lanes, no barrier is needed.
template <int kLanes, int kEntries>
__device__ __forceinline__ int build_block_lists(unsigned char* __restrict__ lists, const unsigned (&masks)[kEntries / kWave], int wave,
                                                 unsigned long long lanes) {
  static_assert(kEntries % kWave == 0 && kEntries < 256, "entry numbers and the padding are bytes");
  constexpr int kPerWave = BlockShape<kLanes>::kPerWave;
  const int lane = __lane_id();
  constexpr unsigned kFill = 0x01010101u * (unsigned) kEntries;
  uint2* fill = (uint2*) lists;
#pragma unroll
  for (int e = 0; e < kPerWave * kEntries / 8; e += kWave) fill[e + lane] = make_uint2(kFill, kFill);
  wave_lds_sync();
  unsigned m[kEntries / kWave];
#pragma unroll
  for (int c = 0; c < kEntries / kWave; ++c) m[c] = masks[c] >> (kPerWave * wave);
  int longest = 0;
#pragma unroll
  for (int g = 0; g < kPerWave; ++g) {
    if ((lanes >> (g * kLanes) & ((1ull << kLanes) - 1ull)) == 0ull) continue;
    int n = 0;
#pragma unroll
    for (int c = 0; c < kEntries / kWave; ++c) {
      const bool on = (m[c] & (1u << g)) != 0u;
      const unsigned long long who = wave_ballot(on);
      const int at = (int) __builtin_amdgcn_mbcnt_hi((unsigned) (who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned) who, n));
      if (on) lists[g * kEntries + at] = (unsigned char) (c * kWave + lane);
      n += (int) __popcll(who);
    }
    longest = max(longest, n);
  }
  wave_lds_sync();
  return longest;
}

// Walks the lists of a wavefront: `load(j)` requests the record of entry j, `work(record, j)` evaluates it and `more()`
// says whether any lane still blends. A wavefront walks alone, so what it would wait for sits on the tile's critical path: the
// record of the next entry is requested before the present one is evaluated, into alternating registers, and the entry
// numbers four at a time one step of four ahead. `work` also gets the step's number. (Reads up to four bytes past the list:
// numbers of another list, or the padding behind the last one; they are loaded but never evaluated.)
template <typename Load, typename Work, typename More>
__device__ __forceinline__ void walk_block_list(const unsigned char* __restrict__ list, int steps, Load load, Work work,
                                                More more) {
  if (steps == 0) return;
  const unsigned* four = (const unsigned*) list;
  unsigned now = four[0];
  auto rec_a = load((int) (now & 255u));
  for (int i = 0;; i += 4) {
    const unsigned next = four[(i >> 2) + 1];
    {
      auto rec_b = load((int) (now >> 8 & 255u));
      work(rec_a, (int) (now & 255u), i);
      if (i + 1 >= steps || !more()) return;
      rec_a = load((int) (now >> 16 & 255u));
      work(rec_b, (int) (now >> 8 & 255u), i + 1);
      if (i + 2 >= steps || !more()) return;
    }
    {
      auto rec_b = load((int) (now >> 24));
      work(rec_a, (int) (now >> 16 & 255u), i + 2);
      if (i + 3 >= steps || !more()) return;
      rec_a = load((int) (next & 255u));
      work(rec_b, (int) (now >> 24), i + 3);
      if (i + 4 >= steps || !more()) return;
    }
    now = next;
  }
}

// The same, one step further ahead (past the list as there: loaded, at most intersected, never blended): `eval(record)`
// forms of an entry what does not depend on the pixel's state, while `work` still deals with the entry before it; `late(j)`
// requests the rest of what `work` reads. Two chains of dependent instructions then stand beside each other. Surfel
// forward, us: 300k 800x800 99.5 -> 95.5, 3M 1352x1014 307 -> 302, 400k 3840x2160 850 -> 832; the 3D Gaussians' and the
// fast path's, whose entries have less in front of the blend, took 1 % longer this way. The record's LDS offset kept for
// both requests instead of formed twice: 96.9, 307, 843.
template <typename Load, typename Late, typename Eval, typename Work, typename More>
__device__ __forceinline__ void walk_block_list_ahead(const unsigned char* __restrict__ list, int steps, Load load, Late late,
                                                      Eval eval, Work work, More more) {
  if (steps == 0) return;
  const unsigned* four = (const unsigned*) list;
  unsigned now = four[0];
  auto rec = load((int) (now & 255u));
  auto a   = eval(rec), b = a;
  rec      = load((int) (now >> 8 & 255u));
  for (int i = 0;; i += 4) {
    const unsigned next = four[(i >> 2) + 1];
    const int j0 = (int) (now & 255u), j1 = (int) (now >> 8 & 255u), j2 = (int) (now >> 16 & 255u), j3 = (int) (now >> 24);
    {
      const auto l = late(j0);
      b   = eval(rec);
      rec = load(j2);
      work(a, l, j0, i);
      if (i + 1 >= steps || !more()) return;
    }
    {
      const auto l = late(j1);
      a   = eval(rec);
      rec = load(j3);
      work(b, l, j1, i + 1);
      if (i + 2 >= steps || !more()) return;
    }
    {
      const auto l = late(j2);
      b   = eval(rec);
      rec = load((int) (next & 255u));
      work(a, l, j2, i + 2);
      if (i + 3 >= steps || !more()) return;
    }
    {
      const auto l = late(j3);
      a   = eval(rec);
      rec = load((int) (next >> 8 & 255u));
      work(b, l, j3, i + 3);
      if (i + 4 >= steps || !more()) return;
    }
    now = next;
  }
}

// ---- which blocks blended an entry ---------------------------------------------------------------------------------------
// A forward kernel (2x4 blocks) can note, per staged entry, the blocks with a pixel that blended it, a byte per block; the
// backward then walks exactly these instead of bounding every footprint again. Block b's byte is b ^ 3: the product below
// gathers the low bits of four bytes, the last byte's first.
constexpr int kHitLanes = 8;  // of a noted block: 32 blocks a tile, which pair_blocks joins to the backward's 4x4
static_assert(BlockShape<kHitLanes>::kPerTile == 32);

__device__ __forceinline__ unsigned hit_bits(const uint4& lo, const uint4& hi) {
  const unsigned w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  unsigned m = 0u;
#pragma unroll
  for (int k = 0; k < 8; ++k) m |= (w[k] * 0x08040201u >> 24) << (4 * k);
  return m;
}

// Mask of the 4x4 blocks that hold a set 2x4 block: pairs of neighbouring bits joined, every second bit kept.
__device__ __forceinline__ unsigned pair_blocks(unsigned m) {
  m = (m | m >> 1) & 0x55555555u;
  m = (m | m >> 1) & 0x33333333u;
  m = (m | m >> 2) & 0x0f0f0f0fu;
  m = (m | m >> 4) & 0x00ff00ffu;
  return (m | m >> 8) & 0xffffu;
}

// ---- lists of the backward kernels: per 4x4 block, with a place for each entry's sums -------------------------------
// A row of 16 lanes sums an entry's gradient components over its 16 pixels with DPP shifts and stores the totals at the
// step's place: an entry's sums from different rows never meet, so nothing is read back, added or ordered while the lists
// are walked. The flush of the batch adds an entry's up to 16 places in a fixed order. The rows share out a pool of places by
// the lengths of their lists; a batch is as many of the staged entries as the pool holds (a long batch evens out the lists'
// lengths and pays the waits between batches less often).
constexpr int kRowBatch = 128;  // entries staged at most: a byte names one, two wavefronts stage them
// Entries that cover their tile take a place in all 16 rows, and a batch is over after 15 of them. Staged anew for each batch, most
// of the 128 would be gathered, bounded and stored eight times; where a batch ends below kRewalkBelow entries, the next one
// takes what is left of the staging. (Above it a fresh staging is the better one: the batch that would be left is short, and its
// lists uneven.) Backward by operators without notes, of 24 / 48 / 80 / 112 entries: 3D Gaussians 300k 800x800 164 / 163 / 158 / 158 us,
// 2000 with deviations of 128 pixels 552 / 524 / 538 / 521; surfels 316 / 317 / 323 / 323 and 967 / 960 / 914 / 932; fast path
// 196 / 193 / 188 / 188 and 866 / 868 / 867 / 869. Never (a staging per batch): 165 and 577, 317 and 1004, 197 and 987; 102400 surfels
// over all of 128x128 with flow 110 -> 91.
constexpr int kRewalkBelow = 80;
// A byte names one of a pool's kPlaces <= 255 places, too; one more behind them, number kPlaces, holds zeros.

__device__ __forceinline__ uint4 no_places(int zeros) {
  const unsigned w = 0x01010101u * (unsigned) zeros;
  return make_uint4(w, w, w, w);
}

// Places that the staged entries up to and with this lane's (64 c + lane, c = 0 and 1) take (`masks`: zero past the last entry); in the
// high half those in the rows of the wavefronts before this one.
struct RowCounts {
  int of[2];
  __device__ __forceinline__ RowCounts(const unsigned (&masks)[2], int wave) {
    const unsigned lower = (1u << (4 * wave)) - 1u;
    of[0] = places(masks[0], lower);
    of[1] = places(masks[1], lower) + __builtin_amdgcn_readlane(of[0], kWave - 1);
  }
  __device__ __forceinline__ int upto(int e) const {  // of the first e > 0 entries
    return e > kWave ? __builtin_amdgcn_readlane(of[1], e - 1 - kWave) : __builtin_amdgcn_readlane(of[0], e - 1);
  }

 private:
  static __device__ __forceinline__ int places(unsigned m, unsigned lower) { return wave_scan(__popc(m) + (__popc(m & lower) << 16)); }
};

// The end of the batch that starts with staged entry `base` of `n`, and `start`, the first place of this wavefront's rows. Every
// wavefront comes to the same batch.
template <int kPlaces>
__device__ __forceinline__ int row_batch(const RowCounts& counts, int base, int n, int& start) {
  static_assert(kPlaces >= 16 && kPlaces <= 255);
  const int taken = base > 0 ? counts.upto(base) : 0, limit = (taken & 0xffff) + kPlaces;
  const int fits = (int) (__popcll(wave_ballot((counts.of[0] & 0xffff) <= limit)) + __popcll(wave_ballot((counts.of[1] & 0xffff) <= limit)));
  n     = min(n, fits);  // an entry takes 16 places at most, so there is always a batch
  start = (counts.upto(n) - taken) >> 16;
  return n;
}

// As build_block_lists, for the four rows of a wavefront: entries [first[r], n) of row r; the rows' places follow each
// other from `start` on, before[r] becomes row r's first. places[e * 16 + row]: where the row will store its sums of entry e
// (the place of zeros was named there before).
__device__ __forceinline__ int build_row_lists(unsigned char* __restrict__ lists, unsigned char* __restrict__ places,
                                               const unsigned (&masks)[2], int wave, const int (&first)[4], int start,
                                               int (&before)[4], int n) {
  const int lane = __lane_id();
  constexpr unsigned kFill = 0x01010101u * (unsigned) kRowBatch;
  ((uint2*) lists)[lane] = make_uint2(kFill, kFill);
  wave_lds_sync();
  const unsigned m[2] = {masks[0] >> (4 * wave), masks[1] >> (4 * wave)};
  int longest = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    int count = 0;
    before[r] = start;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int e = c * kWave + lane;
      const bool on = (m[c] & (1u << r)) != 0u && e >= first[r] && e < n;
      const unsigned long long who = wave_ballot(on);
      const int at = (int) __builtin_amdgcn_mbcnt_hi((unsigned) (who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned) who, count));
      if (on) lists[r * kRowBatch + at] = (unsigned char) e, places[e * 16 + 4 * wave + r] = (unsigned char) (start + at);
      count += (int) __popcll(who);
    }
    start += count;
    longest = max(longest, count);
  }
  wave_lds_sync();
  return longest;
}

// One entry's sums over the rows that hold it: kCount components from `first` on of the places named by the 16 bytes of `places`. All
// places are read (rows that do not hold the entry name the zeros), four at a time: what the registers hold. Up to nine
// components the four rows of a wavefront are added by twos, and the wavefronts in order (of the errors against 64 bits, the 3D
// Gaussians' conic 7.10e-7 -> 6.83e-7, what it was with sums per wavefront, and 3M surfels 781 -> 778 us); with more, that order
// would spill (fast path 130 -> 136 us), and row follows row.
template <int kStride, int kCount>
__device__ __forceinline__ void sum_places(const float* __restrict__ sums, const uint4& places, int first, float (&a)[kCount]) {
  const unsigned w[4] = {places.x, places.y, places.z, places.w};
  auto place = [&](int r) { return sums + (w[r >> 2] >> (8 * (r & 3)) & 255u) * kStride + first; };
#pragma unroll
  for (int c = 0; c < kCount; ++c) a[c] = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r += 4) {
    if constexpr (kCount <= 9) {
      const float *p0 = place(r), *p1 = place(r + 1), *p2 = place(r + 2), *p3 = place(r + 3);
#pragma unroll
      for (int c = 0; c < kCount; ++c) a[c] += (p0[c] + p1[c]) + (p2[c] + p3[c]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float* p = place(r + q);
#pragma unroll
        for (int c = 0; c < kCount; ++c) a[c] += p[c];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace fsgs
