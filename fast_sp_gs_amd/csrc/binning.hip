// Tile binning for gfx950: prefix sum of per-surfel tile counts, then the (tile, depth) ordering of all (surfel, tile)
// instances and the per-tile ranges.
//
// Reference behaviour reproduced bit for bit: fast_2d_gs/_C/src/gaussian_splatting/gaussian_prepare.cu:32-83
// (getHigherMsb, duplicateWithKeys), :192-220 (identifyTileRanges), :222-308 (prepare / GS_prepare, which uses
// cub::DeviceScan::InclusiveSum and cub::DeviceRadixSort::SortPairs on bits [0, 32 + msb(T))).
//
// Wave64 design notes
//  * scan: 2048 counts per 256-lane block, lane-local sums + wave prefix by cross-lane shifts + LDS across the 4 waves.
//  * standard path: bucket the instances by tile (count -> scan -> scatter) and sort every tile's segment on its own
//    (see "binning by tile buckets" below); rectangles above 32 tiles are walked cooperatively by the whole wavefront
//    so one huge surfel cannot serialise a wave.
//  * small views (tile_gather_kernel, tile_place_kernel): every tile's block finds its own list among all surfels' rectangles, a
//    word each, and sorts it: two launches instead of five.
//  * device-wide radix sort (used by the fused corner-test binning of the fast path, whose padding entries and sort width
//    follow the reference): 8-bit digits. Per pass: block histograms -> per-digit scan over blocks -> scatter. The
//    scatter ranks keys with 64-bit ballot match masks (8 ballots per round, popcount of the mask below the lane),
//    which is stable by construction: within a wave lower rounds and lower lanes come first, waves are ordered by an
//    LDS prefix, blocks by the scanned histogram.
#include <algorithm>

#include "binning.hpp"
#include "blend.hpp"
#include "instance_slots.hpp"

namespace fsgs {
namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems   = 8;
constexpr int kScanChunk   = kScanThreads * kScanItems;

constexpr int kSortThreads = 256;
constexpr int kSortWaves   = kSortThreads / kWave;
constexpr int kSortItems   = 8;                          // keys per lane
constexpr int kSortChunk   = kSortThreads * kSortItems;  // keys per block
constexpr int kRadixBits   = 8;
constexpr int kRadix       = 1 << kRadixBits;

__device__ __forceinline__ unsigned long long lanemask_lt() {
  const unsigned lane = __lane_id();
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v) {
  const int lane = __lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const T o = __shfl_up(v, d, kWave);
    if (lane >= d) v += o;
  }
  return v;
}

// Block-wide exclusive prefix of one value per thread (256 threads); also returns the block total.
template <typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* s_wave /*[4]*/, T& total) {
  const int lane = __lane_id(), wave = threadIdx.x / kWave;
  const T inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) s_wave[wave] = inc;
  __syncthreads();
  T base = 0;
  total  = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / kWave; ++w) {
    const T s = s_wave[w];
    if (w < wave) base += s;
    total += s;
  }
  __syncthreads();
  return base + inc - v;
}

// ---- inclusive scan of tiles_touched (int32) into int64 offsets ----------------------------------------------------
__global__ void __launch_bounds__(kScanThreads) scan_block_sums_kernel(int P, const int32_t* __restrict__ in,
                                                                       int64_t* __restrict__ block_sums) {
  __shared__ int64_t s_wave[kScanThreads / kWave];
  const int base = blockIdx.x * kScanChunk + threadIdx.x * kScanItems;
  int64_t sum = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (base + k < P) sum += in[base + k];
  int64_t total;
  block_exclusive_scan<int64_t>(sum, s_wave, total);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

// records (optional): the blend kernels' packed per-surfel records ([P][20] floats); the surfel's exclusive offset goes
// into the last word of its record, so the blend backward finds it in the record it gathers anyway.
__global__ void __launch_bounds__(kScanThreads) scan_apply_kernel(int P, const int32_t* __restrict__ in,
                                                                  const int64_t* __restrict__ block_sums,
                                                                  int64_t* __restrict__ out,
                                                                  float* __restrict__ records) {
  __shared__ int64_t s_wave[kScanThreads / kWave];
  const int base = blockIdx.x * kScanChunk + threadIdx.x * kScanItems;
  int32_t v[kScanItems];
  int64_t sum = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = base + k < P ? in[base + k] : 0;
    sum += v[k];
  }
  // The sum of the chunks in front of this one is formed here, by every block for itself (a few hundred values at most),
  // instead of by a one-block kernel between the two passes: one launch less in front of the host's wait for the count.
  int64_t before = 0;
  for (int i = threadIdx.x; i < (int) blockIdx.x; i += kScanThreads) before += block_sums[i];
  int64_t total;
  block_exclusive_scan<int64_t>(before, s_wave, total);
  const int64_t chunk_start = total;
  int64_t run = chunk_start + block_exclusive_scan<int64_t>(sum, s_wave, total);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (records && base + k < P) records[20 * (size_t) (base + k) + 19] = __int_as_float((int) run);
    run += v[k];
    if (base + k < P) out[base + k] = run;
  }
}

constexpr int kCoopThreshold = 32;  // rectangles with more tiles are walked by the whole wavefront
static_assert(kCoopThreshold == kCullMaskTiles, "a lane's serial walk covers exactly the rectangles that have a keep mask");

// ---- binning by tile buckets -----------------------------------------------------------------------------------------
// The reference sorts all (tile << 32 | depth bits) keys with one device-wide radix sort (6 passes of 8 bits for 2500
// tiles). The same final order -- tiles ascending, inside a tile depth bits ascending, equal depths by surfel index,
// which is what the stable radix sort leaves from the emission order -- is produced here in four steps that touch the
// instances twice instead of twelve times:
//   1. count the instances of every tile: blocks of 1024 lanes walk a slice of the surfels each and count in LDS; a
//      block's counts become one row of a (block x tile) matrix,
//   2. prefix of every matrix column over the blocks and exclusive scan of the column totals over the tiles:
//      ranges[t] = (start, end), final from here on,
//   3. the same walk again scatters (depth bits << 32 | surfel) into the tile's segment; a block's cursor of a tile
//      starts at the tile's start plus its column prefix, so neither step 1 nor step 3 issues a global atomic,
//   4. one block per tile sorts its segment (unique 64-bit keys, so the arbitrary order inside a block's run does not
//      matter): by buckets of the depth bits in LDS for segments up to 2048 entries, by a bitonic network in LDS up to 16384
//      entries and for depths that the buckets cannot part, in global memory beyond that.
// Empty tiles get (0, 0) as the reference's zero-initialised ranges have. Tile grids above kMaxLdsTiles tiles (no room
// for one LDS counter per tile) count and scatter with 64-bit global atomics on ranges[t].y instead (tile_emit_kernel).

// One counter per tile in LDS: 64 KB, two blocks on a compute unit, for grids up to kNarrowTiles; all of a compute unit's
// 160 KB for those up to kMaxLdsTiles (a 4K picture has 32 400 tiles). With device-scope atomics in their place a 4K view of
// 400k surfels spent 292 us counting and 482 us scattering, against 33 and 157 (and 34 against 7 in the scan by one block).
constexpr int kNarrowTiles = 16384, kMaxLdsTiles = 40960;

// Which tiles of a surfel's rectangle are visited: all of them (the reference's lists), those that pass the fast path's
// corner test (CornerTest, from the surfel's adjugate and opacity), or those whose bit is set in the surfel's keep mask
// (cull_mask_kernel, or the preprocess kernels: the tiles some pixel of which can blend the surfel; rectangles above 32 tiles are kept
// whole, or, by the surfels' preprocess in a view without a backward, as a window of them, cull_window).
// kWalkCornerMask is the corner test with its verdicts for rectangles of at most 32 tiles taken from a mask the
// preprocess kernel left (bit x * h + y: x-major, the order of the fast path's key span), so that the test's set-up (a
// double-precision logarithm among it) runs once per surfel and view instead of once per walk; larger rectangles are
// tested here.
enum WalkMode { kWalkAll = 0, kWalkCorner = 1, kWalkMask = 2, kWalkCornerMask = 3 };

// What a mode reads beside centres and radii: kWalkCorner the adjugates and opacities, kWalkMask the keep masks,
// kWalkCornerMask all three.
struct WalkInputs {
  const float* inverse_m;
  const float* opacities;
  const uint32_t* keep_masks;

  WalkMode mode() const {
    if (inverse_m) return keep_masks ? kWalkCornerMask : kWalkCorner;
    return keep_masks ? kWalkMask : kWalkAll;
  }
};

constexpr int kWalkGroup = 4;

// Visits the kept (surfel, tile) pairs of surfel i (P: none); all lanes of a wavefront call it together. `visit` gets up to
// kWalkGroup tiles and how many they are, the surfel and the bits of its depth (zero without `depths`). What a lane loads has arrived before the first visit: loads and
// stores are counted together, so a load that is waited for between two visits' stores waits for the first of them as well.
// With the depth loaded by each visit, every entry of a surfel cost the scatter a round trip to memory: 3M surfels
// 1352x1014 104 -> 91 us, 25k Gaussians 639x361 10.8 -> 7.4, 10k surfels 256x256 5.6 -> 4.5. What bounds it at many entries is
// the rate at which the L2s take single stores, 100 to 140 G/s: 4-byte entries (the sort gathering the depths) took 3840x2160 from
// 152 to 145 us, parts of the picture one after the other, each within the L2s, to 140. So fewer entries is what helps: windows
// of the large rectangles (cull_window) took that view's 10.7M entries to 6.0M, the scatter from 161 to 100 us, the sort from 46
// to 37 and the blend from 950 to 870, with the count at 34 as before (41 with each window worked out by the whole wavefront in
// its turn, 59 with the tiles' columns and rows by division too).
template <int kMode, typename Visit>
__device__ __forceinline__ void for_each_instance(int i, int P, int gx, int gy, const float2* __restrict__ means2D,
                                                  const int32_t* __restrict__ radii, const float* __restrict__ depths,
                                                  const WalkInputs& in, Visit visit) {
  constexpr bool kCorner = kMode == kWalkCorner || kMode == kWalkCornerMask;  // large rectangles are corner-tested
  auto visit_one = [&](int t, int id, uint32_t d) {
    const int tile[kWalkGroup] = {t, t, t, t};
    visit(tile, 1, id, d);
  };
  const int lane = __lane_id();
  int x0 = 0, y0 = 0, w = 0, h = 0;
  float IM[kCorner ? 9 : 1], opacity = 1.0f;
#pragma unroll
  for (int k = 0; k < (kCorner ? 9 : 1); ++k) IM[k] = 0.0f;
  uint32_t keep_mask = 0xffffffffu, depth = 0u;
  if (i < P && radii[i] > 0) {
    const float2 c   = means2D[i];
    if (depths) depth = __float_as_uint(depths[i]);
    const TileRect r = tile_rect(c.x, c.y, radii[i], gx, gy);
    x0 = r.x0, y0 = r.y0, w = max(r.x1 - r.x0, 0), h = max(r.y1 - r.y0, 0);
    if (kMode == kWalkCorner || (kMode == kWalkCornerMask && w * h > kCoopThreshold)) {
      opacity = in.opacities[i];
#pragma unroll
      for (int k = 0; k < 9; ++k) IM[k] = in.inverse_m[9 * (size_t) i + k];
    }
    if (kMode == kWalkMask || kMode == kWalkCornerMask) keep_mask = in.keep_masks[i];
  }
  asm volatile("" : "+v"(keep_mask), "+v"(depth));
  const int count = w * h;
  if (count > 0 && count <= kCoopThreshold) {
    if (kMode == kWalkCorner) {
      const CornerTest ct(IM, opacity);
      for (int y = 0; y < h; ++y)
        for (int x = 0; x < w; ++x)
          if (ct.tile(x0 + x, y0 + y)) visit_one((y0 + y) * gx + (x0 + x), i, depth);
    } else {
      // The kept tiles, kWalkGroup at a time: their counters' answers are on the way together, and a lane's turns are as many as
      // it has tiles (counting kernel: 3M surfels 27.7 -> 24.1 us, 300k 8.4 -> 7.6, 25k Gaussians 5.6 -> 4.5).
      const int line = kMode == kWalkCornerMask ? h : w;  // bits of a row, or of a column
      const unsigned inv = 65536u / (unsigned) line + 1u;  // e / line = e * inv >> 16 for e < 32, line <= 32
      uint32_t bits = (kMode == kWalkAll ? 0xffffffffu : keep_mask) & (0xffffffffu >> (32 - count));
      while (bits) {
        int tile[kWalkGroup], n = 0;
#pragma unroll
        for (int k = 0; k < kWalkGroup; ++k) {
          const unsigned e = bits ? (unsigned) __builtin_ctz(bits) : 0u, q = e * inv >> 16, rest = e - q * line;
          n += bits != 0u;
          bits &= bits - 1u;
          tile[k] = kMode == kWalkCornerMask ? (y0 + (int) rest) * gx + x0 + (int) q : (y0 + (int) q) * gx + x0 + (int) rest;
        }
        visit(tile, n, i, depth);
      }
    }
  }
  unsigned long long big = __ballot(count > kCoopThreshold);
  // Large rectangles with a window: its columns and rows, without those of their tiles that lie outside its diagonals. Each
  // lane works out its own surfel's window, in tiles of the grid, and the wavefront then reads one lane's after the other.
  TileWindow v = {0, 0, 0, 0, 0, 0, 0, 0};
  unsigned inv_width = 0u;
  if (kMode == kWalkMask && big) {
    v = tile_window(keep_mask, w, h);
    v.x0 += x0, v.x1 += x0, v.y0 += y0, v.y1 += y0, v.s0 += x0 + y0, v.s1 += x0 + y0;
    v.d0 += x0 - y0 - (h - 1), v.d1 += x0 - y0 - (h - 1);
    big = __ballot(count > kCoopThreshold && v.x0 <= v.x1);
    inv_width = (unsigned) (65536.0f * __builtin_amdgcn_rcpf((float) max(v.x1 - v.x0 + 1, 1))) + 1u;  // e / width = e * this >> 16 for e <= 64
  }
  while (big) {
    const int src = __ffsll((long long) big) - 1;
    big &= big - 1;
    auto of = [src](int value) { return __builtin_amdgcn_readlane(value, src); };
    const int sx0 = of(x0), sy0 = of(y0), sw = of(w), sid = of(i);
    const uint32_t sdepth = (uint32_t) of((int) depth);
    if (kMode == kWalkMask) {
      // a lane goes on by 64 tiles, `down` rows and `right` columns, so that nothing is divided on the way
      const int left = of(v.x0), end = of(v.x1), bottom = of(v.y1), width = end - left + 1;
      const int s0 = of(v.s0), s1 = of(v.s1), d0 = of(v.d0), d1 = of(v.d1);
      const unsigned inv = (unsigned) of((int) inv_width);
      const int down = (int) (kWave * inv >> 16), right = kWave - down * width, first = (int) (lane * inv >> 16);
      for (int y = of(v.y0) + first, x = left + lane - first * width; y <= bottom; y += down) {
        if (x + y >= s0 && x + y <= s1 && x - y >= d0 && x - y <= d1) visit_one(y * gx + x, sid, sdepth);
        x += right;
        if (x > end) x -= width, ++y;
      }
    } else {
      const int scount = of(count);
      float sIM[kCorner ? 9 : 1];
#pragma unroll
      for (int k = 0; k < (kCorner ? 9 : 1); ++k) sIM[k] = kCorner ? __shfl(IM[k], src, kWave) : 0.0f;
      const CornerTest ct(sIM, kCorner ? __shfl(opacity, src, kWave) : 1.0f);
      for (int e = lane; e < scount; e += kWave) {
        const int y = e / sw, x = e - y * sw;
        if (!kCorner || ct.tile(sx0 + x, sy0 + y)) visit_one((sy0 + y) * gx + (sx0 + x), sid, sdepth);
      }
    }
  }
}

// Counting (kScatter = false) and scattering with global atomics, for tile grids beyond kMaxLdsTiles.
template <int kMode, bool kScatter>
__global__ void __launch_bounds__(256) tile_emit_kernel(int P, int gx, int gy, int64_t R,
    const float2* __restrict__ means2D, const float* __restrict__ depths, const int32_t* __restrict__ radii,
    WalkInputs in, unsigned long long* __restrict__ ranges, uint64_t* __restrict__ entries) {
  for_each_instance<kMode>(blockIdx.x * blockDim.x + threadIdx.x, P, gx, gy, means2D, radii, kScatter ? depths : nullptr, in,
                           [&](const int (&tile)[kWalkGroup], int n, int id, uint32_t depth) {
#pragma unroll
    for (int k = 0; k < kWalkGroup; ++k) {
      if (k >= n) break;
      const unsigned long long pos = atomicAdd(ranges + 2 * (size_t) tile[k] + 1, 1ull);
      if (kScatter && (int64_t) pos < R) entries[pos] = ((uint64_t) depth << 32) | (uint32_t) id;
    }
  });
}

// One lane per 3D Gaussian: the keep mask of its rectangle from its projected mean, conic and opacity.
__global__ void __launch_bounds__(256) conic_cull_mask_kernel(int P, int gx, int gy, const float2* __restrict__ means2D,
    const float4* __restrict__ conic_opacity, const int32_t* __restrict__ radii, uint32_t* __restrict__ masks) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  uint32_t m = 0xffffffffu;
  const int radius = radii[i];
  if (radius > 0) {
    const float2 c    = means2D[i];
    const TileRect r  = tile_rect(c.x, c.y, radius, gx, gy);
    const int w = max(r.x1 - r.x0, 0), h = max(r.y1 - r.y0, 0);
    if (w * h <= kCullMaskTiles) {
      const float4 co     = conic_opacity[i];
      const CullBounds cb = conic_cull_bounds(co.x, co.y, co.z, co.w);
      m = 0u;
      int e = 0;
      for (int y = 0; y < h; ++y)
        for (int x = 0; x < w; ++x, ++e)
          if (cull_keeps_tile(cb, c.x, c.y, r.x0 + x, r.y0 + y)) m |= 1u << e;
    }
  }
  masks[i] = m;
}

// One lane per surfel: the keep mask of its rectangle (see kCullMaskTiles) from its packed record.
__global__ void __launch_bounds__(256) cull_mask_kernel(int P, int gx, int gy, const float4* __restrict__ records,
                                                        const int32_t* __restrict__ radii, uint32_t* __restrict__ masks) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  uint32_t m = 0xffffffffu;
  const int radius = radii[i];
  if (radius > 0) {
    const float4* rec = records + 5 * (size_t) i;
    const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];
    const float M[9] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x};
    const float ox = q2.y, oy = q2.z;
    const TileRect r = tile_rect(ox, oy, radius, gx, gy);
    const int w = max(r.x1 - r.x0, 0), h = max(r.y1 - r.y0, 0);
    if (w * h <= kCullMaskTiles) {
      const CullBounds cb = cull_bounds(M, ox, oy, q2.w);
      m = 0u;
      int e = 0;
      for (int y = 0; y < h; ++y)
        for (int x = 0; x < w; ++x, ++e)
          if (cull_keeps_tile(cb, ox, oy, r.x0 + x, r.y0 + y)) m |= 1u << e;
    }
  }
  masks[i] = m;
}

// Layout of the `bins` buffer of the bucket binning: the queue length of the long segments in front of the B x T matrix
// of per-(walk block, tile) instance counts, whose last row holds the tiles' totals.
constexpr int kPrefixTiles = 64, kPrefixWaves = 16, kPrefixChunk = 32;  // walk blocks <= kPrefixWaves * kPrefixChunk
constexpr int kUnscanned   = 2;    // in front of it, behind the queue's length and the instances in all tiles (see tile_prefix_kernel)
constexpr size_t kBinsSums = 256;  // the instances of every 64 tiles
constexpr size_t kBinsHeader = 4096;
static_assert(kBinsSums + (kMaxLdsTiles / kPrefixTiles) * sizeof(uint32_t) <= kBinsHeader, "the sums fit the header");
struct BinsLayout {
  int blocks;      // walk blocks B (0: the tile grid is too large for LDS counters, the global-atomic path is used)
  int per_block;   // surfels per walk block
  size_t bytes;
};
inline BinsLayout bins_layout(int P, int T) {
  BinsLayout l{0, 0, kBinsHeader};
  if (T > kMaxLdsTiles || P <= 0) return l;
  // one 1024-lane block per 1024 surfels while that keeps every block resident at once (two fit on a compute unit, one
  // with a large grid's counters), beyond that the blocks grow
  const int most = T > kNarrowTiles ? kPrefixWaves * kPrefixChunk / 2 : kPrefixWaves * kPrefixChunk;
  l.per_block = 1024 * std::max(1, div_up(P, 1024 * most));
  l.blocks    = div_up(P, l.per_block);
  l.bytes     = kBinsHeader + align_up((size_t) (l.blocks + 1) * T * sizeof(uint32_t), 256);
  return l;
}

// The matrix row of walk block b of B. Blocks are dealt to the eight dies in turn, and a die's blocks get rows that follow each
// other: in every tile's segment the entries of one die are then neighbours, and the die's L2 gathers its scattered 8-byte
// stores into lines as long as its eighth of all entries fits (4 MB). With rows in block order every line was written by
// all dies and left each of them as a piece of its own: 3M surfels 1352x1014 83 -> 58 us, fast path 150k 1001x667 11.0 -> 9.4, 300k
// 800x800 16.8 -> 15.6; 400k 3840x2160, an eighth of whose entries is 9 MB, 148 -> 152.
__device__ __forceinline__ int walk_row(int b, int B) {
  const int die = b % kOrderRegions;
  return die * (B / kOrderRegions) + min(die, B % kOrderRegions) + b / kOrderRegions;
}

// Step 1: every block counts the instances of its surfels per tile in LDS and writes its row of the matrix with plain
// stores (zeros included, so the matrix needs no clearing). No global atomics: device-scope atomics on one address are
// served one after the other at fabric latency, and with surfels in no spatial order every block touches nearly
// every tile.
template <int kMode, int kTiles>
__global__ void __launch_bounds__(1024) tile_hist_kernel(int P, int per_block, int gx, int gy,
    const float2* __restrict__ means2D, const int32_t* __restrict__ radii, WalkInputs in,
    uint32_t* __restrict__ hist, SlotPublish publish) {
  __shared__ unsigned s_count[kTiles];
  // first of all, so that the instance count reaches the host while the rest of the counting is still running
  if (publish.counters && blockIdx.x == 0 && threadIdx.x < kWave) publish_slot_regions(publish);
  const int T = gx * gy;
  for (int t = threadIdx.x; t < T; t += blockDim.x) s_count[t] = 0u;
  __syncthreads();
  const int first = blockIdx.x * per_block, last = min(P, first + per_block);
  // whole wavefronts stay in the loop together: the traversal uses ballots and shuffles
  const int rounds = (last - first + (int) blockDim.x - 1) / (int) blockDim.x;
  for (int r = 0; r < rounds; ++r) {
    const int i = first + r * blockDim.x + threadIdx.x;
    for_each_instance<kMode>(i < last ? i : P, P, gx, gy, means2D, radii, nullptr, in,
                             [&](const int (&tile)[kWalkGroup], int n, int, uint32_t) {
#pragma unroll
      for (int k = 0; k < kWalkGroup; ++k)
        if (k < n) atomicAdd(&s_count[tile[k]], 1u);
    });
  }
  __syncthreads();
  uint32_t* row = hist + (size_t) walk_row(blockIdx.x, (P + per_block - 1) / per_block) * T;
  for (int t = threadIdx.x; t < T; t += blockDim.x) row[t] = s_count[t];
}

// Step 2: per tile, the exclusive prefix of its column over the walk blocks (in place), the column total, which goes to the row
// behind the blocks' and to ranges[t] (an empty range there) for tile_scan_kernel, and the sum over the block's tiles to
// sums[blockIdx.x]. header[kUnscanned]: whether the scan of the totals is left to the scatter. 64 tiles per block, lane = tile, the
// 16 wavefronts share the walk blocks in contiguous chunks so that a wavefront's loads are all in flight at once.
__global__ void __launch_bounds__(kPrefixTiles * kPrefixWaves) tile_prefix_kernel(int T, int B,
    uint32_t* __restrict__ hist, unsigned long long* __restrict__ ranges, uint32_t* __restrict__ sums, int* __restrict__ header,
    bool unscanned) {
  if (blockIdx.x == 0 && threadIdx.x == 0) header[kUnscanned] = unscanned;
  __shared__ uint32_t s_sum[kPrefixWaves][kPrefixTiles];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x * kPrefixTiles + lane;
  const int chunk = (B + kPrefixWaves - 1) / kPrefixWaves, b0 = wave * chunk;
  // a wavefront's whole chunk of the column is loaded before anything is written back (B <= 512: at most 32 values per
  // lane), eight loads in flight at least: at clamped addresses, for a load under a condition is waited for on the spot
  uint32_t c[kPrefixChunk], sum = 0;
#pragma unroll
  for (int i0 = 0; i0 < kPrefixChunk; i0 += 8) {
    if (i0 < chunk) {  // uniform
#pragma unroll
      for (int i = i0; i < i0 + 8; ++i) c[i] = hist[(size_t) min(b0 + i, B - 1) * T + min(t, T - 1)];
    }
#pragma unroll
    for (int i = i0; i < i0 + 8; ++i) {
      c[i] = t < T && i < chunk && b0 + i < B ? c[i] : 0u;
      sum += c[i];
    }
  }
  s_sum[wave][lane] = sum;
  __syncthreads();
  uint32_t run = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kPrefixWaves; ++w) {
    const uint32_t v = s_sum[w][lane];
    if (w < wave) run += v;
    total += v;
  }
  if (t < T) {
#pragma unroll
    for (int i = 0; i < kPrefixChunk; ++i) {
      const int b = b0 + i;
      if (i < chunk && b < B) hist[(size_t) b * T + t] = run;
      run += c[i];
    }
    if (wave == 0) ranges[2 * (size_t) t] = ranges[2 * (size_t) t + 1] = total, hist[(size_t) B * T + t] = total;
  }
  if (wave == 0) {
    uint32_t all = t < T ? total : 0u;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) all += __shfl_xor(all, d, kWave);
    if (lane == 0) sums[blockIdx.x] = all;
  }
}

// Step 3: the walk of step 1 again; a block's cursor of a tile starts at the tile's start plus the instances of the
// blocks in front of it, so the placement needs no global atomics either.
// kScan: whether the tiles' totals have still to be scanned, always, never, or where the header says so (a binning begun by the count
// of a view and ended by the operators; asking takes 0.4 us, 300k surfels with whole lists 16.9 -> 17.3). Every block does that for
// itself (up to kScanTiles, four a lane) and the first one leaves ranges and header for the kernels behind: what tile_scan_kernel does,
// without a launch on the way. Its 4.2 us and the gap behind it against 1.2 to 2.4 us more here: 300k surfels 800x800 420.9 -> 417.7 us a pass, 300k Gaussians 270.3 -> 265.9,
// fast surfels 150k 1001x667 288 -> 284. Where one block does prefix and scan it is 1.5 us more than that block saves (10k 256x256,
// 25k 639x361), and beyond kScanTiles every block would scan in several steps.
constexpr int kScanTiles = 4096;
enum ScanInScatter { kScanned, kToScan, kAskHeader };

template <int kMode, int kTiles, ScanInScatter kScan>
__global__ void __launch_bounds__(1024) tile_scatter_kernel(int P, int per_block, int gx, int gy, int64_t R,
    const float2* __restrict__ means2D, const float* __restrict__ depths, const int32_t* __restrict__ radii,
    WalkInputs in, const uint32_t* __restrict__ hist, unsigned long long* __restrict__ ranges,
    uint64_t* __restrict__ entries, int* __restrict__ order_table, int* __restrict__ header) {
  __shared__ __attribute__((aligned(8))) unsigned s_cursor[kTiles];  // (64-bit words in it below)
  const int T = gx * gy, B = (P + per_block - 1) / per_block;
  const uint32_t* totals = hist + (size_t) B * T;
  // One block more than the walk needs, when the frame's blockIdx -> tile schedule is still to be built: the tiles' totals are
  // final, nothing in this kernel reads the table, and the per-tile sorts and the blend kernels that follow do.
  if (order_table && blockIdx.x == gridDim.x - 1) {
    static_assert(sizeof(TileOrderLds) <= sizeof(s_cursor), "the schedule's LDS fits the cursor array");
    TileOrderLds& lds = *reinterpret_cast<TileOrderLds*>(s_cursor);
    if (kScan != kScanned) build_tile_order(gx, gy, [&](int t) { return (int64_t) totals[t]; }, order_table, order_table + kMaxOrderedTiles, lds);
    else build_tile_order(gx, gy, [&](int t) { return (int64_t) (ranges[2 * (size_t) t + 1] - ranges[2 * (size_t) t]); }, order_table,
                          order_table + kMaxOrderedTiles, lds);
    return;
  }
  const uint32_t* row = hist + (size_t) walk_row(blockIdx.x, B) * T;
  bool scan = kScan == kToScan;
  if (kScan != kToScan) {
    // on its way with the cursors of the other case. Not cleared in here: other blocks read it, and the next count sets it
    if (kScan == kAskHeader) scan = header[kUnscanned] != 0;
    if ((int64_t) ranges[2 * (size_t) T - 1] > R && !scan) return;  // the last tile's end
    for (int t = threadIdx.x; t < T; t += blockDim.x) s_cursor[t] = (unsigned) ranges[2 * (size_t) t] + row[t];
    __syncthreads();
  }
  if (scan) {
    unsigned long long* s_wave = (unsigned long long*) &s_cursor[kTiles - 32];  // behind the cursors of kScanTiles tiles
    const int lane = __lane_id(), wave = threadIdx.x / kWave, t0 = threadIdx.x * 4;
    unsigned c[4], mine[4];
    unsigned long long sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = t0 + k < T ? totals[t0 + k] : 0u, mine[k] = t0 + k < T ? row[t0 + k] : 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) sum += c[k];
    const unsigned long long inc = wave_inclusive_scan(sum);
    if (lane == kWave - 1) s_wave[wave] = inc;
    __syncthreads();
    unsigned long long run = inc - sum, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const unsigned long long v = s_wave[w];
      if (w < wave) run += v;
      all += v;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (t0 + k < T) {
        s_cursor[t0 + k] = (unsigned) run + mine[k];
        if (blockIdx.x == 0) ranges[2 * (size_t) (t0 + k)] = run, ranges[2 * (size_t) (t0 + k) + 1] = run + c[k];
      }
      run += c[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) header[0] = 0, header[1] = (int) all;  // queue length | instances in all tiles
    if ((int64_t) all > R) return;  // R was a guess, and too small (see gs_view_scatter)
    __syncthreads();
  }
  const int first = blockIdx.x * per_block, last = min(P, first + per_block);
  const int rounds = (last - first + (int) blockDim.x - 1) / (int) blockDim.x;
  for (int r = 0; r < rounds; ++r) {
    const int i = first + r * blockDim.x + threadIdx.x;
    for_each_instance<kMode>(i < last ? i : P, P, gx, gy, means2D, radii, depths, in,
                             [&](const int (&tile)[kWalkGroup], int n, int id, uint32_t depth) {
      unsigned pos[kWalkGroup];
#pragma unroll
      for (int k = 0; k < kWalkGroup; ++k)
        if (k < n) pos[k] = atomicAdd(&s_cursor[tile[k]], 1u);
#pragma unroll
      for (int k = 0; k < kWalkGroup; ++k)
        if (k < n && (int64_t) pos[k] < R) entries[pos[k]] = ((uint64_t) depth << 32) | (uint32_t) id;
    });
  }
}

// Exclusive scan of the per-tile counts, 4 tiles per lane and step.
// With `sums` (the instances of every 64 tiles) block b scans the tiles from 4096 b on and adds what lies in front of them
// itself; without, one block walks all tiles.
// ends = false: ranges[t] = (start, start), for a scatter that advances ranges[t].y; ends = true: (start, end).
__global__ void __launch_bounds__(1024) tile_scan_kernel(int T, unsigned long long* __restrict__ ranges,
                                                         const uint32_t* __restrict__ sums, int* __restrict__ large_count,
                                                         bool ends) {
  __shared__ unsigned long long s_wave[16];
  const int lane = __lane_id(), wave = threadIdx.x / kWave;
  unsigned long long carry = 0;
  const int first = sums ? blockIdx.x * 4096 : 0, last = sums ? min(T, first + 4096) : T;
  if (first > 0) {
    unsigned long long before = 0;
    for (int b = threadIdx.x; b < first / kPrefixTiles; b += blockDim.x) before += sums[b];
    const unsigned long long inc = wave_inclusive_scan(before);
    if (lane == kWave - 1) s_wave[wave] = inc;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; ++w) carry += s_wave[w];
    __syncthreads();
  }
  for (int start = first; start < last; start += 4096) {
    const int t0 = start + threadIdx.x * 4;
    unsigned long long c[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = t0 + k < T ? ranges[2 * (size_t) (t0 + k) + 1] : 0ull, sum += c[k];
    const unsigned long long inc = wave_inclusive_scan(sum);
    if (lane == kWave - 1) s_wave[wave] = inc;
    __syncthreads();
    unsigned long long base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const unsigned long long v = s_wave[w];
      if (w < wave) base += v;
      total += v;
    }
    __syncthreads();
    unsigned long long run = carry + base + inc - sum;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (t0 + k < T) ranges[2 * (size_t) (t0 + k)] = run, ranges[2 * (size_t) (t0 + k) + 1] = ends ? run + c[k] : run;
      run += c[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0 && last == T) large_count[0] = 0, large_count[1] = (int) carry;  // queue length | instances in all tiles
}

// Step 2 and the scan by one block, lane = tile, for at most 1024 tiles and kColumn walk blocks (65 536 surfels): a lane has
// its whole column in flight at once, and a launch less stands on the path of a small picture, which is nothing but a row of
// short launches. 10k surfels 256x256 (256 tiles, 10 blocks): 4.8 + 2.6 -> 4.8 us; 50k 501x403 (832, 49): 5.1 + 2.9 -> 7.0.
constexpr int kColumn = 64;

__global__ void __launch_bounds__(1024) tile_prefix_scan_kernel(int T, int B, uint32_t* __restrict__ hist,
    unsigned long long* __restrict__ ranges, int* __restrict__ large_count) {
  __shared__ uint32_t s_wave[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  uint32_t c[kColumn], sum = 0;
#pragma unroll
  for (int i0 = 0; i0 < kColumn; i0 += 8) {
#pragma unroll
    for (int i = i0; i < i0 + 8; ++i) c[i] = 0u;
    if (i0 < B) {  // uniform
#pragma unroll
      for (int i = i0; i < i0 + 8; ++i) c[i] = hist[(size_t) min(i, B - 1) * T + min(t, T - 1)];
    }
  }
#pragma unroll
  for (int i = 0; i < kColumn; ++i) {
    c[i] = t < T && i < B ? c[i] : 0u;
    sum += c[i];
  }
  uint32_t inc = sum;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t up = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += up;
  }
  if (lane == kWave - 1) s_wave[wave] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const uint32_t v = s_wave[w];
    if (w < wave) before += v;
    all += v;
  }
  if (t < T) {
    const uint32_t start = before + inc - sum;
    ranges[2 * (size_t) t] = start, ranges[2 * (size_t) t + 1] = start + sum;
    uint32_t run = 0;
#pragma unroll
    for (int i = 0; i < kColumn; ++i) {
      if (i < B) hist[(size_t) i * T + t] = run;
      run += c[i];
    }
  }
  if (t == 0) large_count[0] = 0, large_count[1] = (int) all;  // queue length | instances in all tiles
}

// Where element i of a segment sits in LDS. With kPad one slot in five stays empty: the rounds of the sorting network
// whose lanes each own four consecutive elements, or four elements 4 apart, then spread a wavefront's 8-byte accesses
// over all banks instead of piling them sixteen deep on a quarter of them.
template <bool kPad>
__device__ __forceinline__ int lds_slot(int i) { return kPad ? i + (i >> 2) : i; }

template <bool kPad, typename Number>
__device__ __forceinline__ void tile_sort_output(int tile, int64_t start, int n, const uint64_t* sorted_local,
                                                 Number* __restrict__ point_list, int64_t* __restrict__ keys_out) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const uint64_t e = sorted_local[lds_slot<kPad>(k)];
    point_list[start + k] = (Number) (uint32_t) e;
    if (keys_out) keys_out[start + k] = (int64_t) (((uint64_t) (uint32_t) tile << 32) | (e >> 32));
  }
}

// Bitonic sorting network for any length n (all compare-exchanges ascending: the first step of every merge pairs an
// element with its mirror image inside the block, the following steps are plain half-cleaners). Pairs whose upper
// element lies beyond n are skipped, which is the same as padding with +infinity. `sync` separates the steps.
template <typename Index, typename Sync>
__device__ __forceinline__ void bitonic_sort(uint64_t* e, Index n, int threads, Sync sync) {
  Index m = 2;
  while (m < n) m <<= 1;
  int log_half = 0;
  for (Index size = 2; size <= m; size <<= 1, ++log_half) {
    const Index half = size >> 1;
    for (Index k = threadIdx.x; k < (m >> 1); k += threads) {
      const Index blk = k >> log_half, off = k & (half - 1);
      const Index lo = blk * size + off, hi = blk * size + size - 1 - off;
      if (hi < n) {
        const uint64_t a = e[lo], b = e[hi];
        if (a > b) e[lo] = b, e[hi] = a;
      }
    }
    sync();
    for (Index stride = half >> 1; stride > 0; stride >>= 1) {
      for (Index k = threadIdx.x; k < (m >> 1); k += threads) {
        const Index lo = ((k & ~(stride - 1)) << 1) | (k & (stride - 1));  // index with the `stride` bit clear
        const Index hi = lo | stride;
        if (hi < n) {
          const uint64_t a = e[lo], b = e[hi];
          if (a > b) e[lo] = b, e[hi] = a;
        }
      }
      sync();
    }
  }
}

// The same network for a segment held in LDS, two network steps per barrier: a lane loads four elements that are closed
// under two consecutive steps (mirror + first half-cleaner, or two half-cleaners), exchanges them in registers and
// stores them back.
__device__ __forceinline__ void cx(uint64_t& a, uint64_t& b) {
  const uint64_t lo = a < b ? a : b, hi = a < b ? b : a;
  a = lo, b = hi;
}

// A lane's four elements of a round lie inside an aligned span of the array (the merge size for a mirror round, twice
// the larger stride for a pair of half-cleaners), and with quads dealt to lanes in order a wavefront's 64 quads of one
// loop iteration cover one aligned 256-element chunk. Rounds whose span fits such a chunk therefore exchange data only
// between lanes of the same wavefront, which needs no block-wide barrier (a wavefront's LDS operations complete in
// order): of the 33 rounds that sort 2048 entries only 7 end in a barrier.
constexpr int kWaveSpan = 4 * kWave;

__device__ __forceinline__ void end_round(int span, int next_span) {
  if (span <= kWaveSpan && next_span <= kWaveSpan) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Power of two that a segment of n entries is padded to (with +infinity keys) before bitonic_sort_lds.
__device__ __forceinline__ int padded_length(int n) {
  int m = 2;
  while (m < n) m <<= 1;
  return m;
}

// Sorts m = 2^k >= 2 entries; every one of the m slots holds a key (the caller pads with ~0), so no access is
// conditional: bounds checks around the loads and stores made the compiler serialise them, one LDS round trip each.
template <bool kPad>
__device__ __forceinline__ void bitonic_sort_lds(uint64_t* e, int m, int threads) {
  auto ld = [&](int i) { return e[lds_slot<kPad>(i)]; };
  auto st = [&](int i, uint64_t v) { e[lds_slot<kPad>(i)] = v; };
  // one network step on pairs (two pairs per lane and iteration, so that the quads-in-order property above holds)
  auto single = [&](int size, int log_half, int stride) {  // stride == 0: the mirror step of `size`
    for (int q = threadIdx.x; q < (m >> 2); q += threads) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 2 * q + h;
        int lo, hi;
        if (stride == 0) {
          const int blk = k >> log_half, off = k & ((size >> 1) - 1);
          lo = blk * size + off, hi = blk * size + size - 1 - off;
        } else {
          lo = ((k & ~(stride - 1)) << 1) | (k & (stride - 1)), hi = lo | stride;
        }
        uint64_t a = ld(lo), b = ld(hi);
        cx(a, b);
        st(lo, a), st(hi, b);
      }
    }
  };
  int log_half = 0;
  for (int size = 2; size <= m; size <<= 1, ++log_half) {
    const int next_size_span = size < m ? 2 * size : 0;
    if (size == 2) {
      if (m == 2) {
        if (threadIdx.x == 0) {
          uint64_t a = ld(0), b = ld(1);
          cx(a, b);
          st(0, a), st(1, b);
        }
        __syncthreads();
        return;
      }
      single(2, 0, 0);
      end_round(2, next_size_span);
      continue;
    }
    const int quarter = size >> 2;
    for (int q = threadIdx.x; q < (m >> 2); q += threads) {  // mirror step + half-cleaner of stride size / 4
      const int blk = q >> (log_half - 1), off = q & (quarter - 1);
      const int base = blk * size;
      const int ia = base + off, ib = ia + quarter, ja = base + size - 1 - off, jb = ja - quarter;
      uint64_t a = ld(ia), b = ld(ib), bm = ld(jb), am = ld(ja);
      cx(a, am), cx(b, bm);
      cx(a, b), cx(bm, am);
      st(ia, a), st(ib, b), st(jb, bm), st(ja, am);
    }
    int stride = quarter >> 1;
    end_round(size, stride >= 2 ? 2 * stride : (stride == 1 ? 2 : next_size_span));
    for (; stride >= 2; stride >>= 2) {  // half-cleaners of strides `stride` and `stride / 2`
      const int lo_s = stride >> 1;
      for (int q = threadIdx.x; q < (m >> 2); q += threads) {
        const int base = ((q & ~(lo_s - 1)) << 2) | (q & (lo_s - 1));
        const int i0 = base, i1 = base | lo_s, i2 = base | stride, i3 = base | stride | lo_s;
        uint64_t v0 = ld(i0), v1 = ld(i1), v2 = ld(i2), v3 = ld(i3);
        cx(v0, v2), cx(v1, v3);
        cx(v0, v1), cx(v2, v3);
        st(i0, v0), st(i1, v1), st(i2, v2), st(i3, v3);
      }
      const int next = stride >> 2;
      end_round(2 * stride, next >= 2 ? 2 * next : (next == 1 ? 2 : next_size_span));
    }
    if (stride == 1) {
      single(size, log_half, 1);
      end_round(2, next_size_span);
    }
  }
  __syncthreads();
}

constexpr int kSmallSegment = 2048;   // entries sorted by a 256-lane block in 20 KB of LDS (1024 measured: this kernel
                                      // 29.6 -> 19.7 us, and 43 us for the queued segments in the 1024-lane kernel)
                                      // (512 lanes per block instead of 256: 27.5 against 29.6 us)
constexpr int kLargeSegment = 16384;  // entries sorted by a 1024-lane block in 128 KB of LDS

// Sorts n <= 256 entries held in LDS, ~0 behind them, by a 256-lane block: a lane keeps one entry in registers and learns
// where it belongs. First its rank among the 64 of its wavefront's chunk, by counting (LDS broadcasts, no dependent step);
// then runs of 64 and 128 are merged two by two, an entry's place being its place in its own run plus the number of smaller
// entries in the other one, a binary search of log2 + 1 dependent reads. Such a segment is bound by its chain of LDS reads
// and barriers: at most 15 reads and 4 barriers behind the chunks, where the network takes 20 rounds of read, exchange and
// write by the one wavefront in four that has work there. Entries differ (their low halves are surfel numbers, one of each
// in a tile). Takes the segments that the buckets leave. Kernel, lists of about 100 entries: 10k surfels 256x256 7.7 -> 5.3 us, 25k Gaussians 639x361 7.8 -> 5.2, fast
// path 150k 1001x667 11.4 -> 8.5. Not for longer segments: with two to eight entries per lane the 64-bit comparisons of the
// counting outweigh the chain (300k 800x800, lists of about 600: 24 us by the network, 32 this way).
constexpr int kMergeSegment = 256;

__device__ __forceinline__ void merge_sort_lds(uint64_t* e, int n) {
  const int p = threadIdx.x, chunk = p & ~(kWave - 1);
  const bool on = p < n;
  const uint64_t key = e[p];
  int at = p;
  if (chunk < n) {  // the whole wavefront
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < kWave; j += 2) {
      const ulonglong2 two = *(const ulonglong2*) (e + chunk + j);
      rank += two.x < key, rank += two.y < key;
    }
    at = chunk + rank;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // a chunk is read and written by one wavefront
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (on) e[at] = key;
  __syncthreads();
  for (int run = kWave; run < n; run <<= 1) {
    const int other = (at & ~(run - 1)) ^ run;
    int below = 0;
    for (int step = run; step > 0; step >>= 1) {
      const int t      = below + step;
      const bool there = on && t <= run && other + t <= n;
      if (e[there ? other + t - 1 : 0] < key && there) below = t;
    }
    __syncthreads();
    at = (at & ~(2 * run - 1)) + (at & (run - 1)) + below;
    if (on) e[at] = key;
    __syncthreads();
  }
}

// ---- a tile's segment by buckets --------------------------------------------------------------------------------------
constexpr int kSortBuckets = kSmallSegment / 2;  // their counters fill the LDS that the network's empty slots take
constexpr int kBucketLimit = 32;                 // entries of one bucket that are put in order by counting

// Exclusive prefix over the counters of a block of kWaves wavefronts, in place, and the largest one: a lane owns kOwn neighbouring words of
// kHalves counters (32 or 16 bits). s_wave: two words a wavefront. Two barriers; one more before the counters are read.
template <int kOwn, int kHalves, int kWaves = 4>
__device__ __forceinline__ unsigned prefix_counters(unsigned* s_count, unsigned* s_wave) {
  constexpr unsigned kMask = kHalves == 2 ? 0xffffu : ~0u;
  const int wave = threadIdx.x >> 6;
  unsigned own[kOwn], sum = 0, most = 0;
#pragma unroll
  for (int c = 0; c < kOwn; ++c) {
    const unsigned v = own[c] = s_count[kOwn * threadIdx.x + c];
    sum += v & kMask, most = max(most, v & kMask);
    if (kHalves == 2) sum += v >> 16, most = max(most, v >> 16);
  }
  const unsigned inc = (unsigned) wave_scan((int) sum);
  most = wave_max_to_last(most);
  if ((threadIdx.x & 63) == 63) s_wave[2 * wave] = inc, s_wave[2 * wave + 1] = most;
  __syncthreads();
  unsigned at = inc - sum;
  most = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) at += s_wave[2 * w];
    most = max(most, s_wave[2 * w + 1]);
  }
#pragma unroll
  for (int c = 0; c < kOwn; ++c) {
    const unsigned low = own[c] & kMask;
    s_count[kOwn * threadIdx.x + c] = kHalves == 2 ? at | (at + low) << 16 : at;
    at += kHalves == 2 ? low + (own[c] >> 16) : low;
  }
  __syncthreads();
  return most;
}

// Sorts n <= 256 * kPer entries by a 256-lane block and writes list and keys. Bound by its chain of about ten
// LDS round trips and five barriers, whatever n is, where the network takes 33 rounds and 7 barriers for 2048 entries: against
// the network (merging up to 256 entries), 400k surfels 3840x2160 153 -> 41 us, 3M 1352x1014 62 -> 18, 300k 800x800 24 -> 7.6,
// 300k Gaussians 29 -> 7.9, 150k 1001x667 9.2 -> 4.6, 10k 256x256 5.1 -> 3.7. With depths in two thin shells, which take the
// second cut, 1100 entries a tile in 2500 tiles: 140 -> 87..116 us for the whole binning, 200 entries a tile: alike. With one depth for
// all, or one of two, 1100 a tile: 67 -> 19 and 25 us, 80 a tile: 7.1 and 8.0, as by merging (a count of all in one counter, twice, and
// the network behind it took 89 and 81, 10.5 and 9.8).
// The buckets cut the span of the
// segment's depth bits into equal parts, so they are in order among themselves; an entry's place is its bucket's start plus the
// number of smaller entries in the bucket (all 64 bits compared), a few when the depths spread. When some bucket holds more
// than kBucketLimit entries (surfaces at a few depths, a far outlier), every bucket is cut once more into as many parts as it
// has entries, by its depths, or, if it holds a single one, by the surfels' numbers, which decide among equal depths. (To find those
// buckets costs segments without one about 2 us of the 116.) False, with nothing written and the keys in `key`, when that leaves too
// many together as well (numbers in clumps, half a bucket at one depth): the comparing sorts take such a segment.
// load(i): entry i, from memory, or, kHeld, from s_e itself.
template <int kPer, bool kHeld, typename Load, typename Number>
__device__ __forceinline__ bool bucket_sort(int tile, int64_t start, int n, Load load, uint64_t (&key)[kPer], uint64_t* s_e,
                                            Number* __restrict__ point_list, int64_t* __restrict__ keys_out) {
  constexpr int kBuckets = kPer == 1 ? kSortBuckets / 2 : kSortBuckets, kOwn = kBuckets / 256;
  unsigned* s_count = (unsigned*) (s_e + kSmallSegment);
  unsigned* s_wave  = (unsigned*) s_e;  // before the entries come
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < kPer; ++q) key[q] = load(min((int) threadIdx.x + 256 * q, n - 1));
  if (kHeld) __syncthreads();
  unsigned lo = ~0u, hi = 0u;
#pragma unroll
  for (int c = 0; c < kOwn; ++c) s_count[kOwn * threadIdx.x + c] = 0u;
#pragma unroll
  for (int q = 0; q < kPer; ++q) lo = min(lo, (unsigned) (key[q] >> 32)), hi = max(hi, (unsigned) (key[q] >> 32));
  lo = wave_max_to_last(~lo), hi = wave_max_to_last(hi);
  if ((threadIdx.x & 63) == 63) s_wave[2 * wave] = lo, s_wave[2 * wave + 1] = hi;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) lo = w ? max(lo, s_wave[2 * w]) : s_wave[0], hi = w ? max(hi, s_wave[2 * w + 1]) : s_wave[1];
  lo = ~lo;
  const float scale = (float) kBuckets * __builtin_amdgcn_rcpf((float) (hi - lo) + 1.0f);
  auto place  = [&](uint64_t k) { return (float) ((unsigned) (k >> 32) - lo) * scale; };  // monotone, like its integer part
  auto bucket = [&](uint64_t k) { return min((int) place(k), kBuckets - 1); };
  auto emit   = [&](uint64_t e, int first, int end) {
    int to = first;
    for (int i = first; i < end; ++i) to += s_e[i] < e;
    point_list[start + to] = (Number) (uint32_t) e;
    if (keys_out) keys_out[start + to] = (int64_t) (((uint64_t) (uint32_t) tile << 32) | (e >> 32));
  };
  unsigned rank[kPer];
  const bool one_depth = __builtin_amdgcn_readfirstlane(hi - lo) == 0 && n > kBucketLimit;  // every entry would wait for the one counter, to no end
  if (!one_depth) {
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if ((int) threadIdx.x + 256 * q < n) rank[q] = atomicAdd(&s_count[bucket(key[q])], 1u);
  }
  __syncthreads();
  const unsigned most = one_depth ? (unsigned) n : prefix_counters<kOwn, 1>(s_count, s_wave);
  if (__builtin_amdgcn_readfirstlane(most) <= (unsigned) kBucketLimit) {
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if ((int) threadIdx.x + 256 * q < n) s_e[s_count[bucket(key[q])] + rank[q]] = key[q];
    __syncthreads();
    // in bucket order now: a wavefront's lanes look through the same few buckets and write next to each other
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int p = threadIdx.x + 256 * q;
      if (p < n) {
        const uint64_t e = s_e[p];
        const int b = bucket(e);
        emit(e, s_count[b], b + 1 < kBuckets ? (int) s_count[b + 1] : n);
      }
    }
    return true;
  }
  // A bucket is cut by its depths, or, if it holds one depth only, by the surfels' numbers, which come next in the order: over the
  // span of the segment's numbers. Any entry of a bucket names its depth, an entry with another one marks the bucket.
  unsigned* s_depth = s_wave + 16;
  unsigned* s_mixed = s_depth + kBuckets;
  unsigned id_lo = 0u, id_hi = 0u;
#pragma unroll
  for (int q = 0; q < kPer; ++q) id_lo = max(id_lo, ~(unsigned) key[q]), id_hi = max(id_hi, (unsigned) key[q]);
  id_lo = wave_max_to_last(id_lo), id_hi = wave_max_to_last(id_hi);
  if ((threadIdx.x & 63) == 63) s_wave[8 + 2 * wave] = id_lo, s_wave[9 + 2 * wave] = id_hi;
#pragma unroll
  for (int c = 0; c < kOwn; ++c) s_mixed[kOwn * threadIdx.x + c] = 0u;
#pragma unroll
  for (int q = 0; q < kPer; ++q) s_depth[bucket(key[q])] = (unsigned) (key[q] >> 32);
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) id_lo = max(id_lo, s_wave[8 + 2 * w]), id_hi = max(id_hi, s_wave[9 + 2 * w]);
  id_lo = ~id_lo;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int b = bucket(key[q]);
    if (s_depth[b] != (unsigned) (key[q] >> 32)) s_mixed[b] = 1u;
  }
  __syncthreads();
  const float id_scale = __builtin_amdgcn_rcpf((float) (id_hi - id_lo) + 1.0f);
  // part `fine` of n, 16-bit counters in the counters' words
  constexpr int kOwnFine = kPer == 1 ? 1 : kPer / 2;
  uint16_t* s_fine = (uint16_t*) s_count;
  int fine[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int b = bucket(key[q]), first = one_depth ? 0 : (int) s_count[b];
    const int held = (one_depth || b + 1 == kBuckets ? n : (int) s_count[b + 1]) - first;
    const float part = s_mixed[b] ? place(key[q]) - (float) b : (float) ((unsigned) key[q] - id_lo) * id_scale;
    fine[q] = first + min((int) (part * (float) held), max(held - 1, 0));
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kOwnFine; ++c) s_count[kOwnFine * threadIdx.x + c] = 0u;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((int) threadIdx.x + 256 * q < n) {
      const int shift = 16 * (fine[q] & 1);
      rank[q] = (atomicAdd(&s_count[fine[q] >> 1], 1u << shift) >> shift) & 0xffffu;
    }
  __syncthreads();
  if (prefix_counters<kOwnFine, 2>(s_count, s_wave) > (unsigned) kBucketLimit) return false;
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((int) threadIdx.x + 256 * q < n) s_e[s_fine[fine[q]] + rank[q]] = key[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((int) threadIdx.x + 256 * q < n) emit(key[q], s_fine[fine[q]], fine[q] + 1 < n ? (int) s_fine[fine[q] + 1] : n);
  return true;
}

// n <= kSmallSegment entries (see bucket_sort for load and kHeld), by as many a lane as they need; s_e holds kSmallSegment + kSmallSegment / 4.
template <bool kHeld, typename Load, typename Number>
__device__ __forceinline__ void sort_small_segment(int tile, int64_t start, int n, Load load, uint64_t* s_e,
                                                   Number* __restrict__ point_list, int64_t* __restrict__ keys_out) {
  auto sort = [&](auto per) {  // entries per lane
    constexpr int kPer = decltype(per)::value;
    uint64_t key[kPer];
    if (bucket_sort<kPer, kHeld>(tile, start, n, load, key, s_e, point_list, keys_out)) return;
    if constexpr (kPer == 1) {
      s_e[threadIdx.x] = (int) threadIdx.x < n ? key[0] : ~0ull;
      __syncthreads();
      merge_sort_lds(s_e, n);
      tile_sort_output<false>(tile, start, n, s_e, point_list, keys_out);
    } else {
      const int m = padded_length(n);
#pragma unroll
      for (int q = 0; q < kPer; ++q) {
        const int k = threadIdx.x + 256 * q;
        if (k < m) s_e[lds_slot<true>(k)] = k < n ? key[q] : ~0ull;
      }
      __syncthreads();
      bitonic_sort_lds<true>(s_e, m, 256);
      tile_sort_output<true>(tile, start, n, s_e, point_list, keys_out);
    }
  };
  if (n <= kMergeSegment) sort(std::integral_constant<int, 1>());
  else if (n <= 512) sort(std::integral_constant<int, 2>());
  else if (n <= 1024) sort(std::integral_constant<int, 4>());
  else sort(std::integral_constant<int, 8>());
}

// One block per tile: segments up to kSmallSegment entries are sorted in LDS by as many entries per lane as they need (the
// first loads of all are in flight together), longer ones are queued for
// tile_sort_large_kernel; empty tiles get the (0, 0) range the reference's zero-initialised output has.
// Eight wavefronts per SIMD, as many as the LDS leaves room for: 49 -> 41 us at 400k surfels 3840x2160; what spills for it is
// the second cut of segments above 1024 entries.
// `order` (optional): the blend kernels' blockIdx -> tile table, longest lists first, so that the long segments start
// sorting at once instead of wherever the image puts them in tile order (the launch ends with its slowest block).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) tile_sort_small_kernel(int64_t* __restrict__ ranges,
    const uint64_t* __restrict__ entries, int32_t* __restrict__ point_list, int64_t* __restrict__ keys_out,
    int* __restrict__ large_count, int* __restrict__ large_list, const int* __restrict__ order, int n_tiles,
    int64_t R, const int* __restrict__ kept, uint64_t pad_key) {
  __shared__ __align__(16) uint64_t s_e[kSmallSegment + kSmallSegment / 4];
  // Blocks past the tile grid (the fast path launches some): that path reserves one list position per tile of a
  // surfel's rectangle, and the positions behind the instances that passed the corner test hold the reference's padding
  // entries (key = T << 32, value = -1), which its sort leaves at the tail of the list. Written here, beside the sorts,
  // rather than by a launch of its own behind them.
  if ((int) blockIdx.x >= n_tiles) {
    const int64_t stride = (int64_t) (gridDim.x - n_tiles) * blockDim.x;
    for (int64_t o = (int64_t) *kept + (int64_t) (blockIdx.x - n_tiles) * blockDim.x + threadIdx.x; o < R; o += stride) {
      point_list[o] = -1;
      if (keys_out) keys_out[o] = (int64_t) pad_key;
    }
    return;
  }
  const int tile = order ? order[blockIdx.x] : (int) blockIdx.x;
  const int64_t start = ranges[2 * (size_t) tile];
  const int64_t len   = ranges[2 * (size_t) tile + 1] - start;
  if (len == 0) {
    if (threadIdx.x == 0) ranges[2 * (size_t) tile] = 0, ranges[2 * (size_t) tile + 1] = 0;
    return;
  }
  if (len > kSmallSegment) {
    if (threadIdx.x == 0) large_list[atomicAdd(large_count, 1)] = tile;
    return;
  }
  sort_small_segment<false>(tile, start, (int) len, [&](int i) { return entries[start + i]; }, s_e, point_list, keys_out);
}

// The first cut of bucket_sort for the n <= 1024 * kPer entries of a long segment, by a 1024-lane block. False, with nothing written,
// when a bucket holds more than 4 * kBucketLimit entries (16 times in longer segments, whose network works in global memory).
constexpr int kLargeBuckets = 4096;

template <int kPer>
__device__ __forceinline__ bool bucket_sort_large(int tile, int64_t start, int n, const uint64_t* __restrict__ entries, uint64_t* s_e,
                                                  unsigned* s_count, unsigned* s_wave, int32_t* __restrict__ point_list,
                                                  int64_t* __restrict__ keys_out) {
  constexpr int kThreads = 1024, kWaves = kThreads / kWave, kOwn = kLargeBuckets / kThreads;
  const int wave = threadIdx.x >> 6;
  uint64_t key[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) key[q] = entries[start + min((int) threadIdx.x + kThreads * q, n - 1)];
  unsigned lo = ~0u, hi = 0u;
#pragma unroll
  for (int c = 0; c < kOwn; ++c) s_count[kOwn * threadIdx.x + c] = 0u;
#pragma unroll
  for (int q = 0; q < kPer; ++q) lo = min(lo, (unsigned) (key[q] >> 32)), hi = max(hi, (unsigned) (key[q] >> 32));
  lo = wave_max_to_last(~lo), hi = wave_max_to_last(hi);
  if ((threadIdx.x & 63) == 63) s_wave[2 * wave] = lo, s_wave[2 * wave + 1] = hi;
  __syncthreads();
  lo = s_wave[0], hi = s_wave[1];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) lo = max(lo, s_wave[2 * w]), hi = max(hi, s_wave[2 * w + 1]);
  lo = ~lo;
  if (lo == hi) return false;  // one depth: every entry would wait for the one counter
  const float scale = (float) kLargeBuckets * __builtin_amdgcn_rcpf((float) (hi - lo) + 1.0f);
  auto bucket = [&](uint64_t k) { return min((int) ((float) ((unsigned) (k >> 32) - lo) * scale), kLargeBuckets - 1); };
  unsigned rank[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((int) threadIdx.x + kThreads * q < n) rank[q] = atomicAdd(&s_count[bucket(key[q])], 1u);
  __syncthreads();
  if (prefix_counters<kOwn, 1, kWaves>(s_count, s_wave) > 4u * kBucketLimit) return false;
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((int) threadIdx.x + kThreads * q < n) s_e[s_count[bucket(key[q])] + rank[q]] = key[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int p = threadIdx.x + kThreads * q;
    if (p < n) {
      const uint64_t e = s_e[p];
      const int b = bucket(e), first = (int) s_count[b], end = b + 1 < kLargeBuckets ? (int) s_count[b + 1] : n;
      int to = first;
      for (int i = first; i < end; ++i) to += s_e[i] < e;
      point_list[start + to] = (int32_t) (uint32_t) e;
      if (keys_out) keys_out[start + to] = (int64_t) (((uint64_t) (uint32_t) tile << 32) | (e >> 32));
    }
  }
  return true;
}

// A segment that does not fit the LDS, the same way, as many buckets at a time as hold at most kLargeSegment entries: the segment is read
// once to count and once for every such group.
__device__ __forceinline__ bool bucket_sort_huge(int tile, int64_t start, int64_t len, const uint64_t* __restrict__ entries, uint64_t* s_e,
                                                 unsigned* s_count, unsigned* s_wave, int32_t* __restrict__ point_list,
                                                 int64_t* __restrict__ keys_out) {
  constexpr int kThreads = 1024, kWaves = kThreads / kWave, kOwn = kLargeBuckets / kThreads;
  constexpr unsigned kLimit = 16 * kBucketLimit;
  const int wave = threadIdx.x >> 6, n = (int) len;
  unsigned lo = 0u, hi = 0u;  // lo: of the complement
  for (int p = threadIdx.x; p < n; p += kThreads) {
    const unsigned d = (unsigned) (entries[start + p] >> 32);
    lo = max(lo, ~d), hi = max(hi, d);
  }
#pragma unroll
  for (int c = 0; c < kOwn; ++c) s_count[kOwn * threadIdx.x + c] = 0u;
  lo = wave_max_to_last(lo), hi = wave_max_to_last(hi);
  if ((threadIdx.x & 63) == 63) s_wave[2 * wave] = lo, s_wave[2 * wave + 1] = hi;
  __syncthreads();
  lo = s_wave[0], hi = s_wave[1];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) lo = max(lo, s_wave[2 * w]), hi = max(hi, s_wave[2 * w + 1]);
  lo = ~lo;
  if (lo == hi) return false;
  const float scale = (float) kLargeBuckets * __builtin_amdgcn_rcpf((float) (hi - lo) + 1.0f);
  auto bucket = [&](uint64_t k) { return min((int) ((float) ((unsigned) (k >> 32) - lo) * scale), kLargeBuckets - 1); };
  for (int p = threadIdx.x; p < n; p += kThreads) atomicAdd(&s_count[bucket(entries[start + p])], 1u);
  __syncthreads();
  if (prefix_counters<kOwn, 1, kWaves>(s_count, s_wave) > kLimit) return false;
  // s_count[b]: where bucket b starts; once its group has been placed, where it ends, which is where b + 1 starts
  for (int b0 = 0, base = 0; b0 < kLargeBuckets;) {
    int b1 = kLargeBuckets;  // the last bucket whose end is still within the LDS, and one more
    for (int step = kLargeBuckets, at = b0; step >= 1; step >>= 1) {
      if (at + step < kLargeBuckets && (int) s_count[at + step] - base <= kLargeSegment) at += step;
      b1 = at;
    }
    if (n - base <= kLargeSegment) b1 = kLargeBuckets;
    const int end = b1 < kLargeBuckets ? (int) s_count[b1] : n;
    __syncthreads();
    for (int p = threadIdx.x; p < n; p += kThreads) {
      const uint64_t e = entries[start + p];
      const int b = bucket(e);
      if (b >= b0 && b < b1) s_e[atomicAdd(&s_count[b], 1u) - base] = e;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < end - base; p += kThreads) {
      const uint64_t e = s_e[p];
      const int b = bucket(e), first = b > 0 ? (int) s_count[b - 1] : 0, last = (int) s_count[b];
      int to = first;
      for (int i = first; i < last; ++i) to += s_e[i - base] < e;
      point_list[start + to] = (int32_t) (uint32_t) e;
      if (keys_out) keys_out[start + to] = (int64_t) (((uint64_t) (uint32_t) tile << 32) | (e >> 32));
    }
    __syncthreads();
    b0 = b1, base = end;
  }
  return true;
}

struct LargeSortLds {
  uint64_t e[kLargeSegment];
  unsigned count[kLargeBuckets];
  unsigned wave[2 * 1024 / kWave];
};

// A long segment by a block of 1024 lanes: up to kLargeSegment entries in LDS, by buckets or, where their depths lie too close
// together, by the sorting network; longer ones by groups of buckets, or by the network on the global array.
// Against the network, us a launch: 98k surfels 170x120 (lists of 3 to 6 thousand) 52 -> 8, 577k 228x227 108 -> 14, 2M 600x500 96 -> 15;
// lists above 16 384, 2M 160x110: 1760 (the network) -> 258.
__device__ __forceinline__ void sort_large_segment(int tile, int64_t start, int64_t len, uint64_t* __restrict__ entries, LargeSortLds& s,
                                                   int32_t* __restrict__ point_list, int64_t* __restrict__ keys_out) {
  if (len <= kLargeSegment) {
    const int n = (int) len;
    __syncthreads();  // the counters and the entries of the segment before have been read
    bool sorted;
    if (n <= 4096) sorted = bucket_sort_large<4>(tile, start, n, entries, s.e, s.count, s.wave, point_list, keys_out);
    else if (n <= 8192) sorted = bucket_sort_large<8>(tile, start, n, entries, s.e, s.count, s.wave, point_list, keys_out);
    else sorted = bucket_sort_large<16>(tile, start, n, entries, s.e, s.count, s.wave, point_list, keys_out);
    if (sorted) return;
    __syncthreads();
    const int m = padded_length(n);
    for (int k = threadIdx.x; k < m; k += 1024) s.e[k] = k < n ? entries[start + k] : ~0ull;
    __syncthreads();
    bitonic_sort_lds<false>(s.e, m, 1024);
    tile_sort_output<false>(tile, start, n, s.e, point_list, keys_out);
    __syncthreads();
  } else {
    __syncthreads();
    if (bucket_sort_huge(tile, start, len, entries, s.e, s.count, s.wave, point_list, keys_out)) return;
    uint64_t* e = entries + start;
    bitonic_sort<int64_t>(e, len, 1024, [] {
      __threadfence_block();
      __syncthreads();
    });
    tile_sort_output<false>(tile, start, (int) len, e, point_list, keys_out);
  }
}

// A few blocks walk the queue of long segments.
__global__ void __launch_bounds__(1024) tile_sort_large_kernel(const int64_t* __restrict__ ranges,
    uint64_t* __restrict__ entries, int32_t* __restrict__ point_list, int64_t* __restrict__ keys_out,
    const int* __restrict__ large_count, const int* __restrict__ large_list) {
  __shared__ LargeSortLds s;
  const int n_large = *large_count;
  for (int q = blockIdx.x; q < n_large; q += gridDim.x) {
    const int tile = large_list[q];
    const int64_t start = ranges[2 * (size_t) tile];
    sort_large_segment(tile, start, ranges[2 * (size_t) tile + 1] - start, entries, s, point_list, keys_out);
  }
}

// ---- lists of a small view, tile by tile ------------------------------------------------------------------------------
// A small view's counting, prefix, scatter and sort are four or five launches of 2 to 7 us each, most of them latency: its lists are
// formed by the tiles' own blocks instead. A block looks at every surfel's rectangle of tiles (a word each, left by the preprocess kernel:
// three instructions for whether the tile is in it), checks the keep masks of those that contain it, sorts what remains and
// leaves it in a place of its own; a second launch moves the lists together. Bound by the latency of its loads and, from some millions of
// looks on, by its instructions. Kernels, us, count, prefix, scatter and the two sorts -> gather and place: 10k surfels 256x256
// 3.8 + 4.7 + 4.7 + 3.7 + 1.7 -> 6.7 + 3.5; 25k Gaussians 639x361 4.9 + 5.9 + 6.8 + 4.1 + 1.8 -> 11 + 4.1; 50k surfels 501x403
// 4.5 + 7.2 + 6.6 + 4.6 + 1.8 -> 17 + 4.5. (Words tested by a ballot each whether or not one was in, held by the block behind barriers, one
// load ahead: 8.7, 17.6 and 29.)
// The work grows with surfels times tiles, but the others' prefix is one block's up to 1024 tiles. Views, us, so binned -> gathered:
// 5k surfels 640x480 (1200 tiles) 50 -> 42.5, 20k 54.5 -> 51.7, 25k 800x600 (1900, 47.5M looks) 62.2 -> 62.3, 30k Gaussians
// 800x600 (57M) 54.9 -> 56.3; 1024 tiles and fewer: 65k surfels 500x500 90 -> 82, 440x440 91 -> 85, 65k Gaussians 440x440 85 -> 80, one
// surfel 47 -> 44. With many surfels on few tiles those are few blocks, their lists are long, and what is longer than 2048 entries is
// looked for twice: 49 tiles 10k surfels 97.5 -> 93.4, 20k 162 -> 171, 40k 195 -> 228; 100 tiles 20k 91 -> 86, 40k 154 -> 178; 256 tiles
// 40k 91 -> 89, 65k 121 -> 125. Large surfels, up to that line: 8000 surfels 256x256, 1220 entries a tile, 255 -> 235; 60k
// 400x400, 1585 a tile and up to 5381, 470 -> 458.
constexpr int kGatherSide  = 127;    // tiles along either axis: a rectangle is four numbers of seven bits
constexpr int kGatherTiles = 2040;   // two a lane in the second launch, and eight a block: 255 blocks, and one for the schedule
constexpr int kGatherChunk = 16 * kWave;  // surfels that a wavefront looks at in one go
constexpr int kGatherHeld  = 2 * kGatherChunk;  // of them, what a wavefront can hold
constexpr int kGatherMost  = 65535;  // surfels: their numbers are held in 16 bits
constexpr int64_t kGatherLooks = 48000000;  // surfels times tiles, above 1024 tiles (see above)
constexpr int kGatherPerTile   = 200;       // surfels per tile (see above)

// Bytes of a rectangle's word: first column, 127 - last column, first row, 127 - last row. gather_word(tx, ty) less it has the upper
// bit of a byte set where the tile is on the rectangle's side of that bound.
__device__ __forceinline__ uint32_t gather_word(int tx, int ty) {
  return 0x80808080u | (uint32_t) tx | (uint32_t) (127 - tx) << 8 | (uint32_t) ty << 16 | (uint32_t) (127 - ty) << 24;
}
__device__ __forceinline__ bool gather_hit(uint32_t tile, uint32_t rect) { return ((tile - rect) & 0x80808080u) == 0x80808080u; }

// Whether the keep mask of a surfel (its rectangle contains the tile) keeps the tile: what for_each_instance<kWalkMask> visits.
__device__ __forceinline__ bool gather_keeps(uint32_t rect, uint32_t mask, int tx, int ty) {
  const int x0 = (int) (rect & 127u), y0 = (int) (rect >> 16 & 127u), w = 128 - (int) (rect >> 8 & 127u) - x0, h = 128 - (int) (rect >> 24) - y0;
  const int x = tx - x0, y = ty - y0;
  if (w * h <= kCullMaskTiles) return mask >> (y * w + x) & 1u;
  const TileWindow v = tile_window(mask, w, h);
  const int sum = x + y, diff = x - y + h - 1;
  return x >= v.x0 && x <= v.x1 && y >= v.y0 && y <= v.y1 && sum >= v.s0 && sum <= v.s1 && diff >= v.d0 && diff <= v.d1;
}

__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return (int) __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
}

// A place behind `at` (LDS) for each lane that is `on`; all lanes of a wavefront together.
__device__ __forceinline__ int gather_place(bool on, int* at) {
  const unsigned long long m = __ballot(on);
  if (m == 0ull) return 0;
  int base = 0;
  if (__lane_id() == 0) base = atomicAdd(at, (int) __popcll(m));
  return __builtin_amdgcn_readfirstlane(base) + lanes_below(m);
}

__global__ void __launch_bounds__(256) tile_gather_kernel(int P, int gx, const uint32_t* __restrict__ rects,
    const uint32_t* __restrict__ masks, const float* __restrict__ depths, uint32_t* __restrict__ counts, uint16_t* __restrict__ lists,
    SlotPublish publish) {
  constexpr int kWaves = 256 / kWave, kQuads = kGatherChunk / (4 * kWave);  // quads: of four words a lane
  __shared__ __align__(16) uint64_t s_e[kSmallSegment + kSmallSegment / 4];
  __shared__ uint16_t s_held[kWaves][kGatherHeld];  // surfels whose rectangle contains the tile
  __shared__ int s_kept;
  if (blockIdx.x == 0 && threadIdx.x < kWave) publish_slot_regions(publish);
  const int tile = blockIdx.x, ty = tile / gx, tx = tile - ty * gx, lane = __lane_id(), wave = threadIdx.x / kWave;
  const uint32_t word = gather_word(tx, ty);
  uint16_t* const held = s_held[wave];
  int n_held = 0;
  // behind the last surfel the rectangles contain no tile up to a multiple of 256, behind that another quad's are read and not looked at
  auto words = [&](int first, uint4 (&r)[kQuads]) {
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      const int at = first + 4 * kWave * q;
      r[q] = *(const uint4*) (rects + (at < P ? at : 0) + 4 * lane);
    }
  };
  constexpr int kStep = kWaves * kGatherChunk;
  uint4 r[3][kQuads];  // two goes' words are on their way
  const int begin = __builtin_amdgcn_readfirstlane(wave) * kGatherChunk;
  words(begin, r[0]), words(begin + kStep, r[1]);
  if (threadIdx.x == 0) s_kept = 0;
  __syncthreads();
  auto keep_held = [&] {  // of the surfels held, those kept, as entries to be sorted
    wave_lds_sync();
    for (int e0 = 0; e0 < n_held; e0 += kWave) {
      const int e = e0 + lane;
      const int i = held[min(e, n_held - 1)];
      const uint32_t depth = __float_as_uint(depths[i]);
      const bool kept = e < n_held && (!masks || gather_keeps(rects[i], masks[i], tx, ty));
      const int at = gather_place(kept, &s_kept);
      if (kept && at < kSmallSegment) s_e[at] = (uint64_t) depth << 32 | (uint32_t) i;
    }
    wave_lds_sync();
    n_held = 0;
  };
  auto look = [&](int first, const uint4 (&r)[kQuads]) {
    auto one = [&](uint32_t rect, int i) {
      const bool hit = gather_hit(word, rect);
      if (const unsigned long long m = __ballot(hit)) {  // one in five, or fewer
        if (hit) held[n_held + lanes_below(m)] = (uint16_t) i;
        n_held += (int) __popcll(m);
      }
    };
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      const int at = first + 4 * kWave * q;
      if (at >= P) break;
      one(r[q].x, at + 4 * lane), one(r[q].y, at + 4 * lane + 1), one(r[q].z, at + 4 * lane + 2), one(r[q].w, at + 4 * lane + 3);
    }
    if (n_held > kGatherHeld - kGatherChunk) keep_held();
  };
  for (int first = begin; first < P; first += 3 * kStep) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      if (first + u * kStep >= P) break;
      words(first + (u + 2) * kStep, r[(u + 2) % 3]);
      look(first + u * kStep, r[u]);
    }
  }
  keep_held();
  __syncthreads();
  const int n = s_kept;
  if (threadIdx.x == 0) counts[tile] = (uint32_t) n;
  if (n == 0 || n > kSmallSegment) return;  // a longer list is left to tile_place_kernel
  sort_small_segment<true>(tile, (int64_t) tile * kSmallSegment, n, [&](int i) { return s_e[i]; }, s_e, lists, nullptr);
}

// The lists one behind the other, kTiles tiles a block, and the ranges; lists of more than kSmallSegment entries are formed here.
// One block more than that where the blend kernels' schedule is to be built, the first one: it takes longest. A block takes a compute
// unit's LDS, so that there are 256 of them at most (257 took 6.2 us instead of 4.5), and no more tiles share one than have to: 65k
// surfels in 16 tiles, lists of up to 16 817 entries, four a block 961 us a view, one a block 816 (947 by the queue of long segments).
constexpr int kPlaceBlocks = 255;
template <int kTiles>
__global__ void __launch_bounds__(1024) tile_place_kernel(int P, int gx, int gy, int64_t R, const uint32_t* __restrict__ rects,
    const uint32_t* __restrict__ masks, const float* __restrict__ depths, const uint32_t* __restrict__ counts,
    const uint16_t* __restrict__ lists, int64_t* __restrict__ ranges, int32_t* __restrict__ point_list, uint64_t* __restrict__ entries,
    int* __restrict__ order_table) {
  __shared__ LargeSortLds s;
  constexpr int kLanes = 1024 / kTiles;
  __shared__ int s_end[2048];  // of the tiles' lists
  const int T = gx * gy, lane = __lane_id(), wave = threadIdx.x / kWave;
  if (order_table && blockIdx.x == 0) {
    static_assert(sizeof(TileOrderLds) <= sizeof(s.e), "the schedule's LDS fits");
    build_tile_order(gx, gy, [&](int t) { return (int64_t) counts[t]; }, order_table, order_table + kMaxOrderedTiles,
                     *reinterpret_cast<TileOrderLds*>(s.e));
    return;
  }
  const int t0 = 2 * (int) threadIdx.x, low = t0 < T ? (int) counts[t0] : 0, mine = low + (t0 + 1 < T ? (int) counts[t0 + 1] : 0);
  const int block = (int) blockIdx.x - (order_table ? 1 : 0), own = kTiles * block + (int) threadIdx.x / kLanes;  // this lane's tile
  const int k0 = threadIdx.x % kLanes;
  const uint16_t* list = lists + (size_t) min(own, T - 1) * kSmallSegment;
  const int32_t ahead[2] = {list[k0], list[k0 + kLanes]};  // whatever they are: on their way with the counts
  const int inc  = wave_scan(mine);
  if (lane == kWave - 1) s.wave[wave] = (unsigned) inc;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < 1024 / kWave; ++w) before += w < wave ? (int) s.wave[w] : 0;
  s_end[t0] = before + inc - mine + low, s_end[t0 + 1] = before + inc;
  __syncthreads();
  auto start_of = [&](int t) { return t > 0 ? s_end[t - 1] : 0; };
  int is_long = 0;
  if (own < T) {
    const int start = start_of(own), n = s_end[own] - start;
    if (k0 == 0) ranges[2 * (size_t) own] = n ? start : 0, ranges[2 * (size_t) own + 1] = n ? start + n : 0;
    if (n <= kSmallSegment) {
      auto put = [&](int k, int32_t i) {
        if (k < n && start + k < R) point_list[start + k] = i;
      };
      put(k0, ahead[0]), put(k0 + kLanes, ahead[1]);
      for (int k = k0 + 2 * kLanes; k < n; k += kLanes) put(k, list[k]);
    } else {
      is_long = 1;
    }
  }
  if (!__syncthreads_or(is_long)) return;
  for (int q = 0; q < kTiles; ++q) {
    const int t = kTiles * block + q;
    if (t >= T) return;
    const int start = start_of(t), n = s_end[t] - start, ty = t / gx, tx = t - ty * gx;
    if (n <= kSmallSegment || (int64_t) start + n > R) continue;
    const uint32_t word = gather_word(tx, ty);
    int* at = (int*) s.wave;
    __syncthreads();
    if (threadIdx.x == 0) *at = 0;
    __syncthreads();
    for (int i0 = 0; i0 < P; i0 += 1024) {
      const int i = min(i0 + (int) threadIdx.x, P - 1);
      const uint32_t rect = rects[i];
      const bool kept = i0 + (int) threadIdx.x < P && gather_hit(word, rect) && (!masks || gather_keeps(rect, masks[i], tx, ty));
      const int to = gather_place(kept, at);
      if (kept && to < n) entries[start + to] = (uint64_t) __float_as_uint(depths[i]) << 32 | (uint32_t) i;
    }
    __threadfence_block();
    sort_large_segment(t, start, n, entries, s, point_list, nullptr);
  }
}

// ---- radix sort passes ----------------------------------------------------------------------------------------------
// hist[digit * nblocks + block] = number of keys of `block` whose current digit is `digit`
__global__ void __launch_bounds__(kSortThreads) sort_histogram_kernel(int64_t R, int shift, int nblocks,
    const uint64_t* __restrict__ keys, uint32_t* __restrict__ hist) {
  __shared__ uint32_t s_hist[kRadix];
  s_hist[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t) blockIdx.x * kSortChunk;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k) {
    const int64_t idx = base + k * kSortThreads + threadIdx.x;
    if (idx < R) atomicAdd(&s_hist[(keys[idx] >> shift) & (kRadix - 1)], 1u);
  }
  __syncthreads();
  hist[(size_t) threadIdx.x * nblocks + blockIdx.x] = s_hist[threadIdx.x];
}

// One block per digit: exclusive scan of that digit's row over blocks (in place) and the digit total.
__global__ void __launch_bounds__(kScanThreads) sort_scan_rows_kernel(int nblocks, uint32_t* __restrict__ hist,
                                                                      uint32_t* __restrict__ digit_totals) {
  __shared__ uint32_t s_wave[kScanThreads / kWave];
  uint32_t* row  = hist + (size_t) blockIdx.x * nblocks;
  uint32_t carry = 0;
  for (int start = 0; start < nblocks; start += kScanThreads) {
    const int i = start + threadIdx.x;
    const uint32_t v = i < nblocks ? row[i] : 0;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<uint32_t>(v, s_wave, total);
    if (i < nblocks) row[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) digit_totals[blockIdx.x] = carry;
}

__global__ void __launch_bounds__(kSortThreads) sort_scatter_kernel(int64_t R, int shift, int nblocks,
    const uint64_t* __restrict__ keys_in, const int32_t* __restrict__ vals_in, const uint32_t* __restrict__ hist,
    const uint32_t* __restrict__ digit_totals, uint64_t* __restrict__ keys_out, int32_t* __restrict__ vals_out) {
  __shared__ uint32_t s_cnt[kSortWaves][kRadix];  // per-wave running digit counts, then per-wave global bases
  __shared__ uint32_t s_wave[kScanThreads / kWave];
  const int lane = __lane_id(), wave = threadIdx.x / kWave;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) s_cnt[w][threadIdx.x] = 0;
  // digit base = exclusive scan of digit totals (256 values, one per thread) + this block's offset inside the digit
  uint32_t total_unused;
  const uint32_t digit_base = block_exclusive_scan<uint32_t>(digit_totals[threadIdx.x], s_wave, total_unused) +
                              hist[(size_t) threadIdx.x * nblocks + blockIdx.x];
  // block_exclusive_scan ends with a barrier, so s_cnt is zeroed for everyone here.

  const int64_t wave_base = (int64_t) blockIdx.x * kSortChunk + (int64_t) wave * (kSortItems * kWave);
  uint64_t key[kSortItems];
  int32_t val[kSortItems];
  uint32_t pos[kSortItems];
  const unsigned long long lt = lanemask_lt();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wave_base + r * kWave + lane;
    const bool valid  = idx < R;
    key[r] = valid ? keys_in[idx] : 0;
    val[r] = valid ? vals_in[idx] : 0;
    const uint32_t d = (uint32_t) (key[r] >> shift) & (kRadix - 1);
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kRadixBits; ++b) {
      const unsigned long long m = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? m : ~m;
    }
    const uint32_t rank  = __popcll(peers & lt);
    const uint32_t count = __popcll(peers);
    const int leader     = __ffsll((long long) peers) - 1;
    uint32_t old = 0;
    if (valid && lane == leader) {
      old = s_cnt[wave][d];
      s_cnt[wave][d] = old + count;
    }
    old    = __shfl(old, leader < 0 ? 0 : leader, kWave);
    pos[r] = old + rank;
  }
  __syncthreads();
  {  // turn per-wave counts into per-wave global bases for digit == threadIdx.x
    uint32_t run = digit_base;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const uint32_t c = s_cnt[w][threadIdx.x];
      s_cnt[w][threadIdx.x] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wave_base + r * kWave + lane;
    if (idx < R) {
      const uint32_t d   = (uint32_t) (key[r] >> shift) & (kRadix - 1);
      const uint32_t dst = s_cnt[wave][d] + pos[r];
      keys_out[dst] = key[r];
      vals_out[dst] = val[r];
    }
  }
}

__global__ void __launch_bounds__(kWave) publish_slots_kernel(SlotPublish publish) { publish_slot_regions(publish); }

// ---- ranges -----------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) fill_zero_i64_kernel(int64_t n, int64_t* __restrict__ p) {
  const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void __launch_bounds__(256) tile_ranges_kernel(int64_t R, int num_tiles, const uint64_t* __restrict__ keys,
                                                          int64_t* __restrict__ ranges) {
  const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  const uint32_t cur = (uint32_t) (keys[i] >> 32);
  const bool cur_ok  = cur < (uint32_t) num_tiles;
  if (i == 0) {
    if (cur_ok) ranges[2 * (size_t) cur] = 0;
  } else {
    const uint32_t prev = (uint32_t) (keys[i - 1] >> 32);
    if (cur != prev) {
      if (prev < (uint32_t) num_tiles) ranges[2 * (size_t) prev + 1] = i;
      if (cur_ok) ranges[2 * (size_t) cur] = i;
    }
  }
  if (i == R - 1 && cur_ok) ranges[2 * (size_t) cur + 1] = R;
}

}  // namespace

uint32_t higher_msb(uint32_t n) {  // number of bits needed for the tile id, as gaussian_prepare.cu:32-44 computes it
  uint32_t msb = sizeof(n) * 4, step = msb;
  while (step > 1) {
    step /= 2;
    if (n >> msb) msb += step;
    else msb -= step;
  }
  if (n >> msb) msb++;
  return msb;
}

struct SortLayout {
  int nblocks;
  size_t keys0, keys1, vals_alt, hist, totals, bytes;
};

SortLayout sort_layout(int64_t R) {
  SortLayout L;
  L.nblocks = div_up(R > 0 ? R : 1, kSortChunk);
  size_t o  = 0;
  L.keys0 = o, o = align_up(o + (size_t) R * 8, 256);
  L.keys1 = o, o = align_up(o + (size_t) R * 8, 256);
  L.vals_alt = o, o = align_up(o + (size_t) R * 4, 256);
  L.hist = o, o = align_up(o + (size_t) kRadix * L.nblocks * 4, 256);
  L.totals = o, o = align_up(o + (size_t) kRadix * 4, 256);
  L.bytes = o;
  return L;
}


// Stable LSD radix sort of (key, value) pairs on key bits [0, bits). `vals_in` holds the unsorted payload (it is one of
// the two ping-pong buffers); on return the sorted payload is in `vals_out` and *sorted_keys points at the sorted keys
// (inside the workspace). The caller picks vals_in so that the last pass lands in vals_out: see sort_vals_in().
int radix_sort_pairs(int64_t R, int bits, void* workspace, int32_t* vals_out, const uint64_t** sorted_keys,
                     hipStream_t s) {
  const SortLayout L = sort_layout(R);
  char* ws          = (char*) workspace;
  uint64_t* kbuf[2] = {(uint64_t*) (ws + L.keys0), (uint64_t*) (ws + L.keys1)};
  uint32_t* hist    = (uint32_t*) (ws + L.hist);
  uint32_t* totals  = (uint32_t*) (ws + L.totals);
  const int passes  = (bits + kRadixBits - 1) / kRadixBits;
  int32_t* vbuf[2];
  vbuf[passes & 1]       = vals_out;
  vbuf[(passes & 1) ^ 1] = (int32_t*) (ws + L.vals_alt);
  for (int p = 0; p < passes; ++p) {
    const int shift = p * kRadixBits;
    const int a = p & 1, b = a ^ 1;
    hipLaunchKernelGGL(sort_histogram_kernel, dim3(L.nblocks), dim3(kSortThreads), 0, s, R, shift, L.nblocks, kbuf[a],
                       hist);
    hipLaunchKernelGGL(sort_scan_rows_kernel, dim3(kRadix), dim3(kScanThreads), 0, s, L.nblocks, hist, totals);
    hipLaunchKernelGGL(sort_scatter_kernel, dim3(L.nblocks), dim3(kSortThreads), 0, s, R, shift, L.nblocks, kbuf[a],
                       vbuf[a], hist, totals, kbuf[b], vbuf[b]);
  }
  *sorted_keys = kbuf[passes & 1];
  return passes;
}

// Where the unsorted keys / payload must be written before radix_sort_pairs(R, bits, workspace, vals_out, ...).
uint64_t* sort_keys_in(int64_t R, void* workspace) { return (uint64_t*) ((char*) workspace + sort_layout(R).keys0); }
int32_t* sort_vals_in(int64_t R, int bits, void* workspace, int32_t* vals_out) {
  const int passes = (bits + kRadixBits - 1) / kRadixBits;
  return (passes & 1) ? (int32_t*) ((char*) workspace + sort_layout(R).vals_alt) : vals_out;
}
size_t sort_workspace_bytes(int64_t R) { return sort_layout(R).bytes; }

void launch_zero_ranges(int num_tiles, int64_t* ranges, hipStream_t s) {
  hipLaunchKernelGGL(fill_zero_i64_kernel, dim3(div_up(2 * (int64_t) num_tiles, 256)), dim3(256), 0, s,
                     2 * (int64_t) num_tiles, ranges);
}
void launch_tile_ranges(int64_t R, int num_tiles, const uint64_t* sorted_keys, int64_t* ranges, hipStream_t s) {
  hipLaunchKernelGGL(tile_ranges_kernel, dim3(div_up(R, 256)), dim3(256), 0, s, R, num_tiles, sorted_keys, ranges);
}

size_t fast_bucket_bins_bytes(int P, int W, int H) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const BinsLayout bl = bins_layout(P, gx * gy);
  return bl.blocks > 0 ? bl.bytes : 0;
}

namespace {
#define FSGS_BY_WALK_MODE(IN, ...)                                     \
  do {                                                                  \
    switch ((IN).mode()) {                                              \
      case kWalkAll: { constexpr int kMode = kWalkAll; __VA_ARGS__; break; }   \
      case kWalkCorner: { constexpr int kMode = kWalkCorner; __VA_ARGS__; break; } \
      case kWalkMask: { constexpr int kMode = kWalkMask; __VA_ARGS__; break; } \
      case kWalkCornerMask: { constexpr int kMode = kWalkCornerMask; __VA_ARGS__; break; } \
    }                                                                   \
  } while (0)

// Who forms the tile ranges: the prefix kernel itself, the scatter (behind the count of a view), or tile_scan_kernel.
bool scan_in_prefix(int T, int blocks) { return T <= 1024 && blocks <= kColumn; }
bool scan_in_scatter(int T, int blocks) { return !scan_in_prefix(T, blocks) && T <= kScanTiles; }

// First part of the bucket binning, independent of the instance count: per-tile instance counts and the tile ranges
// (start, end); the header of `bins` is set (length of the long-segment queue: 0 | instances in all tiles).
// for_scatter: the scan, and with it ranges and header, may be left to the scatter (scan_in_scatter); the ranges are empty till then.
int fill_count(int P, int W, int H, const float* means2D, const int32_t* radii, const WalkInputs& in, int64_t* ranges,
               void* bins, hipStream_t s, bool for_scatter = false, const SlotPublish& publish = SlotPublish{}) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const int T  = gx * gy;
  unsigned long long* rng = (unsigned long long*) ranges;
  int* header = (int*) bins;
  const BinsLayout bl = bins_layout(P, T);
  if (bl.blocks > 0) {
    uint32_t* hist = (uint32_t*) ((char*) bins + kBinsHeader);
    uint32_t* sums = (uint32_t*) ((char*) bins + kBinsSums);
    FSGS_BY_WALK_MODE(in, {
      auto kernel = T > kNarrowTiles ? tile_hist_kernel<kMode, kMaxLdsTiles> : tile_hist_kernel<kMode, kNarrowTiles>;
      hipLaunchKernelGGL(kernel, dim3(bl.blocks), dim3(1024), 0, s, P, bl.per_block, gx, gy, (const float2*) means2D, radii, in,
                         hist, publish);
    });
    if (scan_in_prefix(T, bl.blocks)) {
      hipLaunchKernelGGL(tile_prefix_scan_kernel, dim3(1), dim3(1024), 0, s, T, bl.blocks, hist, rng, header);
    } else {
      const bool unscanned = for_scatter && scan_in_scatter(T, bl.blocks);
      hipLaunchKernelGGL(tile_prefix_kernel, dim3(div_up(T, kPrefixTiles)), dim3(kPrefixTiles * kPrefixWaves), 0, s, T,
                         bl.blocks, hist, rng, sums, header, unscanned);
      if (!unscanned)
        hipLaunchKernelGGL(tile_scan_kernel, dim3(div_up(T, 4096)), dim3(1024), 0, s, T, rng, sums, header, true);
    }
    // The tiles' totals are final here; the schedule table the blend kernels of this frame are going to use (and the per-tile
    // sorts) is built from them by an extra block of the scatter, in the second part.
  } else {
    // no room for one LDS counter per tile (or no surfels): count straight into ranges[t].y, then scan to (start, start)
    if (publish.counters) hipLaunchKernelGGL(publish_slots_kernel, dim3(1), dim3(kWave), 0, s, publish);
    launch_zero_ranges(T, ranges, s);
    if (P > 0)
      FSGS_BY_WALK_MODE(in, hipLaunchKernelGGL((tile_emit_kernel<kMode, false>), dim3(div_up(P, 256)), dim3(256), 0, s, P, gx,
                                               gy, (int64_t) 0, (const float2*) means2D, (const float*) nullptr, radii, in,
                                               rng, (uint64_t*) nullptr));
    hipLaunchKernelGGL(tile_scan_kernel, dim3(1), dim3(1024), 0, s, T, rng, (const uint32_t*) nullptr, header, false);
  }
  return check_launch("gs_prepare_count");
}

// Second part: scatter (depth bits << 32 | surfel) into the tile segments. R: what there is room for; `entries` is left as it is
// where the instances are more (tile grids within kMaxLdsTiles, whose cursors are not the ranges).
void fill_scatter(int P, int W, int H, const float* means2D, const float* depths, const int32_t* radii, const WalkInputs& in,
                  int64_t R, int64_t* ranges, void* workspace, void* bins, hipStream_t s, bool of_view = false) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const int T  = gx * gy;
  unsigned long long* rng = (unsigned long long*) ranges;
  uint64_t* entries       = sort_keys_in(R, workspace);
  const BinsLayout bl = bins_layout(P, T);
  if (bl.blocks > 0) {
    // The schedule table is built by one extra block of the scatter (the tiles' totals are final since the counting part).
    const int* order = nullptr;
    int* build       = nullptr;
    (void) defer_tile_order(gx, gy, ranges, s, &order, &build);
    // Entries that do not fit the dies' L2s (4 MB each) leave them in pieces, the smaller the more blocks write at once: LDS that
    // nobody uses keeps a second block off the compute unit. 3M surfels 1352x1014, 6M entries: 71 -> 56 us; 300k 800x800, 1.4M: 12.8 -> 13.9.
    const ScanInScatter scan = !scan_in_scatter(T, bl.blocks) ? kScanned : of_view ? kToScan : kAskHeader;
    const size_t alone = T <= kNarrowTiles && R > (int64_t) 4 << 20 ? 32768 : 0;
    FSGS_BY_WALK_MODE(in, {
      auto kernel = scan == kToScan ? tile_scatter_kernel<kMode, kNarrowTiles, kToScan>
                    : scan == kAskHeader ? tile_scatter_kernel<kMode, kNarrowTiles, kAskHeader>
                    : T > kNarrowTiles ? tile_scatter_kernel<kMode, kMaxLdsTiles, kScanned> : tile_scatter_kernel<kMode, kNarrowTiles, kScanned>;
      hipLaunchKernelGGL(kernel, dim3(bl.blocks + (build ? 1 : 0)), dim3(1024), alone, s, P, bl.per_block, gx, gy, R,
                         (const float2*) means2D, depths, radii, in, (const uint32_t*) ((const char*) bins + kBinsHeader), rng,
                         entries, build, (int*) bins);
    });
  } else {
    FSGS_BY_WALK_MODE(in, hipLaunchKernelGGL((tile_emit_kernel<kMode, true>), dim3(div_up(P, 256)), dim3(256), 0, s, P, gx, gy,
                                             R, (const float2*) means2D, depths, radii, in, rng, entries));
  }
}

// Third part: sort every segment. `R` and `workspace` as for the scatter. pad: the list positions behind the kept instances get the
// fast path's padding entries.
void fill_sort(int P, int W, int H, int64_t R, int64_t* ranges, int32_t* point_list, int64_t* sorted_keys_out, void* workspace,
               void* bins, bool pad, hipStream_t s) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  const int T  = gx * gy;
  int* header       = (int*) bins;
  uint64_t* entries = sort_keys_in(R, workspace);
  // queue of long segments: at most R / kSmallSegment tiles, kept behind the entries in the workspace
  int* large_list = (int*) ((char*) workspace + sort_layout(R).keys1);
  // The schedule table: the scatter's, or a launch of its own on the global-atomic path, whose ranges only become final with the
  // scatter.
  const int* order = nullptr;
  (void) launch_tile_order(gx, gy, ranges, s, &order);
  // with padding, 256 blocks more than tiles: they write the entries behind the kept instances
  hipLaunchKernelGGL(tile_sort_small_kernel, dim3(T + (pad ? 256 : 0)), dim3(256), 0, s, ranges, entries, point_list,
                     sorted_keys_out, header, large_list, order, T, R, (const int*) (header + 1),
                     (uint64_t) (uint32_t) T << 32);
  if (P > kSmallSegment)  // a surfel is in a tile's list once
    hipLaunchKernelGGL(tile_sort_large_kernel, dim3(256), dim3(1024), 0, s, ranges, entries, point_list, sorted_keys_out,
                       header, large_list);
}

int fill_lists(int P, int W, int H, const float* means2D, const float* depths, const int32_t* radii, const WalkInputs& in,
               int64_t R, int64_t* ranges, int32_t* point_list, int64_t* sorted_keys_out, void* workspace, void* bins,
               bool pad, hipStream_t s) {
  fill_scatter(P, W, H, means2D, depths, radii, in, R, ranges, workspace, bins, s);
  fill_sort(P, W, H, R, ranges, point_list, sorted_keys_out, workspace, bins, pad, s);
  return check_launch("gs_prepare_fill");
}
}  // namespace

int fast_bucket_fill(int P, int W, int H, const float* means2D, const float* inverse_m, const float* depths,
                     const float* opacities, const int32_t* radii, const uint32_t* keep_masks, int64_t R,
                     int64_t* ranges, int32_t* point_list, int64_t* sorted_keys_out, void* workspace, void* bins,
                     hipStream_t s) {
  const WalkInputs in{inverse_m, opacities, keep_masks};
  if (int rc = fill_count(P, W, H, means2D, radii, in, ranges, bins, s)) return rc;
  return fill_lists(P, W, H, means2D, depths, radii, in, R, ranges, point_list, sorted_keys_out, workspace, bins, true, s);
}

}  // namespace fsgs

using namespace fsgs;

FSGS_API size_t fsgs_gs_prepare_scan_workspace_bytes(int P) {
  return align_up((size_t) div_up(P > 0 ? P : 1, kScanChunk) * 8, 256);
}

namespace {
// One event per host thread marks "the instance count has been copied": waiting on it instead of on the stream lets the
// caller queue work that does not depend on the count behind the copy.
hipEvent_t count_event() {
  static thread_local hipEvent_t ev = nullptr;
  if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) ev = nullptr;
  return ev;
}
thread_local bool t_count_pending = false;  // a scan_begin of this thread has queued a copy nobody has waited for
}  // namespace

FSGS_API int fsgs_gs_prepare_scan_begin(int P, const int32_t* tiles_touched, int64_t* point_offsets, void* workspace,
                                        size_t workspace_bytes, int64_t* num_rendered_host, float* records,
                                        void* stream) {
  FSGS_REQUIRE(P >= 0 && num_rendered_host, "gs_prepare_scan: bad arguments");
  *num_rendered_host = 0;
  t_count_pending    = false;
  if (P == 0) return kOk;  // nothing is queued, nothing to wait for
  hipStream_t s = (hipStream_t) stream;
  hipEvent_t ev = count_event();
  FSGS_REQUIRE(ev != nullptr, "gs_prepare_scan: cannot create an event");
  {
    FSGS_REQUIRE(tiles_touched && point_offsets && workspace, "gs_prepare_scan: null pointer");
    if (workspace_bytes < fsgs_gs_prepare_scan_workspace_bytes(P))
      return fail(kWorkspaceSmall, "gs_prepare_scan: workspace %zu < %zu bytes", workspace_bytes,
                  fsgs_gs_prepare_scan_workspace_bytes(P));
    const int nb      = div_up(P, kScanChunk);
    int64_t* blk_sums = (int64_t*) workspace;
    hipLaunchKernelGGL(scan_block_sums_kernel, dim3(nb), dim3(kScanThreads), 0, s, P, tiles_touched, blk_sums);
    hipLaunchKernelGGL(scan_apply_kernel, dim3(nb), dim3(kScanThreads), 0, s, P, tiles_touched, blk_sums,
                       point_offsets, records);
    if (int rc = check_launch("gs_prepare_scan")) return rc;
    // The number of (surfel, tile) instances sizes the caller's output, so it has to reach the host
    // (the reference blocks for it, gaussian_prepare.cu:238-239).
    FSGS_HIP(hipMemcpyAsync(num_rendered_host, point_offsets + (P - 1), sizeof(int64_t), hipMemcpyDeviceToHost, s));
  }
  FSGS_HIP(hipEventRecord(ev, s));
  t_count_pending = true;
  return kOk;
}

FSGS_API int fsgs_gs_prepare_scan_end(void) {
  if (!t_count_pending) return kOk;
  t_count_pending = false;
  hipEvent_t ev   = count_event();
  FSGS_REQUIRE(ev != nullptr, "gs_prepare_scan: cannot create an event");
  FSGS_HIP(hipEventSynchronize(ev));
  return kOk;
}

FSGS_API int fsgs_gs_prepare_scan(int P, const int32_t* tiles_touched, int64_t* point_offsets, void* workspace,
                                  size_t workspace_bytes, int64_t* num_rendered_host, void* stream) {
  if (int rc = fsgs_gs_prepare_scan_begin(P, tiles_touched, point_offsets, workspace, workspace_bytes,
                                          num_rendered_host, nullptr, stream))
    return rc;
  return fsgs_gs_prepare_scan_end();
}

FSGS_API size_t fsgs_gs_prepare_fill_workspace_bytes(int64_t R) { return sort_layout(R).bytes; }

FSGS_API int fsgs_gs_prepare_sort_bits(int W, int H) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  return 32 + (int) higher_msb((uint32_t) (gx * gy));
}

FSGS_API size_t fsgs_gs_prepare_bins_bytes(int P, int W, int H) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  return bins_layout(P, gx * gy).bytes;
}

FSGS_API int fsgs_gs_prepare_count(int P, int W, int H, const float* means2D, const int32_t* radii, int64_t* ranges,
                                   void* bins, size_t bins_bytes, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && ranges && bins, "gs_prepare_count: bad arguments");
  FSGS_REQUIRE(P == 0 || (means2D && radii), "gs_prepare_count: null pointer");
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_prepare_count: bins %zu < %zu bytes", bins_bytes,
                fsgs_gs_prepare_bins_bytes(P, W, H));
  tile_order_invalidate((hipStream_t) stream);  // the ranges are rewritten: the blend schedule of this stream is stale
  return fill_count(P, W, H, means2D, radii, WalkInputs{}, ranges, bins, (hipStream_t) stream);
}

FSGS_API int fsgs_gs_prepare_fill_counted(int P, int W, int H, const float* means2D, const float* depths,
                                          const int32_t* radii, int64_t R, int64_t* ranges, int32_t* point_list,
                                          int64_t* sorted_keys_out, void* bins, size_t bins_bytes, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && R >= 0 && ranges && bins, "gs_prepare_fill: bad arguments");
  FSGS_REQUIRE(R < (int64_t) 0x7fffffff, "gs_prepare_fill: %lld instances exceed the 2^31-1 limit", (long long) R);
  if (R == 0 || P == 0) return kOk;  // the counting part left every range empty
  FSGS_REQUIRE(means2D && depths && radii && point_list && workspace, "gs_prepare_fill: null pointer");
  if (workspace_bytes < sort_workspace_bytes(R))
    return fail(kWorkspaceSmall, "gs_prepare_fill: workspace %zu < %zu bytes", workspace_bytes,
                sort_workspace_bytes(R));
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_prepare_fill: bins %zu < %zu bytes", bins_bytes,
                fsgs_gs_prepare_bins_bytes(P, W, H));
  return fill_lists(P, W, H, means2D, depths, radii, WalkInputs{}, R, ranges, point_list, sorted_keys_out, workspace, bins,
                   false, (hipStream_t) stream);
}

// Keep masks for the culled binning: a bit per tile of a surfel's rectangle (row-major, rectangles of at most 32 tiles;
// larger ones are kept whole), set when some pixel of the tile can blend the surfel by the blend kernels' own bound.
FSGS_API int fsgs_gs_2d_cull_masks(int P, int W, int H, const float* records, const int32_t* radii, uint32_t* masks,
                                   void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "gs_2d_cull_masks: bad sizes");
  if (P == 0) return kOk;
  FSGS_REQUIRE(records && radii && masks, "gs_2d_cull_masks: null pointer");
  FSGS_REQUIRE(((uintptr_t) records & 15) == 0, "gs_2d_cull_masks: records must be 16-byte aligned");
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  hipLaunchKernelGGL(cull_mask_kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, gx, gy,
                     (const float4*) records, radii, masks);
  return check_launch("gs_2d_cull_masks");
}

// The same for 3D Gaussians, from the tensors their preprocess leaves (gaussian_rasterize's alpha test in place of the
// surfel's).
FSGS_API int fsgs_gs_cull_masks(int P, int W, int H, const float* means2D, const float* conic_opacity,
                                const int32_t* radii, uint32_t* masks, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0, "gs_cull_masks: bad sizes");
  if (P == 0) return kOk;
  FSGS_REQUIRE(means2D && conic_opacity && radii && masks, "gs_cull_masks: null pointer");
  FSGS_REQUIRE(((uintptr_t) conic_opacity & 15) == 0 && ((uintptr_t) means2D & 7) == 0,
               "gs_cull_masks: means2D / conic_opacity must be 8 / 16-byte aligned");
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  hipLaunchKernelGGL(conic_cull_mask_kernel, dim3(div_up(P, 256)), dim3(256), 0, (hipStream_t) stream, P, gx, gy,
                     (const float2*) means2D, (const float4*) conic_opacity, radii, masks);
  return check_launch("gs_cull_masks");
}

// The two phases of the binning over the kept tiles only (masks: fsgs_gs_2d_cull_masks). A process with the culling
// switched off for debugging gets the full lists.
FSGS_API int fsgs_gs_prepare_count_culled(int P, int W, int H, const float* means2D, const int32_t* radii,
                                          const uint32_t* masks, int64_t* ranges, void* bins, size_t bins_bytes,
                                          void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && ranges && bins, "gs_prepare_count_culled: bad arguments");
  FSGS_REQUIRE(P == 0 || (means2D && radii && masks), "gs_prepare_count_culled: null pointer");
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_prepare_count_culled: bins %zu < %zu bytes", bins_bytes,
                fsgs_gs_prepare_bins_bytes(P, W, H));
  tile_order_invalidate((hipStream_t) stream);
  return fill_count(P, W, H, means2D, radii, WalkInputs{nullptr, nullptr, culling_enabled() ? masks : nullptr}, ranges, bins,
                    (hipStream_t) stream);
}

FSGS_API int fsgs_gs_prepare_fill_counted_culled(int P, int W, int H, const float* means2D, const float* depths,
                                                 const int32_t* radii, const uint32_t* masks, int64_t R,
                                                 int64_t* ranges, int32_t* point_list, int64_t* sorted_keys_out,
                                                 void* bins, size_t bins_bytes, void* workspace,
                                                 size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && R >= 0 && ranges && bins, "gs_prepare_fill_culled: bad arguments");
  FSGS_REQUIRE(R < (int64_t) 0x7fffffff, "gs_prepare_fill_culled: %lld instances exceed the 2^31-1 limit", (long long) R);
  if (R == 0 || P == 0) return kOk;
  FSGS_REQUIRE(means2D && depths && radii && masks && point_list && workspace, "gs_prepare_fill_culled: null pointer");
  if (workspace_bytes < sort_workspace_bytes(R))
    return fail(kWorkspaceSmall, "gs_prepare_fill_culled: workspace %zu < %zu bytes", workspace_bytes,
                sort_workspace_bytes(R));
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_prepare_fill_culled: bins %zu < %zu bytes", bins_bytes,
                fsgs_gs_prepare_bins_bytes(P, W, H));
  return fill_lists(P, W, H, means2D, depths, radii, WalkInputs{nullptr, nullptr, culling_enabled() ? masks : nullptr}, R,
                   ranges, point_list, sorted_keys_out, workspace, bins, false, (hipStream_t) stream);
}

// What the views call, for either kind of surfels (inverse_m and opacities: the fast ones) and Gaussians: the counting part, for
// views whose preprocess handed out the record slots (instance_slots.hpp), the scatter and the sort.
namespace {
WalkInputs view_inputs(const float* inverse_m, const float* opacities, const uint32_t* keep_masks) {
  return inverse_m ? WalkInputs{inverse_m, opacities, keep_masks}
                   : WalkInputs{nullptr, nullptr, culling_enabled() ? keep_masks : nullptr};
}
}  // namespace

FSGS_API int fsgs_gs_view_count(int P, int W, int H, const float* means2D, const float* inverse_m, const float* opacities,
                                const int32_t* radii, const uint32_t* keep_masks, uint64_t* slot_counters,
                                int32_t* slot_regions, int64_t* num_rendered_host, int64_t* ranges, void* bins,
                                size_t bins_bytes, void* stream) {
  FSGS_REQUIRE(P > 0 && W > 0 && H > 0 && ranges && bins, "gs_view_count: bad arguments");
  FSGS_REQUIRE(means2D && radii && slot_counters && num_rendered_host && (!inverse_m || (opacities && keep_masks)),
               "gs_view_count: null pointer");
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_view_count: bins %zu < %zu bytes", bins_bytes, fsgs_gs_prepare_bins_bytes(P, W, H));
  tile_order_invalidate((hipStream_t) stream);
  __atomic_store_n(num_rendered_host, (int64_t) -1, __ATOMIC_RELEASE);
  return fill_count(P, W, H, means2D, radii, view_inputs(inverse_m, opacities, keep_masks), ranges, bins, (hipStream_t) stream, true,
                    SlotPublish{(unsigned long long*) slot_counters, slot_regions, num_rendered_host});
}

FSGS_API size_t fsgs_gs_view_lists_workspace_bytes(int64_t capacity) {
  return sort_layout(capacity).keys1 + align_up((size_t) (capacity / kSmallSegment + 1) * sizeof(int), 256);  // entries, queue of long segments
}

namespace {
int check_view_lists(const char* what, int P, int W, int H, const float* means2D, const float* inverse_m, const float* depths,
                     const float* opacities, const int32_t* radii, const uint32_t* keep_masks, int64_t capacity,
                     const int64_t* ranges, const void* bins, size_t bins_bytes, const void* workspace, size_t workspace_bytes) {
  FSGS_REQUIRE(P > 0 && W > 0 && H > 0 && capacity > 0 && ranges && bins && workspace, "%s: bad arguments", what);
  FSGS_REQUIRE(capacity < (int64_t) 0x7fffffff, "%s: %lld instances exceed the 2^31-1 limit", what, (long long) capacity);
  FSGS_REQUIRE(means2D && depths && radii && (!inverse_m || (opacities && keep_masks)), "%s: null pointer", what);
  if (workspace_bytes < fsgs_gs_view_lists_workspace_bytes(capacity) || bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "%s: workspace %zu < %zu or bins %zu < %zu bytes", what, workspace_bytes,
                fsgs_gs_view_lists_workspace_bytes(capacity), bins_bytes, fsgs_gs_prepare_bins_bytes(P, W, H));
  return kOk;
}
bool scatter_can_repeat(int W, int H) {
  return (int64_t) ((W + kTile - 1) / kTile) * ((H + kTile - 1) / kTile) <= kMaxLdsTiles;
}
}  // namespace

// Tile grids beyond kMaxLdsTiles are scattered by cursors in the ranges, which allow it once: with the sort, for the count.
FSGS_API int fsgs_gs_view_scatter(int P, int W, int H, const float* means2D, const float* inverse_m, const float* depths,
                                  const float* opacities, const int32_t* radii, const uint32_t* keep_masks, int64_t capacity,
                                  int64_t* ranges, void* bins, size_t bins_bytes, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  if (int rc = check_view_lists("gs_view_scatter", P, W, H, means2D, inverse_m, depths, opacities, radii, keep_masks, capacity,
                                ranges, bins, bins_bytes, workspace, workspace_bytes))
    return rc;
  if (!scatter_can_repeat(W, H)) return kOk;
  fill_scatter(P, W, H, means2D, depths, radii, view_inputs(inverse_m, opacities, keep_masks), capacity, ranges, workspace, bins,
               (hipStream_t) stream, true);
  return check_launch("gs_view_scatter");
}

FSGS_API int fsgs_gs_view_sort(int P, int W, int H, const float* means2D, const float* inverse_m, const float* depths,
                               const float* opacities, const int32_t* radii, const uint32_t* keep_masks, int64_t R,
                               int64_t capacity, int64_t* ranges, int32_t* point_list, void* bins, size_t bins_bytes,
                               void* workspace, size_t workspace_bytes, void* stream) {
  hipStream_t s = (hipStream_t) stream;
  if (R == 0 && P > 0 && W > 0 && H > 0 && ranges) {
    launch_zero_ranges(((W + kTile - 1) / kTile) * ((H + kTile - 1) / kTile), ranges, s);
    return check_launch("gs_view_sort");
  }
  FSGS_REQUIRE(R > 0 && R <= capacity && point_list, "gs_view_sort: bad arguments (%lld instances, room for %lld)", (long long) R,
               (long long) capacity);
  if (int rc = check_view_lists("gs_view_sort", P, W, H, means2D, inverse_m, depths, opacities, radii, keep_masks, capacity, ranges,
                                bins, bins_bytes, workspace, workspace_bytes))
    return rc;
  if (!scatter_can_repeat(W, H))
    fill_scatter(P, W, H, means2D, depths, radii, view_inputs(inverse_m, opacities, keep_masks), capacity, ranges, workspace, bins, s);
  fill_sort(P, W, H, capacity, ranges, point_list, nullptr, workspace, bins, false, s);
  return check_launch("gs_view_sort");
}

namespace {
struct GatherLayout {
  size_t lists, bytes;
};
GatherLayout gather_layout(int T) {
  GatherLayout l;
  l.lists = align_up((size_t) T * sizeof(uint32_t), 256);
  l.bytes = l.lists + (size_t) T * kSmallSegment * sizeof(uint16_t);
  return l;
}
}  // namespace

FSGS_API int fsgs_gs_view_gathers(int P, int W, int H) {
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  return P > 0 && P <= kGatherMost && gx > 0 && gy > 0 && gx <= kGatherSide && gy <= kGatherSide && gx * gy <= kGatherTiles &&
         P <= kGatherPerTile * gx * gy && (gx * gy <= 1024 || (int64_t) P * gx * gy <= kGatherLooks);
}

FSGS_API size_t fsgs_gs_view_gather_bytes(int W, int H) {
  return gather_layout(((W + kTile - 1) / kTile) * ((H + kTile - 1) / kTile)).bytes;
}

FSGS_API int fsgs_gs_view_gather(int P, int W, int H, const float* depths, const uint32_t* tile_rects, const uint32_t* keep_masks,
                                 uint64_t* slot_counters, int32_t* slot_regions, int64_t* num_rendered_host, void* lists,
                                 size_t lists_bytes, void* stream) {
  FSGS_REQUIRE(fsgs_gs_view_gathers(P, W, H), "gs_view_gather: not a view for it");
  FSGS_REQUIRE(depths && tile_rects && ((uintptr_t) tile_rects & 15) == 0 && slot_counters && lists,
               "gs_view_gather: null pointer, or rectangles off a 16-byte boundary");
  if (lists_bytes < fsgs_gs_view_gather_bytes(W, H))
    return fail(kWorkspaceSmall, "gs_view_gather: lists %zu < %zu bytes", lists_bytes, fsgs_gs_view_gather_bytes(W, H));
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  tile_order_invalidate((hipStream_t) stream);
  if (num_rendered_host) __atomic_store_n(num_rendered_host, (int64_t) -1, __ATOMIC_RELEASE);
  hipLaunchKernelGGL(tile_gather_kernel, dim3(gx * gy), dim3(256), 0, (hipStream_t) stream, P, gx, tile_rects,
                     culling_enabled() ? keep_masks : nullptr, depths, (uint32_t*) lists,
                     (uint16_t*) ((char*) lists + gather_layout(gx * gy).lists),
                     SlotPublish{(unsigned long long*) slot_counters, slot_regions, num_rendered_host});
  return check_launch("gs_view_gather");
}

FSGS_API int fsgs_gs_view_place(int P, int W, int H, const float* depths, const uint32_t* tile_rects, const uint32_t* keep_masks,
                                int64_t R, int64_t* ranges, int32_t* point_list, void* lists, size_t lists_bytes, void* workspace,
                                size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(fsgs_gs_view_gathers(P, W, H) && ranges && R >= 0 && R < (int64_t) 0x7fffffff, "gs_view_place: bad arguments");
  const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
  hipStream_t s = (hipStream_t) stream;
  if (R == 0) {
    launch_zero_ranges(gx * gy, ranges, s);
    return check_launch("gs_view_place");
  }
  FSGS_REQUIRE(depths && tile_rects && point_list && lists && workspace, "gs_view_place: null pointer");
  if (lists_bytes < fsgs_gs_view_gather_bytes(W, H) || workspace_bytes < (size_t) R * sizeof(uint64_t))
    return fail(kWorkspaceSmall, "gs_view_place: lists %zu < %zu or workspace %zu < %zu bytes", lists_bytes,
                fsgs_gs_view_gather_bytes(W, H), workspace_bytes, (size_t) R * sizeof(uint64_t));
  const int* order = nullptr;
  int* build       = nullptr;
  (void) defer_tile_order(gx, gy, ranges, s, &order, &build);
  const int T = gx * gy, tiles = T <= kPlaceBlocks ? 1 : T <= 2 * kPlaceBlocks ? 2 : T <= 4 * kPlaceBlocks ? 4 : 8;
  auto kernel = tiles == 1 ? tile_place_kernel<1> : tiles == 2 ? tile_place_kernel<2> : tiles == 4 ? tile_place_kernel<4> : tile_place_kernel<8>;
  hipLaunchKernelGGL(kernel, dim3(div_up(gx * gy, tiles) + (build ? 1 : 0)), dim3(1024), 0, s, P, gx, gy, R, tile_rects,
                     culling_enabled() ? keep_masks : nullptr, depths, (const uint32_t*) lists,
                     (const uint16_t*) ((const char*) lists + gather_layout(gx * gy).lists), ranges, point_list, (uint64_t*) workspace, build);
  return check_launch("gs_view_place");
}

// Waits until the count has been written. Reading the word is all it takes as long as the stream works; a stream that
// has run dry, or failed, without writing it is an error.
FSGS_API int fsgs_gs_view_wait(const int64_t* num_rendered_host, void* stream) {
  FSGS_REQUIRE(num_rendered_host, "gs_view_wait: null pointer");
  for (unsigned spins = 1;; ++spins) {
    if (__atomic_load_n(num_rendered_host, __ATOMIC_ACQUIRE) >= 0) return kOk;
    if (spins % 65536 == 0) {
      const hipError_t e = hipStreamQuery((hipStream_t) stream);
      if (e == hipErrorNotReady) continue;
      if (__atomic_load_n(num_rendered_host, __ATOMIC_ACQUIRE) >= 0) return kOk;
      return fail(kLaunchFailure, "gs_view_wait: %s", e == hipSuccess ? "the stream ended without an instance count" : hipGetErrorString(e));
    }
    __builtin_ia32_pause();
  }
}

FSGS_API int fsgs_gs_prepare_fill(int P, int W, int H, const float* means2D, const float* depths,
                                  const int32_t* radii, const int64_t* point_offsets, int64_t R, int64_t* ranges,
                                  int32_t* point_list, int64_t* sorted_keys_out, void* bins, size_t bins_bytes,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(P >= 0 && W > 0 && H > 0 && R >= 0 && ranges, "gs_prepare_fill: bad arguments");
  FSGS_REQUIRE(R < (int64_t) 0x7fffffff, "gs_prepare_fill: %lld instances exceed the 2^31-1 limit", (long long) R);
  hipStream_t s = (hipStream_t) stream;
  tile_order_invalidate(s);  // the ranges are rewritten: the blend schedule of this stream is stale
  if (R == 0 || P == 0) {
    const int gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
    hipLaunchKernelGGL(fill_zero_i64_kernel, dim3(div_up(2 * (int64_t) gx * gy, 256)), dim3(256), 0, s,
                       2 * (int64_t) gx * gy, ranges);
    return check_launch("gs_prepare_fill(zero)");
  }
  FSGS_REQUIRE(means2D && depths && radii && point_offsets && point_list && workspace && bins,
               "gs_prepare_fill: null pointer");
  if (workspace_bytes < sort_workspace_bytes(R))
    return fail(kWorkspaceSmall, "gs_prepare_fill: workspace %zu < %zu bytes", workspace_bytes,
                sort_workspace_bytes(R));
  if (bins_bytes < fsgs_gs_prepare_bins_bytes(P, W, H))
    return fail(kWorkspaceSmall, "gs_prepare_fill: bins %zu < %zu bytes", bins_bytes,
                fsgs_gs_prepare_bins_bytes(P, W, H));
  if (int rc = fill_count(P, W, H, means2D, radii, WalkInputs{}, ranges, bins, s)) return rc;
  return fill_lists(P, W, H, means2D, depths, radii, WalkInputs{}, R, ranges, point_list, sorted_keys_out, workspace, bins,
                   false, s);
}
