// Where the gradient records of a (surfel, tile) instance go, and how many instances a view has.
//
// A surfel's instances take consecutive record slots in the order of the tiles of its rectangle. Two ways of handing the
// slots out:
//  * the inclusive prefix scan of tiles_touched (the reference's point_offsets), two kernels of their own;
//  * by regions: the preprocess kernel's block b (256 surfels) takes its slots from region b % 64 with one atomic on that
//    region's counter, so a surfel's offset inside its region is known while its record is written, and no scan, no copy
//    of the count and no second pass over the records is needed (15 us at 300k surfels, 110 us at 3M: the scan's kernel
//    that stored 3M offsets into 80-byte records alone took 91). The regions' first slots follow from the 64 counters
//    afterwards (publish_slot_regions, run by a block of the next kernel), which also hands the instance count to the
//    host. Which block comes first inside a region varies from run to run, the sums do not: a surfel's records are always
//    its own, added in tile order.
// Where the preprocess kernel itself hands the count to the host (ViewOutputs::host_count), a 65th adds up the regions.
// 64 counters keep the atomics on one address few (5 at 300k surfels, 180 at 3M); they are served one after the other.
#pragma once
#include "common.hpp"

namespace fsgs {

constexpr int kSlotRegions = 64;
constexpr int kSlotBlockBits = 8;  // the preprocess kernels' block: 256 surfels

struct SlotSource {
  const int64_t* scan = nullptr;     // [P] inclusive prefix scan, or
  const int32_t* offset = nullptr;   // [P] offset inside the surfel's region,
  const int32_t* region = nullptr;   // [64] first slot of each region,
  const int32_t* tiles = nullptr;    // [P] instances of the surfel
};

__device__ __forceinline__ int slot_region(int i) { return (i >> kSlotBlockBits) & (kSlotRegions - 1); }

// First record slot of a surfel.
__device__ __forceinline__ int64_t slot_first(const SlotSource& s, int i) {
  if (s.region) return (int64_t) s.offset[i] + s.region[slot_region(i)];
  return i > 0 ? s.scan[i - 1] : 0;
}

__device__ __forceinline__ void slot_span(const SlotSource& s, int i, int64_t& first, int& count) {
  if (s.region) {
    first = (int64_t) s.offset[i] + s.region[slot_region(i)];
    count = s.tiles[i];
  } else {
    first = i > 0 ? s.scan[i - 1] : 0;
    count = (int) (s.scan[i] - first);
  }
}

// First part, one call by all 256 lanes of the block: lane-ordered prefix of `count` over the block. `s_wave`: four words
// of LDS. Holds a barrier.
__device__ __forceinline__ int slots_in_block(int count, int* s_wave, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = count;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int up = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += up;
  }
  if (lane == kWave - 1) s_wave[wave] = inc;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int v = s_wave[w];
    if (w < wave) before += v;
    total += v;
  }
  return before + inc - count;
}

// What a view through the native host path asks of a preprocess kernel on top (all optional): the region counters, the
// surfel's first record slot inside its block's region, and the visibility as a byte.
struct ViewOutputs {
  unsigned long long* counters = nullptr;
  int32_t* slot_offsets = nullptr;
  uint8_t* visible = nullptr;
  bool windows = false;  // no backward follows: keep masks of large rectangles may be windows (cull_window)
  float* color_derivs = nullptr;  // [P, 9], for the backward; only where the coefficients' rows are complete (wave_row_floats)
  int64_t* host_count = nullptr;  // pinned host memory: the instance count, as soon as it is known; the counters are 65 then
  uint32_t* tile_rects = nullptr; // [P, up to a multiple of 256] tile_rect_word; grids of at most 127 x 127 tiles
};

// Thread 0 of a block of the preprocess kernel adds the block's instances to its region's counter (`added`: what was there before, of use
// much later). With a host_count the counters count the blocks, too, above their sums: the last block of a region adds the region's
// sum to one counter more, and the last region's block has the instances of the view, while most of the kernel is still to come.
// A small view's binning is over before the host, told by the next kernel, has launched what needs the count: 10k surfels 256x256
// 50 -> 47 us a view.
constexpr int kSlotBlocksShift = 40;
constexpr unsigned long long kSlotSum = (1ull << kSlotBlocksShift) - 1;
__device__ __forceinline__ unsigned long long add_slots(const ViewOutputs& view, int total) {
  return atomicAdd(&view.counters[blockIdx.x & (kSlotRegions - 1)],
                   (unsigned long long) total + (view.host_count ? 1ull << kSlotBlocksShift : 0ull));
}
// In two steps, so that the second counter's answer is not waited for between them.
struct SlotSums {
  unsigned long long sum = 0, before = 0;  // sum: of the region, where this is its last block
  bool last = false;
  __device__ __forceinline__ void add(const ViewOutputs& view, unsigned long long added, int total) {
    const int region = blockIdx.x & (kSlotRegions - 1), blocks = ((int) gridDim.x - region + kSlotRegions - 1) / kSlotRegions;
    last = view.host_count && (int) (added >> kSlotBlocksShift) + 1 == blocks;
    if (!last) return;
    sum    = (added & kSlotSum) + (unsigned long long) total;
    before = atomicAdd(&view.counters[kSlotRegions], sum + (1ull << kSlotBlocksShift));
  }
  __device__ __forceinline__ void publish(const ViewOutputs& view) const {
    if (!last || (int) (before >> kSlotBlocksShift) + 1 != min((int) gridDim.x, kSlotRegions)) return;
    view.counters[kSlotRegions] = 0ull;
    __hip_atomic_store(view.host_count, (int64_t) ((before & kSlotSum) + sum), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

// A rectangle of tiles as a word (ViewOutputs::tile_rects): first column, 127 - last column, first row, 127 - last row.
constexpr uint32_t kNoTiles = 0x7f7f7f7fu;
__device__ __forceinline__ uint32_t tile_rect_word(const TileRect& r) {
  return (uint32_t) r.x0 | (uint32_t) (128 - r.x1) << 8 | (uint32_t) r.y0 << 16 | (uint32_t) (128 - r.y1) << 24;
}

// What the kernel behind the preprocess hands on: see above. `counters` nullptr: nothing to do.
struct SlotPublish {
  unsigned long long* counters = nullptr;  // [64], zeroed again
  int32_t* region = nullptr;               // [64] or nullptr
  int64_t* host_count = nullptr;           // pinned host memory, or nullptr
};

// One wavefront.
__device__ __forceinline__ void publish_slot_regions(const SlotPublish& p) {
  const int lane = threadIdx.x & 63;
  const unsigned long long mine = p.counters[lane] & kSlotSum;
  unsigned long long inc = mine;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const unsigned long long up = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += up;
  }
  if (p.region) p.region[lane] = (int32_t) (inc - mine);
  p.counters[lane] = 0ull;
  if (p.host_count && lane == kWave - 1) __hip_atomic_store(p.host_count, (int64_t) inc, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace fsgs
