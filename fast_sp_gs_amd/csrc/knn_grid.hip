// K nearest control points of many 3D queries through candidate lists per grid cell, for gfx950.
//
// Same result as knn_topk_kernel (point_ops.hip), bit for bit: squared distances dx*dx + dy*dy + dz*dz in single
// precision without contraction, ascending, equal distances by lower index. What bounds the search over all M control
// points is its vector work, 18 to 23 instructions for each of the N * M pairs; all but a few dozen control points can be
// ruled out for a whole cell of a grid over the control points at once:
//   1. knn_cell_lists_kernel: the cells of a G x G x G grid. U = a bound on the K-th nearest distance of ANY point of the
//      cell (the K-th smallest of 64 far-corner distances); the cell's list holds the control points whose nearest-corner
//      distance does not exceed U, with many queries in the order of the distances from the cell's centre (lists_in_order), else of the
//      indices. A block builds the list of one of 8 x 8 x 8 coarse cells and refines it for the (G / 8)^3 cells inside.
//   2. knn_cell_query_kernel: a lane finds its query's cell and walks the cell's list (about 38 entries for 2048 control
//      points and G = 32; in order, about 20 of them: what follows is farther from the centre than the K-th neighbour can be). The walk only keeps the K + 1 smallest keys -- the distance in 2^-20 parts of
//      the cell's bound, then the control point's number -- in a sorted register list, one v_med3_u32 per slot; the K exact
//      distances are formed again afterwards. Queries whose keys cannot separate two neighbours (distances in the same part)
//      walk again with parts of another kind if that can help (kCoarseParts); the others of these, those
//      whose cell has more than 128 candidates, or that lie outside the grid are taken by the whole wavefront one at a
//      time (64 control points per step), or all together by the search over all control points when they are many.
//      (A key of the distance's upper 25 bits and the list position costs three instructions less per candidate, but the
//      numbers have to be fetched from the list again, eight scattered loads a query: 272 us of queries at 3M x 2048, K = 8.)
// The grid planes follow the control points (density to the power 1/2, from a sample), so clusters and far outliers keep
// short lists. 3M queries x 2048 control points, K = 8: 2.43 ms for the search over all pairs, 0.145 ms a call this way
// (traced: lists 0.039, queries 0.118 to 0.129; 0.063 ms for the 324 MB of inputs and outputs alone). In the query kernel neither unit is
// full: the vector units are busy 0.74 of the time (1130 instructions per 64 queries), LDS 0.60, 0.24 in bank conflicts. With lists in
// index order and a row of results stored by each lane for itself it took 0.202 ms and 2180 instructions; in order alone 0.169, its
// memory path busy with stores of 16 bytes each; results through LDS in runs of 512 and 1024 bytes 0.152, and past the caches, which then
// keep the lists (8 MB), 0.118.
// Over all pairs -> this way, calls in a row, queries in a ball (normal): 200 000 x 512, K = 4 57 -> 21 (31) us, 50 000 x 512, K = 3 37 -> 18 (28),
// 5 000 x 512, K = 4 36 -> 6.2 (6.3).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace fsgs {
namespace {

constexpr int kListCap   = 128;   // candidates per cell
constexpr int kCoarse    = 8;     // coarse cells per axis
constexpr int kMaxPoints = 2560;  // control points a block keeps in LDS, 16 bytes each (41 of the list kernel's 72 KB at G = 32, of its 51 KB at G = 16)
constexpr int kMaxK      = 8;
constexpr int kOctantCap = 1024;  // candidates of an octant of a coarse cell
constexpr int kAhead = 4;
constexpr uint32_t kNumberBits = 0xfff;  // of a key: the control point's number, 20 bits of distance above it
static_assert(kMaxPoints + 8 <= (int) kNumberBits, "the numbers behind the last point, too");
// The distances of a key are equal parts of the cell's bound at first (coarse); where control points sit in clusters much tighter
// than their cells, all of a query's neighbours fall into the same few parts. Queries with two neighbours in one part, and that
// below this one (of 2^20), walk their list again with fine parts, which are at least four times as many there; above, equal
// distances are the rule (points on a lattice). A wavefront with kMostLanes queries in cells of kCrowded control points or more
// takes fine parts at once: they cost an instruction more per candidate, and without clusters one query in 700 would need the
// exact search. 128 clusters of 16 among 2048 control points, queries around them, 3M, K = 8, radius 0.01 / 0.001 / 0.0001, us:
// 267 / 2860 / 3150 with coarse parts only, 214 / 263 / 306 with the second walk, 204 / 209 / 207 so; a key of the float's upper
// 25 bits and the list position: 225 / 220 / 221.
constexpr uint32_t kCoarseParts = (1u << 13) * (kNumberBits + 1);
constexpr uint32_t kCrowdedBit = 0x100;  // of a cell's length
constexpr int kCrowded = 8, kMostLanes = 16;
constexpr int kBuildThreads = 512, kQueryThreads = 512;
constexpr uint32_t kLongList = 0xff;
constexpr int kFewQueries = 16384;

// Lists that the wavefront takes one by one once no more than so many of its lanes have candidates left: a lane's eight more cost
// the wavefront 180 instructions, what is left of a list about 80. A third of the candidates' steps is walked for a few lanes else.
constexpr int kFewLists = 4;

enum Scheme { kAllPairs, kAlone, kGrid16, kGrid32 };

// Which search. Measured: an all-pairs walk takes 65 ns per control point however few queries there are (a lane walks
// alone) and N * M / 4e12 s when they fill the chip; a wavefront per query 0.8 (M = 512) to 2.0 ns (M = 2048) a query;
// building the lists 9 us (G = 16, 512 control points, in order or not) to 35 us (G = 32, 2048), in order 39. With G = 16 the lists of more than 640
// control points outgrow their 128 entries; below that the finer grid pays from a million queries on. Behind the limits
// the walk over all pairs takes over at its own price: 3M normal queries, K = 4: 133 us for 2560 control points, 1550 for 2561; 2048
// control points, K = 8: 156 us, K = 9: 5940. 200 000 queries, K = 4: 60 and 187 us.
Scheme knn_scheme(int N, int M, int D, int K) {
  if (D != 3 || K > kMaxK || M > kMaxPoints || M < 96) return kAllPairs;
  if (N <= kFewQueries) return kAlone;
  if (M < 192) return kAllPairs;
  return M > 640 || N >= 1000000 ? kGrid32 : kGrid16;
}

// Whether the lists are put in the order of the distances from their cell's centre, so that a query's walk is over after half of its
// list (below). With G = 32 that costs 4 us (8 when the limits below were measured) whatever the number of queries, with G = 16 1 us; what it saves grows with the queries,
// with K and with the length of the lists, that is, with M. Past about 150 MB of results the stores past the caches, which come with
// the order (kStream), outweigh that. us a call in index order -> in this one, queries in a ball | normal (what two runs differ by: 1 to 3):
//   G = 32, K = 8, M = 2048:  500 000 59 -> 59 | 79 -> 82;  1M 81 -> 76 | 104 -> 100;  3M 183 -> 131 | 204 -> 154
//           K = 8, M = 256:   1.5M 72 -> 73 | 79 -> 83;  1.75M 76 -> 76 | 85 -> 89;  2M 84 -> 81 | 100 -> 97;  2.5M 124 -> 99 | 136 -> 114
//           K = 5, M = 400:   2.2M 71.5 -> 69.8 | 84.8 -> 82.7;  2.5M 77.8 -> 77.0 | 93.8 -> 88.8
//           K = 4, M = 400 (640): 1.7M 58.1 -> 59.7 | 68.7 -> 67.9 (62.5 -> 61.9 | 72.5 -> 71.4)
//           K = 3, M = 640 (1024): 2.1M 65.2 -> 67.4 | 78.6 -> 78.2 (70.2 -> 69.2 | 82.4 -> 81.2)
//           K = 2, 2.5M: M = 640 64.6 -> 69.6 | 76.5 -> 80.1;  1400 71.4 -> 75.3 | 89.3 -> 87.9;  2048 80.1 -> 77.3 | 100 -> 93
//           K = 1, 3M: M = 1024 67.4 -> 69.1 | 79.6 -> 81.3;  2048 78.5 -> 78.7 | 102.5 -> 97.9
//   G = 16, K = 3, M = 512: 50 000 17.8 -> 17.2 | 27.8 -> 27.1;  K = 1: 50 000 16.4 -> 16.2 | 23.2 -> 22.8;  400 000 22.0 -> 20.6 | 29.9 -> 27.7;
//           K = 1, M = 256: 120 000 15.2 -> 15.4 | 21.5 -> 21.8;  400 000 20.1 -> 19.2 | 26.7 -> 26.1
template <int kK, int kG>
constexpr bool kAlwaysOrdered = kG == 16 && kK >= 3;
template <int kK, int kG>
constexpr bool kNeverOrdered = kG == 32 && kK == 1;
template <int kK, int kG>
bool lists_in_order(int64_t N, int M) {
  if (kG == 16) return N >= 400000;
  const int64_t results = N * (kK + 2), entries = M * (kK + 2);
  if (kK == 2) return results >= 10000000 && M >= 1400;
  return results >= (entries >= 3800 ? 10000000 : 17500000);
}

// A cell. `length`: how many candidates its list holds (or kLongList) and kCrowdedBit; `scale`: what takes a squared distance to 2^32 at
// the cell's bound. Where the list is in the order of the distances from the cell's centre, byte g - 1 of the bounds, the first two of
// which are the upper half of `length`, is a lower bound, in cell_step's, on the distances from the 8 g-th entry on (the last one counts
// for what is behind it, too).
constexpr int kBounds = 10;
template <bool kOrder>
struct Cell {
  uint32_t length;
  float scale;
};
template <>
struct __attribute__((aligned(16))) Cell<true> {
  uint32_t length;
  float scale;
  uint32_t bounds[2];
};
struct GridLayout {
  int G;
  size_t planes, cells, lists, bytes;
};
GridLayout grid_layout(Scheme scheme) {
  GridLayout l{scheme == kGrid32 ? 32 : scheme == kGrid16 ? 16 : 0, 0, 0, 0, 0};
  if (l.G == 0) return l;
  const size_t cells = (size_t) l.G * l.G * l.G;
  l.planes  = 0;
  l.cells   = align_up(3 * (size_t) (l.G + 1) * 4, 256);
  l.lists   = align_up(l.cells + cells * sizeof(Cell<true>), 256);
  l.bytes   = l.lists + cells * kListCap * 2;
  return l;
}

__device__ __forceinline__ float distance2(float qx, float qy, float qz, const float4& p) {
#pragma clang fp contract(off)
  const float dx = qx - p.x, dy = qy - p.y, dz = qz - p.z;
  return (dx * dx + dy * dy) + dz * dz;
}

// A control point as the searches take it. One with a NaN is nobody's neighbour: it lies at infinity along every axis, so that
// its distance is infinite and not a NaN, which the keys would order in front of everything (the conversion makes it 0).
__device__ __forceinline__ float4 control_point(const float* __restrict__ y, int i) {
  const float a = y[3 * i], b = y[3 * i + 1], c = y[3 * i + 2];
  const bool known = a == a && b == b && c == c;
  return known ? make_float4(a, b, c, 0.0f) : make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.0f);
}

// Upper bound on the K-th smallest of the 64 lanes' non-negative values: the value's upper bits by bisection on lane masks
// (scalar work), the lower `kDrop` bits rounded up (19: at most 1/16 above the value; 0: the value itself). Infinity when
// fewer than K lanes hold a finite value.
template <int kDrop = 19>
__device__ __forceinline__ float wave_kth_bound(float v, int K) {
  const uint32_t bits = __float_as_uint(v);  // NaN compares above every finite value
  uint32_t low = 0;
#pragma unroll
  for (int b = 30; b >= kDrop; --b) {
    const uint32_t trial = low | (1u << b);
    if ((int) __popcll(wave_ballot(bits < trial)) < K) low = trial;
  }
  return low >= 0x7f800000u ? __builtin_inff() : __uint_as_float(low | ((1u << kDrop) - 1u));
}

// Squared distance of a point to the farthest / nearest point of a box.
__device__ __forceinline__ float box_far2(const float4& p, const float* lo, const float* hi) {
  const float x = fmaxf(fabsf(p.x - lo[0]), fabsf(p.x - hi[0])), y = fmaxf(fabsf(p.y - lo[1]), fabsf(p.y - hi[1])),
              z = fmaxf(fabsf(p.z - lo[2]), fabsf(p.z - hi[2]));
  return x * x + y * y + z * z;
}
__device__ __forceinline__ float box_near2(const float4& p, const float* lo, const float* hi) {
  const float x = fmaxf(fmaxf(lo[0] - p.x, p.x - hi[0]), 0.0f), y = fmaxf(fmaxf(lo[1] - p.y, p.y - hi[1]), 0.0f),
              z = fmaxf(fmaxf(lo[2] - p.z, p.z - hi[2]), 0.0f);
  return x * x + y * y + z * z;
}
// What a nearest-corner distance may reach at most: the bound widened by far more than the rounding of either side (and,
// near the underflow threshold, by an absolute amount), so that a point left out is strictly farther in single precision
// than K points of the list, whatever the query.
__device__ __forceinline__ float widened(float bound2) { return bound2 * 1.00002f + 1e-36f; }

// The unit of a cell's bounds: no entry of its list is farther from its centre than twice the root of 2^32 / scale.
__device__ __forceinline__ float cell_step(float scale) { return __builtin_amdgcn_rsqf(scale) * (2.0f * 65536.0f / 255.0f); }
__device__ __forceinline__ float cell_centre(float lo, float hi) { return 0.5f * (lo + hi); }
__device__ __forceinline__ float centre_distance(float x, float y, float z) { return __builtin_amdgcn_sqrtf(fmaf(x, x, fmaf(y, y, z * z))); }
// Infinite where its square exceeds the floats, from 1.844e19 on: an entry of a list whose K nearest are still in reach may lie there.
// As a lower bound it then says no more than this.
constexpr float kFarthest = 1.84e19f;

__device__ __forceinline__ int lanes_below(unsigned long long mask) {
  return (int) __builtin_amdgcn_mbcnt_hi((uint32_t) (mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) mask, 0u));
}

// Order-preserving 32-bit image of a float (NaN on top), and back.
__device__ __forceinline__ uint32_t ordered_bits(float v) {
  v = v == v ? fminf(fmaxf(v, -3e38f), 3e38f) : 3e38f;
  const uint32_t b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : b | 0x80000000u;
}
__device__ __forceinline__ float from_ordered_bits(uint32_t b) {
  return __uint_as_float((b & 0x80000000u) ? b & 0x7fffffffu : ~b);
}

__device__ __forceinline__ uint32_t med3_u32(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, kCtrl, 0xf, 0xf, true);
}
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kXor3 = 0x1b, kXor7 = 0x141, kXor8 = 0x128, kXor15 = 0x140;  // quad_perm, mirrors, row_ror:8
// The lane's value and that of lane l ^ 16 (l ^ 32), one in a and one in b: after the swap, of the 16-lane (32-lane) rows, a holds the
// even ones and b the odd ones (s_nop: the wait states that the compiler does not count in here).
__device__ __forceinline__ void pair16(uint32_t v, uint32_t& a, uint32_t& b) {
  a = v, b = v;
  asm("s_nop 1\n\tv_permlane16_swap_b32_e32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void pair32(uint32_t v, uint32_t& a, uint32_t& b) {
  a = v, b = v;
  asm("s_nop 1\n\tv_permlane32_swap_b32_e32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
// Bitonic network over the 64 lanes' values. A step keeps the smaller or the larger of a lane's value and its partner's: the median of
// the two and 0 or 2^32 - 1, one instruction behind the partner's value (a minimum, a maximum and a choice between them are three, and
// a mirror image across rows costs a choice more: the merges of rows run over rows of opposite directions instead).
struct WaveSort {
  uint32_t m1, m2, m4, m8, m16, m32;  // all ones in the lanes that have that bit
  __device__ __forceinline__ WaveSort() {
    const int lane = __lane_id();
    auto mask = [&](int bit) { return lane & bit ? ~0u : 0u; };
    m1 = mask(1), m2 = mask(2), m4 = mask(4), m8 = mask(8), m16 = mask(16), m32 = mask(32);
  }
  static __device__ __forceinline__ uint32_t xor4(uint32_t x) { return dpp_u32<kXor3>(dpp_u32<kXor7>(x)); }
  static __device__ __forceinline__ void keep(uint32_t& v, uint32_t other, uint32_t upper) { v = med3_u32(v, other, upper); }
  static __device__ __forceinline__ void keep16(uint32_t& v, uint32_t upper) {
    uint32_t a, b;
    pair16(v, a, b);
    v = med3_u32(a, b, upper);
  }
  static __device__ __forceinline__ void keep32(uint32_t& v, uint32_t upper) {
    uint32_t a, b;
    pair32(v, a, b);
    v = med3_u32(a, b, upper);
  }
  // `down`: all ones in the rows that are to descend
  __device__ __forceinline__ void below4(uint32_t& v, uint32_t down) const { keep(v, dpp_u32<kXor2>(v), m2 ^ down), keep(v, dpp_u32<kXor1>(v), m1 ^ down); }
  __device__ __forceinline__ void below16(uint32_t& v, uint32_t down) const {
    keep(v, dpp_u32<kXor8>(v), m8 ^ down), keep(v, xor4(v), m4 ^ down), below4(v, down);
  }
  __device__ __forceinline__ void below64(uint32_t& v) const { keep32(v, m32), keep16(v, m16), below16(v, 0u); }
  __device__ __forceinline__ void ascending(uint32_t& v) const {
    keep(v, dpp_u32<kXor1>(v), m1 ^ m16);
    keep(v, dpp_u32<kXor3>(v), m2 ^ m16), keep(v, dpp_u32<kXor1>(v), m1 ^ m16);
    keep(v, dpp_u32<kXor7>(v), m4 ^ m16), below4(v, m16);
    keep(v, dpp_u32<kXor15>(v), m8 ^ m16), keep(v, xor4(v), m4 ^ m16), below4(v, m16);
    keep16(v, m16 ^ m32), below16(v, m32);
    below64(v);
  }
  // of 128 values, the lower ones to v
  __device__ __forceinline__ void ascending(uint32_t& v, uint32_t& w) const {
    w = ~w;
    ascending(v), ascending(w);
    const uint32_t down = ~w;  // descending
    w = max(v, down), v = min(v, down);
    below64(v), below64(w);
  }
};

// Of the 64 lanes: all get the least (largest); a lane gets the sum (the largest) of its own and the lanes' below it.
template <bool kMost>
__device__ __forceinline__ float wave_extreme(float v) {
  auto of = [](float a, float b) { return kMost ? fmaxf(a, b) : fminf(a, b); };
  auto partner = [&](auto ctrl) { return __uint_as_float(dpp_u32<decltype(ctrl)::value>(__float_as_uint(v))); };
  v = of(v, partner(std::integral_constant<int, kXor1>())), v = of(v, partner(std::integral_constant<int, kXor2>()));
  v = of(v, partner(std::integral_constant<int, kXor7>())), v = of(v, partner(std::integral_constant<int, kXor15>()));
  uint32_t a, b;
  pair16(__float_as_uint(v), a, b);
  pair32(__float_as_uint(of(__uint_as_float(a), __uint_as_float(b))), a, b);
  return of(__uint_as_float(a), __uint_as_float(b));
}
template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ float dpp_or(float v, float otherwise) {  // `otherwise` where no lane of the row (no such row) is read
  return __uint_as_float((uint32_t) __builtin_amdgcn_update_dpp((int) __float_as_uint(otherwise), (int) __float_as_uint(v), kCtrl, kRows, 0xf, false));
}
constexpr int kShiftRow = 0x110, kShiftWave = 0x138, kLastOfRow = 0x142, kLastOfHalf = 0x143;  // row_shr, wave_shr:1, row_bcast:15 and :31
__device__ __forceinline__ float wave_running_sum(float v) {
  v += dpp_or<kShiftRow + 1>(v, 0.0f), v += dpp_or<kShiftRow + 2>(v, 0.0f), v += dpp_or<kShiftRow + 4>(v, 0.0f);
  v += dpp_or<kShiftRow + 8>(v, 0.0f), v += dpp_or<kLastOfRow, 0xa>(v, 0.0f), v += dpp_or<kLastOfHalf, 0xc>(v, 0.0f);
  return v;
}
__device__ __forceinline__ float wave_running_max(float v) {
  v = fmaxf(v, dpp_or<kShiftRow + 1>(v, v)), v = fmaxf(v, dpp_or<kShiftRow + 2>(v, v)), v = fmaxf(v, dpp_or<kShiftRow + 4>(v, v));
  v = fmaxf(v, dpp_or<kShiftRow + 8>(v, v)), v = fmaxf(v, dpp_or<kLastOfRow, 0xa>(v, v)), v = fmaxf(v, dpp_or<kLastOfHalf, 0xc>(v, v));
  return v;
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float((uint32_t) __builtin_amdgcn_readlane((int) __float_as_uint(v), lane));
}

constexpr float kRim = 0.5f;  // parts of the sample's extent

template <int kG>
struct PlaneLds {
  static constexpr int kSamples = 128;
  float sorted[3][kSamples], along[3][kSamples];
  float plane[3][kG + 1];
  float least[kG > 16 ? 3 : 1][8], most[kG > 16 ? 3 : 1][8];  // of the control points near the sample, per wavefront
};

// The grid planes, from 128 sampled control points per axis (256 cost 6 us more and make the lists no shorter): sorted by
// counting ranks, inner planes at equal steps of the accumulated square root of the gaps (cells shrink with density, but slower
// than quantiles would). Coordinates far outside the others are moved in first, for a gap of a thousand times the others' extent
// would take three quarters of the planes: to half the extent of the sample without its eight outermost on either side, or, where
// most of it lies in one spot (a flat scene), to the extent without the outermost one. The outermost planes lie a tenth of the
// sample's extent beyond it. With many queries (G = 32) they lie beyond all control points within half of its extent, too: a
// query outside the grid costs as much as 30 inside, and there was one in every wavefront (3M normal queries, 2048 normal
// control points); two more planes on either side divide that margin, which a sample's gaps know nothing of: its cells would have
// lists of more than 128. Control points still farther out are left to the far search: the cells in front of the gap would have
// such lists, for every query at the rim. 3M x 2048, K = 8, us, with planes beyond all control points and nothing moved in -> so:
// no outlier 219 -> 219, one at 10 (1000) times the deviation 295 -> 219 (534 -> 220), in the sample 2775 -> 224; normal points
// times exp(normal) 1786 -> 930; points nine tenths of which lie in a plane 324 -> 315.
// Every block computes the planes for itself instead of waiting for another launch: 4.4 us of the list kernel at G = 32, 1.9 at G = 16. A
// wavefront per axis sorts the samples in its registers and sums over its lanes; ranks counted over LDS by all threads, sums by shuffles
// and a barrier behind each step took 6.6 and 4.2.
template <int kG>
__device__ __forceinline__ void make_planes(const float4* s_y, int M, PlaneLds<kG>& s) {
  constexpr int S = PlaneLds<kG>::kSamples, kSpare = kG > 16 ? 2 : 0;
  static_assert(S == 2 * kWave);
  const int t = threadIdx.x, a = t >> 6, lane = t & 63;  // a wavefront per axis, two samples to a lane
  float along = 0.0f;
  if (a < 3) {
    const WaveSort sort;
    uint32_t key[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int j = h * kWave + lane;
      const float4 p = s_y[(int) ((int64_t) j * M / S)];
      key[h] = (ordered_bits(a == 0 ? p.x : a == 1 ? p.y : p.z) & ~(uint32_t) (S - 1)) | (uint32_t) j;
    }
    sort.ascending(key[0], key[1]);
    float v = from_ordered_bits(key[0] & ~(uint32_t) (S - 1)), w = from_ordered_bits(key[1] & ~(uint32_t) (S - 1));
    const float low8 = lane_value(v, 8), low1 = lane_value(v, 1), high8 = lane_value(w, kWave - 9), high1 = lane_value(w, kWave - 2);
    const float inner = high8 - low8, outer = high1 - low1;
    const bool even   = inner > 0.125f * outer;
    const float rim   = even ? kRim * inner : outer > 0.0f ? outer : __builtin_inff();
    const float least = (even ? low8 : low1) - rim, most = (even ? high8 : high1) + rim;
    v = fminf(fmaxf(v, least), most), w = fminf(fmaxf(w, least), most);
    s.sorted[a][lane] = v, s.sorted[a][kWave + lane] = w;
    const float sum  = wave_running_sum(sqrtf(fmaxf(v - dpp_or<kShiftWave>(v, v), 0.0f)));
    const float half = lane_value(sum, kWave - 1);
    const float rest = half + wave_running_sum(sqrtf(fmaxf(w - dpp_or<kShiftWave>(w, lane_value(v, kWave - 1)), 0.0f)));
    s.along[a][lane] = sum, s.along[a][kWave + lane] = rest;
    along = lane_value(rest, kWave - 1);
  }
  if constexpr (kSpare > 0) {
    __syncthreads();
    float lo[3], hi[3], least[3], most[3];  // the sample's extent and kRim of it on either side
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float rim = kRim * (s.sorted[c][S - 1] - s.sorted[c][0]);
      lo[c] = s.sorted[c][0] - rim, hi[c] = s.sorted[c][S - 1] + rim;
      least[c] = __builtin_inff(), most[c] = -__builtin_inff();
    }
    for (int i = t; i < M; i += kBuildThreads) {
      const float4 p    = s_y[i];
      const float at[3] = {p.x, p.y, p.z};
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (at[c] >= lo[c] && at[c] <= hi[c]) least[c] = fminf(least[c], at[c]), most[c] = fmaxf(most[c], at[c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      least[c] = wave_extreme<false>(least[c]), most[c] = wave_extreme<true>(most[c]);
      if (lane == 0) s.least[c][a] = least[c], s.most[c][a] = most[c];
    }
    __syncthreads();
  } else if (a < 3) {
    wave_lds_sync();
  }
  if (a < 3) {
    const float lo = s.sorted[a][0], hi = s.sorted[a][S - 1], ext = hi - lo;
    float first = lo - 0.1f * ext, last = hi + 0.1f * ext;
    if constexpr (kSpare > 0) {
      float least = s.least[a][0], most = s.most[a][0];
#pragma unroll
      for (int w = 1; w < kBuildThreads / kWave; ++w) least = fminf(least, s.least[a][w]), most = fmaxf(most, s.most[a][w]);
      first = fminf(least, first) - 0.05f * ext, last = fmaxf(most, last) + 0.05f * ext;
    }
    float v = -3e38f;
    if (lane <= kG) {
      const int i = lane;
      if (i == 0) v = first;
      else if (i == kG) v = last;
      else if (i < 1 + kSpare) v = lo + (i == 1 ? 0.55f : 0.25f) * (first - lo);
      else if (i > kG - 1 - kSpare) v = hi + (i == kG - 1 ? 0.55f : 0.25f) * (last - hi);
      else {
        const float target = along * ((float) (i - 1 - kSpare) / (float) (kG - 2 - 2 * kSpare));
        int j = 0;  // last sample whose accumulated step does not exceed the target
#pragma unroll
        for (int step = S / 2; step >= 1; step >>= 1)
          if (s.along[a][j + step] <= target) j += step;
        const int n = min(j + 1, S - 1);
        const float w = s.along[a][n] - s.along[a][j];
        v = s.sorted[a][j] + (s.sorted[a][n] - s.sorted[a][j]) * (w > 0.0f ? (target - s.along[a][j]) / w : 0.0f);
      }
    }
    v = wave_running_max(v);  // ascending whatever the roundings did
    if (lane <= kG) s.plane[a][lane] = v;
  }
  __syncthreads();
}

// One block per coarse cell, one wavefront per octant of it: with G = 16 an octant is a cell, with G = 32 it is narrowed
// down once more for its eight cells. 26 M vector instructions (98 us) when the cells were taken from the coarse list
// directly: the coarse lists at the rim of the cloud hold nearly everything. A wavefront forms the lists of its cells side by
// side: a candidate is read once for all of them, its distances to their faces are formed once per axis and half of the octant,
// and nothing waits in a chain of eight (cells one after the other: 25 us of the kernel's 51).
// With G = 32 the octants' lists come from the coarse one the same way: a wavefront looks at an eighth of it for all octants instead of
// at all of it for its own. Bound by the instructions of four wavefronts per SIMD; a median wavefront and the last one (rim of the
// cloud, 1300 candidates of 2048 in the coarse list) of 2048 control points, K = 8, in order, us: control points 1.5, planes 4.4 (5.4),
// coarse list 2.3 (3.4), octants 4.5 (7.8), reach of the cells 2.4 (4.0), lists 2.2 (4.3), order 6.3 (7.5). The kernel, by the steps of
// the sort from three instructions to one, of the planes and of the octants: 46 -> 43 -> 41 -> 39 us, not in order 39.3 -> 37.1 -> 35.1,
// G = 16 with 512 control points 11.9 -> 9.3.
template <int kG, bool kOrder>
__global__ void __launch_bounds__(kBuildThreads) knn_cell_lists_kernel(int M, int K, const float* __restrict__ y,
    float* __restrict__ planes, Cell<kOrder>* __restrict__ cells, uint16_t* __restrict__ lists) {
  constexpr int kWaves = kBuildThreads / kWave;
  static_assert(kWaves == 8, "a wavefront per octant");
  __shared__ float4 s_y[kMaxPoints];
  __shared__ uint16_t s_sub[kMaxPoints];  // the coarse cell's list
  __shared__ uint16_t s_octant[kG > 16 ? kWaves : 1][kG > 16 ? kOctantCap : 1];
  __shared__ PlaneLds<kG> s;
  __shared__ float s_bound[kWaves];
  __shared__ int s_count[kWaves];
  __shared__ uint32_t s_far[kG > 16 ? kWaves : 1][kWave];  // an octant's squared distances to control points' farthest corners, the least of each lane
  __shared__ int s_share[kG > 16 ? kWaves : 1][kWaves];    // what a wavefront has found for each octant
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (kG > 16) s_far[wave][lane] = 0x7f800000u;
  for (int i = t; i < M; i += kBuildThreads) s_y[i] = control_point(y, i);
  __syncthreads();
  make_planes<kG>(s_y, M, s);
  if (blockIdx.x == 0)
    for (int e = t; e < 3 * (kG + 1); e += kBuildThreads) planes[e] = (&s.plane[0][0])[e];

  constexpr int kSub = kG / kCoarse;  // cells per axis inside a coarse cell
  const int cc[3] = {(int) blockIdx.x % kCoarse, (int) blockIdx.x / kCoarse % kCoarse, (int) blockIdx.x / (kCoarse * kCoarse)};
  float lo[3], hi[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) lo[a] = s.plane[a][cc[a] * kSub], hi[a] = s.plane[a][(cc[a] + 1) * kSub];
  // coarse list: every wavefront bounds the K-th distance from the control points it looks at, the best bound counts
  float least = __builtin_inff();
  for (int i = t; i < M; i += kBuildThreads) least = fminf(least, box_far2(s_y[i], lo, hi));
  const float bound = wave_kth_bound(least, K);
  if (lane == 0) s_bound[wave] = bound;
  __syncthreads();
  float limit = s_bound[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) limit = fminf(limit, s_bound[w]);
  limit = widened(limit);
  constexpr int kSteps = kMaxPoints / (kWaves * kWave);  // of 64 control points, a wavefront
  static_assert(kMaxPoints % (kWaves * kWave) == 0);
  const int per = ((M + kWaves - 1) / kWaves + kWave - 1) / kWave * kWave;  // a contiguous share per wavefront: index order
  const int first = wave * per, last = min(M, first + per);
  unsigned long long near[kSteps];
  int n_mine = 0;
#pragma unroll
  for (int u = 0; u < kSteps; ++u) {
    const int i = first + u * kWave + lane;
    near[u] = 0ull;
    if (first + u * kWave < last) near[u] = wave_ballot(i < last) & wave_ballot(box_near2(s_y[min(i, M - 1)], lo, hi) <= limit);
    n_mine += __popcll(near[u]);
  }
  if (lane == 0) s_count[wave] = n_mine;
  __syncthreads();
  int at = 0, n_sub = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) at += s_count[w];
    n_sub += s_count[w];
  }
#pragma unroll
  for (int u = 0; u < kSteps; ++u) {
    if (near[u] >> lane & 1ull) s_sub[at + lanes_below(near[u])] = (uint16_t) (first + u * kWave + lane);
    at += __popcll(near[u]);
  }
  __syncthreads();

  constexpr int kIn = kSub / 2;  // cells per axis inside an octant
  const int corner[3] = {cc[0] * kSub + (wave & 1) * kIn, cc[1] * kSub + ((wave >> 1) & 1) * kIn,
                         cc[2] * kSub + (wave >> 2) * kIn};
  const uint16_t* from = s_sub;
  int n_from = n_sub;
  if constexpr (kG > 16) {
    // The octants' lists, from the coarse one: a wavefront looks at its share of that for all eight octants side by side (as for the
    // cells below), not at all of it for its own.
    constexpr int kHalves = 2;
    float face[3][kHalves + 1];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int h = 0; h <= kHalves; ++h) face[a][h] = s.plane[a][cc[a] * kSub + h * kIn];
    const int share = ((n_sub + kWaves - 1) / kWaves + kWave - 1) / kWave * kWave, begin = wave * share, end = min(n_sub, begin + share);
    float least_far[kWaves];
#pragma unroll
    for (int c = 0; c < kWaves; ++c) least_far[c] = __builtin_inff();
    for (int i0 = begin; i0 < end; i0 += kWave) {
      const float4 p    = s_y[s_sub[min(i0 + lane, end - 1)]];
      const float at[3] = {p.x, p.y, p.z};
      float f[3][kHalves];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int h = 0; h < kHalves; ++h) {
          const float d = fmaxf(fabsf(at[a] - face[a][h]), fabsf(at[a] - face[a][h + 1]));
          f[a][h] = i0 + lane < end ? d * d : __builtin_inff();
        }
#pragma unroll
      for (int c = 0; c < kWaves; ++c) least_far[c] = fminf(least_far[c], (f[0][c & 1] + f[1][c >> 1 & 1]) + f[2][c >> 2]);
    }
    if (begin < end) {
#pragma unroll
      for (int c = 0; c < kWaves; ++c) atomicMin(&s_far[c][lane], __float_as_uint(least_far[c]));
    }
    __syncthreads();
    const float mine = widened(wave_kth_bound(__uint_as_float(s_far[wave][lane]), K));
    if (lane == 0) s_bound[wave] = mine;
    __syncthreads();
    float within[kWaves];
#pragma unroll
    for (int c = 0; c < kWaves; ++c) within[c] = s_bound[c];
    uint32_t in[kSteps];  // bit c: within reach of octant c
    int count[kWaves];
#pragma unroll
    for (int c = 0; c < kWaves; ++c) count[c] = 0;
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int i0 = begin + u * kWave;
      in[u] = 0u;
      if (i0 >= end) continue;
      const float4 p    = s_y[s_sub[min(i0 + lane, end - 1)]];
      const float at[3] = {p.x, p.y, p.z};
      float f[3][kHalves];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int h = 0; h < kHalves; ++h) {
          const float d = fmaxf(fmaxf(face[a][h] - at[a], at[a] - face[a][h + 1]), 0.0f);
          f[a][h] = d * d;
        }
      const unsigned long long there = wave_ballot(i0 + lane < end);
#pragma unroll
      for (int c = 0; c < kWaves; ++c) {
        const bool near = (f[0][c & 1] + f[1][c >> 1 & 1]) + f[2][c >> 2] <= within[c];
        in[u] |= near ? 1u << c : 0u;
        count[c] += (int) __popcll(there & wave_ballot(near));
      }
      if (i0 + lane >= end) in[u] = 0u;
    }
    if (lane == 0) {
#pragma unroll
      for (int c = 0; c < kWaves; ++c) s_share[wave][c] = count[c];
    }
    __syncthreads();
    int place[kWaves];
#pragma unroll
    for (int c = 0; c < kWaves; ++c) place[c] = 0;
    n_from = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
#pragma unroll
      for (int c = 0; c < kWaves; ++c)
        if (w < wave) place[c] += s_share[w][c];
      n_from += s_share[w][wave];
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      if (begin + u * kWave >= end) continue;
      const uint16_t number = s_sub[min(begin + u * kWave + lane, end - 1)];
#pragma unroll
      for (int c = 0; c < kWaves; ++c) {
        const unsigned long long m = wave_ballot((in[u] >> c & 1u) != 0u);
        const int pos = place[c] + lanes_below(m);
        if ((in[u] >> c & 1u) && pos < kOctantCap) s_octant[c][pos] = number;
        place[c] += (int) __popcll(m);
      }
    }
    __syncthreads();
    from = s_octant[wave];
  }
  constexpr int kTogether = kIn > 1 ? 2 : kAhead;
  constexpr int kCells = kIn * kIn * kIn;  // c: half of the octant along x in bit 0, along y in bit 1, along z in bit 2
  float edge[3][kIn + 1];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int h = 0; h <= kIn; ++h) edge[a][h] = s.plane[a][corner[a] + h];
  // an octant with too many candidates: its cells have long lists, too
  const bool too_many = kG > 16 && n_from > kOctantCap;
  if (too_many) n_from = 0;
  float reach[kCells];
  {
    float least_far[kCells];
#pragma unroll
    for (int c = 0; c < kCells; ++c) least_far[c] = __builtin_inff();
#pragma unroll kTogether
    for (int i0 = 0; i0 < n_from; i0 += kWave) {
      const float4 p    = s_y[from[min(i0 + lane, n_from - 1)]];
      const float at[3] = {p.x, p.y, p.z};
      float f[3][kIn];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int h = 0; h < kIn; ++h) {
          const float d = fmaxf(fabsf(at[a] - edge[a][h]), fabsf(at[a] - edge[a][h + 1]));
          f[a][h] = i0 + lane < n_from ? d * d : __builtin_inff();
        }
#pragma unroll
      for (int c = 0; c < kCells; ++c)
        least_far[c] = fminf(least_far[c], (f[0][c % kIn] + f[1][c / kIn % kIn]) + f[2][c / (kIn * kIn)]);
    }
#pragma unroll
    for (int c = 0; c < kCells; ++c) reach[c] = widened(wave_kth_bound(least_far[c], K));
  }
  int n[kCells], inside[kCells];  // candidates, and how many of them lie in the cell itself
  uint16_t* list[kCells];
#pragma unroll
  for (int c = 0; c < kCells; ++c) {
    n[c] = 0, inside[c] = 0;
    list[c] = lists + (size_t) (((corner[2] + c / (kIn * kIn)) * kG + corner[1] + c / kIn % kIn) * kG + corner[0] + c % kIn) * kListCap;
  }
  for (int i0 = 0; i0 < n_from; i0 += kWave) {
    const int i       = from[min(i0 + lane, n_from - 1)];
    const float4 p    = s_y[i];
    const float at[3] = {p.x, p.y, p.z};
    float f[3][kIn];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int h = 0; h < kIn; ++h) {
        const float d = fmaxf(fmaxf(edge[a][h] - at[a], at[a] - edge[a][h + 1]), 0.0f);
        f[a][h] = d * d;
      }
    const unsigned long long there = wave_ballot(i0 + lane < n_from);
    float d2[kCells], nearest = __builtin_inff();
#pragma unroll
    for (int c = 0; c < kCells; ++c) d2[c] = (f[0][c % kIn] + f[1][c / kIn % kIn]) + f[2][c / (kIn * kIn)], nearest = fminf(nearest, d2[c]);
    if (there & wave_ballot(nearest == 0.0f)) {
#pragma unroll
      for (int c = 0; c < kCells; ++c) inside[c] += (int) __popcll(there & wave_ballot(d2[c] == 0.0f));
    }
#pragma unroll
    for (int c = 0; c < kCells; ++c) {
      const unsigned long long m = there & wave_ballot(d2[c] <= reach[c]);
      const int pos = n[c] + lanes_below(m);
      if ((m >> lane & 1ull) && pos < kListCap) list[c][pos] = (uint16_t) i;
      n[c] += (int) __popcll(m);
    }
  }
  // The lists again, to be put in order (ranks counted over LDS instead of the networks: 14 us more): an entry or two per lane, all of them on their way together.
  constexpr int kEntries = kOrder ? kListCap / kWave : 1;
  uint32_t held[kCells][kEntries];
  if constexpr (kOrder) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#pragma unroll
    for (int c = 0; c < kCells; ++c)
#pragma unroll
      for (int h = 0; h < kEntries; ++h) held[c][h] = kWave * h + lane < min(n[c], kListCap) ? list[c][kWave * h + lane] : 0u;
  }
  // the walk takes eight entries at a time: the rest of the last eight is the point at infinity, number M
  Cell<kOrder> cell[kCells];
  const WaveSort sort;
#pragma unroll
  for (int c = 0; c < kCells; ++c) {
    const bool fits = !too_many && n[c] <= kListCap && reach[c] < 3e38f;
    if (fits && lane < 8 && n[c] + lane < (n[c] + 7) / 8 * 8) list[c][n[c] + lane] = (uint16_t) M;
    // the K nearest of any query of the cell are nearer than `reach`: their parts stay below 2^32, the others' may saturate
    cell[c] = Cell<kOrder>{fits ? (uint32_t) n[c] | (inside[c] >= kCrowded ? kCrowdedBit : 0u) : kLongList, fminf(4294967296.0f / reach[c], 3e38f)};
    if constexpr (kOrder) {
      if (!fits || n[c] <= 8) continue;
      uint32_t key[kEntries];
#pragma unroll
      for (int h = 0; h < kEntries; ++h) {
        const float4 p = s_y[held[c][h]];
        const float d  = centre_distance(p.x - cell_centre(edge[0][c % kIn], edge[0][c % kIn + 1]),
                                         p.y - cell_centre(edge[1][c / kIn % kIn], edge[1][c / kIn % kIn + 1]),
                                         p.z - cell_centre(edge[2][c / (kIn * kIn)], edge[2][c / (kIn * kIn) + 1]));
        key[h] = kWave * h + lane < n[c] ? (__float_as_uint(d) & ~kNumberBits) | held[c][h] : ~0u;
      }
      if (n[c] > kWave) sort.ascending(key[0], key[1]);
      else sort.ascending(key[0]);
      const float per_step = 0.9999f * __builtin_amdgcn_rcpf(cell_step(cell[c].scale));  // rounded down, by far more than either side's rounding
      uint32_t bound[kEntries];
#pragma unroll
      for (int h = 0; h < kEntries; ++h) {
        if (kWave * h + lane < n[c]) list[c][kWave * h + lane] = (uint16_t) (key[h] & kNumberBits);
        // (of a place past the end, a NaN, any)
        bound[h] = (uint32_t) fminf(fminf(__uint_as_float(key[h] & ~kNumberBits), kFarthest) * per_step, 255.0f);
      }
      auto at = [&](int g) { return (uint32_t) __builtin_amdgcn_readlane(bound[8 * g / kWave], 8 * g % kWave); };
#pragma unroll
      for (int g = 1; g <= kBounds; ++g) {
        uint32_t& word = g <= 2 ? cell[c].length : cell[c].bounds[(g - 3) / 4];
        word |= at(g) << (g <= 2 ? 8 * g + 8 : (g - 3) % 4 * 8);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kCells; ++c)
    if (lane == 0) cells[(list[c] - lists) / kListCap] = cell[c];
}

__device__ __forceinline__ uint32_t and_or_b32(uint32_t a, uint32_t mask, uint32_t b) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(b));
  return r;
}

// v >= 0 cut to a whole number, 2^32 - 1 from 2^32 on (the conversion in C++ is undefined there)
__device__ __forceinline__ uint32_t saturated_u32(float v) {
  uint32_t r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// The upper 20 bits of a key, with anything below them: of a squared distance times the cell's scale. Coarse: equal parts of the
// cell's bound. Fine: an exponent of five bits and 15 bits behind it, for neighbours that are much nearer than the bound.
template <bool kFine>
__device__ __forceinline__ uint32_t distance_part(float scaled) {
  if constexpr (!kFine) return saturated_u32(scaled);
  constexpr float kBelow = 4294967040.0f;  // the largest float below 2^32
  return (__float_as_uint(__builtin_amdgcn_fmed3f(scaled, 1.0f, kBelow)) << 4) - (0x3f800000u << 4);
}

template <int kK>
__device__ __forceinline__ void store_result(float* __restrict__ dist2, int64_t* __restrict__ index, int n,
                                             const float (&d)[kK], const int (&i)[kK]) {
  float* od   = dist2 + (size_t) n * kK;
  int64_t* oi = index + (size_t) n * kK;
  if constexpr (kK % 4 == 0) {
#pragma unroll
    for (int k = 0; k < kK; k += 4) *(float4*) (od + k) = make_float4(d[k], d[k + 1], d[k + 2], d[k + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < kK; ++k) od[k] = d[k];
  }
  if constexpr (kK % 2 == 0) {
#pragma unroll
    for (int k = 0; k < kK; k += 2) *(longlong2*) (oi + k) = make_longlong2(i[k], i[k + 1]);
  } else {
#pragma unroll
    for (int k = 0; k < kK; ++k) oi[k] = i[k];
  }
}

// The same for 64 queries from n0 on, a lane each, through `lds` (128 words of the wavefront's): rows of 16 to 64 bytes a lane apart make
// a store of every 64 bytes they lie in, whole runs of 512 and 1024 bytes do not. kStream: past the caches.
template <int kK, bool kStream>
__device__ __forceinline__ void store_results(float* __restrict__ dist2, int64_t* __restrict__ index, int n0,
                                              const float (&d)[kK], const int (&i)[kK], float* lds) {
  typedef float Distances __attribute__((ext_vector_type(2)));
  typedef int64_t Numbers __attribute__((ext_vector_type(2)));
  constexpr int kQueries = kK > 4 ? 16 : 32, kPairs = kQueries * kK / 2;
  static_assert(kPairs <= kWave);
  const int lane = __lane_id();
#pragma unroll
  for (int c = 0; c < kWave / kQueries; ++c) {
    const size_t at = ((size_t) n0 + c * kQueries) * kK + 2 * lane;
    const bool mine = lane / kQueries == c, stores = lane < kPairs;
    float* const to = lds + lane % kQueries * kK;
    wave_lds_sync();
    if (mine)
#pragma unroll
      for (int k = 0; k < kK; ++k) to[k] = d[k];
    wave_lds_sync();
    const Distances v = ((const Distances*) lds)[lane];
    if constexpr (kStream) { if (stores) __builtin_nontemporal_store(v, (Distances*) (dist2 + at)); }
    else if (stores) *(Distances*) (dist2 + at) = v;
    wave_lds_sync();
    if (mine)
#pragma unroll
      for (int k = 0; k < kK; ++k) to[k] = __int_as_float(i[k]);
    wave_lds_sync();
    const int2 w = ((const int2*) lds)[lane];
    if constexpr (kStream) { if (stores) __builtin_nontemporal_store(Numbers{w.x, w.y}, (Numbers*) (index + at)); }
    else if (stores) *(Numbers*) (index + at) = Numbers{w.x, w.y};
  }
  wave_lds_sync();
}

// kG == 0: no grid, a wavefront per query. kOrder: the lists are in the order of their cells' centre distances.
template <int kK, int kG, bool kOrder>
__global__ void __launch_bounds__(kQueryThreads) __attribute__((amdgpu_waves_per_eu(8, 8)))
knn_cell_query_kernel(int N, int M, const float* __restrict__ x,
    const float* __restrict__ y, const float* __restrict__ planes, const Cell<kOrder>* __restrict__ cells,
    const uint16_t* __restrict__ lists, float* __restrict__ dist2, int64_t* __restrict__ index) {
  // 60 MB of results and more would push the lists out of the caches; fewer are left there for whoever asked
  constexpr bool kStream = kOrder && kG > 16;
  // Short rows behind long walks are stored by their lanes: by way of LDS, lists in index order, K = 3 took 1.2 % longer (1M x 1024
  // 47.5 -> 48.9 us), K = 4 as long; K = 8 3 % less (800 000 x 700 59.9 -> 56.6).
  constexpr bool kRuns = kK > (kOrder ? 2 : 4);
  // a query alone costs a wavefront about 20 M / 64 + 300 instructions, the all-pairs walk about 20 M for all 64
  const int max_alone = 20 * M / (20 * M / 64 + 300);
  constexpr int kWaves = kQueryThreads / kWave;
  extern __shared__ __attribute__((aligned(16))) char s_dyn[];
  float4* s_y = (float4*) s_dyn;  // [M + 8], the last eight at infinity
  __shared__ float s_plane[3][kG + 1];
  __shared__ __attribute__((aligned(16))) float s_cand[kWaves][2 * kWave];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  float* const s_cand_d = s_cand[wave];  // distances and numbers of a query's candidates, or results on their way out
  int* const s_cand_i   = (int*) &s_cand[wave][kWave];
  for (int i = t; i < M; i += kQueryThreads) s_y[i] = control_point(y, i);
  if (t < 8) s_y[M + t] = make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.0f);
  if (kG > 0)
    for (int e = t; e < 3 * (kG + 1); e += kQueryThreads) (&s_plane[0][0])[e] = planes[e];
  __syncthreads();

  // The whole wavefront on one query: a bound on the K-th distance from the lanes' nearest control points, the control
  // points within it collected in index order, ranked against each other. False when more than 64 are within the bound.
  auto alone = [&](int n, float qx, float qy, float qz) -> bool {
    float least = __builtin_inff();
    for (int i = lane; i < M; i += kWave) least = fminf(least, distance2(qx, qy, qz, s_y[i]));
    auto collect = [&](float bound) {
      int count = 0;
      for (int i0 = 0; i0 < M; i0 += kWave) {
        const int i   = min(i0 + lane, M);
        const float d = distance2(qx, qy, qz, s_y[i]);
        const unsigned long long m = wave_ballot(i < M) & wave_ballot(d <= bound) & wave_ballot(d < __builtin_inff());
        const int pos = count + lanes_below(m);
        if (((m >> lane) & 1ull) && pos < kWave) s_cand_d[pos] = d, s_cand_i[pos] = i;
        count += (int) __popcll(m);
      }
      return count;
    };
    int count = collect(wave_kth_bound(least, kK));
    if (count > kWave) count = collect(wave_kth_bound<0>(least, kK));  // a far query: nearly everything at one distance
    if (count > kWave) return false;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float d = lane < count ? s_cand_d[lane] : __builtin_inff();
    const int i   = lane < count ? s_cand_i[lane] : -1;
    int rank = 0;
    for (int c = 0; c < count; ++c) {
      const float o = s_cand_d[c];
      rank += (int) (o < d) | ((int) (o == d) & (int) (c < lane));
    }
    if (lane >= count) rank = lane;  // slots nobody fills
    if (rank < kK) {
      dist2[(size_t) n * kK + rank] = lane < count ? d : -1.0f;
      index[(size_t) n * kK + rank] = i;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return true;
  };
  // Every lane on its own query, over all control points in index order.
  auto all_pairs = [&](float qx, float qy, float qz, float (&bd)[kK], int (&bi)[kK]) {
#pragma unroll
    for (int k = 0; k < kK; ++k) bd[k] = __builtin_inff(), bi[k] = -1;
    for (int m0 = 0; m0 < M; m0 += 8) {
      float d[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) d[u] = distance2(qx, qy, qz, s_y[m0 + u]);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (d[u] < bd[kK - 1]) {
          bool before[kK];
#pragma unroll
          for (int k = 0; k < kK; ++k) before[k] = d[u] < bd[k];
#pragma unroll
          for (int k = kK - 1; k >= 1; --k) {
            bd[k] = __builtin_amdgcn_fmed3f(bd[k - 1], d[u], bd[k]);
            const int stay = before[k] ? m0 + u : bi[k];
            bi[k] = before[k - 1] ? bi[k - 1] : stay;
          }
          bd[0] = before[0] ? d[u] : bd[0], bi[0] = before[0] ? m0 + u : bi[0];
        }
    }
#pragma unroll
    for (int k = 0; k < kK; ++k)
      if (bi[k] < 0) bd[k] = -1.0f;
  };

  if constexpr (kG == 0) {
    for (int n = blockIdx.x * kWaves + wave; n < N; n += gridDim.x * kWaves) {
      const float qx = x[3 * (size_t) n], qy = x[3 * (size_t) n + 1], qz = x[3 * (size_t) n + 2];
      if (!alone(n, qx, qy, qz)) {
        float bd[kK];
        int bi[kK];
        all_pairs(qx, qy, qz, bd, bi);
        if (lane == 0) store_result<kK>(dist2, index, n, bd, bi);
      }
    }
  } else {
    for (int n0 = (blockIdx.x * kWaves + wave) * kWave; n0 < N; n0 += gridDim.x * kQueryThreads) {
      const int n     = n0 + lane;
      const bool live = n < N;
      const size_t at = 3 * (size_t) (live ? n : N - 1);
      const float q[3] = {x[at], x[at + 1], x[at + 2]};
      bool inside = live;
      int cell = 0;
      float off[3];  // from the cell's centre
#pragma unroll
      for (int a = 2; a >= 0; --a) {
        int i = 0;
#pragma unroll
        for (int step = kG / 2; step >= 1; step >>= 1)
          if (s_plane[a][i + step] <= q[a]) i += step;
        inside = inside && q[a] >= s_plane[a][0] && q[a] < s_plane[a][kG];  // false for NaN
        cell   = cell * kG + i;
        off[a] = q[a] - cell_centre(s_plane[a][i], s_plane[a][i + 1]);
      }
      const Cell<kOrder> here = inside ? cells[cell] : Cell<kOrder>{kLongList, 0.0f};
      const float far_off = kOrder ? 1.0001f * centre_distance(off[0], off[1], off[2]) : 0.0f, step = kOrder ? cell_step(here.scale) : 0.0f;
      const bool listed = (here.length & 0xffu) != kLongList;
      const uint16_t* list = lists + (size_t) cell * kListCap;
      uint32_t key[kK + 1];
      auto insert = [&](uint32_t nk) {
#pragma unroll
        for (int k = kK; k >= 1; --k) key[k] = med3_u32(key[k - 1], nk, key[k]);
        key[0] = min(key[0], nk);
      };
      // The smallest keys of the first n_list candidates and of those that are there already.
      auto walk = [&](auto fine, int n_list) {
        auto key_of = [&](uint32_t i, float qx, float qy, float qz, float scale) {
          return and_or_b32(distance_part<decltype(fine)::value>(distance2(qx, qy, qz, s_y[i]) * scale), ~kNumberBits, i);
        };
        uint4 next = n_list > 0 ? *(const uint4*) list : make_uint4(0, 0, 0, 0);
        int c = 0;
        unsigned long long longer;
        uint32_t now_bounds = here.length >> 16, next_bounds = 0u, last_bounds = 0u;
        if constexpr (kOrder) next_bounds = here.bounds[0], last_bounds = here.bounds[1];
        for (;; c += 8) {
          // An entry at distance d from the centre is at least d - far_off away: past the last one that can be among the smallest
          // keys the list is over.
          if (kOrder && c > 0) {
            const float least = fmaxf(fmaf((float) (now_bounds & 255u), step, -far_off), 0.0f);
            const uint32_t part = distance_part<decltype(fine)::value>(least * least * here.scale);
            if (part > (key[kK] | kNumberBits)) n_list = min(n_list, c);
            if (c == 16) now_bounds = next_bounds;
            else if (c == 48) now_bounds = last_bounds;
            else if (c < 8 * kBounds) now_bounds >>= 8;
          }
          longer = wave_ballot(c < n_list);
          if (__popcll(longer) <= kFewLists) break;
          if (c < n_list) {
            const uint4 now = next;
            if (c + 8 < n_list) next = *(const uint4*) (list + c + 8);
            const uint32_t w[4] = {now.x, now.y, now.z, now.w};
#pragma unroll
            for (int j = 0; j < 8; ++j)
              insert(key_of((j & 1) ? (w[j >> 1] >> 16) : (w[j >> 1] & 0xffffu), q[0], q[1], q[2], here.scale));
          }
        }
        while (longer) {  // what is left of a few long lists: the whole wavefront on one, a candidate per lane
          const int l = __builtin_ctzll(longer);
          longer &= longer - 1;
          const int count = __builtin_amdgcn_readlane(n_list, l), its_cell = __builtin_amdgcn_readlane(cell, l);
          const uint16_t* its_list = lists + (size_t) its_cell * kListCap;
          auto its = [&](float v) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l)); };
          const float qx = its(q[0]), qy = its(q[1]), qz = its(q[2]), scale = its(here.scale);
          for (int e = c; e < count; e += kWave) {
            const uint32_t nk = key_of(its_list[min(e + lane, count - 1)], qx, qy, qz, scale);
            unsigned long long nearer = wave_ballot(e + lane < count) & wave_ballot(nk < (uint32_t) __builtin_amdgcn_readlane(key[kK], l));
            while (nearer) {
              const uint32_t v = __builtin_amdgcn_readlane(nk, __builtin_ctzll(nearer));
              nearer &= nearer - 1;
              insert(lane == l ? v : ~0u);
            }
          }
        }
      };
#pragma unroll
      for (int k = 0; k <= kK; ++k) key[k] = 0xffffffffu;
      const int n_list = listed ? (int) (here.length & 0xffu) : 0;
      // most queries in cells with many control points: fine parts at once
      const bool fine_first = __popcll(wave_ballot(listed && (here.length & kCrowdedBit))) >= kMostLanes;
      if (fine_first) walk(std::true_type(), n_list);
      else walk(std::false_type(), n_list);
      // neighbours in the same part are not in a known order; where the parts saturate (there are not K points at a finite
      // distance, or the bound is next to nothing) nothing is known
      auto same_part = [&](uint32_t below) {
        bool same = false;
#pragma unroll
        for (int k = 0; k < kK; ++k) same |= (key[k] ^ key[k + 1]) <= kNumberBits && key[k] < below;
        return same;
      };
      bool same = same_part(~0u);
      if (!fine_first && wave_ballot(same)) {
        const bool again = listed && same_part(kCoarseParts);
        if (wave_ballot(again)) {
#pragma unroll
          for (int k = 0; k <= kK; ++k) key[k] = again ? 0xffffffffu : key[k];
          walk(std::true_type(), again ? n_list : 0);
          same = same_part(~0u);
        }
      }
      const bool unknown = !listed || same || key[kK - 1] >= ~kNumberBits;
      float bd[kK];
      int bi[kK];
#pragma unroll
      for (int k = 0; k < kK; ++k) {
        bi[k] = unknown ? M : (int) (key[k] & kNumberBits);
        bd[k] = distance2(q[0], q[1], q[2], s_y[bi[k]]);
      }
      if (kRuns && wave_ballot(live && !unknown) == ~0ull) {
        if constexpr (kRuns) store_results<kK, kStream>(dist2, index, n0, bd, bi, s_cand_d);
      } else if (live && !unknown) {
        store_result<kK>(dist2, index, n, bd, bi);
      }

      unsigned long long rest = wave_ballot(live && unknown), together = 0ull;
      if (__popcll(rest) > max_alone) together = rest, rest = 0ull;
      while (rest) {
        const int l = __builtin_ctzll(rest);
        rest &= rest - 1;
        if (!alone(n0 + l, __shfl(q[0], l, kWave), __shfl(q[1], l, kWave), __shfl(q[2], l, kWave))) together |= 1ull << l;
      }
      if (together) {
        all_pairs(q[0], q[1], q[2], bd, bi);
        if ((together >> lane) & 1ull) store_result<kK>(dist2, index, n, bd, bi);
      }
    }
  }
}

template <int kK, int kG, bool kOrder>
void launch_query(int N, int M, const float* x, const float* y, const GridLayout& l, char* ws, float* dist2,
                  int64_t* index, hipStream_t s) {
  const size_t lds = 16 * (size_t) (M + 8);
  // blocks take the queries in strides, so that the control points are staged once for many; two rounds of the four
  // blocks that fit on a compute unit (one round 259 us, two 248, four and more 248 at 3M x 2048)
  const int per_block = kG > 0 ? kQueryThreads : kQueryThreads / kWave;
  const int blocks = std::min(div_up(N, per_block), 256 * 8);
  hipLaunchKernelGGL((knn_cell_query_kernel<kK, kG, kOrder>), dim3(blocks), dim3(kQueryThreads), lds, s, N, M, x, y,
                     (const float*) (ws + l.planes), (const Cell<kOrder>*) (ws + l.cells), (const uint16_t*) (ws + l.lists),
                     dist2, index);
}

template <int kK>
int launch_grid_knn(Scheme scheme, int N, int M, const float* x, const float* y, float* dist2, int64_t* index, char* ws,
                    hipStream_t s) {
  const GridLayout l = grid_layout(scheme);
  auto launch = [&](auto grid, auto order) {
    constexpr int kG = decltype(grid)::value;
    constexpr bool kOrder = decltype(order)::value;
    hipLaunchKernelGGL((knn_cell_lists_kernel<kG, kOrder>), dim3(kCoarse * kCoarse * kCoarse), dim3(kBuildThreads), 0, s, M, kK, y,
                       (float*) (ws + l.planes), (Cell<kOrder>*) (ws + l.cells), (uint16_t*) (ws + l.lists));
    launch_query<kK, kG, kOrder>(N, M, x, y, l, ws, dist2, index, s);
  };
  auto launch_grid = [&](auto grid) {
    constexpr int kG = decltype(grid)::value;
    if constexpr (kAlwaysOrdered<kK, kG>) launch(grid, std::true_type());
    else if constexpr (kNeverOrdered<kK, kG>) launch(grid, std::false_type());
    else if (lists_in_order<kK, kG>(N, M)) launch(grid, std::true_type());
    else launch(grid, std::false_type());
  };
  if (scheme == kAlone) launch_query<kK, 0, false>(N, M, x, y, l, ws, dist2, index, s);
  else if (scheme == kGrid16) launch_grid(std::integral_constant<int, 16>());
  else launch_grid(std::integral_constant<int, 32>());
  return check_launch("knn_topk");
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API int fsgs_knn_topk(int N, int M, int D, int K, const float* x, const float* y, float* dist2, int64_t* index,
                           void* stream);

FSGS_API size_t fsgs_knn_topk_workspace_bytes(int N, int M, int D, int K) {
  return N > 0 && M > 0 ? grid_layout(knn_scheme(N, M, D, K)).bytes : 0;
}

FSGS_API int fsgs_knn_topk_ws(int N, int M, int D, int K, const float* x, const float* y, float* dist2, int64_t* index,
                              void* workspace, size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(N >= 0 && M > 0 && D > 0 && K > 0 && x && y && dist2 && index, "knn_topk: bad arguments");
  const Scheme scheme = knn_scheme(N, M, D, K);
  const bool aligned  = (((uintptr_t) dist2 | (uintptr_t) index) & 15) == 0;  // rows are stored in 16-byte pieces
  if (N == 0 || scheme == kAllPairs || !aligned) return fsgs_knn_topk(N, M, D, K, x, y, dist2, index, stream);
  if (workspace_bytes < grid_layout(scheme).bytes || (grid_layout(scheme).bytes > 0 && !workspace))
    return fail(kWorkspaceSmall, "knn_topk: workspace %zu < %zu bytes", workspace_bytes, grid_layout(scheme).bytes);
  char* ws = (char*) workspace;
  hipStream_t s = (hipStream_t) stream;
  switch (K) {
    case 1: return launch_grid_knn<1>(scheme, N, M, x, y, dist2, index, ws, s);
    case 2: return launch_grid_knn<2>(scheme, N, M, x, y, dist2, index, ws, s);
    case 3: return launch_grid_knn<3>(scheme, N, M, x, y, dist2, index, ws, s);
    case 4: return launch_grid_knn<4>(scheme, N, M, x, y, dist2, index, ws, s);
    case 5: return launch_grid_knn<5>(scheme, N, M, x, y, dist2, index, ws, s);
    case 6: return launch_grid_knn<6>(scheme, N, M, x, y, dist2, index, ws, s);
    case 7: return launch_grid_knn<7>(scheme, N, M, x, y, dist2, index, ws, s);
    default: return launch_grid_knn<8>(scheme, N, M, x, y, dist2, index, ws, s);
  }
}
