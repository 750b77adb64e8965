// Fused SSIM map and its backward for gfx950.
//
// Reference behaviour reproduced: fast_2d_gs/_C/src/other/structural_similarity.cu:187-277 (forward kernel), :279-338
// (backward kernel), :340-380 (host entries): separable 11-tap Gaussian (sigma 1.5, the literal weights of :11-21), zero
// padding, per channel; the forward also returns dm/dmu1, dm/dsigma1^2, dm/dsigma12 for the backward.
//
// The reference convolves one quantity at a time through a shared scratchpad (five passes and ~25 barriers per channel).
// Here a wavefront is on its own: its lanes are 64 columns of one plane, of which 54 become outputs of 7 rows. A lane reads its
// column's 17 pixels of both images straight into registers, filters the five moments (I1, I1^2, I2, I2^2, I1 I2) down the
// column while they come in, and hands them over in LDS one moment after the other; nine lanes a row then form six neighbouring
// outputs each along the row. No barrier, no staged halo, and the channels of a tile on wavefronts of their own, so that
// 3x800x800 is 5175 independent wavefronts. Rows of 118 words keep the 8-byte reads (9 lanes x 6 words a row) off each other's
// banks. Bound by vector issue (about 1000 instructions a wavefront) and the maps' traffic.
// 3x800x800 in loss form, forward 27 -> 18 us, backward 22 -> 13.5 (blocks of 32x32 outputs with the 42x42 halo of both images
// and the moments in LDS, two barriers a channel, the three channels one after the other); 3x1080x1920 64 -> 43 with the sum of the
// partial losses, 54 -> 33; 3x667x1001 27 -> 22, 20 -> 16.
#include "common.hpp"

#include <algorithm>
#include <atomic>
#include <initializer_list>

namespace fsgs {
namespace {

constexpr int kRadius   = 5;
constexpr int kLaneOut  = 6, kRowLanes = 9;                 // along a row: outputs of a lane, lanes
constexpr int kOutCols  = kLaneOut * kRowLanes;             // 54 of the wavefront's 64 columns
constexpr int kOutRows  = 7, kInRows = kOutRows + 2 * kRadius;
constexpr int kLineWords = 118;                             // of a row of moments in LDS, see above
constexpr int kSsimWaves = 4;                               // of a block: a channel each
static_assert(kOutCols + 2 * kRadius == kWave && kOutRows * kRowLanes <= kWave, "a wavefront is a tile");

__constant__ float kGauss[11] = {0.001028380123898387f, 0.0075987582094967365f, 0.036000773310661316f,
                                 0.10936068743467331f,  0.21300552785396576f,   0.26601171493530273f,
                                 0.21300552785396576f,  0.10936068743467331f,   0.036000773310661316f,
                                 0.0075987582094967365f, 0.001028380123898387f};

// The weights in vector registers (a scalar operand halves the rate of a multiply-add); the filter is symmetric.
struct Taps {
  float g[kRadius + 1];
  __device__ __forceinline__ Taps() {
#pragma unroll
    for (int k = 0; k <= kRadius; ++k) {
      g[k] = kGauss[k];
      asm volatile("" : "+v"(g[k]));
    }
  }
  __device__ __forceinline__ float operator[](int k) const { return g[k <= kRadius ? k : 2 * kRadius - k]; }
};

// Where a wavefront works. Consecutive blocks go to the eight dies in turn: each die takes a consecutive eighth of the tiles, so
// that the rows which neighbouring tiles share are in its L2.
struct SsimTile {
  static constexpr int kRaw32 = 0x00027000;    // word 3 of a buffer descriptor: 32-bit data, no swizzle
  static constexpr int kOutside = 1 << 31;     // an offset that is outside of every buffer here
  int x0, y0;              // first output
  int column_offset;       // of this lane's input column, in bytes; kOutside: left of the image
  int line, first;         // this lane's outputs: row of the tile, first column of six
  bool writes;
  __device__ __forceinline__ SsimTile(int H, int W, int tiles_x) {
    const int lane = threadIdx.x & 63, block = blockIdx.x, share = (int) gridDim.x >> 3;
    const int tile = block < share * 8 ? (block & 7) * share + (block >> 3) : block;
    const int row = tile / tiles_x;
    x0 = (tile - row * tiles_x) * kOutCols, y0 = row * kOutRows;
    column_offset = x0 - kRadius + lane < 0 ? kOutside : lane * (int) sizeof(float);
    line = lane / kRowLanes, first = (lane - line * kRowLanes) * kLaneOut;
    writes = line < kOutRows && y0 + line < H;
    if (line >= kOutRows) line = 0, first = 0;
  }
  // The lane's column of a plane, rows y0 - 5 on; zeros outside the image. A row is a buffer of the 64 columns' bytes up to the
  // image's right edge (none above and below the image), so that the address needs one register a lane for all rows and what lies
  // outside reads as zero without a branch.
  __device__ __forceinline__ void load(const float* plane, int H, int W, float (&v)[kInRows]) const {
    const int bytes = min(W - x0 + kRadius, kWave) * (int) sizeof(float);
    int top = y0 - kRadius;
    asm volatile("" : "+s"(top));  // what follows is made again for each plane: kept, it takes most of the scalar registers
    float* row = const_cast<float*>(plane) + (ptrdiff_t) top * W + x0 - kRadius;
#pragma unroll
    for (int r = 0; r < kInRows; ++r, row += W) {
      __builtin_amdgcn_sched_barrier(0);  // a row's descriptor does not outlive its load
      const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(row, 0, (unsigned) (top + r) < (unsigned) H ? bytes : 0, kRaw32);
      v[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buffer, column_offset, 0, 0));
    }
  }
  // Six neighbouring values of a plane, from and to the lane's outputs. `pairs` (see SsimGrid): two at a time straight from and to
  // where they are; else whole rows, a lane to a column, by way of LDS.
  __device__ __forceinline__ void read(const float* plane, int H, int W, bool pairs, float* s_rows, float (&v)[kLaneOut]) const {
    if (pairs) {
      const __amdgpu_buffer_rsrc_t buffer = outputs(plane, W);
#pragma unroll
      for (int q = 0; q < kLaneOut; q += 2) {
        const auto two = __builtin_amdgcn_raw_buffer_load_b64(buffer, output_offset(q, W), 0, 0);
        const unsigned low = two[0], high = two[1];
        v[q] = __uint_as_float(low), v[q + 1] = __uint_as_float(high);
      }
    } else {
      const int lane = threadIdx.x & 63;
      int top = y0;
      asm volatile("" : "+s"(top));
      wave_lds_sync();
#pragma unroll
      for (int o = 0; o < kOutRows; ++o)
        s_rows[o * kLineWords + lane] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(row(plane, H, W, top + o), lane * 4, 0, 0));
      wave_lds_sync();
#pragma unroll
      for (int q = 0; q < kLaneOut; q += 2) {
        const float2 two = *(const float2*) (s_rows + line * kLineWords + first + q);
        v[q] = two.x, v[q + 1] = two.y;
      }
    }
  }
  __device__ __forceinline__ void write(float* plane, int H, int W, bool pairs, float* s_rows, const float (&v)[kLaneOut]) const {
    if (pairs) {
      const __amdgpu_buffer_rsrc_t buffer = outputs(plane, W);
#pragma unroll
      for (int q = 0; q < kLaneOut; q += 2) {
        typedef unsigned Two __attribute__((ext_vector_type(2)));
        const Two two = {__float_as_uint(v[q]), __float_as_uint(v[q + 1])};
        __builtin_amdgcn_raw_buffer_store_b64(two, buffer, output_offset(q, W), 0, 0);
      }
    } else {
      const int lane = threadIdx.x & 63;
      int top = y0;
      asm volatile("" : "+s"(top));
      wave_lds_sync();
      if (lane < kOutRows * kRowLanes) {
#pragma unroll
        for (int q = 0; q < kLaneOut; q += 2) *(float2*) (s_rows + line * kLineWords + first + q) = make_float2(v[q], v[q + 1]);
      }
      wave_lds_sync();
#pragma unroll
      for (int o = 0; o < kOutRows; ++o)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s_rows[o * kLineWords + lane]), row(plane, H, W, top + o), lane * 4, 0, 0);
    }
  }

 private:
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t outputs(const float* plane, int W) const {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(plane) + (size_t) y0 * W + x0, 0, 0x7fffffff, kRaw32);
  }
  __device__ __forceinline__ int output_offset(int q, int W) const {
    return writes && x0 + first + q < W ? (line * W + first + q) * (int) sizeof(float) : kOutside;
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t row(const float* plane, int H, int W, int y) const {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(plane) + (size_t) y * W + x0, 0,
                                             y < H ? min(W - x0, kOutCols) * (int) sizeof(float) : 0, kRaw32);
  }
};

// An input row's share of the outputs of its column.
__device__ __forceinline__ void down(const Taps& g, int r, float v, float (&sum)[kOutRows]) {
#pragma unroll
  for (int o = 0; o < kOutRows; ++o)
    if (r >= o && r - o <= 2 * kRadius) sum[o] = fmaf(g[r - o], v, sum[o]);
}

// The columns' sums through LDS, and along the row to the lane's outputs.
__device__ __forceinline__ void along(const Taps& g, const SsimTile& t, float* s_rows, const float (&column)[kOutRows],
                                      float (&out)[kLaneOut]) {
  const int lane = threadIdx.x & 63;
  __builtin_amdgcn_sched_barrier(0);
  wave_lds_sync();
#pragma unroll
  for (int o = 0; o < kOutRows; ++o) s_rows[o * kLineWords + lane] = column[o];
  wave_lds_sync();
  float v[kLaneOut + 2 * kRadius];
#pragma unroll
  for (int k = 0; k < kLaneOut + 2 * kRadius; k += 2) {
    const float2 two = *(const float2*) (s_rows + t.line * kLineWords + t.first + k);
    v[k] = two.x, v[k + 1] = two.y;
  }
#pragma unroll
  for (int q = 0; q < kLaneOut; ++q) {
    out[q] = 0.0f;
#pragma unroll
    for (int k = 0; k <= 2 * kRadius; ++k) out[q] = fmaf(g[k], v[q + k], out[q]);
  }
}

template <bool kTrain, bool kLoss>
__global__ void __launch_bounds__(kSsimWaves * kWave) __attribute__((amdgpu_waves_per_eu(5)))
ssim_forward_kernel(int H, int W, int CH, int tiles_x, bool pairs, float C1, float C2, const float* __restrict__ img1, const float* __restrict__ img2,
    float* __restrict__ ssim_map, float* __restrict__ dm_dmu1, float* __restrict__ dm_dsigma1_sq,
    float* __restrict__ dm_dsigma12, float* __restrict__ partials) {
  __shared__ __align__(16) float s_rows[kSsimWaves][kOutRows * kLineWords];
  __shared__ float s_sum[kSsimWaves][2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const SsimTile t(H, W, tiles_x);
  const Taps g;
  const size_t plane = (size_t) H * W;
  float sum_ssim = 0.0f, sum_l1 = 0.0f;  // kLoss: this lane's share of the two image sums
  for (int c = wave; c < CH; c += waves) {
    const size_t off = ((size_t) blockIdx.z * CH + c) * plane;
    float a[kInRows], b[kInRows];
    t.load(img1 + off, H, W, a), t.load(img2 + off, H, W, b);
    float down_a[kOutRows] = {}, down_aa[kOutRows] = {}, down_b[kOutRows] = {}, down_bb[kOutRows] = {}, down_ab[kOutRows] = {}, l1 = 0.0f;
#pragma unroll
    for (int r = 0; r < kInRows; ++r) {
      down(g, r, a[r], down_a), down(g, r, a[r] * a[r], down_aa), down(g, r, b[r], down_b), down(g, r, b[r] * b[r], down_bb);
      down(g, r, a[r] * b[r], down_ab);
      if (kLoss && r >= kRadius && r < kRadius + kOutRows) l1 += fabsf(a[r] - b[r]);  // outside the image both are zero
    }
    const int lane = threadIdx.x & 63;
    if (kLoss) sum_l1 += lane >= kRadius && lane < kRadius + kOutCols ? l1 : 0.0f;
    float mu1[kLaneOut], e11[kLaneOut], mu2[kLaneOut], e22[kLaneOut], e12[kLaneOut];
    float* rows = s_rows[wave];
    along(g, t, rows, down_a, mu1), along(g, t, rows, down_aa, e11), along(g, t, rows, down_b, mu2);
    along(g, t, rows, down_bb, e22), along(g, t, rows, down_ab, e12);
    float map[kLaneOut], by_mu1[kLaneOut], by_var[kLaneOut], by_cov[kLaneOut];
#pragma unroll
    for (int q = 0; q < kLaneOut; ++q) {
#pragma clang fp contract(off)  // the same numbers in all forms of the kernel
      const float m1 = mu1[q], m2 = mu2[q];
      const float mu_sq = m1 * m1 + m2 * m2, sigma_sq = fmaf(-m1, m1, e11[q]) + fmaf(-m2, m2, e22[q]);
      const float C = fmaf(2.0f, m1 * m2, C1), D = fmaf(2.0f, fmaf(-m1, m2, e12[q]), C2);
      const float A = mu_sq + C1, B = sigma_sq + C2;
      // SSIM = CD / (AB) as one rounded quotient: of images that are alike exactly 1, and finite where 1 / (AB) is not. The derivatives
      // with reciprocals of either factor for the same reason, and 1 / B - 1 / A = (A - B) / (AB).
      map[q] = (C * D) / (A * B);
      if (kTrain) {
        const float rA = __builtin_amdgcn_rcpf(A), rB = __builtin_amdgcn_rcpf(B);
        by_mu1[q] = 2.0f * fmaf(m2, D - C, m1 * ((A - B) * map[q])) * rA * rB;
        by_var[q] = -map[q] * rB;
        by_cov[q] = 2.0f * C * rA * rB;
      }
      if (kLoss && t.writes && t.x0 + t.first + q < W) sum_ssim += map[q];
    }
    if (!kLoss) t.write(ssim_map + off, H, W, pairs, rows, map);
    if (kTrain) {
      t.write(dm_dmu1 + off, H, W, pairs, rows, by_mu1), t.write(dm_dsigma1_sq + off, H, W, pairs, rows, by_var);
      t.write(dm_dsigma12 + off, H, W, pairs, rows, by_cov);
    }
  }
  if (kLoss) {
    // block sums in a fixed order: lanes by xor butterfly, then the wavefronts in turn
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sum_ssim += __shfl_xor(sum_ssim, d, 64), sum_l1 += __shfl_xor(sum_l1, d, 64);
    if ((threadIdx.x & 63) == 0) s_sum[wave][0] = sum_ssim, s_sum[wave][1] = sum_l1;
    __syncthreads();
    if (threadIdx.x == 0) {
      float a = 0.0f, b = 0.0f;
      for (int w = 0; w < waves; ++w) a += s_sum[w][0], b += s_sum[w][1];
      const size_t block = (size_t) blockIdx.z * gridDim.x + blockIdx.x;
      partials[2 * block] = a, partials[2 * block + 1] = b;
    }
  }
}

// loss_out[0] = (1 - lambda) * mean|img - target| + lambda * (1 - mean SSIM); [1] = the L1 mean, [2] = the SSIM mean.
// One block; the per-block partial sums are added in a fixed order.
constexpr int kFinishLanes = 1024;
__global__ void __launch_bounds__(kFinishLanes) image_loss_finish_kernel(int n_blocks, const float2* __restrict__ partials,
                                                                         float inv_n, float lambda, float* __restrict__ loss_out) {
  __shared__ float s_red[2][kFinishLanes];
  float a = 0.0f, b = 0.0f;
  for (int i = threadIdx.x; i < n_blocks; i += kFinishLanes) {
    const float2 p = partials[i];
    a += p.x, b += p.y;
  }
  s_red[0][threadIdx.x] = a, s_red[1][threadIdx.x] = b;
  __syncthreads();
  for (int d = kFinishLanes / 2; d >= 1; d >>= 1) {
    if ((int) threadIdx.x < d)
      s_red[0][threadIdx.x] += s_red[0][threadIdx.x + d], s_red[1][threadIdx.x] += s_red[1][threadIdx.x + d];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float ssim_mean = s_red[0][0] * inv_n, l1_mean = s_red[1][0] * inv_n;
    loss_out[0] = (1.0f - lambda) * l1_mean + lambda * (1.0f - ssim_mean);
    loss_out[1] = l1_mean, loss_out[2] = ssim_mean;
  }
}

// kLoss: the gradient of the fused image loss. dL/dmap is the same number at every pixel, -lambda / n times the
// upstream gradient of the scalar loss (read from device memory), and (1 - lambda) / n * sign(img1 - img2) is added.
template <bool kLoss>
__global__ void __launch_bounds__(kSsimWaves * kWave) __attribute__((amdgpu_waves_per_eu(5)))
ssim_backward_kernel(int H, int W, int CH, int tiles_x, bool pairs, const float* __restrict__ img1, const float* __restrict__ img2,
    const float* __restrict__ dL_dmap, const float* __restrict__ dm_dmu1, const float* __restrict__ dm_dsigma1_sq,
    const float* __restrict__ dm_dsigma12, float* __restrict__ dL_dimg1, float map_scale, float l1_scale) {
  __shared__ __align__(16) float s_rows[kSsimWaves][kOutRows * kLineWords];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const SsimTile t(H, W, tiles_x);
  const Taps g;
  const size_t plane = (size_t) H * W;
  const float upstream = kLoss ? dL_dmap[0] : 1.0f, everywhere = map_scale * upstream, of_l1 = l1_scale * upstream;
  for (int c = wave; c < CH; c += waves) {
    const size_t off = ((size_t) blockIdx.z * CH + c) * plane;
    float mu[kInRows], var[kInRows], cov[kInRows], map[kInRows];
    t.load(dm_dmu1 + off, H, W, mu), t.load(dm_dsigma1_sq + off, H, W, var), t.load(dm_dsigma12 + off, H, W, cov);
    if (!kLoss) t.load(dL_dmap + off, H, W, map);
    float* rows = s_rows[wave];
    float one[kLaneOut], two[kLaneOut];
    t.read(img1 + off, H, W, pairs, rows, one), t.read(img2 + off, H, W, pairs, rows, two);
    float down_mu[kOutRows] = {}, down_var[kOutRows] = {}, down_cov[kOutRows] = {};
#pragma unroll
    for (int r = 0; r < kInRows; ++r) {
      if (!kLoss) mu[r] *= map[r], var[r] *= map[r], cov[r] *= map[r];
      down(g, r, mu[r], down_mu), down(g, r, var[r], down_var), down(g, r, cov[r], down_cov);
    }
    float a0[kLaneOut], a1[kLaneOut], a2[kLaneOut], grad[kLaneOut];
    along(g, t, rows, down_mu, a0), along(g, t, rows, down_var, a1), along(g, t, rows, down_cov, a2);
#pragma unroll
    for (int q = 0; q < kLaneOut; ++q) {
      grad[q] = a0[q] + one[q] * 2.0f * a1[q] + two[q] * a2[q];
      if (kLoss) {
        const float d = one[q] - two[q];
        grad[q] = everywhere * grad[q] + of_l1 * (d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f));
      }
    }
    t.write(dL_dimg1 + off, H, W, pairs, rows, grad);
  }
}

// The launch of either kernel: a block per tile of an image, a wavefront per channel. Outputs two at a time where rows and planes
// start at multiples of 8 bytes and seven rows are within a buffer's offsets: 3x800x800 backward 13.5 us against 15.5 by rows
// through LDS. Elsewhere by rows: 3x667x1001 forward 22 us against 27 with single words from the lanes, which lie 24 bytes apart.
// By rows, too, once the maps that a call with gradients reads and writes are more than the memory-side cache holds with them: the pairs
// leave the L2s as parts of lines. us pairs | rows: 3x2160x3840 (map and derivatives 597 MB) 238 | 181, in loss form (498 MB) 200 | 163, backward
// (697, 597 MB) 197 | 181 and 165 | 149; in loss form 288 MB 113 | 100, 243 MB 70 | 76; backward 310 MB 89 | 83, 292 MB 75 | 69, 270 MB 61 | 68.
// The map with its derivatives, four maps written: 115 MB 37 | 36, 149 MB 44 | 40, 265 MB 86 | 77. (The map alone: 3x4000x6000 308 | 314.)
constexpr double kPairsMost = 280e6, kPairsMostOfFour = 120e6;
struct SsimGrid {
  int tiles_x, tiles;
  dim3 grid, block;
  bool pairs;
  // planes: those that are written or read a pair at a time; maps: how many the call reads and writes, where it is one with gradients
  SsimGrid(int B, int CH, int H, int W, std::initializer_list<const void*> planes, int maps, double most = kPairsMost) {
    tiles_x = div_up(W, kOutCols), grid = dim3(tiles_x * div_up(H, kOutRows), 1, B), tiles = grid.x * B;
    block = dim3(kWave * std::min(CH, kSsimWaves));
    pairs = W % 2 == 0 && W < (1 << 26) && 4.0 * maps * B * CH * H * W <= most;
    for (const void* p : planes) pairs &= ((uintptr_t) p & 7) == 0;
  }
};
inline int64_t ssim_tiles(int B, int H, int W) { return (int64_t) B * div_up(W, kOutCols) * div_up(H, kOutRows); }

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API int fsgs_fusedssim_forward(int B, int CH, int H, int W, double C1, double C2, const float* img1,
    const float* img2, float* ssim_map, float* dm_dmu1, float* dm_dsigma1_sq, float* dm_dsigma12, void* stream) {
  FSGS_REQUIRE(B >= 0 && CH >= 0 && H >= 0 && W >= 0, "fusedssim: bad sizes");
  if ((size_t) B * CH * H * W == 0) return kOk;
  FSGS_REQUIRE(img1 && img2 && ssim_map, "fusedssim: null pointer");
  const bool train = dm_dmu1 != nullptr;
  FSGS_REQUIRE(!train || (dm_dsigma1_sq && dm_dsigma12), "fusedssim: the three partial-derivative maps go together");
  FSGS_REQUIRE(B <= 65535, "fusedssim: batch %d exceeds the grid limit", B);
  const SsimGrid g(B, CH, H, W, {ssim_map, dm_dmu1, dm_dsigma1_sq, dm_dsigma12}, train ? 6 : 0, kPairsMostOfFour);
  hipLaunchKernelGGL((train ? ssim_forward_kernel<true, false> : ssim_forward_kernel<false, false>), g.grid, g.block, 0,
                     (hipStream_t) stream, H, W, CH, g.tiles_x, g.pairs, (float) C1, (float) C2, img1, img2,
                     ssim_map, dm_dmu1, dm_dsigma1_sq, dm_dsigma12, nullptr);
  return check_launch("fusedssim");
}

FSGS_API int fsgs_fusedssim_backward(int B, int CH, int H, int W, const float* img1, const float* img2,
    const float* dL_dmap, const float* dm_dmu1, const float* dm_dsigma1_sq, const float* dm_dsigma12,
    float* dL_dimg1, void* stream) {
  FSGS_REQUIRE(B >= 0 && CH >= 0 && H >= 0 && W >= 0, "fusedssim_backward: bad sizes");
  if ((size_t) B * CH * H * W == 0) return kOk;
  FSGS_REQUIRE(img1 && img2 && dL_dmap && dm_dmu1 && dm_dsigma1_sq && dm_dsigma12 && dL_dimg1,
               "fusedssim_backward: null pointer");
  FSGS_REQUIRE(B <= 65535, "fusedssim_backward: batch %d exceeds the grid limit", B);
  const SsimGrid g(B, CH, H, W, {img1, img2, dL_dimg1}, 7);
  hipLaunchKernelGGL(ssim_backward_kernel<false>, g.grid, g.block, 0, (hipStream_t) stream, H, W, CH, g.tiles_x, g.pairs, img1, img2, dL_dmap, dm_dmu1, dm_dsigma1_sq, dm_dsigma12, dL_dimg1, 0.0f, 0.0f);
  return check_launch("fusedssim_backward");
}

FSGS_API size_t fsgs_image_loss_workspace_bytes(int B, int H, int W) {
  if (B <= 0 || H <= 0 || W <= 0) return 256;
  return align_up((size_t) ssim_tiles(B, H, W) * 2 * sizeof(float), 256);
}

FSGS_API int fsgs_image_loss_forward(int B, int CH, int H, int W, double C1, double C2, double lambda_dssim,
    const float* img, const float* target, float* loss_out, float* dm_dmu1, float* dm_dsigma1_sq,
    float* dm_dsigma12, void* workspace, size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(B > 0 && CH > 0 && H > 0 && W > 0 && B <= 65535, "image_loss: bad sizes");
  FSGS_REQUIRE(img && target && loss_out && workspace, "image_loss: null pointer");
  const bool train = dm_dmu1 != nullptr;
  FSGS_REQUIRE(!train || (dm_dsigma1_sq && dm_dsigma12), "image_loss: the three partial-derivative maps go together");
  if (workspace_bytes < fsgs_image_loss_workspace_bytes(B, H, W))
    return fail(kWorkspaceSmall, "image_loss: workspace %zu < %zu bytes", workspace_bytes,
                fsgs_image_loss_workspace_bytes(B, H, W));
  const SsimGrid g(B, CH, H, W, {dm_dmu1, dm_dsigma1_sq, dm_dsigma12}, 5);
  hipStream_t s = (hipStream_t) stream;
  float* partials = (float*) workspace;
  hipLaunchKernelGGL((train ? ssim_forward_kernel<true, true> : ssim_forward_kernel<false, true>), g.grid, g.block, 0, s, H, W,
                     CH, g.tiles_x, g.pairs, (float) C1, (float) C2, img, target, nullptr, dm_dmu1,
                     dm_dsigma1_sq, dm_dsigma12, partials);
  const double n = (double) B * CH * H * W;
  hipLaunchKernelGGL(image_loss_finish_kernel, dim3(1), dim3(kFinishLanes), 0, s, g.tiles, (const float2*) partials,
                     (float) (1.0 / n), (float) lambda_dssim, loss_out);
  return check_launch("image_loss");
}

// ---- the same forward for callers that cannot allocate ----------------------------------------------------------------
// The per-block partial sums live in a file-scope device array instead of a caller workspace. Every GPU the library
// runs on holds its own copy of the array at its own address until the process ends; the address is looked up once per
// device and only that pointer is handed to kernels (the array's name is a host-side stand-in, not a device address).
constexpr int kStaticSide = 32, kStaticLossMaxBlocks = 65536;  // 32x32-pixel blocks, e.g. one 8192x8192 image or 40 images of 1280x1280
constexpr int kStaticTiles = (kStaticSide + kOutRows - 1) / kOutRows * kStaticLossMaxBlocks;  // a block touches so many rows of tiles at most
static_assert(kOutCols >= kStaticSide, "and one column of them, counted over the image");
static __device__ __align__(256) float scratch[2 * kStaticTiles];  // 2.5 MiB
constexpr int kMaxDevices = 64;
static std::atomic<float*> g_scratch_ptr[kMaxDevices];

static int static_scratch(float** out) {
  int dev = -1;
  FSGS_HIP(hipGetDevice(&dev));
  FSGS_REQUIRE(dev >= 0 && dev < kMaxDevices, "image_loss_static: device ordinal %d out of range", dev);
  float* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    FSGS_HIP(hipGetSymbolAddress((void**) &p, HIP_SYMBOL(scratch)));
    FSGS_REQUIRE(p != nullptr, "image_loss_static: no device address for the scratch array");
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return kOk;
}

FSGS_API int fsgs_image_loss_static_max_blocks(void) { return kStaticLossMaxBlocks; }

FSGS_API int fsgs_image_loss_forward_static(int B, int CH, int H, int W, double C1, double C2, double lambda_dssim,
    const float* img, const float* target, float* loss_out, float* dm_dmu1, float* dm_dsigma1_sq,
    float* dm_dsigma12, void* stream) {
  FSGS_REQUIRE(B > 0 && CH > 0 && H > 0 && W > 0 && B <= 65535, "image_loss_static: bad sizes");
  const int64_t blocks = (int64_t) B * div_up(W, kStaticSide) * div_up(H, kStaticSide);
  if (blocks > kStaticLossMaxBlocks)
    return fail(kUnsupported, "image_loss_static: %lld blocks of 32x32 pixels exceed the built-in scratch of %d blocks; "
                "use fsgs_image_loss_forward with a workspace", (long long) blocks, kStaticLossMaxBlocks);
  float* partials = nullptr;
  if (int rc = static_scratch(&partials)) return rc;
  return fsgs_image_loss_forward(B, CH, H, W, C1, C2, lambda_dssim, img, target, loss_out, dm_dmu1, dm_dsigma1_sq,
                                 dm_dsigma12, partials, sizeof(scratch), stream);
}

FSGS_API int fsgs_image_loss_backward(int B, int CH, int H, int W, double lambda_dssim, const float* img,
    const float* target, const float* grad_loss, const float* dm_dmu1, const float* dm_dsigma1_sq,
    const float* dm_dsigma12, float* dL_dimg, void* stream) {
  FSGS_REQUIRE(B > 0 && CH > 0 && H > 0 && W > 0 && B <= 65535, "image_loss_backward: bad sizes");
  FSGS_REQUIRE(img && target && grad_loss && dm_dmu1 && dm_dsigma1_sq && dm_dsigma12 && dL_dimg,
               "image_loss_backward: null pointer");
  const SsimGrid g(B, CH, H, W, {img, target, dL_dimg}, 6);
  const double n = (double) B * CH * H * W;
  hipLaunchKernelGGL(ssim_backward_kernel<true>, g.grid, g.block, 0, (hipStream_t) stream, H, W, CH, g.tiles_x, g.pairs, img, target, grad_loss, dm_dmu1, dm_dsigma1_sq, dm_dsigma12, dL_dimg,
                     (float) (-lambda_dssim / n), (float) ((1.0 - lambda_dssim) / n));
  return check_launch("image_loss_backward");
}
