// Block-cooperative movement of per-surfel SH rows between HBM and LDS for the one-lane-per-surfel preprocess kernels.
// A lane that walks its own 192-byte row touches one 128-byte line per instruction and relies on the caches to keep 96
// lines per wavefront alive between touches; moving the block's rows with consecutive lanes on consecutive addresses
// reads (writes) every line once. Used when the active degree is <= 3 (at most 16 coefficients, 48 floats per row).
#pragma once
#include "common.hpp"
#include "sh.hpp"

namespace fsgs {

constexpr int kShStageRows   = 256;  // surfels per block
constexpr int kShStageFloats = 48;   // 16 coefficients x rgb
constexpr int kShStageStride = 49;   // odd stride: a lane reading its own row hits a different bank than its neighbours

// e / d for 0 <= e < 2^20 and 1 <= d <= 256 without an integer division: (e + 0.5) / d is at least 0.5 / d away from any
// integer, far more than the rounding error of the float product.
__device__ __forceinline__ int small_div(int e, float inv_d) { return (int) (((float) e + 0.5f) * inv_d); }

// Copies the first n coefficients (n * 3 floats) of every flagged row of the block into LDS. Row r of the block is
// surfel block_base + r. With sh_rest the DC coefficient comes from shs[P,1,3] and the others from sh_rest[P,n_sh,3].
__device__ __forceinline__ void stage_sh_rows(float* __restrict__ s_rows, const unsigned char* __restrict__ s_flag,
                                              int block_base, int P, int n, int n_sh, const float* __restrict__ shs,
                                              const float* __restrict__ sh_rest) {
  const int per_row = n * 3;
  const int rows    = min(kShStageRows, P - block_base);
  if (sh_rest == nullptr) {
    const size_t stride = (size_t) n_sh * 3;
    const float inv     = 1.0f / (float) per_row;
    for (int e = threadIdx.x; e < rows * per_row; e += blockDim.x) {
      const int r = small_div(e, inv), c = e - r * per_row;
      if (s_flag[r]) s_rows[r * kShStageStride + c] = shs[(size_t) (block_base + r) * stride + c];
    }
  } else {
    for (int e = threadIdx.x; e < rows * 3; e += blockDim.x) {
      const int r = e / 3, c = e - r * 3;
      if (s_flag[r]) s_rows[r * kShStageStride + c] = shs[(size_t) (block_base + r) * 3 + c];
    }
    const int rest    = per_row - 3;
    const size_t stride = (size_t) n_sh * 3;
    const float inv     = 1.0f / (float) max(rest, 1);
    for (int e = threadIdx.x; e < rows * rest; e += blockDim.x) {
      const int r = small_div(e, inv), c = e - r * rest;
      if (s_flag[r]) s_rows[r * kShStageStride + 3 + c] = sh_rest[(size_t) (block_base + r) * stride + c];
    }
  }
}

// Writes the block's staged gradient rows (n * 3 floats each, zeros where the owning lane stored zeros) to
// g_shs / g_sh_rest and zero-fills the coefficients above the active degree, so the caller's tensors need no
// initialisation. With the split layout (has_rest) either output may be absent.
__device__ __forceinline__ void unstage_sh_grads(const float* __restrict__ s_rows, int block_base, int P, int n,
                                                 int n_sh, bool has_rest, float* __restrict__ g_shs,
                                                 float* __restrict__ g_sh_rest) {
  const int rows = min(kShStageRows, P - block_base);
  if (!has_rest) {
    if (g_shs == nullptr) return;
    const int per_row = n_sh * 3, live = n * 3;
    const float inv   = 1.0f / (float) per_row;
    for (int e = threadIdx.x; e < rows * per_row; e += blockDim.x) {
      const int r = small_div(e, inv), c = e - r * per_row;
      g_shs[(size_t) (block_base + r) * per_row + c] = c < live ? s_rows[r * kShStageStride + c] : 0.0f;
    }
    return;
  }
  if (g_shs != nullptr) {
    for (int e = threadIdx.x; e < rows * 3; e += blockDim.x) {
      const int r = e / 3, c = e - r * 3;
      g_shs[(size_t) (block_base + r) * 3 + c] = s_rows[r * kShStageStride + c];
    }
  }
  if (g_sh_rest != nullptr) {
    const int per_row = n_sh * 3, live = n * 3 - 3;
    const float inv   = 1.0f / (float) max(per_row, 1);
    for (int e = threadIdx.x; e < rows * per_row; e += blockDim.x) {
      const int r = small_div(e, inv), c = e - r * per_row;
      g_sh_rest[(size_t) (block_base + r) * per_row + c] = c < live ? s_rows[r * kShStageStride + 3 + c] : 0.0f;
    }
  }
}

// ---- wavefront-private variant for complete rows ---------------------------------------------------------------------
// A [P, kFloats / 3, 3] tensor of complete rows (all coefficients of the active degree and no others) that starts on a
// 16-byte boundary: the 64 rows of a wavefront are 16 * kFloats consecutive 16-byte pieces, whatever the length of a row.
// A wavefront moves them by itself: every load or store instruction covers 1 KB of consecutive addresses, the loads can be
// issued before the data is needed (they are held in registers while the lane does its geometry) and no block-wide barrier
// is involved. Rows of 48 floats are all coefficients of degree 3 in one tensor, of 45 the fifteen above the first where a
// model keeps that one apart, of 27 and 12 degrees 2 and 1. Forward preprocess with 45 floats, 400k surfels (the rows are
// 72 MB of its 150): 127 us through stage_sh_rows (4-byte loads behind a block barrier), 64 us this way.
// In LDS a row has an odd stride, so lanes that read their own rows hit different banks: rows of odd length lie as they
// do in memory (a piece is one 16-byte LDS write), rows of even length get one float more.
// The rows are most of what a pass moves, and each is read once and written once in it: they pass the 256 MB memory-side cache by
// (non-temporal stores, and loads where the rows are 48 MB or more), which then holds the records, the lists and the model's other tensors from kernel to
// kernel. Preprocess forward and backward, us: 3M 1352x1014 238 + 369 -> 216 + 330; 1M 1352x900 96 + 131 -> 85 + 119; 300k 800x800
// 34 + 51 -> 34 + 45. Stores by ordinary and by streaming ones, preprocess backward of small scenes: 10k 10.9 and 11.0, 50k 14.6 and
// 14.2, 100k 19.3 and 18.1, 200k 39.3 and 37.2; colours' backward 10k 6.4 and 6.3, 50k 7.9 and 7.0, 200k 19.0 and 18.0: no size at which
// ordinary ones are better. The SH operators' backward, where it reads the coefficients that their forward has read, uses ordinary
// loads, 1M rows of coefficients 53 + 82 -> 33 + 76 us (with streaming loads
// 36 + 77). Smaller tables stay in the cache from pass to pass: view of 98k surfels 170x120, preprocess 14 us and 16 with streaming
// loads; 200k 22.3 and 23.5; 300k (58 MB) 36.4 and 35.2; 400k 58 and 52.
using ShPiece = float __attribute__((ext_vector_type(4)));

constexpr size_t kStreamBytes = 48u << 20;

template <int kFloats>
struct ShWaveRows {
  static_assert(kFloats % 2 == 1 || kFloats % 4 == 0, "a piece lies in one row or rows are stored without a gap");
  static constexpr int kStride = kFloats | 1;
  static __device__ __forceinline__ bool large(int P) { return (size_t) P * kFloats * 4 >= kStreamBytes; }
  static constexpr int kPieces = 16 * kFloats;          // of 64 rows
  static constexpr int kVecs   = (kPieces + 63) / 64;   // of a lane
  ShPiece v[kVecs];
  float tail;

  // floats of the wavefront's existing rows
  template <int kRows = 64>
  static __device__ __forceinline__ int floats(int wave_base, int P) { return max(min(kRows, P - wave_base), 0) * kFloats; }

  // `flags` has bit r set for the rows that are needed (all of them existing rows); a piece of other rows re-reads the
  // first needed row's instead of branching. flags must not be 0.
  // stream (uniform): the pieces pass the memory-side cache by.
  __device__ __forceinline__ void fetch(unsigned long long flags, int wave_base, int P, const float* __restrict__ src,
                                        bool stream = false) {
    const int all = floats(wave_base, P), whole = all >> 2, lane = (int) __lane_id();
    const int first  = (__builtin_ctzll(flags) * kFloats) >> 2;
    const float* row = src + (size_t) wave_base * kFloats;
    auto piece = [&](int k) {
      const int e = k * 64 + lane;
      const int r0 = (4 * e) / kFloats, r1 = (4 * e + 3) / kFloats;
      const bool on = e < whole && (((flags >> (r0 & 63)) | (flags >> (r1 & 63))) & 1ull);
      return (const ShPiece*) row + (on ? e : first);
    };
    if (stream) {
#pragma unroll
      for (int k = 0; k < kVecs; ++k) v[k] = __builtin_nontemporal_load(piece(k));
    } else {
#pragma unroll
      for (int k = 0; k < kVecs; ++k) v[k] = *piece(k);
    }
    if (kFloats % 4 != 0) {  // up to three floats behind the last piece of the last wavefront
      tail = 0.0f;
      if (lane < (all & 3)) tail = row[4 * whole + lane];
    }
  }

  __device__ __forceinline__ void to_lds(float* __restrict__ s_wave_rows, int wave_base, int P) const {
    const int lane = (int) __lane_id();
#pragma unroll
    for (int k = 0; k < kVecs; ++k) {
      const int e = k * 64 + lane;
      if (kFloats % 2 == 1) {
        if (e < kPieces) *(ShPiece*) (s_wave_rows + 4 * e) = v[k];
      } else {
        const int r = (4 * e) / kFloats;
        float* d = s_wave_rows + r * kStride + (4 * e - r * kFloats);
        d[0] = v[k].x, d[1] = v[k].y, d[2] = v[k].z, d[3] = v[k].w;
      }
    }
    if (kFloats % 4 != 0) {
      const int all = floats(wave_base, P);
      if (lane < (all & 3)) s_wave_rows[(all & ~3) + lane] = tail;
    }
  }

  // Each lane's own row in its registers, 32 rows at a time by way of kHalfFloats floats of LDS, which lets four blocks of a preprocess
  // kernel share a compute unit (120 registers) where room for all 64 rows (50 KB a block) let three: 200k surfels are 782 blocks,
  // a few more than three for each of the 256 units. Rows of 48 floats lie with a stride of 52, in steps of 16 bytes all the way.
  static constexpr int kHalfStride = kFloats == 48 ? 52 : kStride, kHalfFloats = 32 * kHalfStride;
  __device__ __forceinline__ void to_lanes(float (&own)[kFloats], float* __restrict__ s_half, int wave_base, int P) const {
    static_assert(kFloats == 48 || kFloats % 2 == 1);
    constexpr int kHalf = 8 * kFloats;  // pieces of 32 rows
    const int lane = (int) __lane_id();
    const float* row = s_half + (lane & 31) * kHalfStride;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < kVecs; ++k) {
        if (64 * k + 63 < h * kHalf || 64 * k >= (h + 1) * kHalf) continue;
        const int e = k * 64 + lane - h * kHalf;
        if (kFloats == 48) *(ShPiece*) (s_half + 4 * e + e / 12 * 4) = v[k];
        else if (e >= 0 && e < kHalf) *(ShPiece*) (s_half + 4 * e) = v[k];
      }
      if (kFloats % 4 != 0) {
        const int all = floats(wave_base, P), at = (all & ~3) - 4 * h * kHalf;
        if (lane < (all & 3) && at >= 0 && at < 4 * kHalf) s_half[at + lane] = tail;
      }
      wave_lds_sync();
      if (lane >> 5 == h) {
        if (kFloats == 48) {
#pragma unroll
          for (int k = 0; k < 12; ++k) {
            const ShPiece q = *(const ShPiece*) (row + 4 * k);
            own[4 * k] = q.x, own[4 * k + 1] = q.y, own[4 * k + 2] = q.z, own[4 * k + 3] = q.w;
          }
        } else {
#pragma unroll
          for (int k = 0; k < kFloats; ++k) own[k] = row[k];
        }
      }
    }
  }

  // Writes the wavefront's staged rows (every existing row; kRows at most, from wave_base on) to dst.
  template <int kRows = 64>
  static __device__ __forceinline__ void to_global(const float* __restrict__ s_wave_rows, int wave_base, int P,
                                                   float* __restrict__ dst) {
    const int all = floats<kRows>(wave_base, P), whole = all >> 2, lane = (int) __lane_id();
    float* row = dst + (size_t) wave_base * kFloats;
#pragma unroll
    for (int k = 0; k < (kRows * kFloats / 4 + 63) / 64; ++k) {
      const int e = k * 64 + lane;
      if (kFloats % 2 == 1) {
        if (e < whole) __builtin_nontemporal_store(*(const ShPiece*) (s_wave_rows + 4 * e), (ShPiece*) row + e);
      } else if (e < whole) {
        const int r = (4 * e) / kFloats;
        const float* s = s_wave_rows + r * kStride + (4 * e - r * kFloats);
        __builtin_nontemporal_store(ShPiece{s[0], s[1], s[2], s[3]}, (ShPiece*) row + e);
      }
    }
    if (kFloats % 4 != 0 && lane < (all & 3)) row[4 * whole + lane] = s_wave_rows[4 * whole + lane];
  }

  static __device__ __forceinline__ void zeros_to_global(int wave_base, int P, float* __restrict__ dst) {
    const int all = floats(wave_base, P), whole = all >> 2, lane = (int) __lane_id();
    float* row = dst + (size_t) wave_base * kFloats;
#pragma unroll
    for (int k = 0; k < kVecs; ++k)
      if (k * 64 + lane < whole) __builtin_nontemporal_store(ShPiece{0.0f, 0.0f, 0.0f, 0.0f}, (ShPiece*) row + k * 64 + lane);
    if (kFloats % 4 != 0 && lane < (all & 3)) row[4 * whole + lane] = 0.0f;
  }
};

// Writes a wavefront's rows of kFloats floats from LDS, where they lie without gaps as they will in memory, to dst (on a 16-byte
// boundary; a wavefront's rows then start on one, too). With its own stores a lane touches lines that it shares with its
// neighbours' stores of the same kind, an instruction as many lines as its 64 rows cover, for each of its pieces.
template <int kFloats>
__device__ __forceinline__ void wave_rows_out(const float* __restrict__ s_rows, int wave_base, int P, float* __restrict__ dst) {
  const int all = max(min(64, P - wave_base), 0) * kFloats, whole = all >> 2, lane = (int) __lane_id();
  float* row = dst + (size_t) wave_base * kFloats;
#pragma unroll
  for (int k = 0; k < (16 * kFloats + 63) / 64; ++k)
    if (k * 64 + lane < whole) ((ShPiece*) row)[k * 64 + lane] = ((const ShPiece*) s_rows)[k * 64 + lane];
  if (kFloats % 4 != 0 && lane < (all & 3)) row[4 * whole + lane] = s_rows[4 * whole + lane];
}

// Which rows of a preprocess kernel move this way: 48 (one tensor), 45 (the first coefficient apart) or 0 (every other
// degree, number of coefficients or alignment: stage_sh_rows, or the lane's own walk). The gradients' tensors, where there
// are any, have to be aligned like the coefficients'.
inline int wave_row_floats(int sh_degree, int n_sh, const float* shs, const float* sh_rest, const float* g_rows = nullptr) {
  if (sh_degree != 3 || n_sh != (sh_rest ? 15 : 16)) return 0;
  if ((((uintptr_t) (sh_rest ? sh_rest : shs) | (uintptr_t) g_rows) & 15) != 0) return 0;
  return sh_rest ? 45 : 48;
}

// The derivatives of the colours by the direction (sh_color_derivatives) that a view's forward leaves for its backward: a row of
// nine floats per point.
constexpr int kColorDerivs = 9;

// A point's colours and, on request, their derivatives from its complete row of degree 3 (of 45 floats: `dc` in front). Against double
// precision, 10k points: root mean square 2.04e-8, largest 1.11e-7 (summed from LDS: 2.05e-8 and 1.11e-7).
template <int kRow>
__device__ __forceinline__ void sh_lane_colors(const float (&own)[kRow], const float (&dc)[3], int degree, float x, float y, float z,
                                               bool want_derivs, float (&rgb)[3], float (&derivs)[kColorDerivs]) {
  constexpr bool kSplit = kRow == 45;
  auto coef = [&](int l, int c) { return kSplit ? l == 0 ? dc[c] : own[3 * (l > 0 ? l - 1 : 0) + c] : own[kSplit ? 0 : 3 * l + c]; };
  float Y[16];
  sh_eval(degree, x, y, z, Y);
  float r = coef(0, 0) * Y[0], g = coef(0, 1) * Y[0], b = coef(0, 2) * Y[0];
#pragma unroll
  for (int l = 1; l < 16; ++l) r = fmaf(coef(l, 0), Y[l], r), g = fmaf(coef(l, 1), Y[l], g), b = fmaf(coef(l, 2), Y[l], b);
  rgb[0] = fmaxf(0.0f, r + 0.5f), rgb[1] = fmaxf(0.0f, g + 0.5f), rgb[2] = fmaxf(0.0f, b + 0.5f);
  if (want_derivs) sh_color_derivatives(degree, x, y, z, coef, derivs);
}

// Leaves a wavefront's rows of them (`derivs`, of every lane; aligned as wave_rows_out asks) by way of the LDS that held its rows.
__device__ __forceinline__ void wave_derivs_out(float* __restrict__ s_wave_rows, const float (&derivs)[kColorDerivs], int wave_base,
                                                int P, float* __restrict__ dst) {
  const int lane = (int) __lane_id();
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < kColorDerivs; ++k) s_wave_rows[kColorDerivs * lane + k] = derivs[k];
  wave_lds_sync();
  wave_rows_out<kColorDerivs>(s_wave_rows, wave_base, P, dst);
}

// The gradients of a wavefront's rows of kRow coefficients (48, or 45 with the first coefficient apart) where nothing is read from
// them: the products of a lane's colour gradient `g` and basis `Y` (zeros where there is no gradient). Half of the rows at a time
// pass through the LDS, so that it holds 32 rows of a wavefront, and more of them share a compute unit than with room for all 64.
constexpr int kShHalfRows = 32;
template <int kRow>
__device__ __forceinline__ void sh_products_to_global(float* __restrict__ s_half_rows, const float (&g)[3], const float (&Y)[16],
                                                      int wave_base, int P, float* __restrict__ dst) {
  static_assert(kShHalfRows * kRow % 4 == 0);
  constexpr int kStride = kRow | 1, kFirst = (48 - kRow) / 3;
  const int lane = (int) __lane_id();
  float* row = s_half_rows + (lane & (kShHalfRows - 1)) * kStride;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    wave_lds_sync();
    if (lane / kShHalfRows == h) {
#pragma unroll
      for (int l = kFirst; l < 16; ++l)
#pragma unroll
        for (int c = 0; c < 3; ++c) row[3 * (l - kFirst) + c] = g[c] * Y[l];
    }
    wave_lds_sync();
    ShWaveRows<kRow>::template to_global<kShHalfRows>(s_half_rows, wave_base + h * kShHalfRows, P, dst);
  }
}

// A backward's gradient of the view direction `dir`: from the forward's derivatives (kDerivs), or from the coefficients (`rows`:
// coefficient l of channel c at 3 l + c).
template <int kSh, bool kDerivs>
__device__ __forceinline__ void sh_direction_part(int degree, const float (&dir)[3], const float (&g)[3], const float* rows,
                                                  float (&derivs)[kColorDerivs], float& dx, float& dy, float& dz) {
  if constexpr (kSh == 16) {
    if (!kDerivs) sh_color_derivatives(degree, dir[0], dir[1], dir[2], [&](int l, int c) { return rows[3 * l + c]; }, derivs);
    sh_direction_gradient(g, derivs, dx, dy, dz);
  } else {
    const int n = sh_count(degree);
    float tl[kSh];
    tl[0] = 0.0f;
    for (int l = 1; l < n; ++l) tl[l] = g[0] * rows[3 * l] + g[1] * rows[3 * l + 1] + g[2] * rows[3 * l + 2];
    sh_grad_accumulate(degree, dir[0], dir[1], dir[2], tl, dx, dy, dz);
  }
}

}  // namespace fsgs
