// Fused deformation MLP forward and backward on the CDNA4 matrix cores (bf16 operands, fp32 accumulation) for gfx950.
//
// Reference behaviour reproduced (in fp32 there): fast_2d_gs/network.py:1757-1776 -- h = in; for each of the L layers
// h = relu(W_i h + b_i); after layer index `skip` the input is concatenated in front, h = [in | h]; the heads are plain
// linear maps of the last hidden state (gaussian_warp 3, gaussian_rotation 4, gaussian_scaling 3 stacked into one
// [n_out, 256] matrix by the caller).
//
// One block owns 16 rows (control points) and keeps their activations in LDS for the whole network, so the only HBM/L2
// traffic is the weights (about 1 MB in bf16, shared by all blocks through L2) and 40 bytes of output per row.
// Each of the 8 wavefronts computes a 16 x 32 slab of a layer's output with v_mfma_f32_16x16x32_bf16: A fragments
// (activations) come from LDS as one 16-byte read per lane, B fragments (weights, packed in fragment order, see
// frag_index) as one 16-byte global read per lane; both use the same (lane / 16, element) -> k mapping, so the product
// is independent of how the hardware orders k inside a fragment. The input rows are either given or formed here from
// positions and time (the frequency encoding), which spares three launches and a [B][84] tensor.
//
// Training: the forward optionally stores every layer's post-ReLU hidden state and the input rows, in bf16 and with the
// batch innermost ([layer][256][B_pad], B_pad = B rounded up to 32): an accumulator's four consecutive registers are four
// consecutive rows of one column, so that layout takes 8-byte stores, and it is what the weight gradients read. The
// backward (the reference leaves it to torch autograd: one addmm-backward pair and a ReLU mask per layer, ~30 launches)
// is two kernels:
//   * a chain kernel with the forward's structure, one block per 16 rows: dZ_L-1 = (g_out . W_heads) masked by the saved
//     state, then for each layer dH_l-1 = dZ_l . W_l[:, hidden part] on the matrix cores against a transposed bf16 copy
//     of the weights, masked, kept in LDS for the next layer and written to HBM as dZ[l][256][B_pad];
//   * a weight-gradient kernel over all layers at once, dW = dZ^T X: with the batch innermost both operands' fragments are
//     16-byte loads of consecutive memory. A block owns a 64 x 64 tile, its four wavefronts take a share of the batch each
//     with every load of 128 rows in flight, and add their sums through LDS in wavefront order; the first tile column of a
//     layer also sums dZ over the batch for the bias gradient. No atomics: every output element has one writer.
// The chains' time is nine dependent layers of one block, so what a layer costs a compute unit counts: LDS reads, matrix
// products and the epilogue's conversions all halve with 16 rows in place of 32. At B = 512 and 8 layers: forward 39 -> 20
// us, backward chain 41 -> 27, weight gradients (operands transposed through LDS two bytes at a time before) 48 -> 11.
// Gradients with respect to the (frequency-encoded) input are not produced; the reference detaches it
// (network.py:586).
#include <algorithm>

#include "common.hpp"

namespace fsgs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kMlpWidth   = 256;
constexpr int kMlpRows    = 16;                       // rows per block of the chains
constexpr int kMlpRowPad  = 32;                       // the saved tensors' batch is padded to this
constexpr int kMlpMaxIn   = 96;                       // padded input width limit
constexpr int kMlpStride  = kMlpWidth + kMlpMaxIn + 8;  // LDS row stride in bf16 (+8 keeps 16-byte rows off one bank)
constexpr int kMlpThreads = 256;
// Forward and backward chain: eight wavefronts per block, 16 x 32 outputs each. With that little per wavefront a whole
// layer's 16 fragments fit in registers and are requested together.
constexpr int kChainThreads = 512;

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t) ((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t) (u >> 16);
}

// Weights are stored in the order the matrix cores consume them: the [rows_pad][K_pad] matrix is cut into tiles of 32
// rows x 16 columns, tile (row tile nt, k-step ks) at ((nt * K_pad / 16) + ks) * 512 elements, and inside a tile the 8
// consecutive k values that lane l of a wavefront feeds to one MFMA (row l % 32, columns 8 * (l / 32) .. + 7) are
// contiguous at l * 8. One fragment load of a wavefront is then a single 1 KB run instead of 64 rows 2 * K_pad bytes apart.
__device__ __forceinline__ size_t frag_index(int r, int k, int K_pad) {
  const int nt = r >> 5, n = r & 31, ks = k >> 4, kk = k & 15;
  return (((size_t) nt * (K_pad >> 4) + ks) * 64 + n + 32 * (kk >> 3)) * 8 + (kk & 7);
}

__global__ void __launch_bounds__(256) pack_bf16_kernel(int rows, int K, int rows_pad, int K_pad,
                                                        const float* __restrict__ src, uint16_t* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows_pad * K_pad) return;
  const int r = i / K_pad, k = i - r * K_pad;
  dst[frag_index(r, k, K_pad)] = (r < rows && k < K) ? f32_to_bf16(src[(size_t) r * K + k]) : (uint16_t) 0;
}

// Every per-step re-pack of the network in one launch: blockIdx.y selects a job of the table passed by value.
struct PackJob {
  const float* src;
  void* dst;
  int rows, K;            // extent of the source that exists: rows x K values
  int rows_cover, K_pad;  // fragment rows this job writes (zeros past `rows`), padded row length of the fragment matrix
  int dst_row0;           // first fragment row
  int src_ld, col0;       // leading dimension and first column of the source
  int kind;               // 0 fragment pack | 1 fragment pack of the transpose | 2 plain float copy of `rows` values
};
constexpr int kMaxPackJobs = 40;
struct PackTable {
  PackJob job[kMaxPackJobs];
};

__global__ void __launch_bounds__(256) pack_jobs_kernel(PackTable table) {
  const PackJob& j = table.job[blockIdx.y];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (j.kind == 2) {
    if (i < j.rows) ((float*) j.dst)[i] = j.src[i];
    return;
  }
  if (i >= j.rows_cover * j.K_pad) return;
  const int r = i / j.K_pad, k = i - r * j.K_pad;
  float v = 0.0f;
  if (r < j.rows && k < j.K)
    v = j.kind == 0 ? j.src[(size_t) r * j.src_ld + j.col0 + k] : j.src[(size_t) k * j.src_ld + j.col0 + r];
  ((uint16_t*) j.dst)[frag_index(j.dst_row0 + r, k, j.K_pad)] = f32_to_bf16(v);
}

__global__ void __launch_bounds__(256) fill_zero_kernel(size_t n, float* __restrict__ p) {
  for (size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x) p[i] = 0.0f;
}

// D layout of the 32x32 accumulator: register r of lane l holds row 8 * (r / 4) + 4 * (l / 32) + (r % 4), column l % 32.
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

__device__ __forceinline__ int div_up_dev(int a, int b) { return (a + b - 1) / b; }

constexpr int kMaxHeads = 8;
struct MlpHeads {  // the outputs' (or their gradients') columns: head h is [B][width[h]] and holds columns first[h] ..
  float* at[kMaxHeads];
  int first[kMaxHeads + 1];
  int n;
};
__device__ __forceinline__ float* head_cell(const MlpHeads& h, int row, int col) {
  int q = 0;
#pragma unroll
  for (int k = 1; k < kMaxHeads; ++k) q += (k < h.n && col >= h.first[k]) ? 1 : 0;
  float* base = h.at[0];
  int first = h.first[0], width = h.first[1];
#pragma unroll
  for (int k = 1; k < kMaxHeads; ++k)
    if (q == k) base = h.at[k], first = h.first[k], width = h.first[k + 1] - h.first[k];
  return base ? base + (size_t) row * width + (col - first) : nullptr;
}

// The frequency encoding of positions x[B,3] and one time t[1]: [x | sin 2^d s x, cos 2^d s x ...] then the same for t.
struct FreqInput {
  const float* x;
  const float* t;
  int degree_x, degree_t;
  float scale_x, scale_t;
};
__device__ __forceinline__ float encoded(const FreqInput& f, int row, int k) {
  const int wide = 3 * (1 + 2 * f.degree_x);
  int q;
  float v, scale;
  if (k < wide) q = k / 3, v = f.x[3 * (size_t) row + (k - 3 * q)], scale = f.scale_x;
  else q = k - wide, v = f.t[0], scale = f.scale_t;
  if (q == 0) return v;
  v = ldexpf(v * scale, (q - 1) >> 1);
  return ((q - 1) & 1) ? cosf(v) : sinf(v);
}

__device__ __forceinline__ uint2 pack4(const uint16_t* h) {
  return make_uint2((uint32_t) h[0] | ((uint32_t) h[1] << 16), (uint32_t) h[2] | ((uint32_t) h[3] << 16));
}

// Two values rounded to nearest even by the conversion instruction (the chains' epilogues are vector-bound: with the
// rounding written out in integer arithmetic a layer's epilogue was 760 instructions, half of its time).
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 h = {(__bf16) lo, (__bf16) hi};
  return __builtin_bit_cast(uint32_t, h);
}

// A block streams all of the weights, 1.1 MB, through one compute unit, and how fast it can is a matter of latency: about
// 35 GB/s when the lines come from beyond the L2 (30 us). With few row blocks most of the chip is idle, so some blocks more
// fetch the weights into every L2 (blocks go round the 8 XCDs in turn), all of them together from the first layer on.
constexpr int kFetchParts = 8;                // blocks per XCD that fetch
constexpr int kFetchBlocks = 8 * kFetchParts;
constexpr int kFetchBelow = 128;              // row blocks; with more of them the weights are in every L2 soon enough
__device__ __forceinline__ void fetch_to_l2(const uint16_t* __restrict__ data, size_t elems, int part) {
  const uint4* p = (const uint4*) data;
  const size_t n = elems / 8;
  for (size_t e = (size_t) part * kChainThreads + threadIdx.x; e < n; e += (size_t) kFetchParts * kChainThreads * 4) {
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = p[min(e + (size_t) k * kFetchParts * kChainThreads, n - 1)];
#pragma unroll
    for (int k = 0; k < 4; ++k) asm volatile("" ::"v"(v[k].x));
  }
}

// B fragments of a wavefront's two 16-column tiles for k-step kk (32 values of k) of the matrix whose row tile (32 rows, one
// per output) starts at `tile`: tile elements are laid out by frag_index, so a fragment is four runs of 256 bytes. A
// matrix with an odd number of 16-column steps ends in half a step; its missing half re-reads the last one and meets zeros.
__device__ __forceinline__ void load_fragments(const uint16_t* __restrict__ tile, int kk, int last_step, bf16x8 (&b)[2]) {
  const int lane = threadIdx.x & 63, ks = min(2 * kk + (lane >> 5), last_step), half = (lane >> 4) & 1;
#pragma unroll
  for (int t = 0; t < 2; ++t) b[t] = *(const bf16x8*) (tile + ks * 512 + (16 * t + (lane & 15) + 32 * half) * 8);
}

// D layout of the 16x16 accumulator: register r of lane l holds row 4 * (l / 16) + r, column l % 16.
// What the forward stores of the hidden states: nothing; them and the input rows batch innermost (see the file's head); or
// the states alone as rows, [layer][B][256], the form that fsgs_mlp_forward's callers keep.
enum class Keep { kNothing, kBatchInnermost, kRows };
// `in` or `freq.x` gives the input rows; in_t goes with kBatchInnermost.
template <Keep kKeep>
__global__ void __launch_bounds__(kChainThreads) mlp_forward_kernel(int B, int Din, int n_layers, int skip, int n_out,
    const float* __restrict__ in, FreqInput freq, const uint16_t* __restrict__ packed, const float* __restrict__ bias,
    MlpHeads heads, uint16_t* __restrict__ in_t, uint16_t* __restrict__ saved, int row_blocks, size_t packed_elems) {
  if ((int) blockIdx.x >= row_blocks) {
    fetch_to_l2(packed, packed_elems, ((int) blockIdx.x - row_blocks) / 8);
    return;
  }
  __shared__ __attribute__((aligned(16))) uint16_t s_act[2][kMlpRows][kMlpStride];
  __shared__ __attribute__((aligned(16))) uint16_t s_in[kMlpRows][kMlpMaxIn + 8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * kMlpRows;
  const int Din_pad = (Din + 15) & ~15;
  const size_t B_pad = (size_t) row_blocks * kMlpRows;
  const int arow = lane & 15, kofs = 8 * (lane >> 4), col = wave * 32 + (lane & 15);  // and column col + 16

  const uint16_t* W = packed;
  const float* bl   = bias;
  auto tile_of = [&](const uint16_t* Wl, int K_pad_l) { return Wl + wave * (K_pad_l >> 4) * 512; };
  // The weights do not depend on the activations: the first eight k-steps' fragments (and the bias) of the NEXT layer are
  // requested at the start of each layer and arrive while this layer's products, epilogue and barrier run. Nothing else is
  // loaded behind them: loads complete in order, and a wait for a later one would be a wait for all of these.
  // Two register sets take turns: handing one over to the next layer by copies would make the compiler wait for the
  // prefetch where the copies are, in front of the products.
  bf16x8 even[8][2], odd[8][2];
  float bias_even[2] = {bl[col], bl[col + 16]}, bias_odd[2] = {0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (32 * u < Din_pad) load_fragments(tile_of(W, Din_pad), u, (Din_pad >> 4) - 1, even[u]);

  // stage the (bf16) input rows, zero padded to whole k-steps
  constexpr int kInPad = kMlpMaxIn;
  for (int e = threadIdx.x; e < kMlpRows * kInPad; e += kChainThreads) {
    const int r = e / kInPad, k = e - r * kInPad;
    float v = 0.0f;
    if (row0 + r < B && k < Din) v = in ? in[(size_t) (row0 + r) * Din + k] : encoded(freq, row0 + r, k);
    const uint16_t h = f32_to_bf16(v);
    s_in[r][k] = h;
    s_act[0][r][k] = h;
  }
  __syncthreads();
  if (kKeep == Keep::kBatchInnermost) {
    for (int e = threadIdx.x; e < Din * (kMlpRows / 4); e += kChainThreads) {
      const int k = e >> 2, r = (e & 3) * 4;
      const uint16_t h[4] = {s_in[r][k], s_in[r + 1][k], s_in[r + 2][k], s_in[r + 3][k]};
      *(uint2*) (in_t + (size_t) k * B_pad + row0 + r) = pack4(h);
    }
  }

  int cur = 0, K_pad = Din_pad;
  auto run_layer = [&](int layer, const bf16x8 (&b)[8][2], const float (&bv)[2], bf16x8 (&ahead)[8][2], float (&bias_ahead)[2]) {
    floatx4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = 0.0f;
    bf16x8 tail[3][2];
    const int last_step = (K_pad >> 4) - 1;
    if (K_pad > kMlpWidth) {  // the layer behind the re-concatenated input: up to three k-steps more
#pragma unroll
      for (int u = 0; u < 3; ++u) load_fragments(tile_of(W, K_pad), 8 + u, last_step, tail[u]);
    }
    const int K_next = layer == skip ? Din + kMlpWidth : kMlpWidth, K_next_pad = (K_next + 15) & ~15;
    const uint16_t* W_next = W + (size_t) kMlpWidth * K_pad;
    if (layer + 1 < n_layers) {
      bias_ahead[0] = bl[kMlpWidth + col], bias_ahead[1] = bl[kMlpWidth + col + 16];
#pragma unroll
      for (int u = 0; u < 8; ++u) load_fragments(tile_of(W_next, K_next_pad), u, 15, ahead[u]);
    }
    const uint16_t* arow_at = &s_act[cur][arow][kofs];
    auto product = [&](int kk, const bf16x8 (&w)[2]) {
      const bf16x8 a = *(const bf16x8*) (arow_at + 32 * kk);
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[t], acc[t], 0, 0, 0);
    };
    if (K_pad >= kMlpWidth) {
#pragma unroll
      for (int u = 0; u < 8; ++u) product(u, b[u]);
      if (K_pad > kMlpWidth) {
#pragma unroll
        for (int u = 0; u < 3; ++u)
          if (kMlpWidth + 32 * u < K_pad) product(8 + u, tail[u]);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (32 * u < K_pad) product(u, b[u]);
    }
    // bias + ReLU -> bf16 into the other buffer; after the skip layer the input goes in front of the hidden state
    const int nxt = cur ^ 1;
    const int col_shift = (layer == skip) ? Din : 0;
    uint16_t* to = &s_act[nxt][4 * (lane >> 4)][col_shift + col];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = fmaxf(acc[t][k] + bv[t], 0.0f);
      const uint2 h = make_uint2(bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]));
      uint16_t* row = to + 16 * t;
      row[0] = (uint16_t) h.x, row[kMlpStride] = (uint16_t) (h.x >> 16);
      row[2 * kMlpStride] = (uint16_t) h.y, row[3 * kMlpStride] = (uint16_t) (h.y >> 16);
      if (kKeep == Keep::kBatchInnermost)
        *(uint2*) (saved + ((size_t) layer * kMlpWidth + col + 16 * t) * B_pad + row0 + 4 * (lane >> 4)) = h;
      if (kKeep == Keep::kRows) {
        const uint16_t state[4] = {(uint16_t) h.x, (uint16_t) (h.x >> 16), (uint16_t) h.y, (uint16_t) (h.y >> 16)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int r = row0 + 4 * (lane >> 4) + k;
          if (r < B) saved[((size_t) layer * B + r) * kMlpWidth + col + 16 * t] = state[k];
        }
      }
    }
    if (layer == skip) {
      for (int e = threadIdx.x; e < kMlpRows * kInPad; e += kChainThreads) {
        const int r = e / kInPad, k = e - r * kInPad;
        if (k < Din) s_act[nxt][r][k] = s_in[r][k];
        else s_act[nxt][r][kMlpWidth + k] = 0;  // columns Din + 256 .. 256 + kInPad
      }
    }
    lds_barrier();
    W = W_next;
    bl += kMlpWidth;
    K_pad = K_next_pad;
    cur = nxt;
  };
  for (int layer = 0; layer < n_layers; layer += 2) {
    run_layer(layer, even, bias_even, odd, bias_odd);
    if (layer + 1 < n_layers) run_layer(layer + 1, odd, bias_odd, even, bias_even);
  }

  // heads: one padded 32-column tile, wavefront 0 only
  if (wave == 0) {
    bf16x8 b[8][2];
#pragma unroll
    for (int u = 0; u < 8; ++u) load_fragments(W, u, 15, b[u]);
    floatx4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bf16x8 a = *(const bf16x8*) &s_act[cur][arow][kofs + 32 * u];
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[u][t], acc[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int head_col = 16 * t + (lane & 15);
      if (head_col >= n_out) continue;
      const float bv = bl[head_col];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + 4 * (lane >> 4) + r;
        if (row < B) *head_cell(heads, row, head_col) = acc[t][r] + bv;
      }
    }
  }
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t) h << 16); }

// dZ[l] for every layer, back to front, and the outputs' gradient in the same form (g_t[32][B_pad]); in_t (optional): the
// input rows too, for callers whose forward did not leave them. packed_t holds, for l = 1 .. n_layers-1, the hidden part
// of W_l transposed: [256 inputs][256 outputs] bf16. Rows past the batch are zeros in every output.
__global__ void __launch_bounds__(kChainThreads) mlp_backward_chain_kernel(int B, int Din, int n_layers, int n_out,
    const float* __restrict__ in, const float* __restrict__ heads_w /*[n_out][256] fp32*/,
    const uint16_t* __restrict__ packed_t, const uint16_t* __restrict__ saved, MlpHeads heads,
    uint16_t* __restrict__ dz, uint16_t* __restrict__ g_t, uint16_t* __restrict__ in_t, int row_blocks) {
  if ((int) blockIdx.x >= row_blocks) {
    // the last layer's weights are used first: whole layers from the back
    for (int l = n_layers - 1; l >= 1; --l)
      fetch_to_l2(packed_t + (size_t) (l - 1) * kMlpWidth * kMlpWidth, kMlpWidth * kMlpWidth, ((int) blockIdx.x - row_blocks) / 8);
    return;
  }
  constexpr int kStride = kMlpWidth + 8;
  __shared__ __attribute__((aligned(16))) uint16_t s_dz[2][kMlpRows][kStride];
  __shared__ float s_g[kMlpRows][33];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * kMlpRows;
  const size_t B_pad = (size_t) row_blocks * kMlpRows;
  const int arow = lane & 15, kofs = 8 * (lane >> 4), col = wave * 32 + (lane & 15);  // and column col + 16
  auto fetch_weights = [&](int layer, bf16x8 (&b)[8][2]) {
    const uint16_t* tile = packed_t + ((layer - 1) * 8 + wave) * (kMlpWidth / 16) * 512;
#pragma unroll
    for (int u = 0; u < 8; ++u) load_fragments(tile, u, 15, b[u]);
  };
  // the stored states that mask a layer's result: four consecutive rows of a column per load
  auto fetch_mask = [&](int layer, uint2 (&keep)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      keep[t] = *(const uint2*) (saved + ((size_t) layer * kMlpWidth + col + 16 * t) * B_pad + row0 + 4 * (lane >> 4));
  };
  // one layer ahead of their use, the masks in front of the weights (loads complete in order)
  uint2 keep_even[2], keep_odd[2];
  bf16x8 even[8][2], odd[8][2];
  if (n_layers >= 2) fetch_mask(n_layers - 2, keep_even), fetch_weights(n_layers - 1, even);
  for (int e = threadIdx.x; e < kMlpRows * 32; e += kChainThreads) {
    const int r = e >> 5, k = e & 31;
    const float* cell = (row0 + r < B && k < n_out) ? head_cell(heads, row0 + r, k) : nullptr;
    s_g[r][k] = cell ? *cell : 0.0f;
  }
  if (in_t) {
    for (int e = threadIdx.x; e < Din * kMlpRows; e += kChainThreads) {
      const int r = e / Din, k = e - r * Din;
      in_t[(size_t) k * B_pad + row0 + r] = row0 + r < B ? f32_to_bf16(in[(size_t) (row0 + r) * Din + k]) : (uint16_t) 0;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 32 * kMlpRows; e += kChainThreads)
    g_t[(size_t) (e / kMlpRows) * B_pad + row0 + e % kMlpRows] = f32_to_bf16(s_g[e % kMlpRows][e / kMlpRows]);
  {
    // dZ of the last layer: (g_out . W_heads) where the stored state is non-zero. A lane owns 8 rows of one column.
    const int c = threadIdx.x & 255, r0 = 8 * (threadIdx.x >> 8);
    const size_t top = ((size_t) (n_layers - 1) * kMlpWidth + c) * B_pad + row0 + r0;
    const uint4 keep = *(const uint4*) (saved + top);
    float v[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = 0.0f;
    for (int k = 0; k < n_out; ++k) {
      const float wv = heads_w[k * kMlpWidth + c];
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] += s_g[r0 + r][k] * wv;
    }
    const uint32_t words[4] = {keep.x, keep.y, keep.z, keep.w};
    uint32_t h[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool lo = (words[q] & 0xffffu) != 0u && row0 + r0 + 2 * q < B, hi = (words[q] >> 16) != 0u && row0 + r0 + 2 * q + 1 < B;
      h[q] = bf16_pair(lo ? v[2 * q] : 0.0f, hi ? v[2 * q + 1] : 0.0f);
      s_dz[0][r0 + 2 * q][c] = (uint16_t) h[q], s_dz[0][r0 + 2 * q + 1][c] = (uint16_t) (h[q] >> 16);
    }
    *(uint4*) (dz + top) = make_uint4(h[0], h[1], h[2], h[3]);
  }
  __syncthreads();
  int cur = 0;
  auto run_layer = [&](int layer, const bf16x8 (&b)[8][2], const uint2 (&keep)[2], bf16x8 (&ahead)[8][2], uint2 (&keep_ahead)[2]) {
    floatx4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = 0.0f;
    if (layer >= 2) fetch_mask(layer - 2, keep_ahead), fetch_weights(layer - 1, ahead);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bf16x8 a = *(const bf16x8*) &s_dz[cur][arow][32 * u + kofs];
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[u][t], acc[t], 0, 0, 0);
    }
    uint16_t* to = &s_dz[cur ^ 1][4 * (lane >> 4)][col];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float v[4];  // rows past the batch: dZ is zero since the last layer
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = (((k < 2 ? keep[t].x : keep[t].y) >> (16 * (k & 1))) & 0xffffu) != 0u ? acc[t][k] : 0.0f;
      const uint2 h = make_uint2(bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]));
      uint16_t* row = to + 16 * t;
      row[0] = (uint16_t) h.x, row[kStride] = (uint16_t) (h.x >> 16);
      row[2 * kStride] = (uint16_t) h.y, row[3 * kStride] = (uint16_t) (h.y >> 16);
      *(uint2*) (dz + ((size_t) (layer - 1) * kMlpWidth + col + 16 * t) * B_pad + row0 + 4 * (lane >> 4)) = h;
    }
    lds_barrier();
    cur ^= 1;
  };
  for (int layer = n_layers - 1; layer >= 1; layer -= 2) {
    run_layer(layer, even, keep_even, odd, keep_odd);
    if (layer >= 2) run_layer(layer - 1, odd, keep_odd, even, keep_even);
  }
}

// dW_l = dZ_l^T X_l and db_l = row sums of dZ_l for l = 0 .. n_layers (l == n_layers: the heads, whose dZ is g_t).
// X_0 = in, X_{skip+1} = [in | H_skip], X_l = H_{l-1} otherwise, all with the batch innermost. g_w is the layers' [256][K_l]
// gradients back to back followed by the heads' [n_out][256]; g_b has the layout of the forward's bias vector.
constexpr int kWgTile = 64;
constexpr int kWgSteps = 8;  // k-steps of 16 rows that a wavefront has in flight
__global__ void __launch_bounds__(kMlpThreads) mlp_backward_weights_kernel(int B, int Din, int n_layers, int skip,
    int n_out, const uint16_t* __restrict__ in_t, const uint16_t* __restrict__ saved, const uint16_t* __restrict__ dz,
    const uint16_t* __restrict__ g_t, float* __restrict__ g_w, float* __restrict__ g_b) {
  __shared__ float s_sum[kWgTile][kWgTile + 1];
  __shared__ float s_bias[kMlpThreads / kWave][kWgTile];
  // which (layer, output tile, input tile) this block owns
  int layer = 0, K = Din, tile = blockIdx.x;
  size_t w_off = 0;
  for (;; ++layer) {
    const int rows = layer < n_layers ? kMlpWidth : n_out;
    const int tiles = div_up_dev(rows, kWgTile) * div_up_dev(K, kWgTile);
    if (tile < tiles || layer == n_layers) break;
    tile -= tiles;
    w_off += (size_t) rows * K;
    K = (layer == skip) ? Din + kMlpWidth : kMlpWidth;
  }
  const int rows = layer < n_layers ? kMlpWidth : n_out, across = div_up_dev(K, kWgTile);
  const int o0 = (tile / across) * kWgTile, i0 = (tile % across) * kWgTile;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kofs = 8 * (lane >> 5);
  const size_t B_pad = (size_t) ((B + kMlpRowPad - 1) / kMlpRowPad) * kMlpRowPad;
  const int shift = layer == 0 ? Din : (layer == skip + 1 ? Din : 0);  // columns of X_l that are the input
  const uint16_t *arow[2], *brow[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int o = min(o0 + 32 * t + (lane & 31), rows - 1), i = min(i0 + 32 * t + (lane & 31), K - 1);
    arow[t] = (layer < n_layers ? dz + ((size_t) layer * kMlpWidth + o) * B_pad : g_t + (size_t) o * B_pad) + kofs;
    brow[t] = (i < shift ? in_t + (size_t) i * B_pad
                         : saved + ((size_t) (layer - 1) * kMlpWidth + (i - shift)) * B_pad) + kofs;
  }
  floatx16 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0.0f;
  float bias[2] = {0.0f, 0.0f};
  const bool wants_bias = i0 == 0;
  const int last = (int) B_pad - 16;
  constexpr int kChunk = 16 * kWgSteps;
  for (int b0 = wave * kChunk; b0 < (int) B_pad; b0 += (kMlpThreads / kWave) * kChunk) {
    bf16x8 a[2][kWgSteps], b[2][kWgSteps];
#pragma unroll
    for (int u = 0; u < kWgSteps; ++u) {
      const int at = min(b0 + 16 * u, last);
#pragma unroll
      for (int t = 0; t < 2; ++t) a[t][u] = *(const bf16x8*) (arow[t] + at), b[t][u] = *(const bf16x8*) (brow[t] + at);
    }
#pragma unroll
    for (int u = 0; u < kWgSteps; ++u) {
      if (b0 + 16 * u > last) break;  // uniform
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x][u], b[y][u], acc[x][y], 0, 0, 0);
      if (wants_bias) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int k = 0; k < 8; ++k) bias[t] += (float) a[t][u][k];
      }
    }
  }
  if (wants_bias) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bias[t] += __shfl_xor(bias[t], 32, kWave);
      if (lane < 32) s_bias[wave][32 * t + lane] = bias[t];
    }
  }
  // the wavefronts' sums in wavefront order
  for (int w = 0; w < kMlpThreads / kWave; ++w) {
    if (wave == w) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float* cell = &s_sum[32 * x + acc_row(r, lane)][32 * y + (lane & 31)];
            *cell = w == 0 ? acc[x][y][r] : *cell + acc[x][y][r];
          }
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < kWgTile * kWgTile; e += kMlpThreads) {
    const int o = e >> 6, i = e & 63;
    if (o0 + o < rows && i0 + i < K) g_w[w_off + (size_t) (o0 + o) * K + i0 + i] = s_sum[o][i];
  }
  if (wants_bias && threadIdx.x < kWgTile && o0 + (int) threadIdx.x < rows) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kMlpThreads / kWave; ++w) v += s_bias[w][threadIdx.x];
    g_b[(size_t) layer * kMlpWidth + o0 + threadIdx.x] = v;
  }
}

// Hidden states or their gradients between the callers' rows [layer][B][256] and the kernels' [layer][256][B_pad] (zeros
// past the batch), 32 x 32 through LDS: grid (B_pad / 32, 8, layers).
template <bool kToRows>
__global__ void __launch_bounds__(256) mlp_transpose_kernel(int B, int B_pad, const uint16_t* __restrict__ from,
                                                            uint16_t* __restrict__ to) {
  __shared__ uint16_t s_tile[32][33];
  const int x = threadIdx.x & 31, r0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const size_t rows = (size_t) blockIdx.z * B, columns = (size_t) blockIdx.z * kMlpWidth;
  for (int y = threadIdx.x >> 5; y < 32; y += 8) {
    if (kToRows) s_tile[y][x] = from[(columns + c0 + y) * B_pad + r0 + x];
    else s_tile[y][x] = r0 + y < B ? from[(rows + r0 + y) * kMlpWidth + c0 + x] : (uint16_t) 0;
  }
  __syncthreads();
  for (int y = threadIdx.x >> 5; y < 32; y += 8) {
    if (!kToRows) to[(columns + c0 + y) * B_pad + r0 + x] = s_tile[x][y];
    else if (r0 + y < B) to[(rows + r0 + y) * kMlpWidth + c0 + x] = s_tile[x][y];
  }
}

}  // namespace
}  // namespace fsgs

using namespace fsgs;

FSGS_API int fsgs_pack_bf16(int rows, int K, int rows_pad, int K_pad, const float* src, uint16_t* dst, void* stream) {
  FSGS_REQUIRE(rows > 0 && K > 0 && rows_pad >= rows && K_pad >= K && src && dst, "pack_bf16: bad arguments");
  FSGS_REQUIRE(rows_pad % 32 == 0 && K_pad % 16 == 0, "pack_bf16: rows_pad must be a multiple of 32 and K_pad of 16");
  hipLaunchKernelGGL(pack_bf16_kernel, dim3(div_up((int64_t) rows_pad * K_pad, 256)), dim3(256), 0,
                     (hipStream_t) stream, rows, K, rows_pad, K_pad, src, dst);
  return check_launch("pack_bf16");
}

// All buffers the fused network reads, refreshed from the fp32 parameters in one launch: `packed` (what
// fsgs_mlp_forward reads: the layers' fragment matrices, then the heads stacked into one [32][256] matrix), `packed_t`
// (optional; what fsgs_mlp_backward reads: [n_layers - 1][256 in][256 out] fragments of the last 256 input columns of
// layers 1..), `bias_out` (layer biases then head biases) and `heads_w_out` (the heads' fp32 rows stacked).
FSGS_API int fsgs_mlp_pack_all(int Din, int n_layers, int skip, const float* const* weights,
    const float* const* biases, int n_heads, const float* const* head_weights, const float* const* head_biases,
    const int* head_rows, uint16_t* packed, uint16_t* packed_t, float* bias_out, float* heads_w_out, void* stream) {
  FSGS_REQUIRE(Din > 0 && n_layers >= 1 && skip < n_layers - 1 && weights && biases && packed && bias_out,
               "mlp_pack_all: bad arguments");
  FSGS_REQUIRE(n_heads >= 0 && (n_heads == 0 || (head_weights && head_biases && head_rows && heads_w_out)),
               "mlp_pack_all: bad head arguments");
  FSGS_REQUIRE(2 * n_layers + 3 * n_heads + (packed_t ? n_layers - 1 : 0) <= kMaxPackJobs,
               "mlp_pack_all: too many layers / heads for one launch (%d jobs at most)", kMaxPackJobs);
  PackTable table{};
  int n = 0, most = 0;
  auto add = [&](const PackJob& j) {
    most = std::max(most, j.kind == 2 ? j.rows : j.rows_cover * j.K_pad);
    table.job[n++] = j;
  };
  size_t off = 0;
  int K = Din;
  for (int l = 0; l < n_layers; ++l) {
    FSGS_REQUIRE(weights[l] && biases[l], "mlp_pack_all: null layer tensor");
    const int K_pad = (K + 15) & ~15;
    add({weights[l], packed + off, kMlpWidth, K, kMlpWidth, K_pad, 0, K, 0, 0});
    add({biases[l], bias_out + (size_t) l * kMlpWidth, kMlpWidth, 0, 0, 0, 0, 0, 0, 2});
    if (packed_t && l > 0)
      add({weights[l], packed_t + (size_t) (l - 1) * kMlpWidth * kMlpWidth, kMlpWidth, kMlpWidth, kMlpWidth,
           kMlpWidth, 0, K, K - kMlpWidth, 1});
    off += (size_t) kMlpWidth * K_pad;
    K = (l == skip) ? Din + kMlpWidth : kMlpWidth;
  }
  FSGS_REQUIRE(K == kMlpWidth, "mlp_pack_all: the heads must follow a %d-wide layer", kMlpWidth);
  int row0 = 0;
  for (int h = 0; h < n_heads; ++h) {
    FSGS_REQUIRE(head_weights[h] && head_biases[h] && head_rows[h] > 0, "mlp_pack_all: bad head tensor");
    const bool last = h == n_heads - 1;
    FSGS_REQUIRE(row0 + head_rows[h] <= 32, "mlp_pack_all: the heads have more than 32 rows together");
    add({head_weights[h], packed + off, head_rows[h], kMlpWidth, last ? 32 - row0 : head_rows[h], kMlpWidth, row0,
         kMlpWidth, 0, 0});
    add({head_biases[h], bias_out + (size_t) n_layers * kMlpWidth + row0, head_rows[h], 0, 0, 0, 0, 0, 0, 2});
    add({head_weights[h], heads_w_out + (size_t) row0 * kMlpWidth, head_rows[h] * kMlpWidth, 0, 0, 0, 0, 0, 0, 2});
    row0 += head_rows[h];
  }
  if (n_heads == 0) add({weights[0], packed + off, 0, kMlpWidth, 32, kMlpWidth, 0, kMlpWidth, 0, 0});  // zero head block
  hipLaunchKernelGGL(pack_jobs_kernel, dim3(div_up(most, 256), n), dim3(256), 0, (hipStream_t) stream, table);
  return check_launch("mlp_pack_all");
}

// Number of bf16 elements of the packed weight buffer: per layer [256][K_pad_i], then the heads as [32][K_pad_last].
FSGS_API size_t fsgs_mlp_packed_elems(int Din, int n_layers, int skip) {
  size_t n = 0;
  int K = Din;
  for (int l = 0; l < n_layers; ++l) {
    n += (size_t) kMlpWidth * ((K + 15) & ~15);
    K = (l == skip) ? Din + kMlpWidth : kMlpWidth;
  }
  n += (size_t) 32 * ((K + 15) & ~15);
  return n;
}

namespace {
size_t padded_rows(int B) { return (size_t) div_up(std::max(B, 1), kMlpRowPad) * kMlpRowPad; }

bool make_heads(MlpHeads& h, int n_heads, const int* head_rows, float* const* at) {
  if (n_heads < 1 || n_heads > kMaxHeads) return false;
  h.n = n_heads, h.first[0] = 0;
  for (int k = 0; k < n_heads; ++k) {
    if (head_rows[k] < 1) return false;
    h.at[k] = at[k], h.first[k + 1] = h.first[k] + head_rows[k];
  }
  return h.first[n_heads] <= 32;
}
}  // namespace

FSGS_API size_t fsgs_mlp_saved_elems(int B, int n_layers) { return (size_t) n_layers * kMlpWidth * padded_rows(B); }
FSGS_API size_t fsgs_mlp_saved_input_elems(int B, int Din) { return (size_t) Din * padded_rows(B); }

namespace {
int launch_forward(Keep keep, int B, int Din, int width, int n_layers, int skip, int n_heads, const int* head_rows,
    const float* in, const FreqInput& freq, const uint16_t* packed, const float* bias, float* const* outs, uint16_t* saved_in,
    uint16_t* saved, void* stream) {
  FSGS_REQUIRE(B >= 0 && (in || (freq.x && freq.t)) && packed && bias && head_rows && outs, "mlp_forward: bad arguments");
  FSGS_REQUIRE(in || (freq.degree_x >= 0 && freq.degree_t >= 0 && Din == 3 * (1 + 2 * freq.degree_x) + 1 + 2 * freq.degree_t),
               "mlp_forward: the encoding has another width than the network's input");
  FSGS_REQUIRE(width == kMlpWidth, "mlp_forward: width %d is not supported (only %d)", width, kMlpWidth);
  FSGS_REQUIRE(Din > 0 && ((Din + 15) & ~15) <= kMlpMaxIn, "mlp_forward: input width %d exceeds %d", Din, kMlpMaxIn);
  MlpHeads heads{};
  FSGS_REQUIRE(make_heads(heads, n_heads, head_rows, outs), "mlp_forward: bad heads (at most %d with 32 rows)", kMaxHeads);
  for (int h = 0; h < n_heads; ++h) FSGS_REQUIRE(outs[h], "mlp_forward: null output");
  const int n_out = heads.first[n_heads];
  FSGS_REQUIRE(n_layers >= 1 && skip < n_layers - 1, "mlp_forward: bad layer structure (layers %d, skip %d, outputs %d)",
               n_layers, skip, n_out);
  if (B == 0) return kOk;
  auto kernel = keep == Keep::kNothing ? mlp_forward_kernel<Keep::kNothing>
                : keep == Keep::kRows  ? mlp_forward_kernel<Keep::kRows>
                                       : mlp_forward_kernel<Keep::kBatchInnermost>;
  const int row_blocks = (int) (padded_rows(B) / kMlpRows);
  hipLaunchKernelGGL(kernel, dim3(row_blocks + (row_blocks < kFetchBelow ? kFetchBlocks : 0)), dim3(kChainThreads), 0,
                     (hipStream_t) stream, B, Din, n_layers, skip, n_out, in, freq, packed, bias, heads, saved_in, saved,
                     row_blocks, fsgs_mlp_packed_elems(Din, n_layers, skip));
  return check_launch("mlp_forward");
}
}  // namespace

FSGS_API int fsgs_deform_mlp_forward(int B, int Din, int width, int n_layers, int skip, int n_heads, const int* head_rows,
    const float* in, const float* x, const float* t, int degree_x, double scale_x, int degree_t, double scale_t,
    const uint16_t* packed, const float* bias, float* const* outs, uint16_t* saved_in, uint16_t* saved, void* stream) {
  FSGS_REQUIRE((saved == nullptr) == (saved_in == nullptr), "mlp_forward: saved_in and saved go together");
  return launch_forward(saved ? Keep::kBatchInnermost : Keep::kNothing, B, Din, width, n_layers, skip, n_heads, head_rows, in,
                        FreqInput{x, t, degree_x, degree_t, (float) scale_x, (float) scale_t}, packed, bias, outs, saved_in,
                        saved, stream);
}

FSGS_API size_t fsgs_deform_mlp_backward_workspace_bytes(int B, int Din, int n_layers) {
  if (B < 0 || n_layers < 1 || Din < 1) return 0;
  return align_up(((size_t) n_layers * kMlpWidth + 32 + Din) * padded_rows(B) * sizeof(uint16_t), 256);
}

FSGS_API int fsgs_deform_mlp_backward(int B, int Din, int width, int n_layers, int skip, int n_heads, const int* head_rows,
    const float* in, const uint16_t* saved_in, const uint16_t* packed_t, const float* heads_w, const uint16_t* saved,
    const float* const* g_outs, float* g_w, float* g_b, void* workspace, size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(B >= 0 && (in || saved_in) && packed_t && heads_w && saved && head_rows && g_outs && g_w && g_b && workspace,
               "mlp_backward: bad arguments");
  FSGS_REQUIRE(width == kMlpWidth, "mlp_backward: width %d is not supported (only %d)", width, kMlpWidth);
  FSGS_REQUIRE(Din > 0 && ((Din + 15) & ~15) <= kMlpMaxIn, "mlp_backward: input width %d exceeds %d", Din, kMlpMaxIn);
  MlpHeads heads{};
  FSGS_REQUIRE(make_heads(heads, n_heads, head_rows, (float* const*) g_outs), "mlp_backward: bad heads");
  const int n_out = heads.first[n_heads];
  FSGS_REQUIRE(n_layers >= 1 && n_layers <= 64 && skip < n_layers - 1,
               "mlp_backward: bad layer structure (layers %d, skip %d, outputs %d)", n_layers, skip, n_out);
  if (workspace_bytes < fsgs_deform_mlp_backward_workspace_bytes(B, Din, n_layers))
    return fail(kWorkspaceSmall, "mlp_backward: workspace %zu < %zu bytes", workspace_bytes,
                fsgs_deform_mlp_backward_workspace_bytes(B, Din, n_layers));
  hipStream_t s = (hipStream_t) stream;
  const size_t B_pad = padded_rows(B);
  uint16_t* dz   = (uint16_t*) workspace;
  uint16_t* g_t  = dz + (size_t) n_layers * kMlpWidth * B_pad;
  uint16_t* in_t = saved_in ? nullptr : g_t + 32 * B_pad;
  if (B == 0) {  // no rows: the gradients are zeros
    const size_t n_w = (size_t) kMlpWidth * Din * (skip >= 0 ? 2 : 1) + (size_t) (n_layers - 1) * kMlpWidth * kMlpWidth +
                       (size_t) n_out * kMlpWidth;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(256), dim3(256), 0, s, n_w, g_w);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(16), dim3(256), 0, s, (size_t) n_layers * kMlpWidth + n_out, g_b);
    return check_launch("mlp_backward");
  }
  const int row_blocks = (int) (padded_rows(B) / kMlpRows);
  hipLaunchKernelGGL(mlp_backward_chain_kernel, dim3(row_blocks + (row_blocks < kFetchBelow ? kFetchBlocks : 0)),
                     dim3(kChainThreads), 0, s, B, Din, n_layers, n_out, in, heads_w, packed_t, saved, heads, dz, g_t, in_t,
                     row_blocks);
  int tiles = 0, K = Din;
  for (int l = 0; l <= n_layers; ++l) {
    tiles += div_up(l < n_layers ? kMlpWidth : n_out, kWgTile) * div_up(K, kWgTile);
    K = (l == skip) ? Din + kMlpWidth : kMlpWidth;
  }
  hipLaunchKernelGGL(mlp_backward_weights_kernel, dim3(tiles), dim3(kMlpThreads), 0, s, B, Din, n_layers, skip, n_out,
                     saved_in ? saved_in : in_t, saved, dz, g_t, g_w, g_b);
  return check_launch("mlp_backward");
}

// The entry points whose callers keep the states as rows. The backward lays them out for the kernels and its result dZ back.
FSGS_API int fsgs_mlp_forward(int B, int Din, int width, int n_layers, int skip, int n_out, const float* in,
                              const uint16_t* packed, const float* bias, float* out, uint16_t* saved, void* stream) {
  FSGS_REQUIRE(in && out, "mlp_forward: bad arguments");
  return launch_forward(saved ? Keep::kRows : Keep::kNothing, B, Din, width, n_layers, skip, 1, &n_out, in, FreqInput{}, packed,
                        bias, &out, nullptr, saved, stream);
}

namespace {
struct RowsWorkspace {  // dZ as rows | the states batch innermost | the kernels' own, dZ batch innermost in front
  size_t states, own, bytes;
  RowsWorkspace(int B, int n_layers) {
    states = align_up((size_t) n_layers * std::max(B, 1) * kMlpWidth * sizeof(uint16_t), 256);
    own    = states + align_up(fsgs_mlp_saved_elems(B, n_layers) * sizeof(uint16_t), 256);
    bytes  = own + fsgs_deform_mlp_backward_workspace_bytes(B, kMlpMaxIn, n_layers);
  }
};
}  // namespace

FSGS_API size_t fsgs_mlp_backward_workspace_bytes(int B, int n_layers) {
  return B < 0 || n_layers < 1 ? 0 : RowsWorkspace(B, n_layers).bytes;
}

FSGS_API int fsgs_mlp_backward(int B, int Din, int width, int n_layers, int skip, int n_out, const float* in,
    const uint16_t* packed_t, const float* heads_w, const uint16_t* saved, const float* g_out, float* g_w, float* g_b,
    void* workspace, size_t workspace_bytes, void* stream) {
  FSGS_REQUIRE(B >= 0 && in && saved && g_out && workspace, "mlp_backward: bad arguments");
  FSGS_REQUIRE(n_layers >= 1 && n_layers <= 64, "mlp_backward: bad layer structure (%d layers)", n_layers);
  const RowsWorkspace at(B, n_layers);
  if (workspace_bytes < at.bytes) return fail(kWorkspaceSmall, "mlp_backward: workspace %zu < %zu bytes", workspace_bytes, at.bytes);
  uint16_t* rows   = (uint16_t*) workspace;
  uint16_t* states = (uint16_t*) ((char*) workspace + at.states);
  uint16_t* own    = (uint16_t*) ((char*) workspace + at.own);
  const int B_pad = (int) padded_rows(B);
  const dim3 grid(B_pad / 32, kMlpWidth / 32, n_layers);
  if (B > 0)
    hipLaunchKernelGGL(mlp_transpose_kernel<false>, grid, dim3(256), 0, (hipStream_t) stream, B, B_pad, saved, states);
  const int rc = fsgs_deform_mlp_backward(B, Din, width, n_layers, skip, 1, &n_out, in, nullptr, packed_t, heads_w, states,
                                          &g_out, g_w, g_b, own, at.bytes - at.own, stream);
  if (rc != kOk || B == 0) return rc;
  hipLaunchKernelGGL(mlp_transpose_kernel<true>, grid, dim3(256), 0, (hipStream_t) stream, B, B_pad, own, rows);
  return check_launch("mlp_backward");
}
