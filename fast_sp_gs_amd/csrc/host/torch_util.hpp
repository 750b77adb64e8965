// Shared pieces of the native host layer: argument checks with the operators' error texts, output allocation, and the two
// small resources a view needs besides its tensors (a pinned word for the instance count, zeroed slot counters).
//
// This layer does in C++ what the Python operators do for one whole render call: check, allocate, launch, record one
// autograd node. A render of 10k surfels keeps the GPU busy for 0.08 ms and its backward for 0.09 ms; marshalling its 13 to
// 20 launches through Python took 0.14 and 0.4 ms.
#pragma once
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>

#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../../include/fsgs.h"

namespace fsgs_host {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int kTile = 16, kSlotRegions = 64;

[[noreturn]] inline void fail(const std::string& text) { throw std::runtime_error(text); }

inline void check(int rc, const char* what) {
  if (rc == 0) return;
  const char* text = fsgs_last_error();
  fail(std::string(what) + ": " + (text && *text ? text : "error") + " (status " + std::to_string(rc) + ")");
}

std::string shape_text(at::IntArrayRef shape);
std::string dtype_text(at::ScalarType type);

// A device tensor, contiguous, of the given type (the operators' CHECK_INPUT).
void require(const char* what, const char* name, const Tensor& t, at::ScalarType type);
void require_shape(const char* what, const char* name, const Tensor& t, at::IntArrayRef shape);
inline bool has(const OptTensor& t) { return t.has_value() && t->defined(); }
inline Tensor opt(const OptTensor& t) { return has(t) ? *t : Tensor(); }

// Forward-mode derivatives are not implemented; a dual tensor would lose its tangent on the way through a kernel. There
// are dual tensors only while a dual level (torch has one, 0) is open.
inline bool is_dual(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }
inline bool is_dual(const OptTensor& t) { return has(t) && is_dual(*t); }
template <typename... T>
void refuse_duals(const char* what, const T&... t) {
  if (torch::autograd::ForwardADLevel::try_get_by_idx(0) && (is_dual(t) || ...))
    fail(std::string(what) + ": forward-mode differentiation is not implemented");
}

// Stored SH coefficients per point beside the split-off first one: checks [P,M,3] (or [P,1,3] + [P,M,3], or colours [P,3]
// for degree < 0) and returns M.
int sh_coefficients(const char* what, const Tensor& shs, const OptTensor& sh_rest, int sh_degree, int64_t P);
void require_point_mask(const char* what, const OptTensor& culling, int64_t P);
void require_accumulators(const char* what, const OptTensor& max_count, const OptTensor& weights_p,
                          const OptTensor& weights_count, int64_t P);

template <typename T>
T* data(const Tensor& t) {
  return t.defined() ? (T*) t.data_ptr() : nullptr;
}
inline float* f32(const Tensor& t) { return data<float>(t); }
inline int32_t* i32(const Tensor& t) { return data<int32_t>(t); }
inline int64_t* i64(const Tensor& t) { return data<int64_t>(t); }

inline Tensor empty(at::IntArrayRef shape, const Tensor& like, at::ScalarType type = at::kFloat) {
  return at::empty(shape, like.options().dtype(type));
}
inline Tensor contiguous(const Tensor& t) { return t.defined() ? t.contiguous() : t; }

// `part`, a tensor over some of `whole`'s storage made outside the graph, as an output of its own that counts edits with
// `whole`: the backward reads that storage, and an in-place edit of either has to be noticed there.
Tensor sharing_edits(const Tensor& whole, Tensor part);

// A node's gradients come from kernels, outside the graph. Where the backward itself is recorded (create_graph=True) they
// get a node that raises when it is differentiated, reached from what they depend on (the upstream gradients and the saved
// inputs); without it they would pass for constants.
variable_list first_order_only(const variable_list& upstream, const variable_list& inputs, variable_list grads);

inline void* stream_of(const Tensor& t) { return (void*) c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// One uninitialised allocation handed out in 256-byte aligned pieces: a view's scratch, or what only its backward reads.
class Slab {
 public:
  size_t reserve(size_t bytes) {
    const size_t at = size_;
    size_ = (size_ + bytes + 255) / 256 * 256;
    return at;
  }
  void allocate(const Tensor& like) { memory_ = empty({(int64_t) (size_ ? size_ : 1)}, like, at::kByte); }
  template <typename T>
  T* at(size_t offset) const {
    return (T*) ((char*) memory_.data_ptr() + offset);
  }
  const Tensor& memory() const { return memory_; }

 private:
  size_t size_ = 0;
  Tensor memory_;
};

// Page-locked word the instance count of a view is stored to; one per host thread (a thread waits for its count before
// it starts the next view).
int64_t* pinned_count();

// The count of a view whose counting kernel has been queued. The word is the thread's next view's, too, so whoever leaves without
// the count (an allocation that failed) waits for it here.
class PendingCount {
 public:
  PendingCount(int64_t* word, void* stream) : word_(word), stream_(stream) {}
  PendingCount(const PendingCount&) = delete;
  PendingCount& operator=(const PendingCount&) = delete;
  ~PendingCount() {
    if (!known_) (void) fsgs_gs_view_wait(word_, stream_);
  }
  bool arrived() const { return __atomic_load_n(word_, __ATOMIC_ACQUIRE) >= 0; }
  int64_t wait(const char* what) {
    const int rc = fsgs_gs_view_wait(word_, stream_);
    known_ = true;  // or the stream has failed
    check(rc, what);
    return *word_;
  }

 private:
  int64_t* word_;
  void* stream_;
  bool known_ = false;
};

// Room for the instances of a view whose count is not known yet; 0: wait for the count. A surfel has at most one instance per tile,
// and on average fewer than 16 unless the surfels are large (2 to 8 in ordinary scenes); beyond 2^18 surfels the device is busy
// with the counting for longer than the host needs to wait and go on.
inline int64_t instances_to_guess(int64_t P, int64_t T) {
  if (P > (1 << 18) || T > (1 << 14)) return 0;
  return std::min(P * T, std::max<int64_t>(16 * P, 1 << 16));
}

// A view's instances, scattered into its tiles' segments, and their number.
struct Instances {
  Tensor space;      // fsgs_gs_view_lists_workspace_bytes(room) bytes
  int64_t room = 0;  // for that many
  int64_t count = 0;
};

// The scatter is queued for a guess, so that the device has something to do until the host has seen the count and launched the
// sort; only what lives no longer than the view is sized by the guess. A guess that was too small, or that memory does not suffice
// for, costs an empty launch, and the scatter is queued again for the count.
// Six processes each in turn, with the wait in front of the scatter -> so, fastest and median us: view of 10k surfels 256x256 50.7 and
// 57.4 -> 49.4 and 55.7, of 25k Gaussians 639x361 51.1 and 55.4 -> 50.4 and 54.6; dynamic frame of 50k and iteration of 200k equal
// within what the runs of one side differ. Counts above the guess (5000 surfels of 43 pixels 800x800, 1.7M instances): 426, 442
// with the wait and a larger workspace.
// `scatter(instances)` queues the kernel, `meanwhile()` allocates what does not depend on the count (before
// the guess, which can do without).
template <typename Scatter, typename Meanwhile>
Instances scatter_instances(const char* what, PendingCount& pending, int64_t guess, const Tensor& like, Scatter scatter,
                            Meanwhile meanwhile) {
  Instances in;
  auto queue = [&](int64_t room) {
    in.space = empty({(int64_t) fsgs_gs_view_lists_workspace_bytes(room)}, like, at::kByte);
    in.room  = room;
    scatter(in);
  };
  meanwhile();
  if (guess > 0 && !pending.arrived()) {
    try {
      queue(guess);
    } catch (const c10::OutOfMemoryError&) {
    }
  }
  in.count = pending.wait(what);
  if (in.count > in.room) queue(in.count);
  return in;
}

// A view's scratch. A small view (fsgs_gs_view_gathers) has its lists gathered tile by tile, by way of `rects` and `lists`, the others
// are binned by way of `bins`, and so is a small one for whose lists (4 KB a tile) there is no memory.
struct ViewScratch {
  bool small = false;
  size_t depths = 0, masks = 0, bins = 0, bins_bytes = 0, rects = 0, lists = 0, lists_bytes = 0;
  Slab slab;
  ViewScratch(int64_t P, int W, int H, const Tensor& like) {
    if (fsgs_gs_view_gathers((int) P, W, H)) {
      try {
        lay_out(P, W, H, like, true);
        return;
      } catch (const c10::OutOfMemoryError&) {
      }
    }
    lay_out(P, W, H, like, false);
  }
  template <typename T>
  T* at(size_t offset) const {
    return slab.at<T>(offset);
  }
  uint32_t* small_rects() const { return small ? slab.at<uint32_t>(rects) : nullptr; }

 private:
  void lay_out(int64_t P, int W, int H, const Tensor& like, bool as_small) {
    slab = Slab(), small = as_small;
    depths = slab.reserve((size_t) P * 4), masks = slab.reserve((size_t) P * 4);
    lists_bytes = small ? fsgs_gs_view_gather_bytes(W, H) : 0, bins_bytes = small ? 0 : fsgs_gs_prepare_bins_bytes((int) P, W, H);
    if (small) rects = slab.reserve((size_t) (P + 255) / 256 * 1024), lists = slab.reserve(lists_bytes);
    else bins = slab.reserve(bins_bytes);
    slab.allocate(like);
  }
};

// 65 zeroed counters on the tensor's device for one view on its current stream. They go back to a list of that stream
// once the kernel that zeroes them again is queued; a view that fails in between drops them.
class SlotCounters {
 public:
  explicit SlotCounters(const Tensor& like);
  uint64_t* data() const { return (uint64_t*) memory_.data_ptr(); }
  void give_back();

 private:
  Tensor memory_;
  std::pair<int, void*> key_;
};

// Both parts of a small view's binning (`regions` optional), behind a preprocess kernel that stores the count to `count`; `meanwhile()`
// allocates what does not depend on it. Returns the list of as many places as there are instances.
template <typename Meanwhile>
Tensor small_view_lists(const ViewScratch& scratch, int64_t P, int W, int H, const uint32_t* masks, SlotCounters& counters,
                        int32_t* regions, const Tensor& ranges, int64_t* count, void* stream, Meanwhile meanwhile) {
  const char* what = "GS_prepare";
  PendingCount pending(count, stream);
  const float* depths = scratch.at<float>(scratch.depths);
  check(fsgs_gs_view_gather((int) P, W, H, depths, scratch.small_rects(), masks, counters.data(), regions, nullptr,
                            scratch.at<void>(scratch.lists), scratch.lists_bytes, stream),
        what);
  counters.give_back();
  meanwhile();
  // for lists too long to be sorted by their own blocks, as many entries as there may be: nearly always that is enough
  Tensor space;
  try {
    space = empty({16 * P * 8}, ranges, at::kByte);
  } catch (const c10::OutOfMemoryError&) {
  }
  const int64_t R = pending.wait(what);
  const Tensor list = empty({R}, ranges, at::kInt);
  if (!space.defined() || 8 * R > space.numel()) space = empty({8 * std::max<int64_t>(R, 1)}, ranges, at::kByte);
  check(fsgs_gs_view_place((int) P, W, H, depths, scratch.small_rects(), masks, R, i64(ranges), i32(list),
                           scratch.at<void>(scratch.lists), scratch.lists_bytes, space.data_ptr(), space.numel(), stream),
        what);
  return list;
}

}  // namespace fsgs_host
