#include "torch_util.hpp"

#include <torch/csrc/autograd/functions/basic_ops.h>

#include <map>

namespace fsgs_host {

std::string shape_text(at::IntArrayRef shape) {
  std::string s = "(";
  for (size_t i = 0; i < shape.size(); ++i) s += (i ? ", " : "") + std::to_string(shape[i]);
  return s + (shape.size() == 1 ? ",)" : ")");
}

std::string dtype_text(at::ScalarType type) {
  switch (type) {
    case at::kFloat: return "torch.float32";
    case at::kDouble: return "torch.float64";
    case at::kHalf: return "torch.float16";
    case at::kBFloat16: return "torch.bfloat16";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    case at::kBool: return "torch.bool";
    case at::kByte: return "torch.uint8";
    default: return c10::toString(type);
  }
}

void require(const char* what, const char* name, const Tensor& t, at::ScalarType type) {
  if (!t.is_cuda()) fail(std::string(what) + ": " + name + " must be a CUDA tensor");
  if (!t.is_contiguous()) fail(std::string(what) + ": " + name + " must be contiguous");
  if (t.scalar_type() != type)
    fail(std::string(what) + ": " + name + " must have dtype " + dtype_text(type) + ", got " + dtype_text(t.scalar_type()));
}

void require_shape(const char* what, const char* name, const Tensor& t, at::IntArrayRef shape) {
  if (t.sizes() != shape)
    fail(std::string(what) + ": " + name + " must have shape " + shape_text(shape) + ", got " + shape_text(t.sizes()));
}

int sh_coefficients(const char* what, const Tensor& shs, const OptTensor& sh_rest, int sh_degree, int64_t P) {
  const int64_t need = (int64_t) (1 + sh_degree) * (1 + sh_degree);
  const bool rest = has(sh_rest) && sh_rest->numel() > 0;
  const Tensor& table = rest ? *sh_rest : shs;
  if (rest) require(what, "sh_rest", table, at::kFloat);
  if (rest || sh_degree >= 0) {
    const auto s = table.sizes();
    if (!(s.size() == 3 && s[0] == P && s[1] >= need - (rest ? 1 : 0) && s[2] == 3)) fail("Error shape for sh features");
  }
  // what is read of shs itself: the colours, the first coefficients beside sh_rest, or the table above
  if (sh_degree < 0) require_shape(what, "shs", shs, {P, 3});
  else if (rest && shs.numel() < 3 * P) fail("Error shape for sh features");
  return table.dim() == 3 ? (int) table.size(1) : 0;
}

void require_point_mask(const char* what, const OptTensor& culling, int64_t P) {
  if (!has(culling)) return;
  require(what, "culling", *culling, at::kBool);
  require_shape(what, "culling", *culling, {P});
}

void require_accumulators(const char* what, const OptTensor& max_count, const OptTensor& weights_p,
                          const OptTensor& weights_count, int64_t P) {
  auto one = [&](const char* name, const OptTensor& t, at::ScalarType type) {
    if (!has(t)) return;
    require(what, name, *t, type);
    require_shape(what, name, *t, {P});
  };
  one("accum_max_count", max_count, at::kInt);
  one("accum_weights_count", weights_count, at::kInt);
  one("accum_weights_p", weights_p, at::kFloat);
}

Tensor sharing_edits(const Tensor& whole, Tensor part) {
  namespace impl = torch::autograd::impl;
  impl::set_version_counter(part, impl::version_counter(whole));
  return part;
}

variable_list first_order_only(const variable_list& upstream, const variable_list& inputs, variable_list grads) {
  bool recorded = false;
  if (at::GradMode::is_enabled())
    for (const Tensor& g : upstream) recorded = recorded || (g.defined() && g.requires_grad());
  if (!recorded) return grads;
  variable_list from = upstream;
  from.insert(from.end(), inputs.begin(), inputs.end());
  const auto refuse = std::make_shared<torch::autograd::Error>(
      "trying to differentiate twice a function whose backward is differentiable once only",
      torch::autograd::collect_next_edges(from));
  for (Tensor& g : grads)
    if (g.defined()) torch::autograd::create_gradient_edge(g = g.detach(), refuse);
  return grads;
}

int64_t* pinned_count() {
  static thread_local Tensor word;
  if (!word.defined()) word = at::zeros({8}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
  return word.data_ptr<int64_t>();
}

namespace {
constexpr size_t kMostCounters = 64;  // kept in all, over streams and devices
std::mutex g_counters_mu;
std::map<std::pair<int, void*>, std::vector<Tensor>>& free_counters() {
  static auto* m = new std::map<std::pair<int, void*>, std::vector<Tensor>>;  // outlives the allocator's own end
  return *m;
}
size_t g_counters_kept = 0;
}  // namespace

SlotCounters::SlotCounters(const Tensor& like) : key_((int) like.device().index(), stream_of(like)) {
  {
    std::lock_guard<std::mutex> lock(g_counters_mu);
    auto it = free_counters().find(key_);
    if (it != free_counters().end() && !it->second.empty()) {
      memory_ = std::move(it->second.back());
      it->second.pop_back();
      --g_counters_kept;
    }
  }
  if (!memory_.defined()) memory_ = at::zeros({kSlotRegions + 1}, like.options().dtype(at::kLong));
}

void SlotCounters::give_back() {
  std::lock_guard<std::mutex> lock(g_counters_mu);
  if (g_counters_kept >= kMostCounters) return;  // the allocator takes them back
  free_counters()[key_].push_back(std::move(memory_));
  ++g_counters_kept;
}

}  // namespace fsgs_host
