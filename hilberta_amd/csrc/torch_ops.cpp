// The torch operators of namespace hilberta_hip, over the C ABI (include/hilberta_hip.h).
//
// The reference launches its kernels as framework-visible Triton launches (hilberta/paired_kernel.py
// :181-204, hilberta/sparse_kernel.py:315-339) and gathers with index_select (hilberta/flux_adapter.py
// :209-212, :243).  Registered here natively, an operator call costs the host a few microseconds; as
// Python functions behind torch's dispatcher the attention operator took 22 us and a gather 16.5 us,
// more than the kernels of a 512 px attention call or a latents gather.  The shape-only (fake)
// implementations and the CPU kernel of pair_rows, which is plan setup, are in hilberta_amd/ops.py.
#include <ATen/ATen.h>
#include <ATen/DeviceGuard.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/library.h>

#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/hilberta_hip.h"

namespace {

using at::Tensor;

// Key blocks per row hb_pair_rows pairs.
constexpr int64_t PAIR_MAX_BLOCKS = 16384;
constexpr int64_t MIN_WORKSPACE = 1 << 16;

void check(int rc, const char* name) {
  if (rc == 0) return;
  if (rc == 1) TORCH_CHECK_VALUE(false, name, ": ", hb_last_error());
  TORCH_CHECK(false, name, ": ", hb_last_error());
}

int32_t i32(int64_t v, const char* name) {
  TORCH_CHECK_VALUE(v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max(),
                    name, " does not fit 32 bits");
  return static_cast<int32_t>(v);
}

hipStream_t stream_of(const at::Device& device) {
  return c10::hip::getCurrentHIPStream(device.index()).stream();
}

// ------------------------------------------------------------------ attention workspaces
// One workspace per (device, stream): the persistent kernel's work-queue counters (zero-filled once;
// every launch leaves them at zero) and the partial results of split global query tiles.  Launches
// that may overlap in time are on different streams and so never share one.  A call launches two
// kernels over its workspace, so threads of one stream take turns: each holds the workspace (Lease)
// until both are enqueued, or the second thread's first kernel could come between them.  A captured
// launch gets a workspace of its own from the capture's private pool, zero-filled on every replay.
class Workspaces {
  struct Held {
    std::mutex launching;
    Tensor tensor;
  };

 public:
  struct Lease {
    Tensor tensor;
    std::shared_ptr<Held> held;
    std::unique_lock<std::mutex> turn;
  };

  Lease get(const at::Device& device, int64_t need) {
    const auto options = at::TensorOptions().dtype(at::kByte).device(device);
    const int64_t bytes = std::max(need, MIN_WORKSPACE);
    const hipStream_t stream = stream_of(device);
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    TORCH_CHECK(hipStreamIsCapturing(stream, &status) == hipSuccess, "stream capture query failed");
    if (status != hipStreamCaptureStatusNone) return {at::zeros({bytes}, options), nullptr, {}};
    Lease lease;
    {
      const std::lock_guard<std::mutex> lock(mutex_);
      std::shared_ptr<Held>& held = cache_[{device.index(), reinterpret_cast<int64_t>(stream)}];
      if (!held) held = std::make_shared<Held>();
      lease.held = held;
    }
    lease.turn = std::unique_lock<std::mutex>(lease.held->launching);
    Tensor& tensor = lease.held->tensor;
    if (!tensor.defined() || tensor.numel() < need) tensor = at::zeros({bytes}, options);
    lease.tensor = tensor;
    return lease;
  }

  std::vector<int64_t> keys() {
    const std::lock_guard<std::mutex> lock(mutex_);
    std::vector<int64_t> out;
    for (const auto& [key, held] : cache_) {
      out.push_back(key.first);
      out.push_back(key.second);
    }
    return out;
  }

  void clear() {
    std::map<Key, std::shared_ptr<Held>> gone;
    const std::lock_guard<std::mutex> lock(mutex_);
    gone.swap(cache_);
  }

 private:
  using Key = std::pair<int64_t, int64_t>;
  std::mutex mutex_;
  std::map<Key, std::shared_ptr<Held>> cache_;
};

// Never destroyed: at process exit the allocator behind the tensors may be gone first.
Workspaces& workspaces() {
  static Workspaces* w = new Workspaces;
  return *w;
}

Tensor attention_workspace(at::Device device, int64_t need) {
  TORCH_CHECK_VALUE(device.is_cuda(), "workspaces live on a HIP device");
  if (!device.has_index()) device = at::Device(at::kCUDA, c10::hip::current_device());
  const at::OptionalDeviceGuard guard(device);
  return workspaces().get(device, need).tensor;
}

std::vector<int64_t> workspace_keys() { return workspaces().keys(); }
void clear_workspaces() { workspaces().clear(); }

// The C ABI this library was compiled against (ops.py compares it before it binds the operators).
int64_t abi_version() { return HB_ABI_VERSION; }

// ------------------------------------------------------------------ operators
struct Shape {
  int32_t batch, heads, tokens, dim, dtype;
  int64_t strides[12];
};

Shape shape_of(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out) {
  TORCH_CHECK_VALUE(q.dim() == 4 && k.sizes() == q.sizes() && v.sizes() == q.sizes() && out.sizes() == q.sizes(),
                    "Q/K/V/out must have equal [B,H,N,D] shapes");
  TORCH_CHECK_VALUE(q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf,
                    "Q/K/V must be bf16 or fp16");
  Shape s{i32(q.size(0), "batch"), i32(q.size(1), "heads"), i32(q.size(2), "tokens"),
          i32(q.size(3), "head_dim"), q.scalar_type() == at::kHalf ? HB_DTYPE_F16 : HB_DTYPE_BF16, {}};
  int i = 0;
  for (const Tensor* t : {&q, &k, &v, &out})
    for (int d = 0; d < 3; ++d) s.strides[i++] = t->stride(d);
  return s;
}

float* lse_ptr(const std::optional<Tensor>& lse) {
  return lse.has_value() && lse->defined() ? static_cast<float*>(lse->data_ptr()) : nullptr;
}

Workspaces::Lease workspace_for(const Tensor& q, const Shape& s, int32_t global_tokens, int32_t width,
                     int32_t key_block, int32_t paired, bool all_queries) {
  const int64_t need = hb_attention_workspace_bytes(s.batch, s.heads, s.tokens, s.dim, global_tokens, width,
                                                    key_block, paired, all_queries);
  check(need < 0 ? 1 : 0, "hb_attention_workspace_bytes");
  return workspaces().get(q.device(), need);
}

void paired_launch(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                   const std::optional<Tensor>& lse, const Tensor& ids, const Tensor& flags,
                   const Tensor& counts, int64_t global_tokens, int64_t key_block, double scale_log2,
                   bool all_queries, int64_t num_groups) {
  const Shape s = shape_of(q, k, v, out);
  const int32_t width = i32(ids.size(1), "table width"), G = i32(global_tokens, "global_tokens"),
                kb = i32(key_block, "key_block_size");
  const auto ws = workspace_for(q, s, G, width, kb, 1, all_queries);
  check(hb_paired_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse_ptr(lse), s.strides, s.batch,
                      s.heads, s.tokens, s.dim, s.dtype, static_cast<const int32_t*>(ids.data_ptr()),
                      static_cast<const int32_t*>(flags.data_ptr()),
                      static_cast<const int32_t*>(counts.data_ptr()), width, G, kb, all_queries,
                      static_cast<float>(scale_log2), ws.tensor.data_ptr(), ws.tensor.numel(),
                      i32(num_groups, "num_groups"), stream_of(q.device())),
        "hb_paired_fwd");
}

// hb_paired_fwd on the current stream (replaces the _paired_fwd launch, paired_kernel.py:181-204).
void paired_fwd(const Tensor& q, const Tensor& k, const Tensor& v, Tensor out, std::optional<Tensor> lse,
                const Tensor& ids, const Tensor& flags, const Tensor& counts, int64_t global_tokens,
                int64_t key_block, double scale_log2, bool all_queries, int64_t num_groups) {
  const at::OptionalDeviceGuard guard(q.device());
  paired_launch(q, k, v, out, lse, ids, flags, counts, global_tokens, key_block, scale_log2, all_queries,
                num_groups);
}

// hb_pair_rows: rows 2r and 2r + 1 of an unpaired table become paired row r, ascending and
// zero-padded (paired_metadata.py:26-51); an odd row count is paired from the end.
std::tuple<Tensor, Tensor, Tensor> pair_rows(const Tensor& ids, const Tensor& counts, int64_t total_blocks,
                                             int64_t key_block, int64_t paired_width) {
  TORCH_CHECK_VALUE(ids.scalar_type() == at::kInt && counts.scalar_type() == at::kInt && ids.dim() == 2 &&
                        counts.dim() == 1 && counts.size(0) == ids.size(0) && ids.is_contiguous() &&
                        counts.is_contiguous() && ids.device() == counts.device(),
                    "tables must be contiguous int32 kv_indices [rows, width] and kv_counts [rows] on one device");
  const at::OptionalDeviceGuard guard(ids.device());
  const int64_t rows = ids.size(0), prows = (rows + 1) / 2;
  Tensor out = at::empty({prows, paired_width}, ids.options()), flags = at::empty_like(out);
  Tensor out_counts = at::empty({prows}, ids.options());
  check(hb_pair_rows(static_cast<const int32_t*>(ids.data_ptr()), static_cast<const int32_t*>(counts.data_ptr()),
                     i32(rows, "rows"), i32(ids.size(1), "width"), i32(total_blocks, "total_blocks"),
                     i32(key_block, "key_block_size"), static_cast<int32_t*>(out.data_ptr()),
                     static_cast<int32_t*>(flags.data_ptr()), static_cast<int32_t*>(out_counts.data_ptr()),
                     i32(paired_width, "paired_width"), nullptr, stream_of(ids.device())),
        "hb_pair_rows");
  return {out, flags, out_counts};
}

// Unpaired 64-query tables (replaces the _block_sparse_fwd launch, sparse_kernel.py:315-339).
//
// With at most PAIR_MAX_BLOCKS key blocks, rows 2r, 2r + 1 are merged on the device, as pair_metadata
// does (paired_metadata.py:26-51), and run on hb_paired_fwd: a 128-query item keeps two waves per
// SIMD busy where a 64-query item keeps one (1.7-1.85x faster).  An odd row count is paired from the
// end, its first paired row carrying an empty half that reaches into the global prefix and is never
// stored; a global prefix that is an odd multiple of 64 leaves a last global tile whose upper half is
// never stored either.  Every query sees the same key blocks in the same ascending order with the
// same arithmetic; the other half's blocks are masked to exact zeros.  The paired tables are padded
// to min(2 * width, N / 64) entries, which needs no host synchronisation.  Longer sequences run as
// they are on hb_block_sparse_fwd.
void sparse_fwd(const Tensor& q, const Tensor& k, const Tensor& v, Tensor out, std::optional<Tensor> lse,
                const Tensor& ids, const Tensor& counts, int64_t global_tokens, double scale_log2,
                bool all_queries, int64_t num_groups) {
  const at::OptionalDeviceGuard guard(q.device());
  const Shape s = shape_of(q, k, v, out);
  const int64_t blocks = s.tokens / 64;
  if (blocks <= PAIR_MAX_BLOCKS) {
    const auto [pids, pflags, pcounts] = pair_rows(ids, counts, blocks, 64, std::min(2 * ids.size(1), blocks));
    paired_launch(q, k, v, out, lse, pids, pflags, pcounts, global_tokens, 64, scale_log2, all_queries, num_groups);
    return;
  }
  const int32_t width = i32(ids.size(1), "table width"), G = i32(global_tokens, "global_tokens");
  const auto ws = workspace_for(q, s, G, width, 64, 0, all_queries);
  check(hb_block_sparse_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse_ptr(lse), s.strides,
                            s.batch, s.heads, s.tokens, s.dim, s.dtype, static_cast<const int32_t*>(ids.data_ptr()),
                            static_cast<const int32_t*>(counts.data_ptr()), width, G, 64, all_queries,
                            static_cast<float>(scale_log2), ws.tensor.data_ptr(), ws.tensor.numel(),
                            i32(num_groups, "num_groups"), stream_of(q.device())),
        "hb_block_sparse_fwd");
}

// One stride walking every index of the dims before `dim`: {count, stride}, stride -1 if none does.
std::pair<int64_t, int64_t> outer_walk(const Tensor& x, int64_t dim) {
  int64_t outer = 1, last = 0, step = -1;  // step: what the next dim outwards must advance by
  for (int64_t d = 0; d < dim; ++d) outer *= x.size(d);
  if (outer <= 1) return {outer, 0};
  for (int64_t d = dim - 1; d >= 0; --d) {
    if (x.size(d) <= 1) continue;
    if (step < 0) last = x.stride(d);
    else if (x.stride(d) != step) return {outer, -1};
    step = x.stride(d) * x.size(d);
  }
  return {outer, last};
}

// x.index_select(dim, index) by hb_gather_rows (flux_adapter.py:209-212, :243), bit for bit; the
// dims after `dim` must be contiguous.
Tensor gather_rows(const Tensor& input, int64_t dim, const Tensor& index) {
  const int64_t nd = input.dim();
  TORCH_CHECK_INDEX(nd > 0 && dim >= -nd && dim < nd, "dim out of range");
  if (dim < 0) dim += nd;
  TORCH_CHECK_VALUE(index.dim() == 1 && index.scalar_type() == at::kLong && index.device() == input.device(),
                    "index must be a 1-D int64 tensor on x's device");
  int64_t row = 1;
  for (int64_t d = nd - 1; d > dim; --d) {
    TORCH_CHECK_VALUE(input.size(d) <= 1 || input.stride(d) == row,
                      "index_select_rows needs the dims after `dim` to be contiguous");
    row *= input.size(d);
  }
  const at::OptionalDeviceGuard guard(input.device());
  Tensor x = input;
  auto [outer, src_outer] = outer_walk(x, dim);
  if (src_outer < 0) {
    x = x.contiguous();
    std::tie(outer, src_outer) = outer_walk(x, dim);
  }
  const Tensor idx = index.contiguous();
  auto sizes = x.sizes().vec();
  sizes[dim] = idx.numel();
  Tensor out = at::empty(sizes, x.options());
  const int64_t es = x.element_size();
  check(hb_gather_rows(x.data_ptr(), out.data_ptr(), static_cast<const int64_t*>(idx.data_ptr()), idx.numel(),
                       outer, src_outer * es, idx.numel() * row * es, x.stride(dim) * es, row * es, row * es,
                       x.size(dim), nullptr, stream_of(x.device())),
        "hb_gather_rows");
  return out;
}

// The attention operators return nothing and write `out` and `lse`, which torch's own boxed fallbacks
// overlook: they look after returned tensors only.

// No derivative is recorded (the entry points refuse inputs that need one); a transform that takes one
// is refused, as torch refuses an autograd.Function in one, for it would get zeros.
void attention_autograd(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const size_t count = op.schema().arguments().size();
  // (included for as long as any torch.func transform is active)
  const bool transformed = at::GradMode::is_enabled() &&
                           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
  for (const c10::IValue& value : torch::jit::last(stack, count)) {
    if (!value.isTensor() || !value.toTensor().defined()) continue;
    const Tensor& t = value.toTensor();
    TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(/*level=*/0).defined(), "Trying to use forward AD with ",
                                op.schema().name(), " that does not support it.");
    TORCH_CHECK(!(transformed && t.requires_grad()), op.schema().name(), " has no derivative for torch.func transforms");
  }
  const at::AutoDispatchBelowAutograd below;
  op.redispatchBoxed(keys & c10::after_autograd_keyset, stack);
}

// A tensor saved for a backward and then overwritten here has to fail that backward: every written
// argument's version counts up.
void attention_writes(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const auto& arguments = op.schema().arguments();
  const auto values = torch::jit::last(stack, arguments.size());
  c10::SmallVector<Tensor, 2> written;
  for (size_t i = 0; i < arguments.size(); ++i) {
    const c10::AliasInfo* alias = arguments[i].alias_info();
    if (alias && alias->isWrite() && values[i].isTensor() && values[i].toTensor().defined())
      written.push_back(values[i].toTensor());
  }
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    op.redispatchBoxed(keys & c10::after_ADInplaceOrView_keyset, stack);
  }
  for (const Tensor& t : written)
    if (!t.is_inference()) torch::autograd::impl::bump_version(t);
}

}  // namespace

TORCH_LIBRARY(hilberta_hip, m) {
  const std::vector<at::Tag> tags{at::Tag::pt2_compliant_tag};
  m.def("paired_fwd(Tensor q, Tensor k, Tensor v, Tensor(a3!) out, Tensor(a4!)? lse, Tensor kv_indices, "
        "Tensor kv_flags, Tensor kv_counts, SymInt global_tokens, SymInt key_block_size, float scale_log2, "
        "bool all_queries, SymInt num_groups) -> ()", tags);
  m.def("sparse_fwd(Tensor q, Tensor k, Tensor v, Tensor(a3!) out, Tensor(a4!)? lse, Tensor kv_indices, "
        "Tensor kv_counts, SymInt global_tokens, float scale_log2, bool all_queries, SymInt num_groups) -> ()",
        tags);
  m.def("pair_rows(Tensor kv_indices, Tensor kv_counts, SymInt total_blocks, SymInt key_block_size, "
        "SymInt paired_width) -> (Tensor, Tensor, Tensor)", tags);
  m.def("gather_rows(Tensor x, SymInt dim, Tensor index) -> Tensor", tags);
  m.def("_attention_workspace(Device device, int need) -> Tensor");
  m.def("_workspace_keys() -> int[]");
  m.def("_clear_workspaces() -> ()");
  m.def("_abi_version() -> int");
}

TORCH_LIBRARY_IMPL(hilberta_hip, CUDA, m) {
  m.impl("paired_fwd", paired_fwd);
  m.impl("sparse_fwd", sparse_fwd);
  m.impl("pair_rows", pair_rows);
  m.impl("gather_rows", gather_rows);
}

TORCH_LIBRARY_IMPL(hilberta_hip, CompositeExplicitAutograd, m) {
  m.impl("_attention_workspace", attention_workspace);
  m.impl("_workspace_keys", workspace_keys);
  m.impl("_clear_workspaces", clear_workspaces);
  m.impl("_abi_version", abi_version);
}

// gather_rows and pair_rows: a differentiated call fails in its backward.
TORCH_LIBRARY_IMPL(hilberta_hip, Autograd, m) {
  for (const char* name : {"pair_rows", "gather_rows"})
    m.impl(name, torch::autograd::autogradNotImplementedFallback());
  for (const char* name : {"paired_fwd", "sparse_fwd"})
    m.impl(name, torch::CppFunction::makeFromBoxedFunction<&attention_autograd>());
}

TORCH_LIBRARY_IMPL(hilberta_hip, ADInplaceOrView, m) {
  for (const char* name : {"paired_fwd", "sparse_fwd"})
    m.impl(name, torch::CppFunction::makeFromBoxedFunction<&attention_writes>());
}
