// Host side of the Python package's eager path: allocates outputs, launches the kernels of libck_mi355.so through its C ABI
// and records the autograd nodes.
//
// Why native: a small call is bound by the host. An autograd.Function in Python costs 20 to 30 us forward and, because
// the engine's device thread has to win the interpreter lock from the waiting main thread, 30 to 60 us backward, while the
// kernels of such a call take 5 to 20. The nodes here run in the engine's thread without the interpreter. The Python files
// keep the public signatures, their checks and the dispatch to the traced operators (torch.compile).
//
// No state is kept by the address or identity of a tensor. What outlives a call: the workspaces below, one per device and
// stream (calls on one stream are ordered, calls on different streams never share one).
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/extension.h>

#include <atomic>
#include <map>
#include <mutex>
#include <optional>
#include <tuple>

#include "ck_mi355.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- the C ABI, from the library the package loaded ---------------------------------------------------------------
#define CK_API(X)                                                                                                       \
  X(ck_last_error_string) X(ck_count_workspace_words) X(ck_count_offsets) X(ck_route_topk_softmax_all)                  \
  X(ck_route_topk_softmax_bwd) X(ck_route_topk_softmax_bwd_exact) X(ck_sort_max_rows) X(ck_sort_workspace_words)        \
  X(ck_sort_by_expert) X(ck_combine_rows) X(ck_gate_grad_both) X(ck_group_segment_rows) X(ck_swiglu_bwd_grouped)         \
  X(ck_transpose_batched) X(ck_grouped_gemm_workspace_bytes) X(ck_grouped_gemm_uses_workspace) X(ck_grouped_gemm_ws) X(ck_grouped_gemm_nn_ws)             \
  X(ck_grouped_gemm_f32) X(ck_grouped_gemm_dw_f32) X(ck_grouped_gemm_dw) X(ck_grouped_gemm_dw_rows)                     \
  X(ck_quant_rows_e4m3) X(ck_quant_grouped_rows_e4m3) X(ck_grouped_gemm_fp8) X(ck_swiglu_fwd) X(ck_swiglu_bwd) X(ck_gelu_tanh_bwd) X(ck_rmsnorm_route) X(ck_router_rows) \
  X(ck_gelu_tanh_bwd_grouped) X(ck_fused_residual_add_rmsnorm_fwd) X(ck_rmsnorm_fwd) X(ck_rmsnorm_bwd_partial_rows) X(ck_rmsnorm_bwd_typed)         \
  X(ck_softmax_fwd) X(ck_softmax_bwd) X(ck_add_expert_bias) X(ck_expert_bias_grad)

struct Api {
#define CK_MEMBER(f) decltype(&::f) f = nullptr;
  CK_API(CK_MEMBER)
#undef CK_MEMBER
} api;

void init(const std::string& path) {
  void* handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(handle != nullptr, "cannot load ", path, ": ", dlerror());
#define CK_RESOLVE(f)                                                       \
  api.f = reinterpret_cast<decltype(&::f)>(dlsym(handle, #f));              \
  TORCH_CHECK(api.f != nullptr, path, " does not export ", #f);
  CK_API(CK_RESOLVE)
#undef CK_RESOLVE
}

void check(int rc) {
  if (rc != 0) throw std::runtime_error(api.ck_last_error_string());
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CK_F32;
    case at::kHalf: return CK_F16;
    case at::kBFloat16: return CK_BF16;
    default: TORCH_CHECK_NOT_IMPLEMENTED(false, "libck_mi355 has no kernels for dtype ", t);
  }
}
int dtype_code(const Tensor& t) { return dtype_code(t.scalar_type()); }

void require_gpu(const Tensor& t) {
  TORCH_CHECK(!t.defined() || t.is_cuda(), "cute_kernels (MI355X build) runs on the GPU only; got a tensor on ", t.device(),
              ". There is no CPU path.");
}
template <typename... Rest>
void require_gpu(const Tensor& t, const Rest&... rest) {
  require_gpu(t);
  require_gpu(rest...);
}

// A tensor whose sizes a launch is derived from has as many dimensions as the code takes it to have: rows of a [B, S, H]
// tensor read as [T, K] would be addressed past its end.
void require_dims(std::initializer_list<std::pair<const Tensor*, int64_t>> ts) {
  for (const auto& [t, dims] : ts)
    TORCH_CHECK_VALUE(t->dim() == dims, "expected a tensor with ", dims, " dimensions, got shape ", t->sizes());
}

// the device of a call made current, and torch's current stream on it
struct Launch {
  c10::OptionalDeviceGuard guard;
  void* stream;
  explicit Launch(const Tensor& t)
      : guard(t.device()), stream(at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()) {}
};

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const Tensor value_or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
Tensor contiguous(const Tensor& t) { return t.defined() ? t.contiguous() : t; }
OptTensor to_opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }
Tensor new_empty(at::IntArrayRef size, const Tensor& like, at::ScalarType t) { return at::empty(size, like.options().dtype(t)); }
Tensor new_empty(at::IntArrayRef size, const Tensor& like) { return at::empty(size, like.options()); }
Tensor like_contiguous(const Tensor& t) { return at::empty(t.sizes(), t.options()); }

// Whether a call is recorded for autograd. Forward-mode tangents count, in every grad mode: the nodes have no forward-mode
// rule, and recording is what makes torch refuse such a call instead of losing the tangent.
bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(/*level=*/0).defined())) return true;
  return false;
}

// rows of a tensor whose last dimension is one row
int64_t row_count(const Tensor& x) {
  TORCH_CHECK(x.size(-1) > 0, "rows of a tensor of shape ", x.sizes(), " are empty");
  return x.numel() / x.size(-1);
}

// ---- workspaces: one per kind, device and stream. "count" starts zero and its kernel leaves it so; "sort" and "split" need no
// initial contents. Never freed (torch's allocator may be gone at exit); torch has a bounded number of streams.
// A call that is being captured gets a workspace of its own, in the graph's memory: a graph may be replayed on any stream,
// beside eager calls on the one it was captured on, and the zeros of a kept one would be written by the replays of the graph
// that happened to ask first.
enum WorkspaceKind { kCountWs, kSortWs, kSplitWs };
Tensor workspace(WorkspaceKind kind, const Tensor& like, void* stream, int64_t words) {
  static std::mutex mutex;
  static auto* table = new std::map<std::tuple<int, int, void*>, Tensor>();
  const auto options = at::TensorOptions().dtype(at::kInt).device(like.device());
  const auto made = [&](int64_t n) { return kind == kCountWs ? at::zeros({n}, options) : at::empty({n}, options); };
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return made(words);
  const std::tuple<int, int, void*> key{(int)kind, (int)like.device().index(), stream};
  {
    const std::lock_guard<std::mutex> lock(mutex);
    const Tensor& ws = (*table)[key];
    if (ws.defined() && ws.numel() >= words) return ws;
  }
  // not under the lock: making a tensor may run Python (dispatch modes) and wait for its lock
  const Tensor fresh = made(kind == kSplitWs ? words : std::max<int64_t>(words, 1 << 16));
  const std::lock_guard<std::mutex> lock(mutex);
  Tensor& ws = (*table)[key];
  if (!ws.defined() || ws.numel() < words) ws = fresh;
  return ws;
}

// ---- optional per-launch timing of the expert GEMMs (scattermoe.set_launch_timer): timer.time(name, (N, K), launch)
// The backward pass launches from threads that do not hold the interpreter lock, and the timer may be taken off meanwhile:
// the atomic says whether to ask for the lock, the pointer is read under it, and a call keeps a reference of its own.
std::atomic<bool> timed_launches{false};
py::object* launch_timer = nullptr;
void set_launch_timer(py::object timer) {
  timed_launches = false;
  delete launch_timer;
  launch_timer = timer.is_none() ? nullptr : new py::object(std::move(timer));
  timed_launches = launch_timer != nullptr;
}
template <typename F>
void timed(const char* name, int64_t a, int64_t b, F&& launch) {
  if (timed_launches) {
    const py::gil_scoped_acquire gil;
    if (launch_timer != nullptr) {
      const py::object timer = *launch_timer;
      timer.attr("time")(name, py::make_tuple(a, b), py::cpp_function([&] { launch(); }));
      return;
    }
  }
  launch();
}

// ---- count, sort ------------------------------------------------------------------------------------------------
std::tuple<Tensor, OptTensor, OptTensor> count(const Tensor& ids_in, int64_t size, bool want_offsets) {
  require_gpu(ids_in);
  const Tensor ids = ids_in.contiguous();
  const Launch l(ids);
  const Tensor counts = new_empty({size}, ids, at::kUInt32);
  Tensor ends, starts;
  if (want_offsets) {
    ends = new_empty({size}, ids, at::kUInt32);
    starts = new_empty({size}, ids, at::kUInt32);
  }
  const Tensor ws = workspace(kCountWs, ids, l.stream, api.ck_count_workspace_words((int32_t)size));
  check(api.ck_count_offsets(ptr(ids), ids.scalar_type() == at::kLong, ids.numel(), (int32_t)size, (uint32_t*)ptr(counts),
                             (uint32_t*)ptr(ends), (uint32_t*)ptr(starts), (uint32_t*)ptr(ws), l.stream));
  return {counts, to_opt(ends), to_opt(starts)};
}

// `words` 32-bit words of `base` from word `offset` on, as a tensor of its own: no view of base, the way an allocation would be,
// at a quarter of its cost
Tensor words_of(const Tensor& base, int64_t offset, int64_t words, at::ScalarType t) {
  Tensor part = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(), c10::scalarTypeToTypeMeta(t));
  part.unsafeGetTensorImpl()->set_storage_offset(base.storage_offset() + offset);
  part.unsafeGetTensorImpl()->set_sizes_contiguous({words});
  return part;
}

// (sorted_expert_idxs, sorted_scattered_idxs, counts, ends, starts, seg_starts, row_slot, tile_expert, max_rows)
// The tables live and die together: one allocation for those of a word per routed row and one for those of a word per expert, which
// a caller may keep of every step; each table on a 256-byte boundary. apart: eight, for a registered operator, whose outputs may
// not share storage.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, int64_t> sort_by_expert(const Tensor& ids_in,
                                                                                                int64_t E, int64_t align, bool apart) {
  require_gpu(ids_in);
  const Tensor ids = ids_in.contiguous();
  const Launch l(ids);
  const int64_t R = ids.numel();
  const int64_t max_rows = api.ck_sort_max_rows(R, (int32_t)E, (int32_t)align);
  const int64_t slots = std::max<int64_t>(max_rows, 1), tiles = std::max<int64_t>(max_rows / align, 1);
  const auto room = [](int64_t n) { return (n + 63) / 64 * 64; };
  struct Tables {
    Tensor all;
    int64_t used = 0;
  } of_rows, of_experts;
  if (!apart) {
    of_rows.all = new_empty({2 * room(R) + room(slots) + room(tiles)}, ids, at::kInt);
    of_experts.all = new_empty({3 * room(E) + room(E + 1)}, ids, at::kInt);
  }
  const auto next = [&](Tables& from, int64_t n, at::ScalarType t) {
    if (apart) return new_empty({n}, ids, t);
    const Tensor part = words_of(from.all, from.used, n, t);
    from.used += room(n);
    return part;
  };
  const Tensor se = next(of_rows, R, at::kInt), ss = next(of_rows, R, at::kInt), row_slot = next(of_rows, slots, at::kInt);
  const Tensor tile_expert = next(of_rows, tiles, at::kInt), counts = next(of_experts, E, at::kUInt32);
  const Tensor ends = next(of_experts, E, at::kUInt32), starts = next(of_experts, E, at::kUInt32);
  const Tensor seg_starts = next(of_experts, E + 1, at::kInt);
  const Tensor ws = workspace(kSortWs, ids, l.stream, api.ck_sort_workspace_words(R, (int32_t)E));
  check(api.ck_sort_by_expert(ptr(ids), ids.scalar_type() == at::kLong, R, (int32_t)E, (int32_t)align, (int32_t*)ptr(se),
                              (int32_t*)ptr(ss), (uint32_t*)ptr(counts), (uint32_t*)ptr(ends), (uint32_t*)ptr(starts),
                              (int32_t*)ptr(seg_starts), (int32_t*)ptr(row_slot), (int32_t*)ptr(tile_expert),
                              (uint32_t*)ptr(ws), l.stream));
  return {se, ss, counts, ends, starts, seg_starts, row_slot, tile_expert, max_rows};
}

// ---- router -----------------------------------------------------------------------------------------------------
// Side channel between the expert block's backward and the router's. Autograd hands a 16-bit gates tensor a 16-bit
// gradient; the softmax backward then subtracts nearly equal rounded numbers and the router's weight gradient loses digits.
// The expert block leaves its unrounded fp32 d_gates here, and the router's backward uses it when the gradient it receives
// is exactly that tensor rounded (i.e. nothing else contributed to the gates' gradient).
struct GateSlot : torch::CustomClassHolder {
  Tensor d_gates_f32;
};
using SlotPtr = c10::intrusive_ptr<GateSlot>;

// (gates fp32, gates in logits.dtype, selected int32, selected int64); what is not wanted stays undefined
std::tuple<Tensor, Tensor, Tensor, Tensor> route_forward(const Tensor& logits_in, int64_t k, bool want_f32, bool want_i32, bool want_i64) {
  require_dims({{&logits_in, 2}});
  require_gpu(logits_in);
  const Tensor logits = logits_in.contiguous();
  const Launch l(logits);
  const int64_t T = logits.size(0), E = logits.size(1);
  const bool fp32 = logits.scalar_type() == at::kFloat;
  Tensor gates, rounded, sel, sel_long;
  if (want_f32 || fp32) gates = new_empty({T, k}, logits, at::kFloat);
  if (!fp32) rounded = new_empty({T, k}, logits);
  if (want_i32) sel = new_empty({T, k}, logits, at::kInt);
  if (want_i64) sel_long = new_empty({T, k}, logits, at::kLong);
  check(api.ck_route_topk_softmax_all(ptr(logits), dtype_code(logits), T, (int32_t)E, (int32_t)k, (int32_t*)ptr(sel),
                                      (int64_t*)ptr(sel_long), (float*)ptr(gates), ptr(rounded), l.stream));
  return {gates, fp32 ? gates : rounded, sel, sel_long};
}

// exact: the unrounded gradient where the caller has it (used wherever d_gates is that gradient rounded; decided per element
// inside the kernel: no host sync, no extra launches)
Tensor route_backward(const Tensor& gates, const Tensor& selected, const Tensor& d_gates, const Tensor& exact, int64_t E,
                      at::ScalarType dtype) {
  const Launch l(gates);
  const int64_t T = gates.size(0), k = gates.size(1);
  const Tensor d_logits = new_empty({T, E}, gates, dtype);
  if (exact.defined() && exact.sizes() == d_gates.sizes() && d_gates.scalar_type() == dtype && dtype != at::kFloat) {
    const Tensor d = d_gates.contiguous();
    check(api.ck_route_topk_softmax_bwd_exact((const float*)ptr(gates), (const float*)ptr(exact), ptr(d),
                                              (const int32_t*)ptr(selected), T, (int32_t)E, (int32_t)k, ptr(d_logits),
                                              dtype_code(dtype), l.stream));
  } else {
    const Tensor d = d_gates.to(at::kFloat).contiguous();
    check(api.ck_route_topk_softmax_bwd((const float*)ptr(gates), (const float*)ptr(d), (const int32_t*)ptr(selected), T,
                                        (int32_t)E, (int32_t)k, ptr(d_logits), dtype_code(dtype), l.stream));
  }
  return d_logits;
}

struct Route : torch::autograd::Function<Route> {
  static variable_list forward(AutogradContext* ctx, const Tensor& logits, int64_t k, bool long_indices, SlotPtr slot) {
    auto [gates, out, sel, sel_long] = route_forward(logits, k, true, true, long_indices);
    ctx->save_for_backward({gates, sel});
    ctx->saved_data["E"] = logits.size(1);
    ctx->saved_data["dtype"] = (int64_t)logits.scalar_type();
    ctx->saved_data["slot"] = c10::IValue::make_capsule(std::move(slot));
    const Tensor selected = long_indices ? sel_long : sel;
    ctx->mark_non_differentiable({selected});
    ctx->set_materialize_grads(false);
    return {out, selected};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const auto saved = ctx->get_saved_variables();
    const auto capsule = ctx->saved_data["slot"].toCapsule();
    auto* slot = static_cast<GateSlot*>(capsule.get());
    Tensor exact;
    std::swap(exact, slot->d_gates_f32);
    return {route_backward(saved[0], saved[1], grads[0], exact, ctx->saved_data["E"].toInt(),
                           (at::ScalarType)ctx->saved_data["dtype"].toInt()),
            Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor> route(const Tensor& logits, int64_t k, bool long_indices, SlotPtr slot) {
  if (any_requires_grad({&logits})) {
    auto out = Route::apply(logits, k, long_indices, std::move(slot));
    return {out[0], out[1]};
  }
  auto [gates, out, sel, sel_long] = route_forward(logits, k, false, !long_indices, long_indices);
  return {out, long_indices ? sel_long : sel};
}

// ---- expert blocks ----------------------------------------------------------------------------------------------
struct Segments {  // the tables of scattermoe.ExpertSegments
  Tensor seg_starts, counts, tile_expert, row_slot;
  int64_t max_rows = 0, experts = 0, align = 0;

  static Segments of(const py::handle& s) {
    Segments g;
    g.seg_starts = s.attr("seg_starts").cast<Tensor>();
    g.counts = s.attr("counts").cast<Tensor>();
    g.tile_expert = s.attr("tile_expert").cast<Tensor>();
    g.row_slot = s.attr("row_slot").cast<Tensor>();
    g.max_rows = s.attr("max_rows").cast<int64_t>();
    g.experts = s.attr("num_experts").cast<int64_t>();
    g.align = s.attr("align").cast<int64_t>();
    return g;
  }
  // rows_in: table a gathered input is read through; rows_out: table the scatter epilogue writes through (default: rows_in)
  ck_segments c(const Tensor& rows_in = Tensor(), const Tensor& rows_out = Tensor()) const {
    return {(const int32_t*)ptr(seg_starts), (const uint32_t*)ptr(counts), (const int32_t*)ptr(tile_expert),
            (const int32_t*)ptr(rows_in.defined() ? rows_in : row_slot), max_rows, (int32_t)experts, (int32_t)align,
            (const int32_t*)ptr(rows_out)};
  }
};

// scattermoe.Options as bits
enum Flags { kGemmSplit = 1, kBiasFused = 2, kGemmNn = 4, kDwRows = 8 };

const char* epilogue_name(int64_t epilogue, bool nn) {
  switch (epilogue) {
    case CK_EPI_SCATTER: return nn ? "grouped_gemm_nn<scatter>" : "grouped_gemm<scatter>";
    case CK_EPI_SWIGLU:
    case CK_EPI_GLU: return "grouped_gemm<swiglu>";
    case CK_EPI_SWIGLU_BWD: return "grouped_gemm<swiglu_bwd>";
    default: return nn ? "grouped_gemm_nn<grouped>" : "grouped_gemm<grouped>";
  }
}

bool is_f32(const Tensor& t) { return t.scalar_type() == at::kFloat; }

Tensor split_workspace(const Tensor& like, void* stream) {
  return workspace(kSplitWs, like, stream, (api.ck_grouped_gemm_workspace_bytes() + 3) / 4);
}
// whether a launch of contraction K may split its last round
bool may_split(int64_t K, int64_t flags) { return (flags & kGemmSplit) && api.ck_grouped_gemm_uses_workspace((int32_t)K); }

void gemm_f32(const Tensor& a, int64_t gather_div, const Tensor& w, bool w_is_kn, int64_t N, int64_t K, const Segments& seg,
              bool scatter, const Tensor& y, const Tensor& bias, const Tensor& rows_in, const Tensor& rows_out) {
  const Launch l(w);
  const ck_segments cs = seg.c(rows_in, rows_out);
  check(api.ck_grouped_gemm_f32((const float*)ptr(a), (int32_t)gather_div, (const float*)ptr(w), w_is_kn, (int32_t)N, (int32_t)K,
                                &cs, scatter, (float*)ptr(y), (const float*)ptr(bias), l.stream));
}

void gemm(const Tensor& a, int64_t gather_div, const Tensor& w, const Segments& seg, int64_t epilogue, const Tensor& y,
          const Tensor& y_t, const Tensor& aux, const Tensor& aux_in, const Tensor& rows_in, const Tensor& rows_out, int64_t flags) {
  const int64_t N = w.size(1), K = w.size(2);
  if (is_f32(w)) {
    TORCH_CHECK((epilogue == CK_EPI_GROUPED || epilogue == CK_EPI_SCATTER) && !y_t.defined() && !aux.defined(),
                "fp32 expert GEMMs have the grouped and scatter epilogues");
    return gemm_f32(a, gather_div, w, false, N, K, seg, epilogue == CK_EPI_SCATTER, y, aux_in, rows_in, rows_out);
  }
  // gathered rows are addressed with 32-bit byte offsets from the start of `a` (the library is not told how many rows `a` has)
  if (gather_div > 0) TORCH_CHECK((uint64_t)a.numel() * a.element_size() < (1ull << 32),
                                  "the token-order input of a grouped GEMM must stay below 4 GiB");
  timed(epilogue_name(epilogue, false), N, K, [&] {
    const Launch l(w);
    const ck_segments cs = seg.c(rows_in, rows_out);
    const Tensor ws = seg.align == 256 && may_split(K, flags) ? split_workspace(w, l.stream) : Tensor();
    check(api.ck_grouped_gemm_ws(ptr(a), (int32_t)gather_div, ptr(w), (int32_t)N, (int32_t)K, &cs, (int32_t)epilogue, ptr(y), ptr(y_t),
                                 seg.max_rows, ptr(aux), ptr(aux_in), dtype_code(w), l.stream, ptr(ws), ws.defined() ? ws.nbytes() : 0));
  });
}

Tensor transpose_weights(const Tensor& w) {
  const Launch l(w);
  const Tensor w_t = new_empty({w.size(0), w.size(2), w.size(1)}, w);
  check(api.ck_transpose_batched(ptr(w), w.size(0), (int32_t)w.size(1), (int32_t)w.size(2), ptr(w_t), dtype_code(w), l.stream));
  return w_t;
}

// out = d_y @ w[e] per expert, w [E, out_features, in_features] as the forward stores it: the input-gradient GEMM. Reads w
// contraction-strided where the kernel for that exists (256-row tiles, out_features % 64 == 0), else through a transposed copy.
void gemm_dx(const Tensor& d_y, const Tensor& w, const Segments& seg, int64_t epilogue, const Tensor& out, const Tensor& rows_out,
             int64_t flags) {
  const int64_t n_out = w.size(1), n_in = w.size(2);
  if (is_f32(w)) return gemm_f32(d_y, 0, w, true, n_in, n_out, seg, epilogue == CK_EPI_SCATTER, out, Tensor(), Tensor(), rows_out);
  if (seg.align == 256 && n_out % 64 == 0 && (flags & kGemmNn)) {
    return timed(epilogue_name(epilogue, true), n_in, n_out, [&] {
      const Launch l(w);
      const ck_segments cs = seg.c(Tensor(), rows_out);
      const Tensor ws = may_split(n_out, flags) ? split_workspace(w, l.stream) : Tensor();
      check(api.ck_grouped_gemm_nn_ws(ptr(d_y), ptr(w), (int32_t)n_in, (int32_t)n_out, &cs, (int32_t)epilogue, ptr(out), dtype_code(w),
                                      l.stream, ptr(ws), ws.defined() ? ws.nbytes() : 0));
    });
  }
  gemm(d_y, 0, transpose_weights(w), seg, epilogue, out, Tensor(), Tensor(), Tensor(), Tensor(), rows_out, flags);
}

// dw[e] = a_t[:, rows of e] @ b_t[:, rows of e]^T from transposed padded-grouped operands
void gemm_dw(const Tensor& a_t, const Tensor& b_t, const Segments& seg, const Tensor& dw) {
  timed("grouped_gemm<dw>", dw.size(1), dw.size(2), [&] {
    const Launch l(dw);
    const ck_segments cs = seg.c();
    check(api.ck_grouped_gemm_dw(ptr(a_t), ptr(b_t), seg.max_rows, (int32_t)dw.size(1), (int32_t)dw.size(2), &cs, ptr(dw), dtype_code(dw),
                                 l.stream));
  });
}

// dw[e] = a[rows of e]^T @ b[rows of e] from row-major padded-grouped operands (no transposed copies)
void gemm_dw_rows(const Tensor& a, const Tensor& b, const Segments& seg, const Tensor& dw) {
  const int32_t M = (int32_t)dw.size(1), N = (int32_t)dw.size(2);
  const ck_segments cs = seg.c();
  if (is_f32(dw)) {
    const Launch l(dw);
    return check(api.ck_grouped_gemm_dw_f32((const float*)ptr(a), (const float*)ptr(b), M, N, &cs, (float*)ptr(dw), l.stream));
  }
  timed("grouped_gemm_dw_rows", M, N, [&] {
    const Launch l(dw);
    check(api.ck_grouped_gemm_dw_rows(ptr(a), ptr(b), M, N, &cs, ptr(dw), dtype_code(dw), l.stream));
  });
}

// Whether the weight-gradient GEMMs of shapes (M, N), ... read row-major operands (ck_grouped_gemm_dw_rows) instead of
// transposed copies: whenever that kernel takes the shapes. Not writing (and not holding) the transposes outweighs the wider
// tiles the transposed form can use (fine-grained layer 4 % faster, Mixtral-shape layer 0.4 %). A function of sizes only, and
// the one for forward, backward and the traced (fake) implementations, which have to agree on which tensors exist.
bool dw_from_rows(int64_t align, int64_t flags, const std::vector<std::pair<int64_t, int64_t>>& shapes) {
  if (!(flags & kDwRows) || align % 64 != 0) return false;
  for (const auto& [m, n] : shapes)
    if (std::min(m, n) < 256 || m % 8 != 0 || n % 8 != 0) return false;
  return true;
}

// padded grouped copy of `src` rows (fan_out == 0: src is already padded-grouped) and / or its transpose; rows: the table the
// rows are read through (default seg.row_slot)
std::pair<Tensor, Tensor> group_rows(const Tensor& src, const Tensor& coeff, int64_t fan_out, const Segments& seg, bool want_grouped,
                                     bool want_transposed, const Tensor& rows = Tensor()) {
  const int64_t H = src.size(-1);
  Tensor grouped, grouped_t;
  if (want_grouped) grouped = new_empty({seg.max_rows, H}, src);
  if (want_transposed) grouped_t = new_empty({H, seg.max_rows}, src);
  const Launch l(src);
  const ck_segments cs = seg.c(rows);
  check(api.ck_group_segment_rows(ptr(src), ptr(coeff), (int32_t)fan_out, (int32_t)H, &cs, ptr(grouped), ptr(grouped_t), seg.max_rows,
                                  dtype_code(src), l.stream));
  return {grouped, grouped_t};
}

// sum over a token's k slots of gates * expanded (gates undefined: plain sum)
Tensor combine(const Tensor& expanded, const Tensor& gates, int64_t T, int64_t k, int64_t H) {
  const Tensor out = new_empty({T, H}, expanded);
  const Launch l(expanded);
  check(api.ck_combine_rows(ptr(expanded), ptr(gates), T, (int32_t)k, (int32_t)H, ptr(out), nullptr, nullptr, dtype_code(expanded), l.stream));
  return out;
}

// d_gates in fp32 (kept in `slot` for the router's backward) and rounded to the gates' dtype for autograd
Tensor gate_grad(const Tensor& expanded, const Tensor& grad_out, int64_t T, int64_t k, int64_t H, GateSlot* slot) {
  const Tensor d32 = new_empty({T, k}, expanded, at::kFloat), rounded = new_empty({T, k}, expanded);
  const Launch l(expanded);
  check(api.ck_gate_grad_both(ptr(expanded), ptr(grad_out), T, (int32_t)k, (int32_t)H, (float*)ptr(d32), ptr(rounded), dtype_code(expanded), l.stream));
  if (slot != nullptr) slot->d_gates_f32 = d32;
  return rounded;
}

Tensor expert_bias_grad(const Tensor& d_y, const Segments& seg) {
  const Tensor d_bias = new_empty({seg.experts, d_y.size(1)}, d_y);
  const ck_segments cs = seg.c();
  const Launch l(d_y);
  check(api.ck_expert_bias_grad(ptr(d_y), (int32_t)d_y.size(1), &cs, ptr(d_bias), dtype_code(d_y), l.stream));
  return d_bias;
}

// y[r] += bias[expert of row r] in place: padded grouped rows (row_expert undefined) or token-order rows
void add_expert_bias(const Tensor& y, const Tensor& bias, const Segments& seg, const Tensor& row_expert) {
  const ck_segments cs = seg.c();
  const Launch l(y);
  check(api.ck_add_expert_bias(ptr(y), y.size(0), (int32_t)y.size(1), ptr(bias), (const int32_t*)ptr(row_expert),
                               row_expert.defined() ? nullptr : &cs, dtype_code(y), l.stream));
}

// ---- fused gated block: out = combine_k( gates * c_proj( act( c_fc(x) ) ) ), the activation in the c_fc epilogue
struct Block {
  Tensor out, pre, act, act_t, expanded;
};

// keep_pre: whether the c_fc GEMM also writes its pre-activation (a backward pass reads it; without one, two thirds of that
// GEMM's stores go away). keep_act: d_w_proj needs the activation, as it is or, where its GEMM has no row-major form,
// transposed (act_t, a second output of the same epilogue).
Block swiglu_experts_forward(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates, const Segments& seg,
                             int64_t act_kind, bool keep_pre, bool keep_act, int64_t flags) {
  require_dims({{&x, 2}, {&w_fc, 3}, {&w_proj, 3}, {&gates, 2}});
  require_gpu(x, w_fc, w_proj, gates);
  const int64_t T = x.size(0), H = x.size(1), k = gates.size(1), two_i = w_fc.size(1), I = two_i / 2;
  Block b;
  if (keep_pre) b.pre = new_empty({seg.max_rows, two_i}, x);
  b.act = new_empty({seg.max_rows, I}, x);
  if (keep_act && !dw_from_rows(seg.align, flags, {{H, I}, {two_i, H}})) b.act_t = new_empty({I, seg.max_rows}, x);
  const Tensor none;
  gemm(x, k, w_fc, seg, act_kind == CK_ACT_GLU ? CK_EPI_GLU : CK_EPI_SWIGLU, b.pre, b.act_t, b.act, none, none, none, flags);
  b.expanded = new_empty({T * k, H}, x);
  gemm(b.act, 0, w_proj, seg, CK_EPI_SCATTER, b.expanded, none, none, none, none, none, flags);
  b.out = combine(b.expanded, gates, T, k, H);
  return b;
}

struct BlockGrads {
  Tensor d_x, d_w_fc, d_w_proj, d_gates;
};

BlockGrads swiglu_experts_backward(const Tensor& grad_out_in, const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates,
                                   const Tensor& pre, const Tensor& act_saved, const Tensor& expanded, const Segments& seg, int64_t act_kind,
                                   bool need_x, bool need_fc, bool need_proj, bool need_gates, GateSlot* slot, int64_t flags) {
  const int64_t T = x.size(0), H = x.size(1), k = gates.size(1), two_i = w_fc.size(1), I = two_i / 2;
  const Tensor grad_out = grad_out_in.contiguous(), none;
  const bool rows_form = dw_from_rows(seg.align, flags, {{H, I}, {two_i, H}});  // as in forward
  BlockGrads g;
  if (need_gates) g.d_gates = gate_grad(expanded, grad_out, T, k, H, slot);
  if (!(need_x || need_fc || need_proj)) return g;
  // gate-scaled grad_out rows in padded grouped order (+ transpose for d_w_proj unless it reads rows)
  auto [d_y, d_y_t] = group_rows(grad_out, gates, k, seg, true, need_proj && !rows_form);
  if (need_proj) {
    g.d_w_proj = like_contiguous(w_proj);
    if (rows_form) gemm_dw_rows(d_y, act_saved, seg, g.d_w_proj);
    else gemm_dw(d_y_t, act_saved, seg, g.d_w_proj);
    d_y_t.reset();
  }
  if (need_x || need_fc) {
    // d_act = d_y @ w_proj with the leanest epilogue, then one streaming pass for the activation's backward and the transpose
    // d_w_fc needs. (The GEMM can also do this in its epilogue, CK_EPI_SWIGLU_BWD, but with one workgroup per CU the epilogue
    // is time the MFMA units idle, while the streaming pass runs at HBM speed.)
    Tensor d_act = new_empty({seg.max_rows, I}, x);
    gemm_dx(d_y, w_proj, seg, CK_EPI_GROUPED, d_act, none, flags);
    d_y.reset();
    const Tensor d_pre = new_empty({seg.max_rows, two_i}, x);
    Tensor d_pre_t;
    if (need_fc && !rows_form) d_pre_t = new_empty({two_i, seg.max_rows}, x);
    {
      const Launch l(x);
      check(api.ck_swiglu_bwd_grouped(ptr(pre), ptr(d_act), (int32_t)I, (const int32_t*)ptr(seg.seg_starts), (const uint32_t*)ptr(seg.counts),
                                      (const int32_t*)ptr(seg.tile_expert), (int32_t)seg.align, seg.max_rows, ptr(d_pre), ptr(d_pre_t),
                                      seg.max_rows, (int32_t)act_kind, dtype_code(x), l.stream));
    }
    d_act.reset();
    if (need_fc) {
      g.d_w_fc = like_contiguous(w_fc);
      if (rows_form) gemm_dw_rows(d_pre, group_rows(x, none, k, seg, true, false).first, seg, g.d_w_fc);
      else gemm_dw(d_pre_t, group_rows(x, none, k, seg, false, true).second, seg, g.d_w_fc);
      d_pre_t.reset();
    }
    if (need_x) {
      const Tensor d_expanded = new_empty({T * k, H}, x);
      gemm_dx(d_pre, w_fc, seg, CK_EPI_SCATTER, d_expanded, none, flags);
      g.d_x = k == 1 ? d_expanded : combine(d_expanded, none, T, k, H);
    }
  }
  return g;
}

c10::IValue slot_capsule(const SlotPtr& slot) { return slot.defined() ? c10::IValue::make_capsule(slot) : c10::IValue(); }
GateSlot* slot_of(const c10::IValue& v) { return v.isNone() ? nullptr : static_cast<GateSlot*>(v.toCapsule().get()); }

// Tensors, segment tables and integers of a node. The tables are whole numbers that address memory: they are kept beside the
// saved tensors, where no saved-tensor hook (compression, conversion) gets at them.
void save_segments(AutogradContext* ctx, variable_list tensors, const Segments& seg, std::vector<int64_t> ints) {
  ctx->save_for_backward(std::move(tensors));
  ctx->saved_data["tables"] = std::vector<Tensor>{seg.seg_starts, seg.counts, seg.tile_expert, seg.row_slot};
  ints.insert(ints.end(), {seg.max_rows, seg.experts, seg.align});
  ctx->saved_data["ints"] = std::move(ints);
}
Segments saved_segments(AutogradContext* ctx, const std::vector<int64_t>& ints) {
  const std::vector<Tensor> tables = ctx->saved_data["tables"].toTensorVector();
  const size_t i = ints.size() - 3;
  Segments g;
  g.seg_starts = tables[0];
  g.counts = tables[1];
  g.tile_expert = tables[2];
  g.row_slot = tables[3];
  g.max_rows = ints[i];
  g.experts = ints[i + 1];
  g.align = ints[i + 2];
  return g;
}

struct SwigluExperts : torch::autograd::Function<SwigluExperts> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_fc_in, const Tensor& w_proj_in, const Tensor& gates_in,
                        const Segments& seg, int64_t act_kind, SlotPtr slot, int64_t flags) {
    const Tensor x = x_in.contiguous(), w_fc = w_fc_in.contiguous(), w_proj = w_proj_in.contiguous(), gates = gates_in.contiguous();
    const bool need_proj = w_proj_in.requires_grad();
    const Block b = swiglu_experts_forward(x, w_fc, w_proj, gates, seg, act_kind, true, need_proj, flags);
    const Tensor act_saved = b.act_t.defined() ? b.act_t : need_proj ? b.act : Tensor();
    save_segments(ctx, {x, w_fc, w_proj, gates, b.pre, act_saved, b.expanded}, seg,
                  {act_kind, flags, x_in.requires_grad(), w_fc_in.requires_grad(), need_proj, gates_in.requires_grad()});
    ctx->saved_data["slot"] = slot_capsule(slot);
    ctx->set_materialize_grads(false);
    return b.out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(8);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto n = ctx->saved_data["ints"].toIntVector();
    const BlockGrads g = swiglu_experts_backward(grads[0], s[0], s[1], s[2], s[3], s[4], s[5], s[6], saved_segments(ctx, n), n[0], n[2], n[3],
                                                 n[4], n[5], slot_of(ctx->saved_data["slot"]), n[1]);
    out[0] = g.d_x;
    out[1] = g.d_w_fc;
    out[2] = g.d_w_proj;
    out[3] = g.d_gates;
    return out;
  }
};

Tensor swiglu_experts(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates, py::object seg, int64_t act_kind,
                      std::optional<SlotPtr> slot, int64_t flags) {
  const Segments g = Segments::of(seg);
  if (any_requires_grad({&x, &w_fc, &w_proj, &gates}))
    return SwigluExperts::apply(x, w_fc, w_proj, gates, g, act_kind, slot.value_or(SlotPtr()), flags);
  return swiglu_experts_forward(x.contiguous(), w_fc.contiguous(), w_proj.contiguous(), gates.contiguous(), g, act_kind, false, false, flags).out;
}

// ---- c_fc with any activation behind it: y [max_rows, N] (padded grouped), and with gelu the tanh GELU of it, computed in the
// GEMM's epilogue. Pad rows are never written by the kernel: zero_pads makes them zeros, which keeps whatever a caller applies on
// top of them finite; without it they hold anything, which the expert GEMMs and their backward pass do not mind (valid rows
// only), but nobody else may see: inside the node of the whole GELU block.
std::pair<Tensor, Tensor> experts_up_forward(const Tensor& x, const Tensor& w, const Segments& seg, int64_t k, const Tensor& bias, bool gelu,
                                             bool keep_pre, bool zero_pads, int64_t flags) {
  require_dims({{&w, 3}});
  require_gpu(x, w, bias);
  const int64_t N = w.size(1);
  const auto rows = [&] { return zero_pads ? at::zeros({seg.max_rows, N}, x.options()) : at::empty({seg.max_rows, N}, x.options()); };
  Tensor y, act;
  if (keep_pre || !gelu) y = rows();
  if (gelu) act = rows();
  const bool fused_bias = bias.defined() && (gelu || is_f32(x) || (flags & kBiasFused));
  const Tensor none;
  gemm(x, k, w, seg, gelu ? CK_EPI_GELU_TANH : CK_EPI_GROUPED, y, none, act, fused_bias ? bias : none, none, none, flags);
  if (bias.defined() && !fused_bias) add_expert_bias(y, bias, seg, none);
  return {y, act};
}

struct LinearGrads {
  Tensor d_in, d_w, d_gates, d_bias;
};

// pre: the pre-activation where the GELU ran in the epilogue (d_y_in is then d_act), else undefined
LinearGrads experts_up_backward(const Tensor& d_y_in, const Tensor& x, const Tensor& w, const Tensor& pre, const Segments& seg, int64_t k,
                                bool need_x, bool need_w, bool need_bias, int64_t flags) {
  require_dims({{&x, 2}});
  const int64_t T = x.size(0), K = x.size(1);
  Tensor d_y = d_y_in.contiguous();
  const Tensor none;
  if (pre.defined()) {
    const Tensor d_act = d_y;
    d_y = like_contiguous(d_act);
    const Launch l(d_act);
    const int64_t N = pre.size(1);
    const auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    if (N % 8 == 0 && aligned(pre) && aligned(d_act) && aligned(d_y)) {  // whole 16-byte pieces of rows: the pad rows are left out
      const ck_segments cs = seg.c();
      check(api.ck_gelu_tanh_bwd_grouped(ptr(pre), ptr(d_act), (int32_t)N, &cs, ptr(d_y), dtype_code(d_act), l.stream));
    } else {
      check(api.ck_gelu_tanh_bwd(ptr(pre), ptr(d_act), ptr(d_y), d_act.numel(), dtype_code(d_act), l.stream));
    }
  }
  LinearGrads g;
  if (need_bias) g.d_bias = expert_bias_grad(d_y, seg);
  if (need_w) {
    g.d_w = like_contiguous(w);
    if (is_f32(x) || dw_from_rows(seg.align, flags, {{w.size(1), w.size(2)}})) gemm_dw_rows(d_y, group_rows(x, none, k, seg, true, false).first, seg, g.d_w);
    else gemm_dw(group_rows(d_y, none, 0, seg, false, true).second, group_rows(x, none, k, seg, false, true).second, seg, g.d_w);
  }
  if (need_x) {
    const Tensor d_expanded = new_empty({T * k, K}, x);
    gemm_dx(d_y, w, seg, CK_EPI_SCATTER, d_expanded, none, flags);
    g.d_in = k == 1 ? d_expanded : combine(d_expanded, none, T, k, K);
  }
  return g;
}

struct ExpertsUp : torch::autograd::Function<ExpertsUp> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_in, const OptTensor& bias, const Segments& seg, int64_t k,
                        bool gelu, int64_t flags) {
    const Tensor x = x_in.contiguous(), w = w_in.contiguous();
    auto [y, act] = experts_up_forward(x, w, seg, k, contiguous(value_or_undefined(bias)), gelu, true, true, flags);
    save_segments(ctx, {x, w, gelu ? y : Tensor()}, seg,
                  {k, flags, x_in.requires_grad(), w_in.requires_grad(), bias.has_value() && bias->requires_grad()});
    ctx->set_materialize_grads(false);
    return gelu ? act : y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(7);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto n = ctx->saved_data["ints"].toIntVector();
    const LinearGrads g = experts_up_backward(grads[0], s[0], s[1], s[2], saved_segments(ctx, n), n[0], n[2], n[3], n[4], n[1]);
    out[0] = g.d_in;
    out[1] = g.d_w;
    out[2] = g.d_bias;
    return out;
  }
};

Tensor experts_up(const Tensor& x, const Tensor& w, const OptTensor& bias, py::object seg, int64_t k, bool gelu, int64_t flags) {
  const Tensor b = value_or_undefined(bias);
  const Segments g = Segments::of(seg);
  if (any_requires_grad({&x, &w, &b})) return ExpertsUp::apply(x, w, bias, g, k, gelu, flags);
  auto [y, act] = experts_up_forward(x.contiguous(), w.contiguous(), g, k, contiguous(b), gelu, false, true, flags);
  return gelu ? act : y;
}

// expert of every flat (token, slot) index, int32 [R] (the inverse of the sort)
Tensor slot_experts(const Tensor& sorted_expert_idxs, const Tensor& sorted_scattered_idxs) {
  const Tensor slot_expert = at::empty_like(sorted_expert_idxs);
  slot_expert.index_put_({sorted_scattered_idxs.to(at::kLong)}, sorted_expert_idxs);
  return slot_expert;
}

// ---- c_proj: h [max_rows, I] (padded grouped), gates [T, k] -> (out [T, N], expanded [T * k, N]). slot_expert: expert of every flat
// slot, needed where the bias is added by its own kernel
std::pair<Tensor, Tensor> experts_down_forward(const Tensor& h, const Tensor& w, const Tensor& gates, const Segments& seg, const Tensor& bias,
                                               const Tensor& slot_expert, int64_t flags) {
  require_dims({{&w, 3}, {&gates, 2}});
  require_gpu(h, w, gates, bias);
  const int64_t T = gates.size(0), k = gates.size(1), N = w.size(1);
  const Tensor expanded = new_empty({T * k, N}, h), none;
  const bool fused_bias = bias.defined() && (is_f32(h) || (flags & kBiasFused));
  gemm(h, 0, w, seg, CK_EPI_SCATTER, expanded, none, none, fused_bias ? bias : none, none, none, flags);
  // before the gate multiply, as cute_kernels/kernels/scattermoe/torch_implementation.py:160-163
  if (bias.defined() && !fused_bias) add_expert_bias(expanded, bias, seg, slot_expert);
  return {combine(expanded, gates, T, k, N), expanded};
}

LinearGrads experts_down_backward(const Tensor& grad_out_in, const Tensor& h, const Tensor& w, const Tensor& gates, const Tensor& expanded,
                                  const Segments& seg, bool need_h, bool need_w, bool need_gates, bool need_bias, bool zero_pads,
                                  GateSlot* slot, int64_t flags) {
  const int64_t T = gates.size(0), k = gates.size(1), N = w.size(1), K = w.size(2);
  const Tensor grad_out = grad_out_in.contiguous(), none;
  LinearGrads g;
  if (need_gates) g.d_gates = gate_grad(expanded, grad_out, T, k, N, slot);
  if (!(need_h || need_w || need_bias)) return g;
  const bool rows_form = is_f32(h) || dw_from_rows(seg.align, flags, {{N, K}});
  auto [d_y, d_y_t] = group_rows(grad_out, gates, k, seg, true, need_w && !rows_form);
  if (need_bias) g.d_bias = expert_bias_grad(d_y, seg);  // d_y: the gate-scaled grad_out rows in padded grouped order
  if (need_w) {
    g.d_w = like_contiguous(w);
    if (rows_form) gemm_dw_rows(d_y, h, seg, g.d_w);
    else gemm_dw(d_y_t, group_rows(h, none, 0, seg, false, true).second, seg, g.d_w);
  }
  if (need_h) {
    g.d_in = zero_pads ? at::zeros({seg.max_rows, K}, h.options()) : at::empty({seg.max_rows, K}, h.options());
    gemm_dx(d_y, w, seg, CK_EPI_GROUPED, g.d_in, none, flags);
  }
  return g;
}

struct ExpertsDown : torch::autograd::Function<ExpertsDown> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h_in, const Tensor& w_in, const Tensor& gates_in, const OptTensor& bias,
                        const Segments& seg, const OptTensor& slot_expert, SlotPtr slot, int64_t flags) {
    const Tensor h = h_in.contiguous(), w = w_in.contiguous(), gates = gates_in.contiguous();
    auto [out, expanded] = experts_down_forward(h, w, gates, seg, contiguous(value_or_undefined(bias)),
                                                value_or_undefined(slot_expert), flags);
    save_segments(ctx, {h, w, gates, expanded}, seg,
                  {flags, h_in.requires_grad(), w_in.requires_grad(), gates_in.requires_grad(),
                   bias.has_value() && bias->requires_grad()});
    ctx->saved_data["slot"] = slot_capsule(slot);
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(8);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto n = ctx->saved_data["ints"].toIntVector();
    const LinearGrads g = experts_down_backward(grads[0], s[0], s[1], s[2], s[3], saved_segments(ctx, n), n[1], n[2], n[3], n[4], true,
                                                slot_of(ctx->saved_data["slot"]), n[0]);
    out[0] = g.d_in;
    out[1] = g.d_w;
    out[2] = g.d_gates;
    out[3] = g.d_bias;
    return out;
  }
};

Tensor experts_down(const Tensor& h, const Tensor& w, const Tensor& gates, const OptTensor& bias, py::object seg, std::optional<SlotPtr> slot,
                    int64_t flags) {
  const Tensor b = value_or_undefined(bias);
  const Segments g = Segments::of(seg);
  Tensor slot_expert;
  if (b.defined() && !is_f32(h) && !(flags & kBiasFused))
    slot_expert = slot_experts(seg.attr("sorted_expert_idxs").cast<Tensor>(), seg.attr("sorted_scattered_idxs").cast<Tensor>());
  if (any_requires_grad({&h, &w, &gates, &b}))
    return ExpertsDown::apply(h, w, gates, bias, g, to_opt(slot_expert), slot.value_or(SlotPtr()), flags);
  return experts_down_forward(h.contiguous(), w.contiguous(), gates.contiguous(), g, contiguous(b), slot_expert, flags).first;
}

// ---- the tanh-GELU block as one node: out = combine_k( gates * c_proj( gelu( c_fc(x) ) ) ). The activation's gradient, whose
// pad rows nothing writes, stays inside: between two nodes a hook or anomaly mode would read them.
struct GeluExperts : torch::autograd::Function<GeluExperts> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_fc_in, const Tensor& w_proj_in, const Tensor& gates_in,
                        const OptTensor& bias_fc, const OptTensor& bias_proj, const Segments& seg, SlotPtr slot, int64_t flags) {
    const Tensor x = x_in.contiguous(), w_fc = w_fc_in.contiguous(), w_proj = w_proj_in.contiguous(), gates = gates_in.contiguous();
    auto [pre, act] = experts_up_forward(x, w_fc, seg, gates.size(1), contiguous(value_or_undefined(bias_fc)), true, true, false, flags);
    auto [out, expanded] = experts_down_forward(act, w_proj, gates, seg, contiguous(value_or_undefined(bias_proj)), Tensor(), flags);
    const auto needs = [](const OptTensor& b) { return b.has_value() && b->requires_grad(); };
    save_segments(ctx, {x, w_fc, w_proj, gates, pre, act, expanded}, seg,
                  {flags, x_in.requires_grad(), w_fc_in.requires_grad(), w_proj_in.requires_grad(), gates_in.requires_grad(),
                   needs(bias_fc), needs(bias_proj)});
    ctx->saved_data["slot"] = slot_capsule(slot);
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(9);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto n = ctx->saved_data["ints"].toIntVector();
    const Segments seg = saved_segments(ctx, n);
    const bool need_act = n[1] || n[2] || n[5];
    const LinearGrads down = experts_down_backward(grads[0], s[5], s[2], s[3], s[6], seg, need_act, n[3], n[4], n[6], false,
                                                   slot_of(ctx->saved_data["slot"]), n[0]);
    out[2] = down.d_w;
    out[3] = down.d_gates;
    out[5] = down.d_bias;
    if (need_act) {
      const LinearGrads up = experts_up_backward(down.d_in, s[0], s[1], s[4], seg, s[3].size(1), n[1], n[2], n[5], n[0]);
      out[0] = up.d_in;
      out[1] = up.d_w;
      out[4] = up.d_bias;
    }
    return out;
  }
};

// both biases join the accumulators (kBiasFused)
Tensor gelu_experts(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates, const OptTensor& bias_fc,
                    const OptTensor& bias_proj, py::object seg, std::optional<SlotPtr> slot, int64_t flags) {
  require_dims({{&x, 2}, {&w_fc, 3}, {&w_proj, 3}, {&gates, 2}});
  const Tensor b_fc = value_or_undefined(bias_fc), b_proj = value_or_undefined(bias_proj);
  const Segments g = Segments::of(seg);
  if (any_requires_grad({&x, &w_fc, &w_proj, &gates, &b_fc, &b_proj}))
    return GeluExperts::apply(x, w_fc, w_proj, gates, bias_fc, bias_proj, g, slot.value_or(SlotPtr()), flags);
  const Tensor act = experts_up_forward(x.contiguous(), w_fc.contiguous(), g, gates.size(1), contiguous(b_fc), true, false, false, flags).second;
  return experts_down_forward(act, w_proj.contiguous(), gates.contiguous(), g, contiguous(b_proj), Tensor(), flags).first;
}

// ---- quantised-expert forward (inference) ------------------------------------------------------------------------
// seg: x holds the rows of that padded grouped layout; those that stand for nothing stay undefined
std::pair<Tensor, Tensor> quantize_rows(const Tensor& x_in, const Segments* seg = nullptr) {
  require_gpu(x_in);
  const Tensor x = x_in.contiguous();
  const Launch l(x);
  const Tensor q = new_empty({x.size(0), x.size(1)}, x, at::kFloat8_e4m3fn), scale = new_empty({x.size(0)}, x, at::kFloat);
  if (seg != nullptr) {
    const ck_segments cs = seg->c();
    check(api.ck_quant_grouped_rows_e4m3(ptr(x), &cs, (int32_t)x.size(1), ptr(q), (float*)ptr(scale), dtype_code(x), l.stream));
  } else
    check(api.ck_quant_rows_e4m3(ptr(x), x.size(0), (int32_t)x.size(1), ptr(q), (float*)ptr(scale), dtype_code(x), l.stream));
  return {q, scale};
}

void gemm_fp8(const Tensor& a8, const Tensor& a_scale, int64_t gather_div, const Tensor& w8, const Tensor& w_scale, const Segments& seg,
              int64_t epilogue, const Tensor& y, const Tensor& aux, at::ScalarType out_dtype) {
  const int64_t N = w8.size(1), K = w8.size(2);
  if (gather_div > 0) TORCH_CHECK(a8.numel() < (1ll << 32), "the token-order fp8 input of a grouped GEMM must stay below 4 GiB");
  timed(epilogue == CK_EPI_SWIGLU ? "fp8_grouped_gemm<swiglu>" : epilogue == CK_EPI_SCATTER ? "fp8_grouped_gemm<scatter>" : "fp8_grouped_gemm<grouped>",
        N, K, [&] {
          const Launch l(w8);
          const ck_segments cs = seg.c();
          check(api.ck_grouped_gemm_fp8(ptr(a8), (const float*)ptr(a_scale), (int32_t)gather_div, ptr(w8), (const float*)ptr(w_scale), (int32_t)N,
                                        (int32_t)K, &cs, (int32_t)epilogue, ptr(y), ptr(aux), dtype_code(out_dtype), l.stream));
        });
}

Tensor swiglu_experts_e4m3(const Tensor& x, const Tensor& w_fc8, const Tensor& w_fc_scale, const Tensor& w_proj8, const Tensor& w_proj_scale,
                           const Tensor& gates_in, py::object seg, const OptTensor& x8_in, const OptTensor& x_scale_in) {
  require_dims({{&x, 2}, {&w_fc8, 3}, {&w_proj8, 3}, {&gates_in, 2}});
  require_gpu(x, w_fc8, w_proj8, gates_in);
  const at::NoGradGuard no_grad;
  const Segments g = Segments::of(seg);
  const int64_t T = x.size(0), H = x.size(1), k = gates_in.size(1), I = w_fc8.size(1) / 2;
  Tensor x8, x_scale;
  if (x8_in.has_value()) {
    x8 = *x8_in;
    x_scale = *x_scale_in;
  } else {
    std::tie(x8, x_scale) = quantize_rows(x);  // per token
  }
  const Tensor none;
  const Tensor act = new_empty({g.max_rows, I}, x);  // pad rows: never written, quantised perhaps, never used
  gemm_fp8(x8, x_scale, k, w_fc8, w_fc_scale, g, CK_EPI_SWIGLU, none, act, x.scalar_type());
  // per routed row; the look-up that leaves padding out where that may be more than a quarter of the rows (at 6 % it gains nothing)
  auto [act8, act_scale] = quantize_rows(act, 4 * T * k < 3 * g.max_rows ? &g : nullptr);
  const Tensor expanded = new_empty({T * k, H}, x);
  gemm_fp8(act8, act_scale, 0, w_proj8, w_proj_scale, g, CK_EPI_SCATTER, expanded, none, x.scalar_type());
  return combine(expanded, gates_in.to(x.scalar_type()).contiguous(), T, k, H);
}

// ---- SwiGLU -----------------------------------------------------------------------------------------------------
Tensor swiglu_forward(const Tensor& gate, const Tensor& up) {  // contiguous, one flat row
  const Launch l(gate);
  const Tensor out = like_contiguous(gate);
  const int64_t n = gate.numel();
  check(api.ck_swiglu_fwd(ptr(gate), n, ptr(up), n, ptr(out), n, 1, n, dtype_code(gate), l.stream));
  return out;
}
std::tuple<Tensor, Tensor> swiglu_backward(const Tensor& gate, const Tensor& up, const Tensor& grad_in) {
  const Tensor grad = grad_in.contiguous(), d_gate = like_contiguous(gate), d_up = like_contiguous(up);
  const Launch l(gate);
  const int64_t n = gate.numel();
  check(api.ck_swiglu_bwd(ptr(gate), n, ptr(up), n, ptr(grad), n, ptr(d_gate), n, ptr(d_up), n, 1, n, dtype_code(gate), l.stream));
  return {d_gate, d_up};
}

struct Swiglu : torch::autograd::Function<Swiglu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate_in, const Tensor& up_in) {
    const Tensor gate = gate_in.contiguous(), up = up_in.contiguous();
    ctx->save_for_backward({gate, up});
    ctx->set_materialize_grads(false);
    return swiglu_forward(gate, up);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return {Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    auto [d_gate, d_up] = swiglu_backward(s[0], s[1], grads[0]);
    return {d_gate, d_up};
  }
};
Tensor swiglu(const Tensor& gate, const Tensor& up) {
  require_gpu(gate, up);
  if (any_requires_grad({&gate, &up})) return Swiglu::apply(gate, up);
  return swiglu_forward(gate.contiguous(), up.contiguous());
}

// packed: the first half of a row is up, the second half gate (cute_kernels/kernels/swiglu/__init__.py:121), both read in place
// through the row stride
struct Halves {
  int64_t width, half, rows;
  explicit Halves(const Tensor& x) : width(x.size(-1)), half(width / 2), rows(width ? x.numel() / width : 0) {}
  static char* second(const Tensor& x, int64_t half) { return x.numel() ? (char*)x.data_ptr() + half * x.element_size() : (char*)x.data_ptr(); }
};
Tensor swiglu_packed_forward(const Tensor& x) {
  const Launch l(x);
  const Halves h(x);
  auto size = x.sizes().vec();
  size.back() = h.half;
  const Tensor out = at::empty(size, x.options());
  check(api.ck_swiglu_fwd(Halves::second(x, h.half), h.width, ptr(x), h.width, ptr(out), h.half, h.rows, h.half, dtype_code(x), l.stream));
  return out;
}
Tensor swiglu_packed_backward(const Tensor& x, const Tensor& grad_in) {
  const Tensor grad = grad_in.contiguous(), d_x = like_contiguous(x);
  const Launch l(x);
  const Halves h(x);
  check(api.ck_swiglu_bwd(Halves::second(x, h.half), h.width, ptr(x), h.width, ptr(grad), h.half, Halves::second(d_x, h.half), h.width, ptr(d_x),
                          h.width, h.rows, h.half, dtype_code(x), l.stream));
  return d_x;
}
struct SwigluPacked : torch::autograd::Function<SwigluPacked> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in) {
    const Tensor x = x_in.contiguous();
    ctx->save_for_backward({x});
    ctx->set_materialize_grads(false);
    return swiglu_packed_forward(x);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return {Tensor()};
    return {swiglu_packed_backward(ctx->get_saved_variables()[0], grads[0])};
  }
};
Tensor swiglu_packed(const Tensor& x) {
  require_gpu(x);
  if (any_requires_grad({&x})) return SwigluPacked::apply(x);
  return swiglu_packed_forward(x.contiguous());
}

// ---- RMSNorm, with and without the residual add ------------------------------------------------------------------
std::tuple<Tensor, Tensor> rmsnorm_forward(const Tensor& x, const Tensor& weight, double eps, bool want_rstd) {
  const Launch l(x);
  const int64_t H = x.size(-1), B = row_count(x);
  const Tensor out = like_contiguous(x);
  Tensor rstd;
  if (want_rstd) rstd = new_empty({B}, x, at::kFloat);
  check(api.ck_rmsnorm_fwd(ptr(x), ptr(weight), (float)eps, B, (int32_t)H, ptr(out), (float*)ptr(rstd), dtype_code(x), l.stream));
  return {out, rstd};
}
std::tuple<Tensor, Tensor, Tensor> residual_rmsnorm_forward(const Tensor& x, const Tensor& residual, const Tensor& weight, double eps,
                                                            double multiplier, bool want_rstd) {
  const Launch l(x);
  const int64_t H = x.size(-1), B = row_count(x);
  const Tensor out = like_contiguous(x), added = like_contiguous(x);
  Tensor rstd;
  if (want_rstd) rstd = new_empty({B}, x, at::kFloat);
  check(api.ck_fused_residual_add_rmsnorm_fwd(ptr(x), ptr(residual), ptr(weight), (float)eps, (float)multiplier, B, (int32_t)H, ptr(out), ptr(added),
                                              (float*)ptr(rstd), dtype_code(x), l.stream));
  return {out, added, rstd};
}
// x: the normalised tensor (with the residual: the sum). d_added: the gradient that arrives through the residual stream, or
// undefined. Returns (d_x, d_residual, d_weight); without `residual` d_residual stays undefined, with one_buffer it is d_x.
std::tuple<Tensor, Tensor, Tensor> rmsnorm_backward(const Tensor& x, const Tensor& weight, const Tensor& rstd, const Tensor& d_out_in,
                                                    const Tensor& d_added_in, double eps, double multiplier, bool residual, bool one_buffer) {
  const Tensor d_out = d_out_in.contiguous(), d_added = contiguous(d_added_in);
  const Launch l(x);
  const int64_t H = x.size(-1), B = row_count(x);
  const Tensor d_x = like_contiguous(x);
  Tensor d_residual, d_weight, partial;
  if (residual) d_residual = one_buffer ? d_x : like_contiguous(x);
  if (weight.defined()) {
    d_weight = new_empty({H}, x);
    partial = new_empty({std::max<int64_t>(api.ck_rmsnorm_bwd_partial_rows(B), 1), H}, x, at::kFloat);
  }
  check(api.ck_rmsnorm_bwd_typed(ptr(x), ptr(weight), ptr(d_out), ptr(d_added), (const float*)ptr(rstd), (float)eps, (float)multiplier, B, (int32_t)H,
                                 ptr(d_x), ptr(d_residual), (float*)ptr(partial), ptr(d_weight), dtype_code(x), l.stream));
  return {d_x, d_residual, d_weight};
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const OptTensor& weight_in, double eps, bool memory_efficient) {
    const Tensor x = x_in.contiguous(), weight = contiguous(value_or_undefined(weight_in));
    auto [out, rstd] = rmsnorm_forward(x, weight, eps, !memory_efficient);
    ctx->save_for_backward({x, weight, rstd});
    ctx->saved_data["eps"] = eps;
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    auto [d_x, none, d_weight] = rmsnorm_backward(s[0], s[1], s[2], grads[0], Tensor(), ctx->saved_data["eps"].toDouble(), 1.0, false, false);
    return {d_x, d_weight, Tensor(), Tensor()};
  }
};
Tensor rmsnorm(const Tensor& x, const OptTensor& weight, double eps, bool memory_efficient) {
  const Tensor w = value_or_undefined(weight);
  require_gpu(x, w);
  if (any_requires_grad({&x, &w})) return RmsNorm::apply(x, weight, eps, memory_efficient);
  return std::get<0>(rmsnorm_forward(x.contiguous(), contiguous(w), eps, false));
}

struct ResidualRmsNorm : torch::autograd::Function<ResidualRmsNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& residual_in, const OptTensor& weight_in, double eps,
                               double multiplier, bool memory_efficient) {
    const Tensor weight = contiguous(value_or_undefined(weight_in));
    auto [out, added, rstd] = residual_rmsnorm_forward(x_in.contiguous(), residual_in.contiguous(), weight, eps, multiplier, !memory_efficient);
    ctx->save_for_backward({added, weight, rstd});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["multiplier"] = multiplier;
    // multiplier 1: both gradients are the same values, so one tensor serves both (written once: 368 against 497 us at
    // 65,536 x 4,096). Not where x or residual is a leaf: its .grad takes over only a tensor nobody else holds and copies a
    // shared one (16,384 x 4,096, forward and backward: 239 us with that copy, 214 with two stores).
    const auto leaf = [](const Tensor& t) { return t.requires_grad() && t.is_leaf(); };
    ctx->saved_data["one_buffer"] = multiplier == 1.0 && !leaf(x_in) && !leaf(residual_in);
    ctx->set_materialize_grads(false);
    return {out, added};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(6);
    if (!grads[0].defined() && !grads[1].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const Tensor d_out = grads[0].defined() ? grads[0] : at::zeros_like(s[0]);
    auto [d_x, d_residual, d_weight] = rmsnorm_backward(s[0], s[1], s[2], d_out, grads[1], ctx->saved_data["eps"].toDouble(),
                                                        ctx->saved_data["multiplier"].toDouble(), true, ctx->saved_data["one_buffer"].toBool());
    out[0] = d_x;
    out[1] = d_residual;
    out[2] = d_weight;
    return out;
  }
};
std::tuple<Tensor, Tensor> residual_rmsnorm(const Tensor& x, const Tensor& residual, const OptTensor& weight, double eps, double multiplier,
                                            bool memory_efficient) {
  const Tensor w = value_or_undefined(weight);
  require_gpu(x, residual, w);
  if (any_requires_grad({&x, &residual, &w})) {
    auto out = ResidualRmsNorm::apply(x, residual, weight, eps, multiplier, memory_efficient);
    return {out[0], out[1]};
  }
  auto [out, added, rstd] = residual_rmsnorm_forward(x.contiguous(), residual.contiguous(), contiguous(w), eps, multiplier, false);
  return {out, added};
}

// ---- RMSNorm fused ahead of the router ---------------------------------------------------------------------------
struct NormRoute {
  Tensor y, logits, rstd, x8, scale8;
};
// Where ck_router_rows is the faster way from rows to router logits: while its workgroups of 16 rows x 16 experts do not outnumber
// the compute units.
bool router_rows_fit(int64_t B, int64_t H, int64_t E) {
  return H >= 32 && H % 32 == 0 && H <= 4096 && E >= 1 && ((B + 15) / 16) * ((E + 15) / 16) <= 256;
}
bool router_rows_take(const Tensor& x, const Tensor& gate_weight, const OptTensor& norm_weight) {
  if (!x.is_cuda() || x.dim() < 1 || gate_weight.dim() != 2 || (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf)) return false;
  const Tensor nw = value_or_undefined(norm_weight);
  for (const Tensor* t : {&x, &gate_weight, &nw}) {
    if (!t->defined()) continue;
    if (t->device() != x.device()) return false;
    // the kernel reads 16 bytes at a time; what is not contiguous is copied first, to where a new tensor begins
    if (t->is_contiguous() && (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) != 0) return false;
    if (t->_fw_grad(/*level=*/0).defined()) return false;  // forward-mode tangents
  }
  const int64_t H = x.size(-1);
  return x.numel() > 0 && router_rows_fit(x.numel() / H, H, gate_weight.size(0));
}
Tensor router_rows_forward(const Tensor& x_in, const Tensor& gate_weight_in) {
  const int64_t B = x_in.size(0), H = x_in.size(1), E = gate_weight_in.size(0);
  const Tensor x = x_in.contiguous(), gate_weight = gate_weight_in.contiguous();
  const Launch l(x);
  const Tensor logits = new_empty({B, E}, x);
  check(api.ck_router_rows(ptr(x), nullptr, ptr(gate_weight), 0.f, 0, B, (int32_t)H, (int32_t)E, nullptr, nullptr, ptr(logits), nullptr, nullptr,
                           dtype_code(x), l.stream));
  return logits;
}
struct RouterRows : torch::autograd::Function<RouterRows> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& gate_weight) {
    // what a linear layer saves: a tensor that no gradient is computed from may be written to before the backward pass
    ctx->save_for_backward({gate_weight.requires_grad() ? x : Tensor(), x.requires_grad() ? gate_weight : Tensor()});
    return router_rows_forward(x, gate_weight);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {  // as a linear layer's
    const auto s = ctx->get_saved_variables();
    const Tensor& d_logits = grads[0];
    return {ctx->needs_input_grad(0) ? at::mm(d_logits, s[1]) : Tensor(), ctx->needs_input_grad(1) ? at::mm(d_logits.t(), s[0]) : Tensor()};
  }
};
// x @ gate_weight^T of few 16-bit rows (router_rows_take)
Tensor router_rows(const Tensor& x, const Tensor& gate_weight) {
  require_dims({{&x, 2}, {&gate_weight, 2}});
  require_gpu(x, gate_weight);
  TORCH_CHECK(gate_weight.size(1) == x.size(1) && gate_weight.scalar_type() == x.scalar_type(), "router_rows: rows and weight disagree");
  if (any_requires_grad({&x, &gate_weight})) return RouterRows::apply(x, gate_weight);
  return router_rows_forward(x, gate_weight);
}
// few_rows: ck_router_rows, which the caller has found to take the call, instead of ck_rmsnorm_route
NormRoute norm_route_forward(const Tensor& x, const Tensor& norm_weight, const Tensor& gate_weight, double eps, bool quantize, bool want_rstd,
                             bool few_rows) {
  const Launch l(x);
  const int64_t B = x.size(0), H = x.size(1), E = gate_weight.size(0);
  NormRoute r;
  r.y = like_contiguous(x);
  r.logits = new_empty({B, E}, x);
  if (want_rstd) r.rstd = new_empty({B}, x, at::kFloat);
  if (quantize) {
    r.x8 = new_empty({B, H}, x, at::kFloat8_e4m3fn);
    r.scale8 = new_empty({B}, x, at::kFloat);
  }
  if (few_rows) {
    check(api.ck_router_rows(ptr(x), ptr(norm_weight), ptr(gate_weight), (float)eps, 1, B, (int32_t)H, (int32_t)E, ptr(r.y), (float*)ptr(r.rstd),
                             ptr(r.logits), ptr(r.x8), (float*)ptr(r.scale8), dtype_code(x), l.stream));
    return r;
  }
  const Tensor packed = new_empty({(E + 15) / 16 * 16 * H}, x);  // workspace of the call
  check(api.ck_rmsnorm_route(ptr(x), ptr(norm_weight), ptr(gate_weight), (float)eps, B, (int32_t)H, (int32_t)E, ptr(r.y), (float*)ptr(r.rstd),
                             ptr(r.logits), ptr(r.x8), (float*)ptr(r.scale8), ptr(packed), dtype_code(x), l.stream));
  return r;
}

// d_logits^T @ y ([E, tokens] x [tokens, H]). The BLAS library runs this skinny product (E rows, a contraction as long as the
// batch) on a few workgroups; cut into 16 slices of the tokens it is a batched product that fills the chip, and the 16 partial
// results are added in fp32 (measured on MI355X: 55 -> 27 us at 8,192 x 64 x 2,048, 331 -> 104 us at 65,536 x 128 x 4,096).
Tensor gate_weight_grad(const Tensor& d_logits, const Tensor& y) {
  const int64_t tokens = d_logits.size(0), E = d_logits.size(1), slices = 16;
  if (tokens < 4096 || tokens % slices != 0 || !d_logits.is_contiguous() || !y.is_contiguous()) return at::mm(d_logits.t(), y);
  const Tensor parts = at::bmm(d_logits.view({slices, tokens / slices, E}).transpose(1, 2), y.view({slices, tokens / slices, y.size(1)}));
  return at::sum(parts, at::IntArrayRef{0}, false, at::kFloat).to(y.scalar_type());
}

struct NormRouteFn : torch::autograd::Function<NormRouteFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const OptTensor& norm_weight_in, const Tensor& gate_weight_in, double eps,
                               bool few_rows) {
    const Tensor x = x_in.contiguous(), nw = contiguous(value_or_undefined(norm_weight_in)), gw = gate_weight_in.contiguous();
    NormRoute r = norm_route_forward(x, nw, gw, eps, false, true, few_rows);
    ctx->save_for_backward({x, nw, gw, r.rstd, r.y});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["need_gate"] = gate_weight_in.requires_grad();
    ctx->set_materialize_grads(false);
    return {r.y, r.logits};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(5);
    const auto s = ctx->get_saved_variables();
    Tensor d_total = grads[0];
    if (grads[1].defined()) {
      if (ctx->saved_data["need_gate"].toBool()) out[2] = gate_weight_grad(grads[1], s[4]);
      // y's own gradient joins the product's fp32 sums: one pass over the rows less than adding it afterwards
      d_total = d_total.defined() ? at::addmm(d_total, grads[1], s[2]) : at::mm(grads[1], s[2]);
    }
    if (!d_total.defined()) return out;
    auto [d_x, none, d_weight] = rmsnorm_backward(s[0], s[1], s[3], d_total, Tensor(), ctx->saved_data["eps"].toDouble(), 1.0, false, false);
    out[0] = d_x;
    out[1] = d_weight;
    return out;
  }
};
// x [B, H]: (y, logits, x8, scale8)
std::tuple<Tensor, Tensor, OptTensor, OptTensor> norm_route(const Tensor& x, const OptTensor& norm_weight, const Tensor& gate_weight, double eps,
                                                            bool quantize, bool few_rows) {
  const Tensor nw = value_or_undefined(norm_weight);
  require_gpu(x, nw, gate_weight);
  if (any_requires_grad({&x, &nw, &gate_weight})) {
    auto out = NormRouteFn::apply(x, norm_weight, gate_weight, eps, few_rows);
    OptTensor x8, scale8;
    if (quantize) std::tie(x8, scale8) = quantize_rows(out[0].detach());
    return {out[0], out[1], x8, scale8};
  }
  NormRoute r = norm_route_forward(x.contiguous(), contiguous(nw), gate_weight.contiguous(), eps, quantize, false, few_rows);
  return {r.y, r.logits, to_opt(r.x8), to_opt(r.scale8)};
}

// ---- softmax ----------------------------------------------------------------------------------------------------
Tensor softmax_forward(const Tensor& x, double multiplier) {
  const Launch l(x);
  const int64_t H = x.size(-1);
  const Tensor out = like_contiguous(x);
  check(api.ck_softmax_fwd(ptr(x), (float)multiplier, row_count(x), (int32_t)H, ptr(out), dtype_code(x), l.stream));
  return out;
}
Tensor softmax_backward(const Tensor& y, const Tensor& grad_in, double multiplier) {
  const Tensor grad = grad_in.contiguous(), d_x = like_contiguous(y);
  const Launch l(y);
  const int64_t H = y.size(-1);
  check(api.ck_softmax_bwd(ptr(y), ptr(grad), (float)multiplier, row_count(y), (int32_t)H, ptr(d_x), dtype_code(y), l.stream));
  return d_x;
}
struct Softmax : torch::autograd::Function<Softmax> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, double multiplier) {
    const Tensor out = softmax_forward(x.contiguous(), multiplier);
    ctx->save_for_backward({out});
    ctx->saved_data["multiplier"] = multiplier;
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return {Tensor(), Tensor()};
    return {softmax_backward(ctx->get_saved_variables()[0], grads[0], ctx->saved_data["multiplier"].toDouble()), Tensor()};
  }
};
Tensor softmax(const Tensor& x, double multiplier) {
  require_gpu(x);
  if (any_requires_grad({&x})) return Softmax::apply(x, multiplier);
  return softmax_forward(x.contiguous(), multiplier);
}

}  // namespace

PYBIND11_MODULE(_ck_host, m) {
  py::class_<GateSlot, SlotPtr>(m, "GateSlot")
      .def(py::init([] { return c10::make_intrusive<GateSlot>(); }))
      .def_property(
          "d_gates_f32", [](const GateSlot& s) { return to_opt(s.d_gates_f32); },
          [](GateSlot& s, const OptTensor& t) { s.d_gates_f32 = value_or_undefined(t); })
      // gates are copied and saved with their attributes; what is in a slot belongs to one backward pass: a copy is empty
      .def("__reduce__", [](const py::object& s) { return py::make_tuple(py::type::of(s), py::tuple()); })
      .attr("__module__") = "cute_kernels._ck_host";
#define DEF(name, fn) m.def(name, torch::wrap_pybind_function(fn))
  DEF("init", init);
  m.def("set_launch_timer", set_launch_timer);
  // for tests: a launch as the autograd engine's threads make it, without the interpreter lock
  m.def("timed_without_lock", [](const std::string& name, int64_t a, int64_t b, const py::function& launch) {
    const py::gil_scoped_release release;
    timed(name.c_str(), a, b, [&] {
      const py::gil_scoped_acquire gil;
      launch();
    });
  });
  DEF("count", count);
  DEF("sort_by_expert", sort_by_expert);
  DEF("route", route);
  DEF("swiglu_experts", swiglu_experts);
  DEF("experts_up", experts_up);
  DEF("experts_down", experts_down);
  DEF("gelu_experts", gelu_experts);
  DEF("quantize_rows", ([](const Tensor& x) { return quantize_rows(x); }));
  DEF("swiglu_experts_e4m3", swiglu_experts_e4m3);
  DEF("swiglu", swiglu);
  DEF("swiglu_packed", swiglu_packed);
  DEF("rmsnorm", rmsnorm);
  DEF("residual_rmsnorm", residual_rmsnorm);
  DEF("norm_route", norm_route);
  DEF("router_rows_take", router_rows_take);
  DEF("router_rows", router_rows);
  DEF("softmax", softmax);
  // without autograd, for the traced operators and the kernel tests
  DEF("route_forward", ([](const Tensor& logits, int64_t k) {
        auto [gates, out, sel, sel_long] = route_forward(logits, k, true, true, false);
        return std::make_tuple(gates, sel);
      }));
  DEF("route_backward", ([](const Tensor& gates, const Tensor& selected, const Tensor& d_gates, int64_t E, const Tensor& like) {
        return route_backward(gates, selected, d_gates, Tensor(), E, like.scalar_type());
      }));
  DEF("swiglu_forward", ([](const Tensor& gate, const Tensor& up) { return require_gpu(gate, up), swiglu_forward(gate.contiguous(), up.contiguous()); }));
  DEF("swiglu_backward", ([](const Tensor& gate, const Tensor& up, const Tensor& grad) { return swiglu_backward(gate.contiguous(), up.contiguous(), grad); }));
  DEF("swiglu_packed_forward", ([](const Tensor& x) { return require_gpu(x), swiglu_packed_forward(x.contiguous()); }));
  DEF("swiglu_packed_backward", ([](const Tensor& x, const Tensor& grad) { return swiglu_packed_backward(x.contiguous(), grad); }));
  DEF("rmsnorm_forward", ([](const Tensor& x, const OptTensor& w, double eps, bool want_rstd) {
        require_gpu(x, value_or_undefined(w));
        auto [y, rstd] = rmsnorm_forward(x.contiguous(), contiguous(value_or_undefined(w)), eps, want_rstd);
        return std::make_tuple(y, to_opt(rstd));
      }));
  DEF("residual_rmsnorm_forward", ([](const Tensor& x, const Tensor& residual, const OptTensor& w, double eps, double multiplier, bool want_rstd) {
        require_gpu(x, residual, value_or_undefined(w));
        auto [y, added, rstd] = residual_rmsnorm_forward(x.contiguous(), residual.contiguous(), contiguous(value_or_undefined(w)), eps, multiplier, want_rstd);
        return std::make_tuple(y, added, to_opt(rstd));
      }));
  DEF("rmsnorm_backward", ([](const Tensor& x, const OptTensor& w, const OptTensor& rstd, const Tensor& d_out, const OptTensor& d_added, double eps,
                              double multiplier, bool residual) {
        auto [d_x, d_residual, d_w] = rmsnorm_backward(x.contiguous(), contiguous(value_or_undefined(w)), value_or_undefined(rstd), d_out,
                                                       value_or_undefined(d_added), eps, multiplier, residual, false);
        return std::make_tuple(d_x, to_opt(d_residual), to_opt(d_w));
      }));
  DEF("softmax_forward", ([](const Tensor& x, double multiplier) { return require_gpu(x), softmax_forward(x.contiguous(), multiplier); }));
  DEF("softmax_backward", ([](const Tensor& y, const Tensor& grad, double multiplier) { return softmax_backward(y.contiguous(), grad, multiplier); }));
  DEF("swiglu_experts_forward", ([](const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates, py::object seg, int64_t act_kind,
                                    bool keep_pre, bool keep_act, int64_t flags) {
        Block b = swiglu_experts_forward(x.contiguous(), w_fc.contiguous(), w_proj.contiguous(), gates.contiguous(), Segments::of(seg), act_kind,
                                         keep_pre, keep_act, flags);
        return std::make_tuple(b.out, to_opt(b.pre), to_opt(b.act_t.defined() ? b.act_t : keep_act ? b.act : Tensor()), b.expanded);
      }));
  DEF("swiglu_experts_backward", ([](const Tensor& grad, const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, const Tensor& gates, const Tensor& pre,
                                     const OptTensor& act, const Tensor& expanded, py::object seg, int64_t act_kind, bool need_x, bool need_fc,
                                     bool need_proj, bool need_gates, int64_t flags) {
        BlockGrads g = swiglu_experts_backward(grad, x.contiguous(), w_fc.contiguous(), w_proj.contiguous(), gates.contiguous(), pre, value_or_undefined(act),
                                               expanded, Segments::of(seg), act_kind, need_x, need_fc, need_proj, need_gates, nullptr, flags);
        return std::make_tuple(to_opt(g.d_x), to_opt(g.d_w_fc), to_opt(g.d_w_proj), to_opt(g.d_gates));
      }));
  DEF("experts_up_forward", ([](const Tensor& x, const Tensor& w, const OptTensor& bias, py::object seg, int64_t k, bool gelu, int64_t flags) {
        auto [y, act] = experts_up_forward(x.contiguous(), w.contiguous(), Segments::of(seg), k, contiguous(value_or_undefined(bias)), gelu, true, true, flags);
        return std::make_tuple(y, to_opt(act));
      }));
  DEF("experts_up_backward", ([](const Tensor& d_y, const Tensor& x, const Tensor& w, const OptTensor& pre, py::object seg, int64_t k, bool need_x,
                                 bool need_w, bool need_bias, int64_t flags) {
        LinearGrads g = experts_up_backward(d_y, x.contiguous(), w.contiguous(), value_or_undefined(pre), Segments::of(seg), k, need_x, need_w, need_bias, flags);
        return std::make_tuple(to_opt(g.d_in), to_opt(g.d_w), to_opt(g.d_bias));
      }));
  DEF("experts_down_forward", ([](const Tensor& h, const Tensor& w, const Tensor& gates, const OptTensor& bias, const OptTensor& slot_expert, py::object seg,
                                  int64_t flags) {
        return experts_down_forward(h.contiguous(), w.contiguous(), gates.contiguous(), Segments::of(seg), contiguous(value_or_undefined(bias)),
                                    value_or_undefined(slot_expert), flags);
      }));
  DEF("experts_down_backward", ([](const Tensor& grad, const Tensor& h, const Tensor& w, const Tensor& gates, const Tensor& expanded, py::object seg,
                                   bool need_h, bool need_w, bool need_gates, bool need_bias, int64_t flags) {
        LinearGrads g = experts_down_backward(grad, h.contiguous(), w.contiguous(), gates.contiguous(), expanded, Segments::of(seg), need_h, need_w,
                                              need_gates, need_bias, true, nullptr, flags);
        return std::make_tuple(to_opt(g.d_in), to_opt(g.d_w), to_opt(g.d_gates), to_opt(g.d_bias));
      }));
  // single launches
  DEF("gemm", ([](const Tensor& a, int64_t gather_div, const Tensor& w, py::object seg, int64_t epilogue, const OptTensor& y, const OptTensor& y_t,
                  const OptTensor& aux, const OptTensor& aux_in, const OptTensor& rows_in, const OptTensor& rows_out, int64_t flags) {
        gemm(a, gather_div, w, Segments::of(seg), epilogue, value_or_undefined(y), value_or_undefined(y_t), value_or_undefined(aux),
             value_or_undefined(aux_in), value_or_undefined(rows_in), value_or_undefined(rows_out), flags);
      }));
  DEF("gemm_f32", ([](const Tensor& a, int64_t gather_div, const Tensor& w, bool w_is_kn, int64_t N, int64_t K, py::object seg, bool scatter,
                      const Tensor& y, const OptTensor& bias, const OptTensor& rows_in, const OptTensor& rows_out) {
        gemm_f32(a, gather_div, w, w_is_kn, N, K, Segments::of(seg), scatter, y, value_or_undefined(bias), value_or_undefined(rows_in), value_or_undefined(rows_out));
      }));
  DEF("gemm_dx", ([](const Tensor& d_y, const Tensor& w, py::object seg, int64_t epilogue, const Tensor& out, const OptTensor& rows_out, int64_t flags) {
        gemm_dx(d_y, w, Segments::of(seg), epilogue, out, value_or_undefined(rows_out), flags);
      }));
  DEF("gemm_dw", ([](const Tensor& a_t, const Tensor& b_t, py::object seg, const Tensor& dw) { gemm_dw(a_t, b_t, Segments::of(seg), dw); }));
  DEF("gemm_dw_rows", ([](const Tensor& a, const Tensor& b, py::object seg, const Tensor& dw) { gemm_dw_rows(a, b, Segments::of(seg), dw); }));
  DEF("gemm_fp8", ([](const Tensor& a8, const Tensor& a_scale, int64_t gather_div, const Tensor& w8, const Tensor& w_scale, py::object seg, int64_t epilogue,
                      const OptTensor& y, const OptTensor& aux, const Tensor& like) {
        gemm_fp8(a8, a_scale, gather_div, w8, w_scale, Segments::of(seg), epilogue, value_or_undefined(y), value_or_undefined(aux), like.scalar_type());
      }));
  m.def("dw_from_rows", dw_from_rows);
  DEF("transpose_weights", transpose_weights);
  DEF("group_rows", ([](const Tensor& src, const OptTensor& coeff, int64_t fan_out, py::object seg, bool want_grouped, bool want_transposed,
                        const OptTensor& rows) {
        auto [a, b] = group_rows(src, value_or_undefined(coeff), fan_out, Segments::of(seg), want_grouped, want_transposed, value_or_undefined(rows));
        return std::make_tuple(to_opt(a), to_opt(b));
      }));
  DEF("gate_grad", ([](const Tensor& expanded, const Tensor& grad_out, int64_t T, int64_t k, int64_t H, std::optional<SlotPtr> slot) {
        return gate_grad(expanded, grad_out, T, k, H, slot.has_value() ? slot->get() : nullptr);
      }));
  DEF("add_expert_bias", ([](const Tensor& y, const Tensor& bias, py::object seg, const OptTensor& row_expert) {
        add_expert_bias(y, bias, Segments::of(seg), value_or_undefined(row_expert));
      }));
  DEF("expert_bias_grad", ([](const Tensor& d_y, py::object seg) { return expert_bias_grad(d_y, Segments::of(seg)); }));
  DEF("slot_experts", slot_experts);
  DEF("split_workspace", ([](const Tensor& like) { return split_workspace(like, Launch(like).stream); }));
}
