// The autograd nodes of the plain path and the segment build in C++: the same calls of the library in the same order as the
// classes of ops.py, without the interpreter.  What bounds a small or middle-sized pass is the host: a forward and backward
// of one projection with 16 adapters took 215 us of it, 155 in the backward (33 gradients through Python objects, on a thread
// that waits for the interpreter), next to 210 us of kernels for 16384 rows.
//
// Every function returns None for a call that is anything but plain (another device or dtype, a shape that does not fit,
// tensor subclasses, transforms, tracing): the caller then takes the Python path, which has the checks and their messages.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <mutex>
#include <vector>

#include "twinkle_amd.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

// (the exception types of _lib.check)
void check(int64_t code, const char* what) {
  if (code >= 0) return;
  if (code == TK_ERR_INVALID || code == TK_ERR_UNSUPPORTED)
    TORCH_CHECK_VALUE(false, what, ": ", tk_error_string((int)code), " (", code, ")");
  TORCH_CHECK(false, what, ": ", tk_error_string((int)code), " (", code, ")");
}
tk_stream_t stream() { return (tk_stream_t)c10::hip::getCurrentHIPStream().stream(); }

Tensor bytes_of(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

using c10::DispatchKey;
const c10::DispatchKeySet kUnusual({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Conjugate,
                                    DispatchKey::Negative, DispatchKey::ZeroTensor, DispatchKey::Functionalize,
                                    DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                    DispatchKey::Batched});
// nothing but autograd between a call and the kernels
bool plain_mode() {
  static const c10::DispatchKeySet modes({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::PythonDispatcher,
                                          DispatchKey::Functionalize, DispatchKey::FuncTorchDynamicLayerFrontMode,
                                          DispatchKey::FuncTorchDynamicLayerBackMode, DispatchKey::VmapMode});
  return !c10::impl::tls_local_dispatch_key_set().included_.has_any(modes) && !torch::jit::tracer::isTracing() &&
         !at::impl::torch_function_mode_enabled();
}
bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kUnusual);
}
bool plain_rows(const Tensor& t, int64_t rows, int64_t width, at::ScalarType dtype) {
  return plain(t) && t.dim() == 2 && t.size(0) == rows && t.size(1) == width && t.stride(1) == 1 && t.scalar_type() == dtype;
}

// A tensor as Python holds it; undefined for a subclass, also one without a dispatch key of its own (__torch_function__ only),
// and for what is no tensor at all.
Tensor exact(py::handle h) { return THPVariable_CheckExact(h.ptr()) ? THPVariable_Unpack(h.ptr()) : Tensor(); }

// One side (lora_A or lora_B) of an AdapterGroups object.
struct Side {
  std::vector<Tensor> tensors;
  std::vector<int64_t> index, offset;   // of every group: its tensor, elements into it
  std::vector<bool> live;               // of every tensor: a group of positive rank reads it
  std::vector<int64_t> at;              // of every tensor: elements into the gradients' buffer
  int64_t elems = 0;                    // of that buffer
  Tensor grads_at;                      // device: bytes into it, per group
  Tensor pointers;                      // device: the groups' matrices
  std::vector<const void*> known;       // where the tensors were when `pointers` was made

  bool moved() const {
    for (size_t i = 0; i < tensors.size(); ++i)
      if (tensors[i].const_data_ptr() != known[i]) return true;
    return false;
  }
  void look() {
    known.resize(tensors.size());
    for (size_t i = 0; i < tensors.size(); ++i) known[i] = tensors[i].const_data_ptr();
  }
  void refresh() {
    look();
    const int64_t elt = tensors[0].element_size();
    Tensor host = at::empty({(int64_t)index.size()}, at::kLong);
    for (size_t g = 0; g < index.size(); ++g)
      host.data_ptr<int64_t>()[g] = (int64_t)known[index[g]] + offset[g] * elt;
    pointers = host.to(tensors[0].device());
  }
  // the gradients: tensors of their own that share the buffer's storage
  void views(const Tensor& buffer, variable_list& out) const {
    for (size_t i = 0; i < tensors.size(); ++i) {
      if (!live[i]) {
        out.emplace_back();
        continue;
      }
      auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(buffer.storage()), buffer.key_set(), buffer.dtype());
      impl->set_sizes_and_strides(tensors[i].sizes(), tensors[i].strides(), at[i]);
      out.emplace_back(std::move(impl));
    }
  }
};

struct Groups {
  Side a, b;
  Tensor rank, scale;
  tk_lora_desc base{};
  at::ScalarType dtype, weight_dtype;
  bool zeros = false;  // the gradients' buffers have to start at zero
  std::mutex mutex;

  // The description of a call; `keep` holds the pointer tables it refers to (another thread may replace them).
  tk_lora_desc desc(int64_t rows, bool map_rows, const Tensor& seg, Tensor (&keep)[2]) {
    std::lock_guard<std::mutex> guard(mutex);
    if (a.moved()) a.refresh();
    if (b.moved()) b.refresh();
    keep[0] = a.pointers;
    keep[1] = b.pointers;
    tk_lora_desc d = base;
    d.rows = rows;
    d.map_rows = map_rows;
    d.seg_ws = seg.const_data_ptr();
    d.lora_A = (const void* const*)a.pointers.const_data_ptr();
    d.lora_B = (const void* const*)b.pointers.const_data_ptr();
    return d;
  }
  Tensor buffer(const Side& side, int64_t rows) const {
    const auto options = rank.options().dtype(weight_dtype);
    return zeros || rows == 0 ? at::zeros({side.elems}, options) : at::empty({side.elems}, options);
  }
  // with fp32 adapters under bf16 activations the forward's weight copies at the end of h need not live until the backward
  Tensor h_for_backward(const Tensor& h, tk_lora_desc d) const {
    if (!d.weights_f32) return h;
    d.weights_f32 = 0;
    return h.narrow(0, 0, tk_lora_h_bytes(&d)).clone();
  }
};
using GroupsPtr = std::shared_ptr<Groups>;

std::shared_ptr<Groups> make_groups(const py::dict& v) {
  auto g = std::make_shared<Groups>();
  auto side = [&](const char* s, Side& o) {
    const std::string p = std::string(s) + "_";
    auto get = [&](const char* name) { return v[(p + name).c_str()]; };
    o.tensors = get("tensors").cast<std::vector<Tensor>>();
    o.index = get("index").cast<std::vector<int64_t>>();
    o.offset = get("offset").cast<std::vector<int64_t>>();
    o.live = get("live").cast<std::vector<bool>>();
    o.at = get("at").cast<std::vector<int64_t>>();
    o.elems = get("elems").cast<int64_t>();
    o.grads_at = get("grads_at").cast<Tensor>();
    o.pointers = get("pointers").cast<Tensor>();
    o.look();
  };
  side("a", g->a);
  side("b", g->b);
  g->rank = v["rank"].cast<Tensor>();
  g->scale = v["scale"].cast<Tensor>();
  g->weight_dtype = g->a.tensors[0].scalar_type();
  tk_lora_desc& d = g->base;
  d.in_features = v["in_features"].cast<int>();
  d.out_features = v["out_features"].cast<int>();
  d.num_groups = (int32_t)g->a.index.size();
  d.max_rank = v["max_rank"].cast<int>();
  d.dtype = v["dtype"].cast<int>();
  d.lda = v["lda"].cast<int64_t>();
  d.ldb = v["ldb"].cast<int64_t>();
  d.rank = (const int32_t*)g->rank.const_data_ptr();
  d.scale = (const float*)g->scale.const_data_ptr();
  d.weights_f32 = v["weights_f32"].cast<int>();
  d.rank_classes = v["rank_classes"].cast<int>();
  g->dtype = d.dtype == TK_DTYPE_BF16 ? at::kBFloat16 : at::kFloat;
  return g;
}

// What a node keeps of its call besides tensors.
struct Call : torch::CustomClassHolder {
  Tensor seg;
  int64_t rows = 0;
  bool map_rows = true;
  std::vector<GroupsPtr> groups;
  std::vector<bool> has_bias;
};
using CallPtr = c10::intrusive_ptr<Call>;
CallPtr call_of(AutogradContext* ctx) {
  return c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
}

bool any_grad(AutogradContext* ctx, size_t from, size_t n) {
  for (size_t i = 0; i < n; ++i)
    if (ctx->needs_input_grad(from + i)) return true;
  return false;
}

// Backward of one projection's LoRA term: dx (written when store_dx, else added onto; undefined: not wanted) and the weight
// gradients, appended to `out` in the order of the adapters (undefined where not wanted).
void lora_backward(Call& call, Groups& g, const Tensor& dy, const Tensor& x, const Tensor& h, const Tensor& dx, bool store_dx,
                   bool needs_a, bool needs_b, variable_list& out) {
  Tensor keep[2], da, db;
  const tk_lora_desc d = g.desc(call.rows, call.map_rows, call.seg, keep);
  if (needs_a && g.a.elems) da = g.buffer(g.a, call.rows);
  if (needs_b && g.b.elems) db = g.buffer(g.b, call.rows);
  const int64_t n = tk_lora_bwd_workspace_bytes(&d);
  check(n, "tk_lora_bwd_workspace_bytes");
  const Tensor ws = bytes_of(n, dy);
  check(tk_lora_bwd_into(&d, dy.const_data_ptr(), dy.stride(0), x.const_data_ptr(), x.stride(0), h.const_data_ptr(),
                         dx.defined() ? dx.mutable_data_ptr() : nullptr, dx.defined() ? dx.stride(0) : 0, store_dx,
                         da.defined() ? g.a.grads_at.const_data_ptr<int64_t>() : nullptr,
                         da.defined() ? da.mutable_data_ptr() : nullptr,
                         db.defined() ? g.b.grads_at.const_data_ptr<int64_t>() : nullptr,
                         db.defined() ? db.mutable_data_ptr() : nullptr, ws.mutable_data_ptr(), n, stream()),
        "tk_lora_bwd_into");
  if (da.defined()) g.a.views(da, out);
  else out.resize(out.size() + g.a.tensors.size());
  if (db.defined()) g.b.views(db, out);
  else out.resize(out.size() + g.b.tensors.size());
}

Tensor lora_forward(Call& call, Groups& g, const Tensor& x, const Tensor& y, bool keep_h) {
  Tensor keep[2];
  const tk_lora_desc d = g.desc(call.rows, call.map_rows, call.seg, keep);
  const int64_t n = tk_lora_h_bytes(&d);
  check(n, "tk_lora_h_bytes");
  const Tensor h = bytes_of(n, x);
  check(tk_lora_fwd(&d, x.const_data_ptr(), x.stride(0), y.mutable_data_ptr(), y.stride(0), h.mutable_data_ptr(), stream()),
        "tk_lora_fwd");
  return keep_h ? g.h_for_backward(h, d) : Tensor();
}

// ops.py::_LoraDelta
struct LoraDelta : torch::autograd::Function<LoraDelta> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const CallPtr& call, at::TensorList weights) {
    const Tensor h = lora_forward(*call, *call->groups[0], x, y, true);
    ctx->mark_dirty({y});
    ctx->save_for_backward({x, h});
    ctx->saved_data["call"] = c10::IValue::make_capsule(call);
    return y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &h = saved[1];
    const CallPtr call = call_of(ctx);
    Groups& g = *call->groups[0];
    const size_t na = g.a.tensors.size(), nb = g.b.tensors.size();
    const Tensor dy = grads[0].contiguous();
    const Tensor dx = ctx->needs_input_grad(0) ? at::empty_like(x) : Tensor();
    variable_list out{dx, dy, Tensor()};
    lora_backward(*call, g, dy, x, h, dx, true, any_grad(ctx, 2, na), any_grad(ctx, 2 + na, nb), out);
    return out;
  }
};

// ops.py::_LoraLinear (one projection) and _LoraLinearShared: inputs = x, the weights, the biases there are, the adapters
struct LoraLinear : torch::autograd::Function<LoraLinear> {
  static variable_list forward(AutogradContext* ctx, const CallPtr& call, at::TensorList inputs) {
    const size_t n = call->groups.size();
    const Tensor& x = inputs[0];
    variable_list ys, saved{x};
    for (size_t p = 0, bias = 1 + n; p < n; ++p) {
      ys.push_back(at::linear(x, inputs[1 + p], call->has_bias[p] ? std::optional<Tensor>(inputs[bias]) : std::nullopt));
      bias += call->has_bias[p];
      saved.push_back(inputs[1 + p]);
    }
    if (n == 1) {
      saved.push_back(lora_forward(*call, *call->groups[0], x, ys[0], true));
    } else {
      std::vector<tk_lora_desc> d(n);
      std::vector<const tk_lora_desc*> dp(n);
      std::vector<Tensor> keep(2 * n), hs(n);
      std::vector<void*> y(n), h(n);
      std::vector<int64_t> ldy(n);
      for (size_t p = 0; p < n; ++p) {
        Tensor k[2];
        d[p] = call->groups[p]->desc(call->rows, call->map_rows, call->seg, k);
        keep[2 * p] = k[0];
        keep[2 * p + 1] = k[1];
        const int64_t bytes = tk_lora_h_bytes(&d[p]);
        check(bytes, "tk_lora_h_bytes");
        hs[p] = bytes_of(bytes, x);
        dp[p] = &d[p];
        y[p] = ys[p].mutable_data_ptr();
        ldy[p] = ys[p].stride(0);
        h[p] = hs[p].mutable_data_ptr();
      }
      check(tk_lora_fwd_shared(dp.data(), (int32_t)n, x.const_data_ptr(), x.stride(0), y.data(), ldy.data(), h.data(), stream()),
            "tk_lora_fwd_shared");
      for (const Tensor& t : hs) saved.push_back(t);
    }
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["call"] = c10::IValue::make_capsule(call);
    return ys;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const CallPtr call = call_of(ctx);
    const size_t n = call->groups.size();
    const auto saved = ctx->get_saved_variables();
    const Tensor& x = saved[0];
    variable_list dy(n), out(2);  // (the call itself, then the inputs)
    for (size_t p = 0; p < n; ++p)
      dy[p] = grads[p].defined() ? grads[p].contiguous()
                                 : at::zeros({call->rows, call->groups[p]->base.out_features}, x.options());
    const bool needs_dx = ctx->needs_input_grad(0);
    if (needs_dx || n > 1) {
      out[1] = at::mm(dy[0], saved[1]);
      for (size_t p = 1; p < n; ++p) out[1].addmm_(dy[p], saved[1 + p]);
    }
    size_t edge = 1;  // input the next gradient belongs to
    for (size_t p = 0; p < n; ++p, ++edge) out.push_back(ctx->needs_input_grad(edge) ? at::mm(dy[p].t(), x) : Tensor());
    for (size_t p = 0; p < n; ++p) {
      if (!call->has_bias[p]) continue;
      out.push_back(ctx->needs_input_grad(edge) ? dy[p].sum(0) : Tensor());
      ++edge;
    }
    if (n == 1) {
      Groups& g = *call->groups[0];
      const size_t na = g.a.tensors.size(), nb = g.b.tensors.size();
      lora_backward(*call, g, dy[0], x, saved[2], out[1], false, any_grad(ctx, edge, na), any_grad(ctx, edge + na, nb), out);
      return out;
    }
    std::vector<tk_lora_desc> d(n);
    std::vector<const tk_lora_desc*> dp(n);
    std::vector<Tensor> keep(2 * n), ws(n), buffers(2 * n);
    std::vector<const void*> dyp(n), hp(n);
    std::vector<int64_t> lddy(n), bytes(n);
    std::vector<const int64_t*> at_a(n), at_b(n);
    std::vector<void*> base_a(n), base_b(n), wsp(n);
    for (size_t p = 0; p < n; ++p) {
      Groups& g = *call->groups[p];
      Tensor k[2];
      d[p] = g.desc(call->rows, call->map_rows, call->seg, k);
      keep[2 * p] = k[0];
      keep[2 * p + 1] = k[1];
      dp[p] = &d[p];
      bytes[p] = tk_lora_bwd_workspace_bytes(&d[p]);
      check(bytes[p], "tk_lora_bwd_workspace_bytes");
      ws[p] = bytes_of(bytes[p], x);
      buffers[2 * p] = g.buffer(g.a, call->rows);
      buffers[2 * p + 1] = g.buffer(g.b, call->rows);
      dyp[p] = dy[p].const_data_ptr();
      lddy[p] = dy[p].stride(0);
      hp[p] = saved[1 + n + p].const_data_ptr();
      at_a[p] = g.a.grads_at.const_data_ptr<int64_t>();
      at_b[p] = g.b.grads_at.const_data_ptr<int64_t>();
      base_a[p] = buffers[2 * p].mutable_data_ptr();
      base_b[p] = buffers[2 * p + 1].mutable_data_ptr();
      wsp[p] = ws[p].mutable_data_ptr();
    }
    check(tk_lora_bwd_shared_into(dp.data(), (int32_t)n, dyp.data(), lddy.data(), x.const_data_ptr(), x.stride(0), hp.data(),
                                  out[1].mutable_data_ptr(), out[1].stride(0), at_a.data(), base_a.data(), at_b.data(),
                                  base_b.data(), wsp.data(), bytes.data(), stream()),
          "tk_lora_bwd_shared_into");
    if (!needs_dx) out[1] = Tensor();
    for (size_t p = 0; p < n; ++p) {
      call->groups[p]->a.views(buffers[2 * p], out);
      call->groups[p]->b.views(buffers[2 * p + 1], out);
    }
    return out;
  }
};

CallPtr make_call(const Tensor& seg, int64_t rows, bool map_rows) {
  auto call = c10::make_intrusive<Call>();
  call->seg = seg;
  call->rows = rows;
  call->map_rows = map_rows;
  return call;
}
bool plain_weights(const Groups& g) {
  for (const Side* s : {&g.a, &g.b})
    for (const Tensor& t : s->tensors)
      if (!plain(t)) return false;
  return true;
}
bool wants_grad(const Groups& g) {
  for (const Side* s : {&g.a, &g.b})
    for (const Tensor& t : s->tensors)
      if (t.requires_grad()) return true;
  return false;
}

// ops.py::multi_lora_delta
std::optional<Tensor> delta(py::handle x_, py::handle y_, const Tensor& seg, int64_t rows, int64_t num_groups,
                            const GroupsPtr& g, bool map_rows) {
  const Tensor x = exact(x_), y = exact(y_);
  // (an inference tensor is not updated outside of that mode: the Python node says so)
  if (y.defined() && y.is_inference() && !c10::InferenceMode::is_enabled()) return std::nullopt;
  if (!plain_mode() || num_groups != g->base.num_groups || !plain(seg) ||
      !plain_rows(x, rows, g->base.in_features, g->dtype) || !plain_rows(y, rows, g->base.out_features, g->dtype) ||
      !plain_weights(*g))
    return std::nullopt;
  py::gil_scoped_release release;
  const CallPtr call = make_call(seg, rows, map_rows);
  call->groups = {g};
  if (!at::GradMode::is_enabled() || !(x.requires_grad() || y.requires_grad() || wants_grad(*g))) {
    lora_forward(*call, *g, x, y, false);
    if (!y.is_inference()) y.unsafeGetTensorImpl()->bump_version();
    return y;
  }
  variable_list weights(g->a.tensors);
  weights.insert(weights.end(), g->b.tensors.begin(), g->b.tensors.end());
  return LoraDelta::apply(x, y, call, at::TensorList(weights));
}

// ops.py::multi_lora_linear (one projection) and multi_lora_linear_shared
std::optional<variable_list> linear(py::handle x_, const std::vector<py::object>& weights, const std::vector<py::object>& biases,
                                    const Tensor& seg, int64_t rows, int64_t num_groups, const std::vector<GroupsPtr>& groups,
                                    bool map_rows) {
  const size_t n = groups.size();
  const Tensor x = exact(x_);
  // (autocast, which lifts its key from the excluded ones, would run the base GEMM in a type of its own)
  if (!c10::impl::tls_local_dispatch_key_set().excluded_.has(DispatchKey::AutocastCUDA)) return std::nullopt;
  if (!plain_mode() || n < 1 || n > TK_MAX_SHARED || weights.size() != n || biases.size() != n || !plain(x) || !plain(seg) ||
      !at::GradMode::is_enabled())
    return std::nullopt;
  variable_list inputs{x};
  const CallPtr call = make_call(seg, rows, map_rows);
  bool grad = x.requires_grad();
  variable_list given;  // the biases there are
  for (size_t p = 0; p < n; ++p) {
    const Groups& g = *groups[p];
    const Tensor weight = exact(weights[p]);
    if (num_groups != g.base.num_groups || !plain_rows(x, rows, g.base.in_features, g.dtype) ||
        !plain_rows(weight, g.base.out_features, g.base.in_features, g.dtype) || !plain_weights(g) ||
        (n > 1 && (g.a.elems == 0 || g.b.elems == 0)))
      return std::nullopt;
    inputs.push_back(weight);
    grad = grad || weight.requires_grad() || wants_grad(g);
    call->has_bias.push_back(!biases[p].is_none());
    if (biases[p].is_none()) continue;
    const Tensor bias = exact(biases[p]);
    if (!(plain(bias) && bias.dim() == 1 && bias.size(0) == g.base.out_features && bias.scalar_type() == g.dtype))
      return std::nullopt;
    given.push_back(bias);
    grad = grad || bias.requires_grad();
  }
  if (!grad) return std::nullopt;
  inputs.insert(inputs.end(), given.begin(), given.end());
  for (size_t p = 0; p < n; ++p)
    for (const Side* s : {&groups[p]->a, &groups[p]->b}) inputs.insert(inputs.end(), s->tensors.begin(), s->tensors.end());
  call->groups = groups;
  py::gil_scoped_release release;
  return LoraLinear::apply(call, at::TensorList(inputs));
}

// segments.py::build_segments: workspace, permutation, offsets
std::optional<std::tuple<Tensor, std::optional<Tensor>, std::optional<Tensor>>> segment_build(py::handle keys_, int64_t num_groups,
                                                                                               bool want_perm,
                                                                                               bool want_offsets) {
  const Tensor keys = exact(keys_);
  if (!plain_mode() || !plain(keys)) return std::nullopt;
  const bool i32 = keys.scalar_type() == at::kInt;
  if (!(i32 || keys.scalar_type() == at::kLong) || !keys.is_contiguous() || num_groups <= 0 ||
      num_groups > TK_MAX_GROUPS)
    return std::nullopt;
  const int64_t rows = keys.numel(), n = tk_segment_workspace_bytes(rows, (int32_t)num_groups);
  if (n < 0) return std::nullopt;
  const Tensor ws = bytes_of(n, keys);
  std::optional<Tensor> perm, offsets;
  if (want_perm) perm = at::empty({rows}, keys.options().dtype(at::kLong));
  if (want_offsets) offsets = at::empty({num_groups + 1}, keys.options().dtype(at::kLong));
  check(tk_segment_build(rows ? keys.const_data_ptr() : nullptr, i32 ? TK_KEY_I32 : TK_KEY_I64, rows, (int32_t)num_groups,
                         perm ? perm->data_ptr<int64_t>() : nullptr, offsets ? offsets->data_ptr<int64_t>() : nullptr,
                         ws.mutable_data_ptr(), n, stream()),
        "tk_segment_build");
  return std::make_tuple(ws, perm, offsets);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  py::class_<Groups, GroupsPtr>(m, "Groups").def_readwrite("zeros", &Groups::zeros);
  m.def("plain_mode", &plain_mode);
  m.def("make_groups", &make_groups);
  m.def("delta", &delta);
  m.def("linear", &linear);
  m.def("segment_build", &segment_build);
}
