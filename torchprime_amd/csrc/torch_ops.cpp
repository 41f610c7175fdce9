// The ``tprime`` operators: registration with torch's dispatcher, autograd nodes and the Python entry points, over the
// C ABI of libtprime_hip.so.
//
// Why this file is native: a pass over a small problem is nothing but host work.  With the operators defined in Python
// (torch.library.custom_op around ctypes calls) one operator cost 25-45 us of host time forward and 50-80 us with its
// backward, five to ten times what its kernel runs for at small sizes, and the gradients of outputs nobody uses (the
// LSE, the 1 / rms) were zero-filled tensors, one more launch each.  Here an operator is one allocation per output, one
// launch and one autograd node.
//
// What an operator is made of:
//   *_cuda      checks, output allocation, the launch (registered for the CUDA key)
//   *_autograd  saves what the backward needs in a node and redispatches below autograd (registered for the Autograd
//               key).  The nodes call the backward operators through the dispatcher as well, so traces (fake tensors,
//               AOT autograd) see tprime::*_bwd.
// The backward operators have no derivative of their own: differentiating through one raises.
#include <torch/extension.h>
#include <torch/library.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <tuple>
#include <unordered_map>

#include "../../include/tprime_hip.h"

namespace {

using at::Tensor;
using c10::optional;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
typedef const std::optional<Tensor>& OptTensor;
typedef std::array<int64_t, 3> Strides3;

// ---- helpers ---------------------------------------------------------------------------------------------------
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return TP_BF16;
    case at::kHalf: return TP_F16;
    case at::kFloat: return TP_F32;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t, "; supported: bfloat16, float16, float32");
  }
}

// status of a C ABI call -> the exception the Python binding (_lib.call) raises for it
void check(int rc, const char* name) {
  if (C10_LIKELY(rc == TP_OK)) return;
  const char* msg = tp_last_error();
  if (rc == TP_ERR_BAD_ARG) TORCH_CHECK_VALUE(false, name, " failed (status ", rc, "): ", msg);
  if (rc == TP_ERR_UNSUPPORTED) TORCH_CHECK_NOT_IMPLEMENTED(false, name, " failed (status ", rc, "): ", msg);
  TORCH_CHECK(false, name, " failed (status ", rc, "): ", msg);
}

// All tensors on one GPU; the kernels have no CPU implementation.
struct OneGpu {
  optional<c10::Device> dev;
  void add(const Tensor& t) {
    if (!t.defined()) return;
    TORCH_CHECK(t.is_cuda(), "torchprime_amd ops run on MI355X only: got a tensor on '", t.device(),
                "'. Move the inputs to the GPU (there is no CPU path).");
    if (!dev) dev = t.device();
    else TORCH_CHECK(t.device() == *dev, "tensors on different devices: ", *dev, " and ", t.device());
  }
  void add(OptTensor t) { if (t.has_value()) add(*t); }
};
template <typename... Ts>
c10::Device require_gpu(const Ts&... ts) {
  OneGpu g;
  (g.add(ts), ...);
  return *g.dev;
}

void* stream_of(c10::Device dev) { return (void*)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

const Tensor& undef() { static const Tensor t; return t; }
const Tensor& val(OptTensor t) { return t.has_value() ? *t : undef(); }
void* opt_ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor empty_f32(at::IntArrayRef size, const Tensor& like) { return at::empty(size, like.options().dtype(at::kFloat)); }

// (..., n) seen as rows of n elements: the tensor itself where its memory already is rows at one stride
struct Rows {
  Tensor t;  // keeps a copy alive
  int64_t rows, cols, stride;
  void* ptr() const { return t.data_ptr(); }
};
Rows rows_of(const Tensor& x, bool align16) {
  const int64_t h = x.size(-1);
  if (x.is_contiguous()) {
    const int64_t rows = h > 0 ? x.numel() / h : 0;
    if (!align16 || ((reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0) && (h * x.element_size()) % 16 == 0)) return {x, rows, h, h};
  }
  Tensor x2 = x.reshape({-1, h});
  const bool bad = align16 ? (x2.stride(-1) != 1 || (x2.stride(0) * x2.element_size()) % 16 != 0 ||
                              reinterpret_cast<uintptr_t>(x2.data_ptr()) % 16 != 0)
                           : (x2.stride(-1) != 1 || (x2.size(0) > 1 && x2.stride(0) < h));
  if (bad) x2 = x2.contiguous();
  return {x2, x2.size(0), h, x2.size(0) > 1 ? x2.stride(0) : h};
}

bool at16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
// t with its elements side by side from a 16-byte address, copied only if they are not: for launches that are handed a
// bare pointer.  (A gradient may be a contiguous piece of a larger tensor at any address; a tensor that comes back through
// a saved-tensor hook may have other strides than the one that went in.)
Tensor packed16(const Tensor& t) {
  const Tensor c = t.contiguous();
  return at16(c) ? c : c.clone(at::MemoryFormat::Contiguous);
}

// New (B,H,S,D') tensor.  Head-minor inputs (the (B,S,H,D)-memory views the attention modules build with
// .view(B,S,H,D).transpose(1,2)) get the same head-minor memory order, so the caller's transpose(1,2).contiguous()
// afterwards is free; anything else gets plain contiguous memory.
Tensor empty_like_heads(const Tensor& x, int64_t D) {
  const int64_t B = x.size(0), H = x.size(1), S = x.size(2);
  if (x.stride(1) < x.stride(2)) return at::empty_strided({B, H, S, D}, {S * H * D, D, H * D, 1}, x.options());
  return at::empty({B, H, S, D}, x.options());
}
// 16-byte rows with a unit inner stride, copied only if they are not
Tensor prep_heads(const Tensor& t) {
  const int64_t e = t.element_size();
  const bool ok = t.stride(3) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && (t.stride(0) * e) % 16 == 0 &&
                  (t.stride(1) * e) % 16 == 0 && (t.stride(2) * e) % 16 == 0;
  return ok ? t : t.contiguous();
}
Strides3 strides3(const Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }

template <typename F>
struct Op;  // typed handle of one operator, looked up once
template <typename R, typename... A>
struct Op<R(A...)> {
  c10::TypedOperatorHandle<R(A...)> h;
  explicit Op(const char* name) : h(c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<R(A...)>()) {}
  R operator()(A... a) const { return h.call(std::forward<A>(a)...); }
};
#define TP_OP(fn, ...)                                  \
  static const auto& op_##fn() {                        \
    static const Op<__VA_ARGS__> op("tprime::" #fn);    \
    return op;                                          \
  }

typedef std::tuple<Tensor, Tensor> T2;
typedef std::tuple<Tensor, Tensor, Tensor> T3;
TP_OP(rmsnorm_fwd, T2(const Tensor&, const Tensor&, double))
TP_OP(rmsnorm_bwd, T2(const Tensor&, const Tensor&, const Tensor&, const Tensor&))
TP_OP(add_rmsnorm_fwd, T3(const Tensor&, const Tensor&, const Tensor&, double))
TP_OP(add_rmsnorm_bwd, T2(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&))
TP_OP(rope_table, T2(const Tensor&, const Tensor&, double, at::ScalarType))
TP_OP(rope_apply, T2(const Tensor&, const Tensor&, const Tensor&, const Tensor&, OptTensor, int64_t, bool))
TP_OP(attn_fwd, T2(const Tensor&, const Tensor&, const Tensor&, OptTensor, double, bool))
TP_OP(attn_bwd, T3(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, OptTensor, double, bool))
TP_OP(attn_fwd_masked, T2(const Tensor&, const Tensor&, const Tensor&, OptTensor, OptTensor, double, bool, int64_t, int64_t, int64_t,
                          double, OptTensor))
TP_OP(attn_bwd_masked, T3(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, OptTensor, OptTensor,
                          double, bool, int64_t, int64_t, int64_t, double, OptTensor))
TP_OP(attn_fwd_pairs, T3(const Tensor&, const Tensor&, const Tensor&, const Tensor&, double, bool))
TP_OP(attn_bwd_pairs, T3(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, int64_t, double, bool))
TP_OP(l2norm_fwd, T2(const Tensor&, double))
TP_OP(l2norm_bwd, Tensor(const Tensor&, const Tensor&, const Tensor&))
TP_OP(scale_rows, Tensor(const Tensor&, const Tensor&))
TP_OP(swiglu_fwd, Tensor(const Tensor&, const Tensor&))
TP_OP(swiglu_bwd, T2(const Tensor&, const Tensor&, const Tensor&))
TP_OP(cross_entropy_fwd, T3(const Tensor&, const Tensor&, int64_t, bool))
TP_OP(cross_entropy_bwd, Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, int64_t))

// ---- autograd plumbing -----------------------------------------------------------------------------------------
// A node with its saved tensors in one array.  ``bwd`` runs the backward operator: below autograd in an ordinary
// backward, through it when a graph of the backward is being recorded (the operator then raises when that graph is
// differentiated).
struct OpNode : torch::autograd::Node {
  std::vector<SavedVariable> saved;
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto& s : saved) s.reset_data();
  }
  Tensor get(size_t i) { return saved[i].unpack(shared_from_this()); }
  void keep(const Tensor& t, bool is_output = false) { saved.emplace_back(t, is_output); }
  virtual variable_list bwd(variable_list&& grads) = 0;
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (at::GradMode::is_enabled()) return bwd(std::move(grads));
    at::AutoDispatchBelowADInplaceOrView below;
    return bwd(std::move(grads));
  }
};
template <typename N, typename... Ts>
std::shared_ptr<N> make_node(const Ts&... inputs) {
  const bool fw = (torch::autograd::isFwGradDefined(inputs) || ...);
  TORCH_CHECK_NOT_IMPLEMENTED(!fw, "the tprime operators have no forward-mode derivative");
  if (!torch::autograd::compute_requires_grad(inputs...)) return nullptr;
  std::shared_ptr<N> n(new N(), torch::autograd::deleteNode);
  n->set_next_edges(torch::autograd::collect_next_edges(inputs...));
  return n;
}
variable_list list2(T2&& r) { return {std::move(std::get<0>(r)), std::move(std::get<1>(r))}; }

// ---- RMSNorm ---------------------------------------------------------------------------------------------------
void check_weight(const Tensor& weight, int64_t hidden) {
  TORCH_CHECK_VALUE(weight.dim() == 1 && weight.size(0) == hidden, "weight shape (", weight.sizes(), ") does not match hidden size ", hidden);
}

T2 rmsnorm_fwd_cuda(const Tensor& x, const Tensor& weight, double eps) {
  const c10::Device dev = require_gpu(x, weight);
  check_weight(weight, x.size(-1));
  c10::DeviceGuard guard(dev);
  const Rows r = rows_of(x, false);
  const Tensor w = weight.contiguous();
  Tensor y = at::empty(x.sizes(), x.options().dtype(at::result_type(weight, x)));
  Tensor rstd = empty_f32({r.rows}, x);
  if (r.rows)
    check(tp_rmsnorm_fwd(r.ptr(), w.data_ptr(), y.data_ptr(), (float*)rstd.data_ptr(), r.rows, (int)r.cols, r.stride, r.cols, (float)eps,
                         dtype_code(x.scalar_type()), dtype_code(w.scalar_type()), stream_of(dev)), "tp_rmsnorm_fwd");
  return {y, rstd};
}

T2 rmsnorm_bwd_cuda(const Tensor& dy, const Tensor& x, const Tensor& weight, const Tensor& rstd) {
  const c10::Device dev = require_gpu(dy, x, weight, rstd);
  c10::DeviceGuard guard(dev);
  const Rows xr = rows_of(x, false), gr = rows_of(dy, false);
  const Tensor w = weight.contiguous();
  Tensor dx = at::empty(x.sizes(), x.options()), dw = at::empty({xr.cols}, w.options());
  if (xr.rows == 0) return {dx, dw.zero_()};
  Tensor ws = empty_f32({(int64_t)tp_rmsnorm_bwd_workspace_bytes(xr.rows, (int)xr.cols) / 4}, x);
  check(tp_rmsnorm_bwd(gr.ptr(), xr.ptr(), w.data_ptr(), (const float*)rstd.data_ptr(), dx.data_ptr(), dw.data_ptr(), (float*)ws.data_ptr(),
                       xr.rows, (int)xr.cols, gr.stride, xr.stride, xr.cols, dtype_code(x.scalar_type()), dtype_code(w.scalar_type()),
                       stream_of(dev)), "tp_rmsnorm_bwd");
  return {dx, dw};
}

struct RmsNormNode : OpNode {
  std::string name() const override { return "TprimeRmsNormBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    const Tensor x = get(0), w = get(1);
    return list2(op_rmsnorm_bwd()(g[0].to(at::result_type(w, x)), x, w, get(2)));
  }
};
T2 rmsnorm_fwd_autograd(const Tensor& x, const Tensor& weight, double eps) {
  auto node = make_node<RmsNormNode>(x, weight);
  T2 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_rmsnorm_fwd()(x, weight, eps); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(x); node->keep(weight); node->keep(std::get<1>(r));
  }
  return r;
}

// (y, h, rstd): h = residual + x, y = RMSNorm(h) * weight, in one pass
T3 add_rmsnorm_fwd_cuda(const Tensor& x, const Tensor& residual, const Tensor& weight, double eps) {
  const c10::Device dev = require_gpu(x, residual, weight);
  TORCH_CHECK_VALUE(residual.sizes() == x.sizes() && residual.scalar_type() == x.scalar_type(), "residual (", residual.sizes(), ")/",
                    residual.scalar_type(), " must match x (", x.sizes(), ")/", x.scalar_type());
  check_weight(weight, x.size(-1));
  c10::DeviceGuard guard(dev);
  const Rows xr = rows_of(x, false), rr = rows_of(residual, false);
  const Tensor w = weight.contiguous();
  Tensor y = at::empty(x.sizes(), x.options().dtype(at::result_type(weight, x))), h = at::empty(x.sizes(), x.options());
  Tensor rstd = empty_f32({xr.rows}, x);
  if (xr.rows)
    check(tp_add_rmsnorm_fwd(xr.ptr(), rr.ptr(), w.data_ptr(), h.data_ptr(), y.data_ptr(), (float*)rstd.data_ptr(), xr.rows, (int)xr.cols,
                             xr.stride, rr.stride, xr.cols, xr.cols, (float)eps, dtype_code(x.scalar_type()), dtype_code(w.scalar_type()),
                             stream_of(dev)), "tp_add_rmsnorm_fwd");
  return {y, h, rstd};
}

T2 add_rmsnorm_bwd_cuda(const Tensor& dy, const Tensor& dh, const Tensor& h, const Tensor& weight, const Tensor& rstd) {
  const c10::Device dev = require_gpu(dy, dh, h, weight, rstd);
  c10::DeviceGuard guard(dev);
  const Rows hr = rows_of(h, false), gr = rows_of(dy, false), dr = rows_of(dh, false);
  const Tensor w = weight.contiguous();
  Tensor dx = at::empty(h.sizes(), h.options()), dw = at::empty({hr.cols}, w.options());
  if (hr.rows == 0) return {dx, dw.zero_()};
  Tensor ws = empty_f32({(int64_t)tp_rmsnorm_bwd_workspace_bytes(hr.rows, (int)hr.cols) / 4}, h);
  check(tp_add_rmsnorm_bwd(gr.ptr(), dr.ptr(), hr.ptr(), w.data_ptr(), (const float*)rstd.data_ptr(), dx.data_ptr(), dw.data_ptr(),
                           (float*)ws.data_ptr(), hr.rows, (int)hr.cols, gr.stride, dr.stride, hr.stride, hr.cols,
                           dtype_code(h.scalar_type()), dtype_code(w.scalar_type()), stream_of(dev)), "tp_add_rmsnorm_bwd");
  return {dx, dw};
}

struct AddRmsNormNode : OpNode {
  std::string name() const override { return "TprimeAddRmsNormBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined() && !g[1].defined()) return {Tensor(), Tensor(), Tensor()};
    const Tensor h = get(0), w = get(1), rstd = get(2);
    const auto out_dtype = at::result_type(w, h);
    const Tensor dy = g[0].defined() ? g[0].to(out_dtype) : at::zeros_like(h, h.options().dtype(out_dtype));
    T2 r = g[1].defined() ? op_add_rmsnorm_bwd()(dy, g[1].to(h.scalar_type()), h, w, rstd) : op_rmsnorm_bwd()(dy, h, w, rstd);
    return {std::get<0>(r), std::get<0>(r), std::get<1>(r)};
  }
};
T3 add_rmsnorm_fwd_autograd(const Tensor& x, const Tensor& residual, const Tensor& weight, double eps) {
  auto node = make_node<AddRmsNormNode>(x, residual, weight);
  T3 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_add_rmsnorm_fwd()(x, residual, weight, eps); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    torch::autograd::set_history(std::get<1>(r), node);
    node->keep(std::get<1>(r), true); node->keep(weight); node->keep(std::get<2>(r));
  }
  return r;
}

// ---- rotary ----------------------------------------------------------------------------------------------------
// cos/sin tables (Bp, S, 2*half) from inv_freq (half) and position_ids (Bp, S)
T2 rope_table_cuda(const Tensor& inv_freq, const Tensor& position_ids, double attention_scaling, at::ScalarType dtype) {
  const c10::Device dev = require_gpu(inv_freq, position_ids);
  TORCH_CHECK_VALUE(position_ids.dim() == 2 && inv_freq.dim() == 1, "expected inv_freq (half,) and position_ids (batch, seq)");
  c10::DeviceGuard guard(dev);
  const Tensor f = inv_freq.to(at::kFloat).contiguous(), p = position_ids.to(at::kFloat).contiguous();
  const int64_t Bp = p.size(0), S = p.size(1), half = f.size(0);
  Tensor cos = at::empty({Bp, S, 2 * half}, f.options().dtype(dtype)), sin = at::empty({Bp, S, 2 * half}, f.options().dtype(dtype));
  check(tp_rope_table((const float*)f.data_ptr(), (const float*)p.data_ptr(), cos.data_ptr(), sin.data_ptr(), (int)Bp, (int)S, (int)half,
                      (float)attention_scaling, dtype_code(dtype), stream_of(dev)), "tp_rope_table");
  return {cos, sin};
}

// cos[position_ids] raises IndexError for ids outside the table (model/mixtral/model.py:136-137); so does this.  The
// check is a device reduction and a host synchronisation, so its verdict is kept per tensor object (a weak reference
// and the version counter, never the address alone): a model hands the same position_ids to every layer and to the
// backward of each.
void check_positions(const Tensor& pos, int64_t table_rows) {
  struct Entry { c10::weak_intrusive_ptr<c10::TensorImpl> ref; uint32_t version; int64_t numel, rows; };
  static std::mutex mu;
  static std::unordered_map<c10::TensorImpl*, Entry> verdicts;
  c10::TensorImpl* impl = pos.unsafeGetTensorImpl();
  const bool tracked = !pos.is_inference();
  const uint32_t version = tracked ? (uint32_t)pos._version() : 0;
  if (tracked) {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = verdicts.find(impl);
    if (it != verdicts.end() && !it->second.ref.expired() && it->second.version == version && it->second.numel == pos.numel() &&
        it->second.rows == table_rows) return;
  }
  int64_t lo = 0, hi = 0;
  if (pos.numel()) {
    const Tensor both = at::stack({pos.min(), pos.max()}).cpu();
    lo = both.const_data_ptr<int64_t>()[0];
    hi = both.const_data_ptr<int64_t>()[1];
  }
  TORCH_CHECK_INDEX(lo >= -table_rows && hi < table_rows, "position id ", hi >= table_rows ? hi : lo,
                    " is out of bounds for a rotary table of ", table_rows, " rows");
  TORCH_CHECK_NOT_IMPLEMENTED(lo >= 0, "negative position ids (indexing the table from its end) are not supported");
  if (!tracked) return;
  std::lock_guard<std::mutex> lock(mu);
  if (verdicts.size() >= 64) {  // drop what died; if all live, start over
    for (auto it = verdicts.begin(); it != verdicts.end();) it = it->second.ref.expired() ? verdicts.erase(it) : std::next(it);
    if (verdicts.size() >= 64) verdicts.clear();
  }
  verdicts.insert_or_assign(impl, Entry{c10::weak_intrusive_ptr<c10::TensorImpl>(pos.getIntrusivePtr()), version, pos.numel(), table_rows});
}

// interleaved: 0 rotate-half, 1 DeepSeek ([evens | odds] output), 2 adjacent pairs in place (Llama-4)
T2 rope_apply_cuda(const Tensor& q_, const Tensor& k_, const Tensor& cos_, const Tensor& sin_, OptTensor pos_, int64_t interleaved,
                   bool backward) {
  const c10::Device dev = require_gpu(q_, k_, cos_, sin_, pos_);
  TORCH_CHECK_VALUE(q_.dim() == 4 && k_.dim() == 4, "rotary apply expects (batch, heads, seq, dim) tensors");
  c10::DeviceGuard guard(dev);
  const int64_t B = q_.size(0), Hq = q_.size(1), S = q_.size(2), D = q_.size(3);
  TORCH_CHECK_VALUE(k_.size(0) == B && k_.size(2) == S && k_.size(3) == D && k_.scalar_type() == q_.scalar_type(), "q (", q_.sizes(),
                    ") and k (", k_.sizes(), ") disagree on batch/seq/dim or dtype");
  Tensor cos = cos_.to(q_.scalar_type()), sin = sin_.to(q_.scalar_type()), pos;
  const Tensor q = prep_heads(q_), k = prep_heads(k_);
  int64_t cs_b, cs_s, pos_b = 0, table_rows = 0;
  if (pos_.has_value()) {
    // table gather (Mixtral): cos/sin are (T, D), pos is (B or 1, S) integer
    TORCH_CHECK_VALUE(cos.dim() == 2, "with position_ids the cos/sin tables must be (max_pos, dim)");
    cos = cos.contiguous();
    sin = sin.contiguous();
    pos = pos_->to(at::kLong).contiguous();
    if (pos.dim() == 1) pos = pos.unsqueeze(0);
    TORCH_CHECK_VALUE(pos.size(-1) == S && (pos.size(0) == 1 || pos.size(0) == B), "position_ids shape (", pos.sizes(),
                      ") does not match (batch, seq) = (", B, ", ", S, ")");
    check_positions(pos, cos.size(0));
    cs_b = 0; cs_s = cos.stride(0); pos_b = pos.size(0) == B && B > 1 ? pos.stride(0) : 0; table_rows = cos.size(0);
  } else {
    if (cos.dim() == 2) { cos = cos.unsqueeze(0); sin = sin.unsqueeze(0); }
    TORCH_CHECK_VALUE(cos.dim() == 3 && cos.size(1) == S && cos.size(2) == D && (cos.size(0) == 1 || cos.size(0) == B), "cos/sin shape (",
                      cos.sizes(), ") does not broadcast to (batch, seq, dim) = (", B, ", ", S, ", ", D, ")");
    if (cos.stride(-1) != 1 || sin.strides() != cos.strides()) { cos = cos.contiguous(); sin = sin.contiguous(); }
    cs_b = cos.size(0) == B && B > 1 ? cos.stride(0) : 0;
    cs_s = cos.stride(1);
  }
  Tensor qo = empty_like_heads(q, D), ko = empty_like_heads(k, D);
  const Strides3 qs = strides3(q), ks = strides3(k), qos = strides3(qo), kos = strides3(ko);
  check(tp_rope_apply(q.data_ptr(), k.data_ptr(), cos.data_ptr(), sin.data_ptr(), (const int64_t*)opt_ptr(pos), qo.data_ptr(), ko.data_ptr(),
                      (int)B, (int)Hq, (int)k.size(1), (int)S, (int)D, qs.data(), ks.data(), qos.data(), kos.data(), cs_b, cs_s, pos_b,
                      table_rows, (int)interleaved, (int)backward, dtype_code(q.scalar_type()), stream_of(dev)), "tp_rope_apply");
  return {qo, ko};
}

struct RopeNode : OpNode {
  bool has_pos, backward;
  int64_t interleaved;
  // a gradient that did not arrive (only one of the two outputs is used) is zero
  std::array<std::vector<int64_t>, 2> sizes;
  at::TensorOptions opts;
  std::string name() const override { return "TprimeRopeApplyBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined() && !g[1].defined()) return {Tensor(), Tensor()};
    for (int i = 0; i < 2; i++)
      if (!g[i].defined()) g[i] = at::zeros(sizes[i], opts);
    const optional<Tensor> pos = has_pos ? optional<Tensor>(get(2)) : std::nullopt;
    // the transpose of the transposed rotation is the rotation itself
    return list2(op_rope_apply()(g[0], g[1], get(0), get(1), pos, interleaved, !backward));
  }
};
T2 rope_apply_autograd(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, OptTensor pos, int64_t interleaved, bool backward) {
  auto node = make_node<RopeNode>(q, k);
  T2 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_rope_apply()(q, k, cos, sin, pos, interleaved, backward); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    torch::autograd::set_history(std::get<1>(r), node);
    node->keep(cos); node->keep(sin);
    if (pos.has_value()) node->keep(*pos);
    node->has_pos = pos.has_value();
    node->interleaved = interleaved;
    node->backward = backward;
    node->sizes = {q.sizes().vec(), k.sizes().vec()};
    node->opts = q.options();
  }
  return r;
}

// ---- attention -------------------------------------------------------------------------------------------------
struct AttnShape { int B, Hq, Hkv, Sq, Skv, Dqk, Dv; };
AttnShape check_attn(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& seg) {
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "attention expects (batch, heads, seq, dim) tensors");
  const AttnShape s{(int)q.size(0), (int)q.size(1), (int)k.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3), (int)v.size(3)};
  TORCH_CHECK_VALUE(k.size(0) == s.B && k.size(3) == s.Dqk && v.size(0) == s.B && v.size(1) == s.Hkv && v.size(2) == s.Skv, "q (", q.sizes(),
                    "), k (", k.sizes(), "), v (", v.sizes(), ") are inconsistent");
  TORCH_CHECK_VALUE(s.Hkv != 0 && s.Hq % s.Hkv == 0, "num query heads ", s.Hq, " must be a multiple of num kv heads ", s.Hkv);
  const auto t = q.scalar_type();
  TORCH_CHECK_TYPE((t == at::kBFloat16 || t == at::kHalf || t == at::kFloat) && k.scalar_type() == t && v.scalar_type() == t,
                   "attention kernels take bfloat16, float16 or float32 q/k/v of one dtype, got ", t, "/", k.scalar_type(), "/", v.scalar_type());
  const bool square = s.Dqk == s.Dv && (s.Dqk == 64 || s.Dqk == 128);
  TORCH_CHECK_NOT_IMPLEMENTED(square || (t != at::kFloat && s.Dqk == 192 && s.Dv == 128), "head dims (qk=", s.Dqk, ", v=", s.Dv,
                              ") not built for ", t, "; supported: (64, 64), (128, 128)", t == at::kFloat ? "" : ", (192, 128)");
  // kernel_utils.py:238-241: segment ids must cover the whole (unsharded) sequence
  if (seg.defined() && !(seg.dim() == 2 && seg.size(0) == s.B && seg.size(1) == s.Skv && s.Sq == s.Skv)) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(PyExc_AssertionError, "Sharding along sequence dimension not allowed in tpu kernel attention");
    throw py::error_already_set();
  }
  return s;
}
Tensor prep_ids(const Tensor& seg) { return seg.defined() ? seg.to(at::kInt).contiguous() : seg; }
Tensor prep_qpos(const Tensor& qpos, int64_t Sq) {
  if (!qpos.defined()) return qpos;
  TORCH_CHECK_VALUE(qpos.dim() == 1 && qpos.size(0) == Sq, "q_positions must have shape (", Sq, ",), got (", qpos.sizes(), ")");
  return qpos.to(at::kInt).contiguous();
}
// fp32 tensor with a contiguous key axis, its (batch, head, query) strides with 0 on broadcast axes
Tensor prep_bias(const Tensor& bias, const AttnShape& s, Strides3& st) {
  if (!bias.defined()) return bias;
  TORCH_CHECK_VALUE(bias.dim() == 4 && (bias.size(0) == 1 || bias.size(0) == s.B) && (bias.size(1) == 1 || bias.size(1) == s.Hq) &&
                    bias.size(2) == s.Sq && bias.size(3) == s.Skv, "mask must have shape (1|", s.B, ", 1|", s.Hq, ", ", s.Sq, ", ", s.Skv,
                    "), got (", bias.sizes(), ")");
  Tensor b = bias.to(at::kFloat);
  if (b.stride(-1) != 1) b = b.contiguous();
  st = {b.size(0) == 1 ? 0 : b.stride(0), b.size(1) == 1 ? 0 : b.stride(1), b.stride(2)};
  return b;
}

T2 attn_fwd_cuda(const Tensor& q_, const Tensor& k_, const Tensor& v_, OptTensor seg_, double sm_scale, bool causal) {
  const c10::Device dev = require_gpu(q_, k_, v_, seg_);
  const AttnShape s = check_attn(q_, k_, v_, val(seg_));
  c10::DeviceGuard guard(dev);
  const Tensor q = prep_heads(q_), k = prep_heads(k_), v = prep_heads(v_), seg = prep_ids(val(seg_));
  Tensor out = empty_like_heads(q, s.Dv), lse = empty_f32({s.B, s.Hq, s.Sq}, q);
  if (out.numel()) {
    const Strides3 qs = strides3(q), ks = strides3(k), vs = strides3(v), os = strides3(out);
    check(tp_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const int32_t*)opt_ptr(seg), out.data_ptr(), (float*)lse.data_ptr(), s.B, s.Hq,
                      s.Hkv, s.Sq, s.Skv, s.Dqk, s.Dv, qs.data(), ks.data(), vs.data(), os.data(), (float)sm_scale, (int)causal,
                      dtype_code(q.scalar_type()), stream_of(dev)), "tp_attn_fwd");
  }
  return {out, lse};
}

// the parts of a backward problem that do not depend on its mask, and the launch
struct BwdCall {
  c10::Device dev;
  AttnShape s;
  c10::DeviceGuard guard;
  Tensor q, k, v, out, dout, lse, dq, dk, dv;
  tp_attn_bwd_problem p{};
  BwdCall(c10::Device device, const Tensor& dout_, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& out_, const Tensor& lse_,
          const Tensor& seg_, double sm_scale)
      : dev(device), s(check_attn(q_, k_, v_, seg_)), guard(device), q(prep_heads(q_)), k(prep_heads(k_)), v(prep_heads(v_)),
        out(prep_heads(out_)), dout(prep_heads(dout_)), lse(lse_.contiguous()), dq(empty_like_heads(q, s.Dqk)), dk(empty_like_heads(k, s.Dqk)),
        dv(empty_like_heads(v, s.Dv)) {
    p.dout = dout.data_ptr(); p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.out = out.data_ptr();
    p.lse = (const float*)lse.data_ptr();
    p.dq = dq.data_ptr(); p.dk = dk.data_ptr(); p.dv = dv.data_ptr();
    p.B = s.B; p.Hq = s.Hq; p.Hkv = s.Hkv; p.Sq = s.Sq; p.Skv = s.Skv; p.Dqk = s.Dqk; p.Dv = s.Dv;
    const auto st = [](int64_t (&d)[3], const Tensor& t) { for (int i = 0; i < 3; i++) d[i] = t.stride(i); };
    st(p.do_strides, dout); st(p.q_strides, q); st(p.k_strides, k); st(p.v_strides, v); st(p.o_strides, out);
    st(p.dq_strides, dq); st(p.dk_strides, dk); st(p.dv_strides, dv);
    p.sm_scale = (float)sm_scale;
    p.window_left = p.window_right = -1;
    p.dtype = dtype_code(q.scalar_type());
  }
  T3 run() {
    if (dq.numel() == 0 || dk.numel() == 0) return {dq.zero_(), dk.zero_(), dv.zero_()};
    // one workspace: the row vectors, then the pieces of split key tiles (none for most problems)
    const size_t rows = tp_attn_bwd_workspace_bytes(s.B, s.Hq, s.Sq), at = (rows + 255) / 256 * 256;
    tp_attn_bwd_plan plan;
    p.parts_bytes = tp_attn_bwd_make_plan(&p, &plan);
    const Tensor ws = empty_f32({(int64_t)((p.parts_bytes ? at + p.parts_bytes : rows) / 4)}, q);
    p.ws = (float*)ws.data_ptr();
    p.parts = p.parts_bytes ? (char*)ws.data_ptr() + at : nullptr;
    check(tp_attn_bwd_run_planned(&p, &plan, stream_of(dev), nullptr), "tp_attn_bwd_run");
    return {dq, dk, dv};
  }
};

T3 attn_bwd_cuda(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse, OptTensor seg_,
                 double sm_scale, bool causal) {
  BwdCall c(require_gpu(dout, q, k, v, out, lse, seg_), dout, q, k, v, out, lse, val(seg_), sm_scale);
  const Tensor seg = prep_ids(val(seg_));
  c.p.seg = (const int32_t*)opt_ptr(seg);
  c.p.causal = causal;
  return c.run();
}

struct AttnNode : OpNode {
  bool has_seg, causal;
  double sm_scale;
  std::string name() const override { return "TprimeAttnBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const optional<Tensor> seg = has_seg ? optional<Tensor>(get(5)) : std::nullopt;
    T3 r = op_attn_bwd()(g[0], get(0), get(1), get(2), get(3), get(4), seg, sm_scale, causal);
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r)};
  }
};
T2 attn_fwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, OptTensor seg, double sm_scale, bool causal) {
  auto node = make_node<AttnNode>(q, k, v);
  T2 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_attn_fwd()(q, k, v, seg, sm_scale, causal); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(q); node->keep(k); node->keep(v); node->keep(std::get<0>(r), true); node->keep(std::get<1>(r));
    if (seg.has_value()) node->keep(*seg);
    node->has_seg = seg.has_value();
    node->causal = causal;
    node->sm_scale = sm_scale;
  }
  return r;
}

// mask extensions: sliding window, soft cap, query rows in another order than the keys, additive masks
T2 attn_fwd_masked_cuda(const Tensor& q_, const Tensor& k_, const Tensor& v_, OptTensor seg_, OptTensor qpos_, double sm_scale, bool causal,
                        int64_t causal_offset, int64_t window_left, int64_t window_right, double soft_cap, OptTensor bias_) {
  const c10::Device dev = require_gpu(q_, k_, v_, seg_, qpos_, bias_);
  const AttnShape s = check_attn(q_, k_, v_, val(seg_));
  c10::DeviceGuard guard(dev);
  const Tensor q = prep_heads(q_), k = prep_heads(k_), v = prep_heads(v_), seg = prep_ids(val(seg_)), qpos = prep_qpos(val(qpos_), s.Sq);
  Tensor out = empty_like_heads(q, s.Dv), lse = empty_f32({s.B, s.Hq, s.Sq}, q);
  Strides3 bs{};
  const Tensor bias = prep_bias(val(bias_), s, bs);
  if (out.numel()) {
    const Strides3 qs = strides3(q), ks = strides3(k), vs = strides3(v), os = strides3(out);
    const auto launch = [&](auto fn, const char* name, auto... bias_args) {
      check(fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const int32_t*)opt_ptr(seg), (const int32_t*)opt_ptr(qpos), bias_args...,
               out.data_ptr(), (float*)lse.data_ptr(), s.B, s.Hq, s.Hkv, s.Sq, s.Skv, s.Dqk, s.Dv, qs.data(), ks.data(), vs.data(), os.data(),
               (float)sm_scale, (int)causal, (int)causal_offset, (int)window_left, (int)window_right, (float)soft_cap,
               dtype_code(q.scalar_type()), stream_of(dev)), name);
    };
    if (bias.defined()) launch(tp_attn_fwd_biased, "tp_attn_fwd_biased", (const float*)bias.data_ptr(), (const int64_t*)bs.data());
    else launch(tp_attn_fwd_masked, "tp_attn_fwd_masked");
  }
  return {out, lse};
}

T3 attn_bwd_masked_cuda(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
                        OptTensor seg_, OptTensor qpos_, double sm_scale, bool causal, int64_t causal_offset, int64_t window_left,
                        int64_t window_right, double soft_cap, OptTensor bias_) {
  BwdCall c(require_gpu(dout, q, k, v, out, lse, seg_, qpos_, bias_), dout, q, k, v, out, lse, val(seg_), sm_scale);
  Strides3 bs{};
  const Tensor seg = prep_ids(val(seg_)), qpos = prep_qpos(val(qpos_), c.s.Sq), bias = prep_bias(val(bias_), c.s, bs);
  c.p.seg = (const int32_t*)opt_ptr(seg);
  c.p.q_positions = (const int32_t*)opt_ptr(qpos);
  c.p.bias = (const float*)opt_ptr(bias);
  std::copy(bs.begin(), bs.end(), c.p.bias_strides);
  c.p.causal = causal;
  c.p.causal_offset = (int)causal_offset;
  c.p.window_left = (int)window_left;
  c.p.window_right = (int)window_right;
  c.p.soft_cap = (float)soft_cap;
  return c.run();
}

struct AttnMaskedNode : OpNode {
  int has_seg, has_qpos, has_bias;
  bool causal;
  double sm_scale, soft_cap;
  int64_t causal_offset, window_left, window_right;
  std::string name() const override { return "TprimeAttnMaskedBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const auto opt = [&](int has, int at) { return has ? optional<Tensor>(get(at)) : std::nullopt; };
    const optional<Tensor> seg = opt(has_seg, 5), qpos = opt(has_qpos, 5 + has_seg), bias = opt(has_bias, 5 + has_seg + has_qpos);
    T3 r = op_attn_bwd_masked()(g[0], get(0), get(1), get(2), get(3), get(4), seg, qpos, sm_scale, causal, causal_offset, window_left,
                                window_right, soft_cap, bias);
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r)};
  }
};
T2 attn_fwd_masked_autograd(const Tensor& q, const Tensor& k, const Tensor& v, OptTensor seg, OptTensor qpos, double sm_scale, bool causal,
                            int64_t causal_offset, int64_t window_left, int64_t window_right, double soft_cap, OptTensor bias) {
  auto node = make_node<AttnMaskedNode>(q, k, v);
  T2 r = [&] {
    at::AutoDispatchBelowADInplaceOrView below;
    return op_attn_fwd_masked()(q, k, v, seg, qpos, sm_scale, causal, causal_offset, window_left, window_right, soft_cap, bias);
  }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(q); node->keep(k); node->keep(v); node->keep(std::get<0>(r), true); node->keep(std::get<1>(r));
    for (const auto* t : {&seg, &qpos, &bias})
      if (t->has_value()) node->keep(**t);
    node->has_seg = seg.has_value(); node->has_qpos = qpos.has_value(); node->has_bias = bias.has_value();
    node->causal = causal; node->sm_scale = sm_scale; node->soft_cap = soft_cap;
    node->causal_offset = causal_offset; node->window_left = window_left; node->window_right = window_right;
  }
  return r;
}

// additive masks that only drop pairs (tp_mask_pairs): a (1|B, 1, Sq, Skv) mask in any of the three dtypes
struct PairsIn { Tensor mask; int batches; std::array<int64_t, 2> strides; };
PairsIn prep_pairs(const Tensor& mask, int64_t Sq, int64_t Skv) {
  TORCH_CHECK_VALUE(mask.dim() == 4 && mask.size(1) == 1 && mask.size(2) == Sq && mask.size(3) == Skv, "mask must have shape (1|batch, 1, ", Sq,
                    ", ", Skv, "), got (", mask.sizes(), ")");
  const Tensor m = mask.stride(3) != 1 ? mask.contiguous() : mask;
  return {m, (int)m.size(0), {m.size(0) == 1 ? 0 : m.stride(0), m.stride(2)}};
}
Tensor make_pairs(const PairsIn& m, int64_t Sq, int64_t Skv, bool verdict, void* stream) {
  Tensor pairs = at::empty({(int64_t)tp_mask_pairs_bytes(m.batches, (int)Sq, (int)Skv) / 4}, m.mask.options().dtype(at::kInt));
  if (verdict) pairs.slice(0, 0, 16).zero_();
  check(tp_mask_pairs(m.mask.data_ptr(), m.strides.data(), m.batches, (int)Sq, (int)Skv, dtype_code(m.mask.scalar_type()), pairs.data_ptr(),
                      (int)verdict, stream), "tp_mask_pairs");
  return pairs;
}
// (out, lse, pairs): the bits are made once per forward and kept for the backward
T3 attn_fwd_pairs_cuda(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& mask, double sm_scale, bool /*causal_padded*/) {
  const c10::Device dev = require_gpu(q_, k_, v_, mask);
  const AttnShape s = check_attn(q_, k_, v_, undef());
  TORCH_CHECK_VALUE(mask.size(0) == 1 || mask.size(0) == s.B, "mask batch ", mask.size(0), " does not broadcast to ", s.B);
  c10::DeviceGuard guard(dev);
  const Tensor q = prep_heads(q_), k = prep_heads(k_), v = prep_heads(v_);
  const PairsIn m = prep_pairs(mask, s.Sq, s.Skv);
  const Tensor pairs = make_pairs(m, s.Sq, s.Skv, false, stream_of(dev));
  Tensor out = empty_like_heads(q, s.Dv), lse = empty_f32({s.B, s.Hq, s.Sq}, q);
  const Strides3 qs = strides3(q), ks = strides3(k), vs = strides3(v), os = strides3(out);
  check(tp_attn_fwd_pairs(q.data_ptr(), k.data_ptr(), v.data_ptr(), pairs.data_ptr(), m.batches, out.data_ptr(), (float*)lse.data_ptr(), s.B, s.Hq,
                          s.Hkv, s.Sq, s.Skv, s.Dqk, s.Dv, qs.data(), ks.data(), vs.data(), os.data(), (float)sm_scale,
                          dtype_code(q.scalar_type()), stream_of(dev)), "tp_attn_fwd_pairs");
  return {out, lse, pairs};
}
T3 attn_bwd_pairs_cuda(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
                       const Tensor& pairs, int64_t mask_batches, double sm_scale, bool causal_padded) {
  BwdCall c(require_gpu(dout, q, k, v, out, lse, pairs), dout, q, k, v, out, lse, undef(), sm_scale);
  TORCH_CHECK_VALUE(pairs.is_contiguous() && pairs.scalar_type() == at::kInt && mask_batches > 0 &&
                    pairs.numel() == (int64_t)tp_mask_pairs_bytes((int)mask_batches, c.s.Sq, c.s.Skv) / 4, "pairs were not made for this problem");
  c.p.pairs = pairs.data_ptr();
  c.p.mask_batches = (int)mask_batches;
  c.p.pairs_causal = causal_padded;
  return c.run();
}
struct AttnPairsNode : OpNode {
  int64_t mask_batches;
  double sm_scale;
  bool causal_padded;
  std::string name() const override { return "TprimeAttnPairsBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    T3 r = op_attn_bwd_pairs()(g[0], get(0), get(1), get(2), get(3), get(4), get(5), mask_batches, sm_scale, causal_padded);
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r)};
  }
};
T3 attn_fwd_pairs_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, double sm_scale, bool causal_padded) {
  auto node = make_node<AttnPairsNode>(q, k, v);
  T3 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_attn_fwd_pairs()(q, k, v, mask, sm_scale, causal_padded); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(q); node->keep(k); node->keep(v); node->keep(std::get<0>(r), true); node->keep(std::get<1>(r)); node->keep(std::get<2>(r));
    node->mask_batches = mask.size(0);
    node->sm_scale = sm_scale;
    node->causal_padded = causal_padded;
  }
  return r;
}

// ---- L2 norm, temperature scale ----------------------------------------------------------------------------------
T2 l2norm_fwd_cuda(const Tensor& x, double eps) {
  const c10::Device dev = require_gpu(x);
  c10::DeviceGuard guard(dev);
  const Rows r = rows_of(x, true);
  Tensor y = at::empty(x.sizes(), x.options()), rstd = empty_f32({r.rows}, x);
  if (r.rows)
    check(tp_l2norm_fwd(r.ptr(), y.data_ptr(), (float*)rstd.data_ptr(), r.rows, (int)r.cols, r.stride, r.cols, (float)eps,
                        dtype_code(x.scalar_type()), stream_of(dev)), "tp_l2norm_fwd");
  return {y, rstd};
}
Tensor l2norm_bwd_cuda(const Tensor& dy, const Tensor& x, const Tensor& rstd) {
  const c10::Device dev = require_gpu(dy, x, rstd);
  c10::DeviceGuard guard(dev);
  const Rows xr = rows_of(x, true), gr = rows_of(dy, true);
  Tensor dx = at::empty(x.sizes(), x.options());
  if (xr.rows)
    check(tp_l2norm_bwd(gr.ptr(), xr.ptr(), (const float*)rstd.data_ptr(), dx.data_ptr(), xr.rows, (int)xr.cols, gr.stride, xr.stride, xr.cols,
                        dtype_code(x.scalar_type()), stream_of(dev)), "tp_l2norm_bwd");
  return dx;
}
struct L2NormNode : OpNode {
  std::string name() const override { return "TprimeL2NormBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    const Tensor x = get(0);
    return {op_l2norm_bwd()(g[0].to(x.scalar_type()), x, get(1))};
  }
};
T2 l2norm_fwd_autograd(const Tensor& x, double eps) {
  auto node = make_node<L2NormNode>(x);
  T2 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_l2norm_fwd()(x, eps); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(x); node->keep(std::get<1>(r));
  }
  return r;
}

// x (B, S, N, D) times scale (S) fp32 per position, rounded to x's dtype
Tensor scale_rows_cuda(const Tensor& x, const Tensor& scale) {
  const c10::Device dev = require_gpu(x, scale);
  TORCH_CHECK_VALUE(x.dim() == 4 && scale.dim() == 1 && scale.size(0) == x.size(1), "expected x (batch, seq, heads, dim) and scale (seq,), got (",
                    x.sizes(), ") and (", scale.sizes(), ")");
  c10::DeviceGuard guard(dev);
  const Rows r = rows_of(x, true);
  const Tensor s = scale.to(at::kFloat).contiguous();
  Tensor y = at::empty(x.sizes(), x.options());
  if (y.numel())
    check(tp_scale_rows(r.ptr(), (const float*)s.data_ptr(), y.data_ptr(), r.rows, (int)r.cols, r.stride, r.cols, (int)x.size(2), (int)x.size(1),
                        dtype_code(x.scalar_type()), stream_of(dev)), "tp_scale_rows");
  return y;
}
struct ScaleRowsNode : OpNode {
  std::string name() const override { return "TprimeScaleRowsBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    return {op_scale_rows()(g[0], get(0))};
  }
};
Tensor scale_rows_autograd(const Tensor& x, const Tensor& scale) {
  auto node = make_node<ScaleRowsNode>(x);
  Tensor r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_scale_rows()(x, scale); }();
  if (node) {
    torch::autograd::set_history(r, node);
    node->keep(scale);
  }
  return r;
}

// ---- SwiGLU ------------------------------------------------------------------------------------------------------
Tensor swiglu_fwd_cuda(const Tensor& gate, const Tensor& up) {
  const c10::Device dev = require_gpu(gate, up);
  TORCH_CHECK_VALUE(gate.sizes() == up.sizes() && gate.scalar_type() == up.scalar_type(), "gate (", gate.sizes(), ")/", gate.scalar_type(),
                    " and up (", up.sizes(), ")/", up.scalar_type(), " must match");
  c10::DeviceGuard guard(dev);
  const Rows g = rows_of(gate, true), u = rows_of(up, true);
  Tensor out = at::empty(gate.sizes(), gate.options());
  if (out.numel())
    check(tp_swiglu_fwd(g.ptr(), u.ptr(), out.data_ptr(), g.rows, (int)g.cols, g.stride, u.stride, g.cols, dtype_code(gate.scalar_type()),
                        stream_of(dev)), "tp_swiglu_fwd");
  return out;
}
T2 swiglu_bwd_cuda(const Tensor& dout, const Tensor& gate, const Tensor& up) {
  const c10::Device dev = require_gpu(dout, gate, up);
  c10::DeviceGuard guard(dev);
  const Rows d = rows_of(dout, true), g = rows_of(gate, true), u = rows_of(up, true);
  Tensor dg = at::empty(gate.sizes(), gate.options()), du = at::empty(up.sizes(), up.options());
  if (dg.numel())
    check(tp_swiglu_bwd(d.ptr(), g.ptr(), u.ptr(), dg.data_ptr(), du.data_ptr(), g.rows, (int)g.cols, d.stride, g.stride, u.stride, g.cols, g.cols,
                        dtype_code(gate.scalar_type()), stream_of(dev)), "tp_swiglu_bwd");
  return {dg, du};
}
struct SwigluNode : OpNode {
  std::string name() const override { return "TprimeSwigluBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    const Tensor gate = get(0);
    return list2(op_swiglu_bwd()(g[0].to(gate.scalar_type()), gate, get(1)));
  }
};
Tensor swiglu_fwd_autograd(const Tensor& gate, const Tensor& up) {
  auto node = make_node<SwigluNode>(gate, up);
  Tensor r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_swiglu_fwd()(gate, up); }();
  if (node) {
    torch::autograd::set_history(r, node);
    node->keep(gate); node->keep(up);
  }
  return r;
}

// ---- cross entropy -----------------------------------------------------------------------------------------------
Tensor prep_labels(const Tensor& labels) {
  Tensor l = labels.to(at::kLong);
  return l.stride(1) != 1 ? l.contiguous() : l;
}
// (loss (scalar fp32), lse (B*S), loss_and_count (2)) of the shifted next-token cross entropy; scored_only: the lse of rows
// without a target is 0 (they are not read)
T3 cross_entropy_fwd_cuda(const Tensor& logits_, const Tensor& labels_, int64_t ignore_index, bool scored_only) {
  const c10::Device dev = require_gpu(logits_, labels_);
  TORCH_CHECK_VALUE(logits_.dim() == 3 && labels_.dim() == 2 && labels_.size(0) == logits_.size(0) && labels_.size(1) == logits_.size(1),
                    "expected logits (batch, seq, vocab) and labels (batch, seq), got (", logits_.sizes(), ") and (", labels_.sizes(), ")");
  TORCH_CHECK_TYPE(logits_.scalar_type() == at::kFloat || logits_.scalar_type() == at::kBFloat16,
                   "cross entropy takes float32 or bfloat16 logits, got ", logits_.scalar_type());
  c10::DeviceGuard guard(dev);
  const int64_t B = logits_.size(0), S = logits_.size(1), V = logits_.size(2);
  const Tensor logits = logits_.stride(2) != 1 ? logits_.contiguous() : logits_, labels = prep_labels(labels_);
  Tensor lse = empty_f32({B * S}, logits), row_loss = empty_f32({B * S}, logits), lc = empty_f32({2}, logits), loss = empty_f32({}, logits);
  check(tp_cross_entropy_fwd_loss(logits.data_ptr(), (const int64_t*)labels.data_ptr(), (float*)lse.data_ptr(), (float*)row_loss.data_ptr(),
                                  (float*)lc.data_ptr(), (float*)loss.data_ptr(), (int)B, (int)S, (int)V, logits.stride(0), logits.stride(1),
                                  labels.stride(0), (int)ignore_index, (int)scored_only, dtype_code(logits.scalar_type()), stream_of(dev)),
        "tp_cross_entropy_fwd_loss");
  return {loss, lse, lc};
}
Tensor cross_entropy_bwd_cuda(const Tensor& dloss, const Tensor& logits_, const Tensor& labels_, const Tensor& lse, const Tensor& lc,
                              int64_t ignore_index) {
  const c10::Device dev = require_gpu(dloss, logits_, labels_, lse, lc);
  c10::DeviceGuard guard(dev);
  const int64_t B = logits_.size(0), S = logits_.size(1), V = logits_.size(2);
  const Tensor logits = logits_.stride(2) != 1 ? logits_.contiguous() : logits_, labels = prep_labels(labels_);
  const Tensor dl = dloss.to(at::kFloat).contiguous();
  Tensor dlogits = at::empty({B, S, V}, logits.options());
  check(tp_cross_entropy_bwd(logits.data_ptr(), (const int64_t*)labels.data_ptr(), (const float*)lse.data_ptr(), (const float*)lc.data_ptr(),
                             (const float*)dl.data_ptr(), dlogits.data_ptr(), (int)B, (int)S, (int)V, logits.stride(0), logits.stride(1),
                             labels.stride(0), dlogits.stride(0), dlogits.stride(1), (int)ignore_index, dtype_code(logits.scalar_type()),
                             stream_of(dev)), "tp_cross_entropy_bwd");
  return dlogits;
}
struct CrossEntropyNode : OpNode {
  int64_t ignore_index;
  std::string name() const override { return "TprimeCrossEntropyBackward"; }
  variable_list bwd(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    return {op_cross_entropy_bwd()(g[0], get(0), get(1), get(2), get(3), ignore_index)};
  }
};
T3 cross_entropy_fwd_autograd(const Tensor& logits, const Tensor& labels, int64_t ignore_index, bool scored_only) {
  auto node = make_node<CrossEntropyNode>(logits);
  T3 r = [&] { at::AutoDispatchBelowADInplaceOrView below; return op_cross_entropy_fwd()(logits, labels, ignore_index, scored_only); }();
  if (node) {
    torch::autograd::set_history(std::get<0>(r), node);
    node->keep(logits); node->keep(labels); node->keep(std::get<1>(r)); node->keep(std::get<2>(r));
    node->ignore_index = ignore_index;
  }
  return r;
}

// ---- projections -------------------------------------------------------------------------------------------------
// One input through one to three nn.Linear weights (no bias): tp_linears where the products are small, at::linear where
// they are not, or where anything but plain eager tensors is involved.
//
// These calls do not go through the dispatcher: nothing that acts there (dispatch modes, transforms, autocast, tensors with
// __torch_dispatch__) may be waiting for them.  What acts on Python calls (__torch_function__) is asked for in linear.py
// and blocks.py, before a tensor becomes a C++ argument.
bool plain_eager(const Tensor& t) {
  static const c10::DispatchKeySet usual({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
  const c10::DispatchKeySet on = c10::impl::tls_local_dispatch_key_set().included_;
  return (on - usual).empty() && !at::autocast::is_autocast_enabled(at::kCUDA) && t.is_cuda() && !t.unsafeGetTensorImpl()->is_python_dispatch() &&
         t.layout() == at::kStrided && !torch::autograd::isFwGradDefined(t);
}

// The native nodes below have no second derivative.  A backward that records a graph (create_graph) gets its gradients all
// the same; only differentiating through them raises, as for the operators' own backwards.
struct NoDerivative : torch::autograd::Node {
  const char* what;
  std::string name() const override { return "TprimeNoDerivative"; }
  variable_list apply(variable_list&&) override { TORCH_CHECK_NOT_IMPLEMENTED(false, "derivative for the backward of ", what, " is not implemented"); }
};
void end_of_graph(const char* what, const variable_list& grads, const torch::autograd::Node& from, variable_list& outs) {
  if (!at::GradMode::is_enabled()) return;
  std::shared_ptr<NoDerivative> n(new NoDerivative(), torch::autograd::deleteNode);
  n->what = what;
  torch::autograd::edge_list edges = from.next_edges();
  for (const auto& g : grads) edges.push_back(g.defined() ? torch::autograd::impl::gradient_edge(g) : torch::autograd::Edge());
  n->set_next_edges(std::move(edges));
  for (auto& o : outs)
    if (o.defined() && !o.requires_grad()) torch::autograd::set_history(o, n);  // (two inputs may share one gradient)
}
// The line between the two, in multiply-adds of the whole group.  Measured with the host's time, us, tp_linears against
// at::linear, forward | forward + backward:  bf16 512 x 512 through three 512 x 512: 8 : 62 | 83 : 296;  1024 x 1024 through
// three 1024 x 1024 (3.2e9): 17 : 60 | 81 : 291;  1024 x 2048 through 2048 x 2048 (4.3e9): 18 : 20 | 52 : 114.  Beyond that
// the library's larger tiles win on the device.  fp32: 2048 x 512 through three 512 x 512 (1.6e9): 39 : 60 | 126 : 287;
// 3.2e9: 69 : 60 | 208 : 290;  4.3e9: 76 : 62 | 270 : 188.
int64_t lin_max_work(at::ScalarType t) { return t == at::kFloat ? 1ll << 31 : 1ll << 32; }
// tp_linears addresses an operand with 32-bit byte offsets, up to 64 rows past its end
bool lin_reach(int64_t rows, int64_t stride, int64_t esize) { return (rows + 64) * stride * esize < (1ll << 31); }
// The matrices of one product m x k by n x k, its output and that output's gradient, stored row after row, are in reach.
bool lin_fits(int64_t m, int64_t n, int64_t k, int64_t esize) { return lin_reach(m, k, esize) && lin_reach(n, k, esize) && lin_reach(m, n, esize); }
// x as rows that tp_linears reads, for matrices that lin_fits: a copy where the view's rows lie too far apart (the last token
// of every sequence of a batch), on top of each other (the expanded gradient of a sum) or off the 16-byte addresses.
Rows lin_rows(const Tensor& x) {
  Rows r = rows_of(x, true);
  if (at16(r.t) && r.stride >= r.cols && lin_reach(r.rows, r.stride, x.element_size())) return r;
  return {r.t.reshape({r.rows, r.cols}).clone(at::MemoryFormat::Contiguous), r.rows, r.cols, r.cols};
}
bool linears_take(const Tensor& x, const std::vector<Tensor>& ws) {
  const auto t = x.scalar_type();
  if (ws.empty() || ws.size() > 3 || x.dim() < 1 || x.numel() == 0 || !plain_eager(x)) return false;
  if (t != at::kBFloat16 && t != at::kHalf && t != at::kFloat) return false;
  const int64_t k = x.size(-1), m = x.numel() / k, vec = 16 / x.element_size();
  int64_t n = 0;
  for (const auto& w : ws) {
    if (!plain_eager(w) || w.dim() != 2 || w.scalar_type() != t || w.device() != x.device() || w.size(1) != k || !w.is_contiguous()) return false;
    if (w.size(0) == 0 || w.size(0) % vec || !at16(w)) return false;
    if (!lin_fits(m, w.size(0), k, x.element_size())) return false;
    n += w.size(0);
  }
  return k % vec == 0 && m * n * k <= lin_max_work(t);
}

// (x is kept where a weight wants a gradient, the weights where x does: what is not kept may be freed or changed in place)
struct LinearsNode : torch::autograd::Node {
  SavedVariable x;
  std::vector<SavedVariable> ws;
  at::TensorOptions opts;
  std::vector<int64_t> x_sizes, features;
  std::string name() const override { return "TprimeLinearsBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data();
    for (auto& w : ws) w.reset_data();
  }
  variable_list apply(variable_list&& g) override;
};
// c[m, n] = a b over one segment of k; further pairs of operands are added to the sum
tp_linear_problem lin_problem(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t k, bool a_kmajor, bool b_kmajor, int64_t m,
                              int64_t n, void* c) {
  tp_linear_problem p{};
  p.a[0] = a; p.b[0] = b; p.lda[0] = lda; p.ldb[0] = ldb; p.k[0] = (int)k; p.segments = 1;
  p.a_kmajor = a_kmajor; p.b_kmajor = b_kmajor; p.m = (int)m; p.n = (int)n; p.c = c; p.ldc = n;
  return p;
}
void add_segment(tp_linear_problem& p, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t k) {
  const int i = p.segments++;
  p.a[i] = a; p.b[i] = b; p.lda[i] = lda; p.ldb[i] = ldb; p.k[i] = (int)k;
}
variable_list LinearsNode::apply(variable_list&& g) {
  std::lock_guard<std::mutex> lock(mutex_);
  const size_t nw = ws.size();
  variable_list out(1 + nw);
  const bool want_x = task_should_compute_output(0);
  const auto want_w = [&](size_t i) { return g[i].defined() && task_should_compute_output(1 + i); };
  bool any_w = false, plain = !at::GradMode::is_enabled();
  for (size_t i = 0; i < nw; i++) {
    any_w = any_w || want_w(i);
    plain = plain && (!g[i].defined() || (plain_eager(g[i]) && g[i].scalar_type() == opts.dtype().toScalarType()));
  }
  const Tensor xt = any_w ? x.unpack() : Tensor();
  std::vector<Tensor> wt(nw);
  for (size_t i = 0; i < nw && want_x; i++) wt[i] = ws[i].unpack();
  if (!plain) {  // a graph of the backward is being recorded, or the gradients are not plain tensors
    for (size_t i = 0; i < nw; i++) {
      if (!g[i].defined()) continue;
      if (want_x) {
        const Tensor d = at::matmul(g[i], wt[i]);
        out[0] = out[0].defined() ? out[0] + d : d;
      }
      if (want_w(i)) out[1 + i] = at::mm(g[i].reshape({-1, g[i].size(-1)}).t(), xt.reshape({-1, xt.size(-1)}));
    }
    return out;
  }
  at::AutoDispatchBelowADInplaceOrView below;
  c10::DeviceGuard guard(opts.device());
  const int64_t k = x_sizes.back();
  std::vector<Rows> gr;  // (keep copies of strided gradients alive until the launch)
  gr.reserve(nw);
  std::array<tp_linear_problem, 4> p;
  int n = 0;
  for (size_t i = 0; i < nw; i++) {
    if (!g[i].defined()) continue;
    gr.push_back(lin_rows(g[i]));
    const Rows& r = gr.back();
    if (!want_x) continue;
    wt[i] = packed16(wt[i]);
    if (n == 0) {
      out[0] = at::empty(x_sizes, opts);
      p[n++] = lin_problem(r.ptr(), r.stride, wt[i].data_ptr(), k, features[i], true, false, r.rows, k, out[0].data_ptr());
    } else {
      add_segment(p[0], r.ptr(), r.stride, wt[i].data_ptr(), k, features[i]);
    }
  }
  const optional<Rows> xr = any_w ? optional<Rows>(lin_rows(xt)) : std::nullopt;
  size_t j = 0;
  for (size_t i = 0; i < nw; i++) {
    if (!g[i].defined()) continue;
    const Rows& r = gr[j++];
    if (!want_w(i)) continue;
    out[1 + i] = at::empty({features[i], k}, opts);
    p[n++] = lin_problem(r.ptr(), r.stride, xr->ptr(), xr->stride, r.rows, false, false, features[i], k, out[1 + i].data_ptr());
  }
  if (n) check(tp_linears(p.data(), n, dtype_code(opts.dtype().toScalarType()), stream_of(opts.device())), "tp_linears");
  return out;
}

std::vector<Tensor> py_linears(const Tensor& x, const std::vector<Tensor>& ws) {
  std::vector<Tensor> out;
  out.reserve(ws.size());
  if (!linears_take(x, ws)) {
    for (const auto& w : ws) out.push_back(at::linear(x, w));
    return out;
  }
  std::shared_ptr<LinearsNode> node;
  bool req = at::GradMode::is_enabled() && x.requires_grad();
  for (const auto& w : ws) req = req || (at::GradMode::is_enabled() && w.requires_grad());
  if (req) {
    node = std::shared_ptr<LinearsNode>(new LinearsNode(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges{torch::autograd::impl::gradient_edge(x)};
    for (const auto& w : ws) edges.push_back(torch::autograd::impl::gradient_edge(w));
    node->set_next_edges(std::move(edges));
  }
  {
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(x.device());
    const Rows xr = lin_rows(x);
    std::array<tp_linear_problem, 4> p;
    auto sizes = x.sizes().vec();
    for (size_t i = 0; i < ws.size(); i++) {
      sizes.back() = ws[i].size(0);
      out.push_back(at::empty(sizes, x.options()));
      p[i] = lin_problem(xr.ptr(), xr.stride, ws[i].data_ptr(), xr.cols, xr.cols, true, true, xr.rows, ws[i].size(0), out[i].data_ptr());
    }
    check(tp_linears(p.data(), (int)ws.size(), dtype_code(x.scalar_type()), stream_of(x.device())), "tp_linears");
  }
  if (req) {
    bool any_w = false;
    for (const auto& w : ws) any_w = any_w || w.requires_grad();
    if (any_w) node->x = SavedVariable(x, false);
    node->ws.resize(ws.size());
    node->opts = x.options();
    node->x_sizes = x.sizes().vec();
    for (size_t i = 0; i < ws.size(); i++) {
      if (x.requires_grad()) node->ws[i] = SavedVariable(ws[i], false);
      node->features.push_back(ws[i].size(0));
      torch::autograd::set_history(out[i], node);
    }
  }
  return out;
}

// ---- a decoder layer ---------------------------------------------------------------------------------------------
// The Llama decoder layer with its residual adds deferred (blocks.LlamaDecoderLayer.forward_deferred) as one call and one
// autograd node, for layers whose projections are small (linears_take): norm, q / k / v, rotary, attention, output
// projection, add + norm, gate / up, SwiGLU, down, the same kernels in the same order with the same roundings as the
// modules, so the results are theirs bit for bit.  A layer of that size is 21 launches of 3 to 12 us; taken module by
// module the host spent 30 us per launch on them (Python, one autograd node and its edges per operator, views, a tensor
// per intermediate).  Intermediates lie in one allocation, the rotary runs in place, the backward's in another.
struct LayerShape { int64_t B, S, H, Hq, Hkv, D, I, rows; int dtype; bool causal, residual; double eps1, eps2; };
enum LayerParam { LP_N1, LP_Q, LP_K, LP_V, LP_O, LP_N2, LP_G, LP_U, LP_D, LP_COUNT };

// offsets of the forward's intermediates in one buffer
struct LayerBuf {
  size_t h, n1, q, k, v, attn, n2, gate, up, act, rstd1, rstd2, lse, bytes;
  explicit LayerBuf(const LayerShape& s) {
    const size_t e = s.dtype == TP_F32 ? 4 : 2;
    size_t at = 0;
    const auto take = [&](size_t n) { const size_t o = at; at += (n + 255) / 256 * 256; return o; };
    h = take(s.residual ? s.rows * s.H * e : 0);
    n1 = take(s.rows * s.H * e);
    q = take(s.rows * s.Hq * s.D * e); k = take(s.rows * s.Hkv * s.D * e); v = take(s.rows * s.Hkv * s.D * e);
    attn = take(s.rows * s.Hq * s.D * e);
    n2 = take(s.rows * s.H * e);
    gate = take(s.rows * s.I * e); up = take(s.rows * s.I * e); act = take(s.rows * s.I * e);
    rstd1 = take(s.rows * 4); rstd2 = take(s.rows * 4); lse = take(s.rows * s.Hq * 4);
    bytes = at;
  }
};
// (batch, head, seq) strides of heads side by side in a row
Strides3 head_strides(const LayerShape& s, int64_t heads) { return {s.S * heads * s.D, s.D, heads * s.D}; }
// cos / sin rows: batch stride (0: one table for all batches)
int64_t table_stride(const Tensor& cos, const LayerShape& s) { return cos.size(0) == s.B && s.B > 1 ? cos.stride(0) : 0; }

void layer_rope(const LayerShape& s, void* q, void* k, const Tensor& cos, const Tensor& sin, bool backward, void* st) {
  const Strides3 qs = head_strides(s, s.Hq), ks = head_strides(s, s.Hkv);
  check(tp_rope_apply(q, k, cos.data_ptr(), sin.data_ptr(), nullptr, q, k, (int)s.B, (int)s.Hq, (int)s.Hkv, (int)s.S, (int)s.D, qs.data(),
                      ks.data(), qs.data(), ks.data(), table_stride(cos, s), cos.stride(1), 0, 0, 0, (int)backward, s.dtype, st), "tp_rope_apply");
}

// Which gradients a layer's backward forms on its way down, for what is asked for: of the layer's input; of the first
// norm's output; through attention and rotary; of h, the residual after the attention; of the second norm's output; of gate
// and up.  With the lower parameters frozen and an input without a gradient the way ends where the modules' would: an MLP
// that is tuned alone runs neither the attention's backward nor any product below it, and keeps nothing for them.
struct LayerWants {
  bool in, n1, attn, h, n2, mlp;
  template <typename F>
  LayerWants(bool input, F param) {
    in = input;
    n1 = in || param(LP_N1);
    attn = n1 || param(LP_Q) || param(LP_K) || param(LP_V);
    h = attn || param(LP_O);
    n2 = h || param(LP_N2);
    mlp = n2 || param(LP_G) || param(LP_U);
  }
  bool weight(int i) const {
    switch (i) {
      case LP_D: return mlp;
      case LP_G: case LP_U: case LP_N2: return n2;
      case LP_O: return attn;
      default: return n1;
    }
  }
};

struct LayerNode : torch::autograd::Node {
  LayerShape s;
  at::ScalarType scalar;
  SavedVariable x, buf, h2, cos, sin;
  std::vector<SavedVariable> params;
  std::string name() const override { return "TprimeLlamaLayerBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* v : {&x, &buf, &h2, &cos, &sin}) v->reset_data();
    for (auto& p : params) p.reset_data();
  }
  variable_list apply(variable_list&& g) override;
};

variable_list LayerNode::apply(variable_list&& g) {
  std::lock_guard<std::mutex> lock(mutex_);
  variable_list out(2 + LP_COUNT);  // x, residual, the parameters
  if (!g[0].defined() && !g[1].defined()) return out;
  const auto need = [&](int i) { return task_should_compute_output(2 + i); };
  const LayerWants want(task_should_compute_output(0) || task_should_compute_output(1), need);
  const Tensor B = packed16(buf.unpack());
  std::array<Tensor, LP_COUNT> w;
  for (int i = 0; i < LP_COUNT; i++)
    if (want.weight(i)) w[i] = packed16(params[i].unpack());
  Tensor H2, C, Sn, X;
  if (want.n2) H2 = packed16(h2.unpack(shared_from_this()));
  if (want.attn) { C = packed16(cos.unpack()); Sn = packed16(sin.unpack()); }
  if (want.n1 && !s.residual) X = packed16(x.unpack());
  at::AutoDispatchBelowADInplaceOrView below;
  c10::DeviceGuard guard(B.device());
  void* st = stream_of(B.device());
  const LayerBuf f(s);
  char* base = (char*)B.data_ptr();
  const int64_t R = s.rows, NQ = s.Hq * s.D, NK = s.Hkv * s.D;
  const size_t e = s.dtype == TP_F32 ? 4 : 2;
  const auto opts = B.options().dtype(scalar);
  const std::array<int64_t, 3> hidden{s.B, s.S, s.H};
  const auto grad_in = [&](const Tensor& t) { return t.defined() ? packed16(t.to(scalar)) : at::zeros(hidden, opts); };
  const Tensor go = grad_in(g[0]);
  const auto grad_of = [&](int i) {
    const int64_t n[] = {s.H, NQ, NK, NK, s.H, s.H, s.I, s.I, s.H}, k[] = {0, s.H, s.H, s.H, NQ, 0, s.H, s.H, s.I};
    return out[2 + i] = k[i] ? at::empty({n[i], k[i]}, opts) : at::empty({n[i]}, opts);
  };
  // scratch
  tp_attn_bwd_problem ab{};
  ab.B = (int)s.B; ab.Hq = (int)s.Hq; ab.Hkv = (int)s.Hkv; ab.Sq = ab.Skv = (int)s.S; ab.Dqk = ab.Dv = (int)s.D;
  ab.causal = s.causal; ab.window_left = ab.window_right = -1; ab.dtype = s.dtype; ab.sm_scale = (float)(1.0 / std::sqrt((double)s.D));
  tp_attn_bwd_plan plan;
  ab.parts_bytes = want.attn ? tp_attn_bwd_make_plan(&ab, &plan) : 0;
  size_t at = 0;
  const auto take = [&](bool used, size_t n) { const size_t o = at; at += used ? (n + 255) / 256 * 256 : 0; return o; };
  const size_t o_act = take(want.mlp, R * s.I * e), o_dg = take(want.mlp, R * s.I * e), o_du = take(want.mlp, R * s.I * e);
  const size_t o_dn = take(want.n2, R * s.H * e), o_ds = take(want.n2, R * s.H * e);
  const size_t o_da = take(want.attn, R * NQ * e), o_dq = take(want.attn, R * NQ * e), o_dk = take(want.attn, R * NK * e), o_dv = take(want.attn, R * NK * e);
  const size_t o_ws = take(want.attn, tp_attn_bwd_workspace_bytes((int)s.B, (int)s.Hq, (int)s.S));
  const size_t o_norm = take(want.n2, tp_rmsnorm_bwd_workspace_bytes(R, (int)s.H)), o_dw = take(want.n2, s.H * e), o_parts = take(want.attn, ab.parts_bytes);
  const Tensor scratch = at::empty({(int64_t)at}, opts.dtype(at::kByte));
  char* t = (char*)scratch.data_ptr();
  std::array<tp_linear_problem, 4> p;
  int n = 0;
  const auto wgrad = [&](int i, const void* gr, int64_t nf, const void* in, int64_t k) {
    if (need(i)) p[n++] = lin_problem(gr, nf, in, k, R, false, false, nf, k, grad_of(i).data_ptr());
  };
  const auto run = [&]() { if (n) check(tp_linears(p.data(), n, s.dtype, st), "tp_linears"); n = 0; };
  // down projection
  if (want.mlp) p[n++] = lin_problem(go.data_ptr(), s.H, w[LP_D].data_ptr(), s.I, s.H, true, false, R, s.I, t + o_act);
  wgrad(LP_D, go.data_ptr(), s.H, base + f.act, s.I);
  run();
  // gate, up
  if (want.mlp)
    check(tp_swiglu_bwd(t + o_act, base + f.gate, base + f.up, t + o_dg, t + o_du, R, (int)s.I, s.I, s.I, s.I, s.I, s.I, s.dtype, st), "tp_swiglu_bwd");
  if (want.n2) {
    p[n] = lin_problem(t + o_dg, s.I, w[LP_G].data_ptr(), s.H, s.I, true, false, R, s.H, t + o_dn);
    add_segment(p[n++], t + o_du, s.I, w[LP_U].data_ptr(), s.H, s.I);
  }
  wgrad(LP_G, t + o_dg, s.I, base + f.n2, s.H);
  wgrad(LP_U, t + o_du, s.I, base + f.n2, s.H);
  run();
  // norm 2 and the residual's gradient
  const auto norm_bwd = [&](int i, const void* dy, const void* dh, const void* hh, size_t rstd, void* dx) {
    void* dw = need(i) ? grad_of(i).data_ptr() : t + o_dw;
    check(tp_add_rmsnorm_bwd(dy, dh, hh, w[i].data_ptr(), (const float*)(base + rstd), dx, dw, (float*)(t + o_norm), R, (int)s.H, s.H, s.H, s.H, s.H,
                             s.dtype, s.dtype, st), "tp_add_rmsnorm_bwd");
  };
  if (want.n2) {
    const Tensor gh = grad_in(g[1]);
    norm_bwd(LP_N2, t + o_dn, gh.data_ptr(), H2.data_ptr(), f.rstd2, t + o_ds);
  }
  // output projection
  if (want.attn) p[n++] = lin_problem(t + o_ds, s.H, w[LP_O].data_ptr(), NQ, s.H, true, false, R, NQ, t + o_da);
  wgrad(LP_O, t + o_ds, s.H, base + f.attn, NQ);
  run();
  if (want.attn) {  // attention, rotary
    ab.dout = t + o_da; ab.q = base + f.q; ab.k = base + f.k; ab.v = base + f.v; ab.out = base + f.attn; ab.lse = (const float*)(base + f.lse);
    ab.dq = t + o_dq; ab.dk = t + o_dk; ab.dv = t + o_dv; ab.ws = (float*)(t + o_ws);
    ab.parts = ab.parts_bytes ? t + o_parts : nullptr;
    const Strides3 qs = head_strides(s, s.Hq), ks = head_strides(s, s.Hkv);
    for (int i = 0; i < 3; i++) {
      ab.do_strides[i] = ab.q_strides[i] = ab.o_strides[i] = ab.dq_strides[i] = qs[i];
      ab.k_strides[i] = ab.v_strides[i] = ab.dk_strides[i] = ab.dv_strides[i] = ks[i];
    }
    check(tp_attn_bwd_run_planned(&ab, &plan, st, nullptr), "tp_attn_bwd_run");
    layer_rope(s, t + o_dq, t + o_dk, C, Sn, true, st);
  }
  // q, k, v
  if (want.n1) {
    p[n] = lin_problem(t + o_dq, NQ, w[LP_Q].data_ptr(), s.H, NQ, true, false, R, s.H, t + o_dn);
    add_segment(p[n], t + o_dk, NK, w[LP_K].data_ptr(), s.H, NK);
    add_segment(p[n++], t + o_dv, NK, w[LP_V].data_ptr(), s.H, NK);
  }
  wgrad(LP_Q, t + o_dq, NQ, base + f.n1, s.H);
  wgrad(LP_K, t + o_dk, NK, base + f.n1, s.H);
  wgrad(LP_V, t + o_dv, NK, base + f.n1, s.H);
  run();
  // norm 1; x and the residual get the same gradient
  if (want.n1) {
    const Tensor dx = at::empty(hidden, opts);
    norm_bwd(LP_N1, t + o_dn, t + o_ds, s.residual ? base + f.h : (char*)X.data_ptr(), f.rstd1, dx.data_ptr());
    if (want.in) out[0] = dx;
    if (want.in && s.residual) out[1] = dx;
  }
  end_of_graph("a decoder layer", g, *this, out);
  return out;
}

// (mlp output, residual), or nothing where this layer is one for the modules
std::vector<Tensor> py_llama_layer(const Tensor& x, OptTensor residual_, const std::vector<Tensor>& w, const Tensor& cos, const Tensor& sin,
                                   int64_t Hq, int64_t Hkv, double eps1, double eps2, bool causal) {
  const Tensor& residual = val(residual_);
  if (w.size() != LP_COUNT || x.dim() != 3 || !x.is_contiguous() || x.numel() == 0) return {};
  const auto dt = x.scalar_type();
  LayerShape s;
  s.B = x.size(0); s.S = x.size(1); s.H = x.size(2); s.Hq = Hq; s.Hkv = Hkv; s.rows = s.B * s.S; s.causal = causal; s.eps1 = eps1; s.eps2 = eps2;
  s.residual = residual.defined();
  const auto rows_ok = [&](const Tensor& t) { return t.dim() == 1 && t.size(0) == s.H && t.scalar_type() == dt && t.is_contiguous() && plain_eager(t) && t.device() == x.device(); };
  if (!linears_take(x, {w[LP_Q], w[LP_K], w[LP_V]}) || !linears_take(x, {w[LP_G], w[LP_U]}) || !rows_ok(w[LP_N1]) || !rows_ok(w[LP_N2])) return {};
  if (s.residual && (residual.sizes() != x.sizes() || residual.scalar_type() != dt || !residual.is_contiguous() || !plain_eager(residual) || residual.device() != x.device())) return {};
  s.dtype = dtype_code(dt);
  s.I = w[LP_G].size(0);
  const int64_t NQ = w[LP_Q].size(0), NK = w[LP_K].size(0), vec = 16 / x.element_size();
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || NQ % Hq) return {};
  s.D = NQ / Hq;
  if ((s.D != 64 && s.D != 128) || NK != Hkv * s.D || w[LP_V].size(0) != NK || w[LP_U].size(0) != s.I || s.H % vec) return {};
  // the two projections whose input is made here: shape, layout, and the same line on size
  const auto lin_ok = [&](const Tensor& t, int64_t n, int64_t k) {
    return t.dim() == 2 && t.size(0) == n && t.size(1) == k && t.scalar_type() == dt && t.is_contiguous() && plain_eager(t) && t.device() == x.device() &&
           at16(t) && s.rows * n * k <= lin_max_work(dt) && lin_fits(s.rows, n, k, x.element_size());
  };
  if (!lin_ok(w[LP_O], s.H, NQ) || !lin_ok(w[LP_D], s.H, s.I)) return {};
  for (const Tensor* t : {&cos, &sin})
    if (t->dim() != 3 || (t->size(0) != 1 && t->size(0) != s.B) || t->size(1) != s.S || t->size(2) != s.D || t->scalar_type() != dt ||
        !t->is_contiguous() || !plain_eager(*t) || t->device() != x.device() || t->requires_grad()) return {};
  for (const Tensor* t : {&x, &residual})
    if (t->defined() && !at16(*t)) return {};

  std::shared_ptr<LayerNode> node;
  if (at::GradMode::is_enabled()) {
    bool req = x.requires_grad() || (s.residual && residual.requires_grad());
    for (const auto& t : w) req = req || t.requires_grad();
    if (req) {
      node = std::shared_ptr<LayerNode>(new LayerNode(), torch::autograd::deleteNode);
      torch::autograd::edge_list edges;
      edges.reserve(2 + LP_COUNT);
      edges.push_back(torch::autograd::impl::gradient_edge(x));
      edges.push_back(s.residual ? torch::autograd::impl::gradient_edge(residual) : torch::autograd::Edge());
      for (const auto& t : w) edges.push_back(torch::autograd::impl::gradient_edge(t));
      node->set_next_edges(std::move(edges));
    }
  }
  Tensor out, h2, buf;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(x.device());
    void* st = stream_of(x.device());
    const LayerBuf f(s);
    buf = at::empty({(int64_t)f.bytes}, x.options().dtype(at::kByte));
    out = at::empty(x.sizes(), x.options());
    h2 = at::empty(x.sizes(), x.options());
    char* b = (char*)buf.data_ptr();
    const int64_t R = s.rows;
    std::array<tp_linear_problem, 4> p;
    const auto lin = [&](int i, const void* in, int64_t k, int wi, void* c) { p[i] = lin_problem(in, k, w[wi].data_ptr(), k, k, true, true, R, w[wi].size(0), c); };
    const auto run = [&](int n) { check(tp_linears(p.data(), n, s.dtype, st), "tp_linears"); };
    if (s.residual)
      check(tp_add_rmsnorm_fwd(x.data_ptr(), residual.data_ptr(), w[LP_N1].data_ptr(), b + f.h, b + f.n1, (float*)(b + f.rstd1), R, (int)s.H, s.H, s.H,
                               s.H, s.H, (float)eps1, s.dtype, s.dtype, st), "tp_add_rmsnorm_fwd");
    else
      check(tp_rmsnorm_fwd(x.data_ptr(), w[LP_N1].data_ptr(), b + f.n1, (float*)(b + f.rstd1), R, (int)s.H, s.H, s.H, (float)eps1, s.dtype, s.dtype, st),
            "tp_rmsnorm_fwd");
    lin(0, b + f.n1, s.H, LP_Q, b + f.q); lin(1, b + f.n1, s.H, LP_K, b + f.k); lin(2, b + f.n1, s.H, LP_V, b + f.v);
    run(3);
    layer_rope(s, b + f.q, b + f.k, cos, sin, false, st);
    const Strides3 qs = head_strides(s, s.Hq), ks = head_strides(s, s.Hkv);
    check(tp_attn_fwd(b + f.q, b + f.k, b + f.v, nullptr, b + f.attn, (float*)(b + f.lse), (int)s.B, (int)s.Hq, (int)s.Hkv, (int)s.S, (int)s.S, (int)s.D,
                      (int)s.D, qs.data(), ks.data(), ks.data(), qs.data(), (float)(1.0 / std::sqrt((double)s.D)), (int)causal, s.dtype, st), "tp_attn_fwd");
    lin(0, b + f.attn, NQ, LP_O, out.data_ptr());  // (the output's memory is free until the last projection)
    run(1);
    const void* h = s.residual ? (const void*)(b + f.h) : x.data_ptr();
    check(tp_add_rmsnorm_fwd(out.data_ptr(), h, w[LP_N2].data_ptr(), h2.data_ptr(), b + f.n2, (float*)(b + f.rstd2), R, (int)s.H, s.H, s.H, s.H, s.H,
                             (float)eps2, s.dtype, s.dtype, st), "tp_add_rmsnorm_fwd");
    lin(0, b + f.n2, s.H, LP_G, b + f.gate); lin(1, b + f.n2, s.H, LP_U, b + f.up);
    run(2);
    check(tp_swiglu_fwd(b + f.gate, b + f.up, b + f.act, R, (int)s.I, s.I, s.I, s.I, s.dtype, st), "tp_swiglu_fwd");
    lin(0, b + f.act, s.I, LP_D, out.data_ptr());
    run(1);
  }
  if (node) {
    node->s = s;
    node->scalar = dt;
    torch::autograd::set_history(out, node);
    torch::autograd::set_history(h2, node);
    const LayerWants want(x.requires_grad() || (s.residual && residual.requires_grad()), [&](int i) { return w[i].requires_grad(); });
    node->buf = SavedVariable(buf, false);
    if (want.n2) node->h2 = SavedVariable(h2, true);
    if (want.attn) { node->cos = SavedVariable(cos, false); node->sin = SavedVariable(sin, false); }
    if (want.n1 && !s.residual) node->x = SavedVariable(x, false);
    node->params.resize(LP_COUNT);
    for (int i = 0; i < LP_COUNT; i++)
      if (want.weight(i)) node->params[i] = SavedVariable(w[i], false);
  }
  return {out, h2};
}

// ---- the two ends of a small model ---------------------------------------------------------------------------------
// Embedding rows: the library's where the vocabulary or the batch is not small, or anything but plain tensors is involved.
struct EmbeddingNode : torch::autograd::Node {
  SavedVariable ids;
  int64_t vocab, hidden;
  at::TensorOptions opts;
  std::string name() const override { return "TprimeEmbeddingBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    ids.reset_data();
  }
  variable_list apply(variable_list&& g) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!g[0].defined()) return {Tensor()};
    const Tensor kept = ids.unpack();
    if (at::GradMode::is_enabled() || !plain_eager(g[0])) return {at::embedding_dense_backward(g[0], kept, vocab, -1, false)};
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(kept.device());
    const Tensor dy = packed16(g[0].to(opts.dtype().toScalarType())), i = packed16(kept);
    Tensor dt = at::empty({vocab, hidden}, opts);
    check(tp_embedding_bwd(dy.data_ptr(), (const int64_t*)i.data_ptr(), dt.data_ptr(), i.numel(), (int)vocab, (int)hidden,
                           dtype_code(dt.scalar_type()), stream_of(i.device())), "tp_embedding_bwd");
    return {dt};
  }
};
Tensor py_embedding(const Tensor& ids, const Tensor& table) {
  const auto t = table.scalar_type();
  const bool small = plain_eager(table) && plain_eager(ids) && ids.device() == table.device() && table.dim() == 2 && table.is_contiguous() &&
                     (t == at::kBFloat16 || t == at::kHalf || t == at::kFloat) && ids.scalar_type() == at::kLong && ids.numel() > 0 &&
                     table.size(0) > 0 && table.size(1) > 0 && at16(table) && table.size(1) % 2 == 0 && table.size(0) * ids.numel() <= (1ll << 24) &&
                     ids.numel() * table.size(1) <= (1ll << 24);
  if (!small) return at::embedding(table, ids);
  auto node = make_node<EmbeddingNode>(table);
  Tensor out;
  const Tensor i = ids.contiguous();
  {
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(table.device());
    auto sizes = ids.sizes().vec();
    sizes.push_back(table.size(1));
    out = at::empty(sizes, table.options());
    check(tp_embedding_fwd(table.data_ptr(), (const int64_t*)i.data_ptr(), out.data_ptr(), i.numel(), (int)table.size(0), (int)table.size(1),
                           dtype_code(t), stream_of(table.device())), "tp_embedding_fwd");
  }
  if (node) {
    torch::autograd::set_history(out, node);
    node->ids = SavedVariable(i, false);
    node->vocab = table.size(0);
    node->hidden = table.size(1);
    node->opts = table.options();
  }
  return out;
}

// final add + norm, lm_head, .float(): fp32 logits rounded through the model's type.  An undefined tensor where the
// projection is one for the library.
struct HeadNode : torch::autograd::Node {
  SavedVariable h, n, rstd, norm_w, lm_w;
  std::vector<int64_t> sizes;  // of the hidden states
  at::TensorOptions opts;
  std::string name() const override { return "TprimeLlamaHeadBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* v : {&h, &n, &rstd, &norm_w, &lm_w}) v->reset_data();
  }
  variable_list apply(variable_list&& g) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list out(4);  // x, residual, norm weight, lm_head weight
    if (!g[0].defined()) return out;
    const bool dx = task_should_compute_output(0) || task_should_compute_output(1) || task_should_compute_output(2), dw = task_should_compute_output(3);
    Tensor H, N, R, nw, lw;
    if (dx) { H = packed16(h.unpack()); R = packed16(rstd.unpack()); nw = packed16(norm_w.unpack()); lw = packed16(lm_w.unpack()); }
    if (dw) N = packed16(n.unpack());
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(opts.device());
    void* st = stream_of(opts.device());
    const int64_t k = sizes.back(), V = g[0].size(-1), rows = g[0].numel() / V;
    const auto type = opts.dtype().toScalarType();
    const int code = dtype_code(type);
    const Tensor go = packed16(g[0].to(type));
    Tensor dn;
    std::array<tp_linear_problem, 2> p;
    int c = 0;
    if (dx) {
      dn = at::empty(sizes, opts);
      p[c++] = lin_problem(go.data_ptr(), V, lw.data_ptr(), k, V, true, false, rows, k, dn.data_ptr());
    }
    if (dw) {
      out[3] = at::empty({V, k}, opts);
      p[c++] = lin_problem(go.data_ptr(), V, N.data_ptr(), k, rows, false, false, V, k, out[3].data_ptr());
    }
    if (c) check(tp_linears(p.data(), c, code, st), "tp_linears");
    if (dx) {
      const Tensor ws = empty_f32({(int64_t)tp_rmsnorm_bwd_workspace_bytes(rows, (int)k) / 4}, H);
      out[0] = at::empty(sizes, opts);
      out[2] = at::empty({k}, opts);
      check(tp_rmsnorm_bwd(dn.data_ptr(), H.data_ptr(), nw.data_ptr(), (const float*)R.data_ptr(), out[0].data_ptr(), out[2].data_ptr(),
                           (float*)ws.data_ptr(), rows, (int)k, k, k, k, code, code, st), "tp_rmsnorm_bwd");
      out[1] = out[0];
    }
    end_of_graph("a model head", g, *this, out);
    return out;
  }
};
std::optional<Tensor> py_llama_head(const Tensor& x, const Tensor& residual, const Tensor& norm_w, double eps, const Tensor& lm_w) {
  const auto dt = x.scalar_type();
  if (!linears_take(x, {lm_w}) || !x.is_contiguous() || !residual.is_contiguous() || residual.sizes() != x.sizes() || residual.scalar_type() != dt ||
      !plain_eager(residual) || residual.device() != x.device() || norm_w.dim() != 1 || norm_w.size(0) != x.size(-1) || norm_w.scalar_type() != dt ||
      !norm_w.is_contiguous() || !plain_eager(norm_w) || norm_w.device() != x.device()) return std::nullopt;
  for (const Tensor* t : {&x, &residual})
    if (!at16(*t)) return std::nullopt;
  auto node = make_node<HeadNode>(x, residual, norm_w, lm_w);
  Tensor h, n, rstd, logits;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(x.device());
    void* st = stream_of(x.device());
    const int64_t k = x.size(-1), rows = x.numel() / k, V = lm_w.size(0);
    const int code = dtype_code(dt);
    h = at::empty(x.sizes(), x.options());
    n = at::empty(x.sizes(), x.options());
    rstd = empty_f32({rows}, x);
    auto sizes = x.sizes().vec();
    sizes.back() = V;
    logits = empty_f32(sizes, x);
    check(tp_add_rmsnorm_fwd(x.data_ptr(), residual.data_ptr(), norm_w.data_ptr(), h.data_ptr(), n.data_ptr(), (float*)rstd.data_ptr(), rows, (int)k,
                             k, k, k, k, (float)eps, code, code, st), "tp_add_rmsnorm_fwd");
    tp_linear_problem p = lin_problem(n.data_ptr(), k, lm_w.data_ptr(), k, k, true, true, rows, V, logits.data_ptr());
    p.c_float = 1;
    check(tp_linears(&p, 1, code, st), "tp_linears");
  }
  if (node) {
    torch::autograd::set_history(logits, node);
    node->sizes = x.sizes().vec();
    node->opts = x.options();
    if (x.requires_grad() || residual.requires_grad() || norm_w.requires_grad()) {
      node->h = SavedVariable(h, false);
      node->rstd = SavedVariable(rstd, false);
      node->norm_w = SavedVariable(norm_w, false);
      node->lm_w = SavedVariable(lm_w, false);
    }
    if (lm_w.requires_grad()) node->n = SavedVariable(n, false);
  }
  return logits;
}

// ---- Python entry points -----------------------------------------------------------------------------------------
// What the Python functions of ops.py call: the GPU check with its own message, then the operator.
Tensor py_rmsnorm(const Tensor& x, const Tensor& w, double eps) { require_gpu(x, w); return std::get<0>(op_rmsnorm_fwd()(x, w, eps)); }
T2 py_add_rmsnorm(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  require_gpu(x, r, w);
  T3 o = op_add_rmsnorm_fwd()(x, r, w, eps);
  return {std::get<0>(o), std::get<1>(o)};
}
T2 py_rope_table(const Tensor& f, const Tensor& p, double scaling, const Tensor& like) {
  require_gpu(f, p, like);
  return op_rope_table()(f, p, scaling, like.scalar_type());
}
T2 py_rope_apply(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, OptTensor pos, int64_t interleaved) {
  require_gpu(q, k, cos, sin, pos);
  return op_rope_apply()(q, k, cos, sin, pos, interleaved, false);
}
Tensor py_attention(const Tensor& q, const Tensor& k, const Tensor& v, OptTensor seg, double sm_scale, bool causal) {
  require_gpu(q, k, v, seg);
  return std::get<0>(op_attn_fwd()(q, k, v, seg, sm_scale, causal));
}
Tensor py_attention_masked(const Tensor& q, const Tensor& k, const Tensor& v, OptTensor seg, OptTensor qpos, double sm_scale, bool causal,
                           int64_t causal_offset, int64_t window_left, int64_t window_right, double soft_cap, OptTensor bias) {
  require_gpu(q, k, v, seg, qpos, bias);
  return std::get<0>(op_attn_fwd_masked()(q, k, v, seg, qpos, sm_scale, causal, causal_offset, window_left, window_right, soft_cap, bias));
}
Tensor py_attention_pairs(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, double sm_scale, bool causal_padded) {
  require_gpu(q, k, v, mask);
  return std::get<0>(op_attn_fwd_pairs()(q, k, v, mask, sm_scale, causal_padded));
}
// What a (1|B, 1, Sq, Skv) mask is: 1 the exact causal mask, 2 one that only drops pairs, 3 one that is causality and
// padding, 0 anything else.  Two short kernels and one synchronisation (for each 65535 masks, as many as their grid takes).
int64_t py_mask_verdict(const Tensor& mask) {
  const c10::Device dev = require_gpu(mask);
  TORCH_CHECK_VALUE(mask.dim() == 4, "expected a 4-D mask");
  if (mask.numel() == 0) return 0;
  c10::DeviceGuard guard(dev);
  at::AutoDispatchBelowADInplaceOrView below;
  constexpr int64_t MOST = 65535;
  const int64_t Sq = mask.size(2), Skv = mask.size(3);
  int other = 0, not_causal = 0, empty_finite = 0, not_padded = 0;
  for (int64_t b = 0; b < mask.size(0); b += MOST) {
    const PairsIn m = prep_pairs(mask.size(0) <= MOST ? mask : mask.slice(0, b, b + MOST), Sq, Skv);
    const Tensor flags = make_pairs(m, Sq, Skv, true, stream_of(dev)).slice(0, 0, 16).cpu();
    const int* f = flags.const_data_ptr<int>();
    other |= f[0]; not_causal |= f[1]; empty_finite |= f[2]; not_padded |= f[3];
  }
  return !not_causal ? 1 : other || empty_finite ? 0 : not_padded ? 2 : 3;
}
Tensor py_l2norm(const Tensor& x, double eps) { return std::get<0>(op_l2norm_fwd()(x, eps)); }
Tensor py_swiglu(const Tensor& g, const Tensor& u) { return op_swiglu_fwd()(g, u); }
Tensor py_cross_entropy(const Tensor& l, const Tensor& y, int64_t ignore) { return std::get<0>(op_cross_entropy_fwd()(l, y, ignore, true)); }

}  // namespace

TORCH_LIBRARY(tprime, m) {
  m.def("rmsnorm_fwd(Tensor x, Tensor weight, float eps) -> (Tensor, Tensor)");
  m.def("rmsnorm_bwd(Tensor dy, Tensor x, Tensor weight, Tensor rstd) -> (Tensor, Tensor)");
  m.def("add_rmsnorm_fwd(Tensor x, Tensor residual, Tensor weight, float eps) -> (Tensor, Tensor, Tensor)");
  m.def("add_rmsnorm_bwd(Tensor dy, Tensor dh, Tensor h, Tensor weight, Tensor rstd) -> (Tensor, Tensor)");
  m.def("rope_table(Tensor inv_freq, Tensor position_ids, float attention_scaling, ScalarType dtype) -> (Tensor, Tensor)");
  m.def("rope_apply(Tensor q, Tensor k, Tensor cos, Tensor sin, Tensor? pos, int interleaved, bool backward) -> (Tensor, Tensor)");
  m.def("attn_fwd(Tensor q, Tensor k, Tensor v, Tensor? seg, float sm_scale, bool causal) -> (Tensor, Tensor)");
  m.def("attn_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor out, Tensor lse, Tensor? seg, float sm_scale, bool causal) "
        "-> (Tensor, Tensor, Tensor)");
  m.def("attn_fwd_masked(Tensor q, Tensor k, Tensor v, Tensor? seg, Tensor? qpos, float sm_scale, bool causal, int causal_offset, "
        "int window_left, int window_right, float soft_cap, Tensor? bias=None) -> (Tensor, Tensor)");
  m.def("attn_bwd_masked(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor out, Tensor lse, Tensor? seg, Tensor? qpos, float sm_scale, "
        "bool causal, int causal_offset, int window_left, int window_right, float soft_cap, Tensor? bias=None) -> (Tensor, Tensor, Tensor)");
  m.def("attn_fwd_pairs(Tensor q, Tensor k, Tensor v, Tensor mask, float sm_scale, bool causal_padded=False) -> (Tensor, Tensor, Tensor)");
  m.def("attn_bwd_pairs(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor out, Tensor lse, Tensor pairs, int mask_batches, float sm_scale, bool causal_padded=False) "
        "-> (Tensor, Tensor, Tensor)");
  m.def("l2norm_fwd(Tensor x, float eps) -> (Tensor, Tensor)");
  m.def("l2norm_bwd(Tensor dy, Tensor x, Tensor rstd) -> Tensor");
  m.def("scale_rows(Tensor x, Tensor scale) -> Tensor");
  m.def("swiglu_fwd(Tensor gate, Tensor up) -> Tensor");
  m.def("swiglu_bwd(Tensor dout, Tensor gate, Tensor up) -> (Tensor, Tensor)");
  m.def("cross_entropy_fwd(Tensor logits, Tensor labels, int ignore_index, bool scored_only=False) -> (Tensor, Tensor, Tensor)");
  m.def("cross_entropy_bwd(Tensor dloss, Tensor logits, Tensor labels, Tensor lse, Tensor loss_and_count, int ignore_index) -> Tensor");
}

TORCH_LIBRARY_IMPL(tprime, CUDA, m) {
  m.impl("rmsnorm_fwd", rmsnorm_fwd_cuda);
  m.impl("rmsnorm_bwd", rmsnorm_bwd_cuda);
  m.impl("add_rmsnorm_fwd", add_rmsnorm_fwd_cuda);
  m.impl("add_rmsnorm_bwd", add_rmsnorm_bwd_cuda);
  m.impl("rope_table", rope_table_cuda);
  m.impl("rope_apply", rope_apply_cuda);
  m.impl("attn_fwd", attn_fwd_cuda);
  m.impl("attn_bwd", attn_bwd_cuda);
  m.impl("attn_fwd_masked", attn_fwd_masked_cuda);
  m.impl("attn_bwd_masked", attn_bwd_masked_cuda);
  m.impl("attn_fwd_pairs", attn_fwd_pairs_cuda);
  m.impl("attn_bwd_pairs", attn_bwd_pairs_cuda);
  m.impl("l2norm_fwd", l2norm_fwd_cuda);
  m.impl("l2norm_bwd", l2norm_bwd_cuda);
  m.impl("scale_rows", scale_rows_cuda);
  m.impl("swiglu_fwd", swiglu_fwd_cuda);
  m.impl("swiglu_bwd", swiglu_bwd_cuda);
  m.impl("cross_entropy_fwd", cross_entropy_fwd_cuda);
  m.impl("cross_entropy_bwd", cross_entropy_bwd_cuda);
}

TORCH_LIBRARY_IMPL(tprime, Autograd, m) {
  m.impl("rmsnorm_fwd", rmsnorm_fwd_autograd);
  m.impl("add_rmsnorm_fwd", add_rmsnorm_fwd_autograd);
  m.impl("rope_apply", rope_apply_autograd);
  m.impl("attn_fwd", attn_fwd_autograd);
  m.impl("attn_fwd_masked", attn_fwd_masked_autograd);
  m.impl("attn_fwd_pairs", attn_fwd_pairs_autograd);
  m.impl("l2norm_fwd", l2norm_fwd_autograd);
  m.impl("scale_rows", scale_rows_autograd);
  m.impl("swiglu_fwd", swiglu_fwd_autograd);
  m.impl("cross_entropy_fwd", cross_entropy_fwd_autograd);
  for (const char* name : {"rope_table", "rmsnorm_bwd", "add_rmsnorm_bwd", "attn_bwd", "attn_bwd_masked", "attn_bwd_pairs", "l2norm_bwd",
                           "swiglu_bwd", "cross_entropy_bwd"})
    m.impl(name, torch::autograd::autogradNotImplementedFallback());
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // Other Python threads run meanwhile: some of these wait for the device (mask_verdict, rope_apply with positions), and any
  // launch or allocation may.
  const py::call_guard<py::gil_scoped_release> no_gil;
  m.def("rmsnorm", &py_rmsnorm, no_gil);
  m.def("add_rmsnorm", &py_add_rmsnorm, no_gil);
  m.def("rope_table", &py_rope_table, no_gil);
  m.def("rope_apply", &py_rope_apply, no_gil);
  m.def("attention", &py_attention, no_gil);
  m.def("attention_masked", &py_attention_masked, no_gil);
  m.def("attention_pairs", &py_attention_pairs, no_gil);
  m.def("mask_verdict", &py_mask_verdict, no_gil);
  m.def("mask_pairs_words", [](int64_t Bm, int64_t Sq, int64_t Skv) { return (int64_t)tp_mask_pairs_bytes((int)Bm, (int)Sq, (int)Skv) / 4; });
  m.def("attention_pairs_fit", [](int64_t Bm, int64_t Sq, int64_t Skv, int64_t Dqk, int64_t Dv) {
    const auto is_int = [](int64_t v) { return v >= 0 && v < (1ll << 31); };
    return is_int(Bm) && is_int(Sq) && is_int(Skv) && is_int(Dqk) && is_int(Dv) && tp_attn_pairs_fit((int)Bm, (int)Sq, (int)Skv, (int)Dqk, (int)Dv) != 0;
  });
  m.def("linears", &py_linears, no_gil);
  m.def("llama_layer", &py_llama_layer, no_gil);
  m.def("llama_head", &py_llama_head, no_gil);
  m.def("embedding", &py_embedding, no_gil);
  m.def("l2norm", &py_l2norm, no_gil);
  m.def("swiglu", &py_swiglu, no_gil);
  m.def("cross_entropy", &py_cross_entropy, no_gil);
}
