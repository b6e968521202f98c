// Host path of the per-call entry points for ordinary eager calls: argument checks, allocations,
// autograd and the C-ABI call in one native call each.
//
// Why: through torch.library's Python ops the host needed ~215 us for a forward and backward of one
// attention layer, ~400 us for RoPE, attention and their backward, ~24 us for a forward without
// gradients and ~60 us for a decode step with its KV update, more than the kernels take at most sizes.
// Measured per call on MI355X: attention forward and backward, B8 H12 N2048 D64, 222 -> 171 us (its
// kernels' time); RoPE + attention with gradients, B4 H12 N2048 D64, 402 -> 147 us; forward, B2 H8
// N1024 D64, 24 -> 13.5 us; decode step with update, 16 sequences, 61 -> 37 us a layer. The forward
// also returns O alone to autograd, so no zero gradients are made for LSE and the workspace.
//
// Every function here takes only the calls whose handling needs nothing but the kernels: exact
// torch.Tensor / Parameter arguments on one GPU, in the types, layouts and shapes the kernels read in
// place, with no dispatch or function mode (torch.set_default_device is one), functorch transform, tracer or
// forward-mode dual number about; with gradients, q, k and v (and RoPE's frequencies) also have to be dense, so
// slices of one projection go the general way there. For any other call it returns None before doing anything, and the Python caller takes its
// general path (the torch.library ops, conversions, error messages), so nothing here raises for a
// malformed argument. The autograd functions save tensors through the ordinary hooks and, where their
// backward meets such a case (create_graph, batched gradients), call the same torch.library ops.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cmath>
#include <limits>
#include <optional>

#include "../../include/sps_attn.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------------------------------------------
// Which calls are taken.
// ---------------------------------------------------------------------------------------------
bool plain_thread() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  const c10::DispatchKeySet modes({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                   c10::DispatchKey::PythonDispatcher, c10::DispatchKey::Tracer,
                                   c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                   c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::PreDispatch,
                                   c10::DispatchKey::TESTING_ONLY_GenericMode});
  return !tls.included_.has_any(modes) && c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0;
}

bool plain_tensor(const Tensor& t) {
  static const c10::DispatchKeySet other(
      {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched, c10::DispatchKey::Functionalize,
       c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(other) &&
         !t.unsafeGetTensorImpl()->is_python_dispatch() && !t._fw_grad(0).defined();
}

// The tensor of an exact torch.Tensor / Parameter object fit for a native call; undefined otherwise.
Tensor plain(py::handle o) {
  if (!THPVariable_CheckExact(o.ptr())) return {};
  const Tensor& t = THPVariable_Unpack(o.ptr());
  return plain_tensor(t) ? t : Tensor();
}

bool fits_int(int64_t x) { return x >= std::numeric_limits<int>::min() && x <= std::numeric_limits<int>::max(); }

std::optional<int> as_int(py::handle o) {
  if (!PyLong_CheckExact(o.ptr())) return std::nullopt;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o.ptr(), &overflow);
  if (overflow || !fits_int(x)) return std::nullopt;
  return (int)x;
}

int float_code(at::ScalarType t) {
  return t == at::kBFloat16 ? SPS_DTYPE_BF16 : t == at::kHalf ? SPS_DTYPE_F16 : t == at::kFloat ? SPS_DTYPE_F32 : -1;
}
int index_code(at::ScalarType t) { return t == at::kLong ? SPS_DTYPE_I64 : t == at::kInt ? SPS_DTYPE_I32 : -1; }

bool decode_head_dim(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }

// Unit last stride and every row start 16-byte aligned.
bool rows16(const Tensor& t) {
  const auto st = t.strides();
  const int64_t el = t.element_size();
  if (st.back() != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return false;
  int64_t bits = 0;
  for (size_t i = 0; i + 1 < st.size(); ++i) bits |= st[i];
  return (bits * el) % 16 == 0;
}

void* stream_of(const Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream());
}

// Raises sps_amd._native.NativeError, as the Python callers do.
void check(const char* fn, int status) {
  if (status == SPS_OK) return;
  char msg[1024];
  sps_last_error(msg, sizeof(msg));
  py::gil_scoped_acquire gil;
  py::object cls = py::module_::import("sps_amd._native").attr("NativeError");
  py::object err = cls(fn, status, std::string(msg));
  PyErr_SetObject(cls.ptr(), err.ptr());
  python_error e;
  e.persist();
  throw e;
}

// ---------------------------------------------------------------------------------------------
// Attention.
// ---------------------------------------------------------------------------------------------
struct AttnParams {
  double sm_scale;
  int family, window, has_pkw, pkw;
};

bool attn_readable(const Tensor& t) { return rows16(t) && t.strides()[2] >= 0; }

struct AttnOut {
  Tensor o, lse, ws;
};

// Dense memory in some order, so that empty_like keeps the strides (and with them the row alignment).
bool dense(const Tensor& t) { return t.is_non_overlapping_and_dense(); }

AttnOut attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& docs, const AttnParams& p,
                     bool keep_layout) {
  RECORD_FUNCTION("sps_amd::attention_fwd", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(q.device());
  const auto s = q.sizes();
  const int b = (int)s[0], h = (int)s[1], n = (int)s[2], d = (int)s[3];
  AttnOut r;
  r.o = at::empty({b, n, h, d}, q.options()).transpose(1, 2);
  r.lse = at::empty({b, h, n}, q.options().dtype(at::kFloat));
  const bool has_docs = docs.defined();
  const size_t bytes = sps_attn_workspace_bytes(p.family, b, h, n, has_docs, keep_layout && has_docs);
  if (bytes) r.ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
  check("sps_attn_fwd",
        sps_attn_fwd(p.family, b, h, n, d, float_code(q.scalar_type()), q.data_ptr(), q.strides().data(), k.data_ptr(),
                     k.strides().data(), v.data_ptr(), v.strides().data(), r.o.data_ptr(), r.o.strides().data(),
                     r.lse.data_ptr<float>(), has_docs ? docs.data_ptr() : nullptr,
                     has_docs ? index_code(docs.scalar_type()) : 0, has_docs ? docs.stride(0) : 0, (float)p.sm_scale,
                     p.window, p.has_pkw, p.pkw, bytes ? r.ws.data_ptr() : nullptr, bytes, stream_of(q)));
  return r;
}

struct AttentionFunction : torch::autograd::Function<AttentionFunction> {
  // Compiled autograd may trace the backward (its tensors are then not plain, so it goes through the
  // registered op); otherwise each call would be a graph break, and an error with fullgraph.
  static constexpr bool is_traceable = true;

  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const std::optional<Tensor>& docs_opt, double sm_scale, int64_t family, int64_t window,
                        bool has_pkw, int64_t pkw) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor docs = docs_opt.value_or(Tensor());
    const AttnParams p{sm_scale, (int)family, (int)window, has_pkw, (int)pkw};
    AttnOut r = attn_forward(q, k, v, docs, p, true);
    if (!docs.defined()) r.ws = Tensor();
    ctx->save_for_backward({q, k, v, r.o, r.lse, docs, r.ws});
    ctx->saved_data["sm_scale"] = sm_scale;
    ctx->saved_data["mask"] = std::vector<int64_t>{family, window, has_pkw, pkw};
    return r.o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4], &docs = saved[5];
    Tensor ws = saved[6];
    const double sm_scale = ctx->saved_data["sm_scale"].toDouble();
    const auto mask = ctx->saved_data["mask"].toIntVector();
    Tensor dout = grads[0];
    if (!dout.defined()) dout = at::zeros_like(o);
    // (Saved-tensor hooks may hand back tensors other than those saved.)
    bool native = !at::GradMode::is_enabled() && plain_thread() && lse.is_contiguous();
    for (const Tensor* t : std::initializer_list<const Tensor*>{&q, &k, &v, &o, &dout})
      native = native && plain_tensor(*t) && t->scalar_type() == q.scalar_type() && t->device() == q.device();
    for (const Tensor* t : std::initializer_list<const Tensor*>{&lse, &docs, &ws})
      native = native && (!t->defined() || (plain_tensor(*t) && t->is_contiguous() && t->device() == q.device()));
    for (const Tensor* t : {&q, &k, &v, &o}) native = native && attn_readable(*t) && dense(*t);
    if (!native) {
      // The registered op: refuses a second differentiation, and is what vmap and modes work on.
      static auto op = c10::Dispatcher::singleton().findSchemaOrThrow("sps_amd::attention_bwd", "");
      std::vector<c10::IValue> stack{
          dout, q, k, v, o, lse, docs.defined() ? c10::IValue(docs) : c10::IValue(),
          ws.defined() ? ws : at::empty({0}, q.options().dtype(at::kByte)), sm_scale, mask[0], mask[1],
          mask[2] ? c10::IValue(mask[3]) : c10::IValue()};
      op.callBoxed(&stack);
      return {stack[0].toTensor(), stack[1].toTensor(), stack[2].toTensor(), {}, {}, {}, {}, {}, {}};
    }
    RECORD_FUNCTION("sps_amd::attention_bwd", std::vector<c10::IValue>());
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard on_device(q.device());
    if (!attn_readable(dout)) dout = dout.contiguous();
    const auto s = q.sizes();
    const int b = (int)s[0], h = (int)s[1], n = (int)s[2], d = (int)s[3];
    const bool has_docs = docs.defined();
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    if (!ws.defined())
      ws = at::empty({(int64_t)sps_attn_workspace_bytes((int)mask[0], b, h, n, 0, 1)}, q.options().dtype(at::kByte));
    check("sps_attn_bwd_pass",
          sps_attn_bwd_pass(SPS_BWD_DQ | SPS_BWD_DKDV | (has_docs ? SPS_BWD_REUSE_LAYOUT : 0), (int)mask[0], b, h, n, d,
                            float_code(q.scalar_type()), q.data_ptr(), q.strides().data(), k.data_ptr(),
                            k.strides().data(), v.data_ptr(), v.strides().data(), o.data_ptr(), o.strides().data(),
                            dout.data_ptr(), dout.strides().data(), lse.data_ptr<float>(), dq.data_ptr(),
                            dq.strides().data(), dk.data_ptr(), dk.strides().data(), dv.data_ptr(), dv.strides().data(),
                            has_docs ? docs.data_ptr() : nullptr, has_docs ? index_code(docs.scalar_type()) : 0,
                            has_docs ? docs.stride(0) : 0, (float)sm_scale, (int)mask[1], (int)mask[2], (int)mask[3],
                            ws.data_ptr(), (size_t)ws.numel(), stream_of(q)));
    return {dq, dk, dv, {}, {}, {}, {}, {}, {}};
  }
};

// Whether autograd would record an operation on these tensors.
bool records(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  if (c10::impl::tls_local_dispatch_key_set().excluded_.has(c10::DispatchKey::AutogradCUDA)) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

py::object attention(py::handle q_, py::handle k_, py::handle v_, py::handle scale_, int family, py::handle window_,
                     py::handle docs_, py::handle pkw_) {
  if (!plain_thread() || !(PyFloat_CheckExact(scale_.ptr()) || PyLong_CheckExact(scale_.ptr()))) return py::none();
  const double sm_scale = PyFloat_AsDouble(scale_.ptr());
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return py::none();
  }
  const Tensor q = plain(q_), k = plain(k_), v = plain(v_);
  if (!q.defined() || !k.defined() || !v.defined()) return py::none();
  const auto window = as_int(window_);
  const std::optional<int> pkw = pkw_.is_none() ? std::optional<int>(-1) : as_int(pkw_);
  if (!window || !pkw || !std::isfinite((float)sm_scale)) return py::none();
  const auto type = q.scalar_type();
  if ((type != at::kBFloat16 && type != at::kHalf) || k.scalar_type() != type || v.scalar_type() != type ||
      q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes() || k.device() != q.device() ||
      v.device() != q.device() || q.numel() == 0 || !decode_head_dim(q.size(3)))
    return py::none();
  const int64_t n = q.size(2);
  if ((family != SPS_FAMILY_FULL && n % 2) || !fits_int(q.size(0)) || !fits_int(q.size(1)) || !fits_int(n) ||
      !attn_readable(q) || !attn_readable(k) || !attn_readable(v))
    return py::none();
  Tensor docs;
  if (!docs_.is_none()) {
    docs = plain(docs_);
    if (!docs.defined() || docs.dim() != 2 || docs.size(0) != q.size(0) || docs.size(1) != n ||
        index_code(docs.scalar_type()) < 0 || docs.device() != q.device() || !docs.is_contiguous())
      return py::none();
  }
  const bool grad = records({&q, &k, &v});
  if (grad && !(dense(q) && dense(k) && dense(v))) return py::none();
  py::gil_scoped_release nogil;
  Tensor o;
  if (grad) {
    o = AttentionFunction::apply(q, k, v, docs.defined() ? std::optional<Tensor>(docs) : std::nullopt, sm_scale, (int64_t)family, (int64_t)*window, !pkw_.is_none(),
                                 (int64_t)*pkw);
  } else {
    at::AutoDispatchBelowADInplaceOrView below;
    o = attn_forward(q, k, v, docs, AttnParams{sm_scale, family, *window, !pkw_.is_none(), *pkw}, false).o;
  }
  py::gil_scoped_acquire gil;
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(o));
}

// ---------------------------------------------------------------------------------------------
// RoPE.
// ---------------------------------------------------------------------------------------------
bool rope_readable(const Tensor& t) { return rows16(t); }

// Strides {b, n} in floats of complex64 frequencies [N, D/2] or [B, N, D/2] readable in place.
bool rope_freqs(const Tensor& f, int64_t b, int64_t n, int64_t d, std::array<int64_t, 2>& st) {
  if (f.scalar_type() != at::kComplexFloat || reinterpret_cast<uintptr_t>(f.data_ptr()) % 16) return false;
  const bool batched = f.dim() == 3;
  if (!batched && f.dim() != 2) return false;
  if ((batched && f.size(0) != b) || f.size(-2) != n || f.size(-1) != d / 2) return false;
  if (f.stride(-1) != 1 || f.stride(-2) % 2 || (batched && f.stride(0) % 2)) return false;
  st = {batched ? 2 * f.stride(0) : 0, 2 * f.stride(-2)};
  return true;
}

// RoPE of q and k (and a copy of v when defined), [B, N, H, D] in, contiguous [B, N, H, D] out.
std::vector<Tensor> rope_launch(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& freqs,
                                const std::array<int64_t, 2>& fst, at::ScalarType out_type) {
  RECORD_FUNCTION("sps_amd::rope_qkv", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(q.device());
  const auto opts = q.options().dtype(out_type);
  const int b = (int)q.size(0), n = (int)q.size(1), h = (int)q.size(2), d = (int)q.size(3);
  std::vector<Tensor> out;
  for (int i = 0; i < (v.defined() ? 3 : 2); ++i) out.push_back(at::empty({b, n, h, d}, opts));
  check("sps_rope_qkv",
        sps_rope_qkv(b, n, h, d, float_code(q.scalar_type()), q.data_ptr(), q.strides().data(), k.data_ptr(),
                     k.strides().data(), v.defined() ? v.data_ptr() : nullptr,
                     v.defined() ? v.strides().data() : nullptr, static_cast<const float*>(freqs.data_ptr()), fst.data(),
                     float_code(out_type), out[0].data_ptr(), out[0].strides().data(), out[1].data_ptr(),
                     out[1].strides().data(), v.defined() ? out[2].data_ptr() : nullptr,
                     v.defined() ? out[2].strides().data() : nullptr, stream_of(q)));
  return out;
}

// v undefined: RoPE of a pair, outputs [B, N, H, D]; defined: outputs are [B, H, N, D] views.
struct RopeFunction : torch::autograd::Function<RopeFunction> {
  static constexpr bool is_traceable = true;  // as AttentionFunction's

  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k,
                                                const std::optional<Tensor>& v_opt, const Tensor& freqs,
                                                int64_t out_type) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor v = v_opt.value_or(Tensor());
    std::array<int64_t, 2> fst;
    TORCH_INTERNAL_ASSERT(rope_freqs(freqs, q.size(0), q.size(1), q.size(3), fst));
    auto out = rope_launch(q, k, v, freqs, fst, (at::ScalarType)out_type);
    if (v.defined())
      for (auto& t : out) t = t.transpose(1, 2);
    ctx->save_for_backward({freqs});
    ctx->saved_data["in_type"] = (int64_t)q.scalar_type();
    ctx->saved_data["triple"] = v.defined();
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const Tensor freqs = ctx->get_saved_variables()[0];
    const bool triple = ctx->saved_data["triple"].toBool();
    const auto in_type = (at::ScalarType)ctx->saved_data["in_type"].toInt();
    Tensor ref;
    for (const auto& g : grads)
      if (!ref.defined()) ref = g;
    if (!ref.defined()) return {{}, {}, {}, {}, {}};
    bool native = !at::GradMode::is_enabled() && plain_thread();
    for (auto& g : grads) {
      if (!g.defined()) g = at::zeros_like(ref);
      if (g.scalar_type() != grads[0].scalar_type()) g = g.to(grads[0].scalar_type());
      if (triple) g = g.transpose(1, 2);
      native = native && plain_tensor(g) && g.device() == freqs.device();
    }
    const Tensor conj = at::resolve_conj(at::conj(freqs));
    std::array<int64_t, 2> fst;
    native = native && plain_tensor(conj) &&
             rope_freqs(conj, grads[0].size(0), grads[0].size(1), grads[0].size(3), fst);
    if (!native) {
      static auto op3 = c10::Dispatcher::singleton().findSchemaOrThrow("sps_amd::rope_qkv", "");
      static auto op2 = c10::Dispatcher::singleton().findSchemaOrThrow("sps_amd::rope_pair", "");
      std::vector<c10::IValue> stack{grads[0], grads[1]};
      if (triple) stack.emplace_back(grads[2]);
      stack.emplace_back(conj);
      if (triple) stack.emplace_back((int64_t)in_type);
      (triple ? op3 : op2).callBoxed(&stack);
      return {stack[0].toTensor(), stack[1].toTensor(), triple ? stack[2].toTensor() : Tensor(), {}, {}};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    for (auto& g : grads)
      if (!rope_readable(g)) g = g.contiguous();
    auto out = rope_launch(grads[0], grads[1], triple ? grads[2] : Tensor(), conj, fst, in_type);
    return {out[0], out[1], triple ? out[2] : Tensor(), {}, {}};
  }
};

py::object rope(py::handle q_, py::handle k_, py::handle v_, py::handle freqs_, py::handle out_dtype_) {
  if (!plain_thread()) return py::none();
  const bool triple = !v_.is_none();
  const Tensor q = plain(q_), k = plain(k_), freqs = plain(freqs_), v = triple ? plain(v_) : Tensor();
  if (!q.defined() || !k.defined() || !freqs.defined() || (triple && !v.defined())) return py::none();
  if (!out_dtype_.is_none() && !THPDtype_Check(out_dtype_.ptr())) return py::none();
  const auto out_type = out_dtype_.is_none() ? q.scalar_type()
                                             : reinterpret_cast<THPDtype*>(out_dtype_.ptr())->scalar_type;
  const auto type = q.scalar_type();
  std::array<int64_t, 2> fst;
  if (float_code(type) < 0 || float_code(out_type) < 0 || k.scalar_type() != type || q.dim() != 4 ||
      k.sizes() != q.sizes() || k.device() != q.device() || freqs.device() != q.device() || q.numel() == 0 ||
      q.size(3) % 8 || !rope_readable(q) || !rope_readable(k) || !fits_int(q.size(0)) || !fits_int(q.size(1)) ||
      !fits_int(q.size(2)) || !rope_freqs(freqs, q.size(0), q.size(1), q.size(3), fst))
    return py::none();
  if (triple && (v.scalar_type() != type || v.sizes() != q.sizes() || v.device() != q.device() || !rope_readable(v)))
    return py::none();
  // A differentiated call keeps the frequencies' conjugate for its backward in the same layout.
  const bool grad = records({&q, &k}) || (triple && records({&v}));
  if (records({&freqs}) || (grad && !dense(freqs))) return py::none();
  std::vector<Tensor> out;
  {
    py::gil_scoped_release nogil;
    if (grad) {
      out = RopeFunction::apply(q, k, triple ? std::optional<Tensor>(v) : std::nullopt, freqs, (int64_t)out_type);
    } else {
      at::AutoDispatchBelowADInplaceOrView below;
      out = rope_launch(q, k, v, freqs, fst, out_type);
      if (triple)
        for (auto& t : out) t = t.transpose(1, 2);
    }
  }
  py::tuple r(out.size());
  for (size_t i = 0; i < out.size(); ++i) r[i] = py::reinterpret_steal<py::object>(THPVariable_Wrap(out[i]));
  return std::move(r);
}

// ---------------------------------------------------------------------------------------------
// KV update and decode.
// ---------------------------------------------------------------------------------------------
struct Update {
  // sps_kv_update's arguments; the tensors stay with the caller for the call.
  int kv_dtype, ring_storage = 0, window, ret_storage, len_dtype, new_dtype, active_dtype;
  void *ring_k = nullptr, *ring_v = nullptr, *ring_len = nullptr, *ring_pos = nullptr, *ret_k, *ret_v, *ret_len;
  int64_t ring_st[6] = {0, 0, 0, 0, 0, 0}, ring_len_st[2] = {0, 0}, ret_st[6], ret_len_st[2], new_st[8], active_st;
  const void *kw, *vw, *kr, *vr, *active;
  int B, H, D;
  c10::Device device{c10::kCPU};
};

bool cache_strides(const Tensor& k, const Tensor& v, int64_t* out) {
  if (k.stride(3) != 1 || v.stride(3) != 1) return false;
  for (int i = 0; i < 3; ++i) {
    out[i] = k.stride(i);
    out[3 + i] = v.stride(i);
  }
  return true;
}

// Reads the keyword arguments of fused_sps_kv_update, in its order; false: not a call for this path.
bool read_update(const py::tuple& t, Update& u) {
  if (t.size() != 13) return false;
  const auto window = as_int(t[12]);
  if (!window) return false;
  u.window = *window;
  const bool ring = u.window > 0;
  const Tensor br_k = plain(t[4]), br_v = plain(t[5]), br_len = plain(t[6]), kr = plain(t[9]), vr = plain(t[10]),
               active = plain(t[11]);
  for (const Tensor* x : {&br_k, &br_v, &br_len, &kr, &vr, &active})
    if (!x->defined() || x->device() != br_k.device()) return false;
  u.kv_dtype = float_code(br_k.scalar_type());
  u.new_dtype = float_code(kr.scalar_type());
  u.len_dtype = index_code(br_len.scalar_type());
  if (kr.dim() != 3 || br_k.dim() != 4 || vr.sizes() != kr.sizes() || br_v.sizes() != br_k.sizes() || kr.numel() == 0)
    return false;
  const int64_t b = kr.size(0), h = kr.size(1), d = kr.size(2);
  if (br_k.size(0) != b || br_k.size(1) != h || br_k.size(3) != d || br_len.dim() != 2 || br_len.size(0) != b ||
      br_len.size(1) != h || u.kv_dtype < 0 || u.new_dtype < 0 || u.len_dtype < 0 ||
      br_v.scalar_type() != br_k.scalar_type() || vr.scalar_type() != kr.scalar_type() || kr.stride(2) != 1 ||
      vr.stride(2) != 1 || active.dim() != 1 || active.size(0) != b || !fits_int(b) || !fits_int(h) || !fits_int(d) ||
      !fits_int(br_k.size(2)) || !cache_strides(br_k, br_v, u.ret_st))
    return false;
  const auto flag = active.scalar_type();
  u.active_dtype = flag == at::kBool || flag == at::kByte || flag == at::kChar ? SPS_DTYPE_U8 : index_code(flag);
  if (u.active_dtype < 0) return false;
  u.B = (int)b;
  u.H = (int)h;
  u.D = (int)d;
  u.device = br_k.device();
  u.kr = kr.data_ptr();
  u.vr = vr.data_ptr();
  u.kw = u.kr;
  u.vw = u.vr;
  const int64_t rs[4] = {kr.stride(0), kr.stride(1), vr.stride(0), vr.stride(1)};
  for (int i = 0; i < 4; ++i) u.new_st[i] = u.new_st[4 + i] = rs[i];
  if (ring) {
    const Tensor nw_k = plain(t[0]), nw_v = plain(t[1]), nw_len = plain(t[2]), nw_pos = plain(t[3]),
                 kw = plain(t[7]), vw = plain(t[8]);
    for (const Tensor* x : {&nw_k, &nw_v, &nw_len, &nw_pos, &kw, &vw})
      if (!x->defined() || x->device() != u.device) return false;
    if (nw_k.dim() != 4 || nw_v.sizes() != nw_k.sizes() || nw_k.size(0) != b || nw_k.size(1) != h ||
        nw_k.size(3) != d || nw_len.dim() != 1 || nw_len.size(0) != b || nw_pos.dim() != 1 || nw_pos.size(0) != b ||
        kw.sizes() != kr.sizes() || vw.sizes() != kr.sizes() || nw_k.scalar_type() != br_k.scalar_type() ||
        nw_v.scalar_type() != br_k.scalar_type() || nw_len.scalar_type() != br_len.scalar_type() ||
        nw_pos.scalar_type() != br_len.scalar_type() || u.window > nw_k.size(2) || !fits_int(nw_k.size(2)) ||
        kw.scalar_type() != kr.scalar_type() || vw.scalar_type() != kr.scalar_type() || kw.stride(2) != 1 ||
        vw.stride(2) != 1 || !cache_strides(nw_k, nw_v, u.ring_st))
      return false;
    u.ring_k = nw_k.data_ptr();
    u.ring_v = nw_v.data_ptr();
    u.ring_storage = (int)nw_k.size(2);
    u.ring_len = nw_len.data_ptr();
    u.ring_pos = nw_pos.data_ptr();
    u.ring_len_st[0] = nw_len.stride(0);
    u.ring_len_st[1] = nw_pos.stride(0);
    u.kw = kw.data_ptr();
    u.vw = vw.data_ptr();
    const int64_t ws[4] = {kw.stride(0), kw.stride(1), vw.stride(0), vw.stride(1)};
    for (int i = 0; i < 4; ++i) u.new_st[i] = ws[i];
  }
  u.ret_k = br_k.data_ptr();
  u.ret_v = br_v.data_ptr();
  u.ret_storage = (int)br_k.size(2);
  u.ret_len = br_len.data_ptr();
  u.ret_len_st[0] = br_len.stride(0);
  u.ret_len_st[1] = br_len.stride(1);
  u.active = active.data_ptr();
  u.active_st = active.stride(0);
  return true;
}

// Runs fused_sps_kv_update on a tuple of its arguments; false: the caller takes the general path.
bool kv_update(py::handle args) {
  Update u;
  if (!plain_thread() || !PyTuple_Check(args.ptr()) || !read_update(py::reinterpret_borrow<py::tuple>(args), u))
    return false;
  c10::DeviceGuard on_device(u.device);
  void* stream = static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(u.device.index()).stream());
  py::gil_scoped_release nogil;
  check("sps_kv_update",
        sps_kv_update(u.B, u.H, u.D, u.kv_dtype, u.ring_k, u.ring_v, u.ring_st, u.ring_storage, u.window, u.ring_len,
                      u.ring_pos, u.ring_len_st, u.ret_k, u.ret_v, u.ret_st, u.ret_storage, u.ret_len, u.ret_len_st,
                      u.len_dtype, u.new_dtype, u.kw, u.vw, u.kr, u.vr, u.new_st, u.active, u.active_dtype,
                      u.active_st, stream));
  return true;
}

// Segmented decode of one (nq = 1, q [B, H, D]) or two (q [B, 2, H, D]) queries over a list of
// KVSegments and a list of up to two extra (k, v) pairs (nq = 2: the first is seen by both queries, the
// second by query 1), with the KV update folded in when `update` is given.
py::object decode(py::handle q_, int nq, py::handle segments_, py::handle extras_, py::handle attn_dtype,
                  py::handle update) {
  if (!plain_thread() || !THPDtype_Check(attn_dtype.ptr()) || !PyList_Check(segments_.ptr()) ||
      !(extras_.is_none() || PyList_Check(extras_.ptr())))
    return py::none();
  const py::list segments = py::reinterpret_borrow<py::list>(segments_);
  const py::list extras = extras_.is_none() ? py::list() : py::reinterpret_borrow<py::list>(extras_);
  const auto type = reinterpret_cast<THPDtype*>(attn_dtype.ptr())->scalar_type;
  const Tensor q = plain(q_);
  if (!q.defined() || q.scalar_type() != type || float_code(type) < 0 || q.dim() != (nq == 1 ? 3 : 4) ||
      q.stride(-1) != 1 || (nq == 2 && q.size(1) != 2))
    return py::none();
  const int64_t b = q.size(0), h = q.size(-2), d = q.size(-1);
  const int n_seg = (int)segments.size(), n_extra = (int)extras.size();
  if (n_seg < 1 || n_seg > (nq == 1 ? 3 : 2) || n_extra > 2 || q.numel() == 0 || !decode_head_dim(d) || !fits_int(b) ||
      !fits_int(h))
    return py::none();
  static PyObject* const names[4] = {PyUnicode_InternFromString("k"), PyUnicode_InternFromString("v"),
                                     PyUnicode_InternFromString("lengths"), PyUnicode_InternFromString("max_len_cap")};
  const void *sk[3], *sv[3], *sl[3], *ek[2], *ev[2];
  int64_t skst[9], svst[9], scan[3], est[2] = {0, 0};
  int ldt[3], lph[3], emask[2];
  at::ScalarType kv_type = at::kBFloat16;
  for (int i = 0; i < n_seg; ++i) {
    py::object f[4];
    for (int j = 0; j < 4; ++j) {
      f[j] = py::reinterpret_steal<py::object>(PyObject_GetAttr(segments[i].ptr(), names[j]));
      if (!f[j]) {
        PyErr_Clear();
        return py::none();
      }
    }
    const Tensor k = plain(f[0]), v = plain(f[1]), len = plain(f[2]);
    if (!k.defined() || !v.defined() || !len.defined() || k.device() != q.device() || v.device() != q.device() ||
        len.device() != q.device())
      return py::none();
    if (i == 0) kv_type = k.scalar_type();
    if (float_code(kv_type) < 0 || k.scalar_type() != kv_type || v.scalar_type() != kv_type || k.dim() != 4 ||
        v.sizes() != k.sizes() || k.size(0) != b || k.size(1) != h || k.size(3) != d || !k.is_contiguous() ||
        !v.is_contiguous() || !rows16(k) || !rows16(v) || index_code(len.scalar_type()) < 0 || !len.is_contiguous())
      return py::none();
    const bool per_head = len.dim() == 2;
    if (per_head ? (len.size(0) != b || len.size(1) != h) : (len.dim() != 1 || len.size(0) != b)) return py::none();
    scan[i] = k.size(2);
    if (!f[3].is_none()) {
      const auto cap = as_int(f[3]);
      if (!cap || *cap < 0) return py::none();
      if (scan[i] > 0) scan[i] = std::max<int64_t>(1, std::min<int64_t>(scan[i], *cap));
    }
    sk[i] = k.data_ptr();
    sv[i] = v.data_ptr();
    sl[i] = len.data_ptr();
    ldt[i] = index_code(len.scalar_type());
    lph[i] = per_head;
    for (int j = 0; j < 3; ++j) {
      skst[3 * i + j] = k.stride(j);
      svst[3 * i + j] = v.stride(j);
    }
  }
  for (int i = 0; i < n_extra; ++i) {
    const py::object item = extras[i];
    if (!PyTuple_Check(item.ptr())) return py::none();
    const py::tuple pair = py::reinterpret_borrow<py::tuple>(item);
    if (pair.size() != 2) return py::none();
    const Tensor k = plain(pair[0]), v = plain(pair[1]);
    for (const Tensor* x : {&k, &v}) {
      if (!x->defined() || x->device() != q.device() || x->scalar_type() != type || x->dim() != 3 || x->size(0) != b ||
          x->size(1) != h || x->size(2) != d || x->stride(2) != 1)
        return py::none();
      if (i == 0 && x == &k) {
        est[0] = k.stride(0);
        est[1] = k.stride(1);
      } else if (x->stride(0) != est[0] || x->stride(1) != est[1]) {
        return py::none();
      }
    }
    ek[i] = k.data_ptr();
    ev[i] = v.data_ptr();
    emask[i] = nq == 1 ? 1 : i == 0 ? 0b11 : 0b10;
  }
  Update u;
  const bool with_update = !update.is_none();
  if (with_update && (!PyTuple_Check(update.ptr()) || !read_update(py::reinterpret_borrow<py::tuple>(update), u) ||
                      u.device != q.device() || u.kv_dtype != float_code(kv_type) || u.B != b || u.H != h || u.D != d))
    return py::none();
  Tensor out;
  {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard on_device(q.device());
    out = nq == 1 ? at::empty({b, h, d}, q.options().dtype(at::kFloat))
                  : at::empty({b, 2, h, d}, q.options().dtype(at::kFloat));
    const int64_t qst[3] = {q.stride(0), nq == 1 ? q.stride(0) : q.stride(1), q.stride(-2)};
    const int64_t ost[3] = {out.stride(0), nq == 1 ? out.stride(0) : out.stride(1), out.stride(-2)};
    const int kvd = float_code(kv_type);
    const size_t bytes = std::max<size_t>(
        1, with_update ? sps_decode_kv_update_workspace_bytes((int)b, (int)h, (int)d, nq, kvd, n_seg, scan)
                       : sps_decode_workspace_bytes((int)b, (int)h, (int)d, nq, kvd, n_seg, scan));
    const Tensor ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    const float scale = (float)(1.0 / std::sqrt((double)d));
    const int e_dtype = n_extra ? float_code(type) : SPS_DTYPE_F32;
    if (with_update)
      check("sps_decode_kv_update",
            sps_decode_kv_update((int)b, (int)h, (int)d, nq, q.data_ptr(), float_code(type), qst, kvd, n_seg, sk, skst,
                                 sv, svst, sl, ldt, lph, scan, n_extra, ek, ev, e_dtype, est, emask, scale,
                                 out.data_ptr<float>(), ost, u.ring_k, u.ring_v, u.ring_st, u.ring_storage, u.window,
                                 u.ring_len, u.ring_pos, u.ring_len_st, u.ret_k, u.ret_v, u.ret_st, u.ret_storage,
                                 u.ret_len, u.ret_len_st, u.len_dtype, u.new_dtype, u.kw, u.vw, u.kr, u.vr, u.new_st,
                                 u.active, u.active_dtype, u.active_st, ws.data_ptr(), bytes, stream_of(q)));
    else
      check("sps_decode", sps_decode((int)b, (int)h, (int)d, nq, q.data_ptr(), float_code(type), qst, kvd, n_seg, sk,
                                     skst, sv, svst, sl, ldt, lph, scan, n_extra, ek, ev, e_dtype, est, emask, scale,
                                     out.data_ptr<float>(), ost, ws.data_ptr(), bytes, stream_of(q)));
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

}  // namespace

PYBIND11_MODULE(_torch_binding, m) {
  m.def("attention", &attention);
  m.def("rope", &rope);
  m.def("kv_update", &kv_update);
  m.def("decode", &decode);
}
