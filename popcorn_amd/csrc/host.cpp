// The call path of popcorn_amd.impls for the inputs a model passes: plain HIP
// tensors in layouts the kernels read where they lie. Each function checks that
// the call is one of these, allocates the outputs, enqueues the kernels on
// torch's current stream and, when a gradient is to be recorded, makes the
// autograd node, all without entering the interpreter; the nodes' backward runs
// on autograd's threads without it too. A short call is bound by this work and
// not by its kernels: an rms_norm of 64 rows with its gradients spent 80 us on
// the host in Python and ctypes.
//
// For any other call a function returns NotImplemented before it does anything,
// and impls.py takes it: tensor subclasses and calls under tracing, dispatch or
// function modes or function transforms, layouts that need a copy, empty tensors,
// and every call that has to be refused. So what is accepted and how errors read is
// said there, and here only what the fast path covers.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cmath>
#include <optional>
#include <string>

#include "../../include/popcorn_amd.h"

namespace {

using at::ScalarType;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

PyObject* kernel_error = nullptr;    // popcorn_amd._lib.KernelError
PyObject* device_context = nullptr;  // torch.utils._device.DeviceContext

// Raises KernelError, from any thread.
void check(int status) {
  if (status == PK_OK) return;
  const std::string text = pk_last_error();
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(kernel_error, ("popcorn_amd: " + (text.empty() ? "status " + std::to_string(status) : text)).c_str());
  python_error e;
  e.persist();
  throw e;
}

int code_of(ScalarType t) { return t == at::kFloat ? PK_F32 : (t == at::kBFloat16 ? PK_BF16 : PK_F16); }
bool is_half(ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
bool is_float(ScalarType t) { return t == at::kFloat || is_half(t); }
ScalarType promoted(ScalarType a, ScalarType b) { return a == b ? a : at::kFloat; }  // of the three types above

// A plain strided HIP tensor of a float type: no subclass behaviour, wrapper,
// pending negation or tangent that reading its memory would miss.
bool plain(const Tensor& t) {
  const auto keys = t.key_set();
  static constexpr c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                              c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::Negative,
                                              c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor});
  return keys.has(c10::DispatchKey::CUDA) && !keys.has_any(other) && t.layout() == at::kStrided && t.has_storage() &&
         is_float(t.scalar_type()) && t.numel() > 0 && !t._fw_grad(0).defined();
}

// Whether a torch function mode is active that could look at the torch calls
// inside one of these. The one behind torch.set_default_device and `with
// torch.device(..)` only gives a device to calls that name none.
bool function_mode() {
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < at::impl::PythonTorchFunctionTLS::stack_len(); ++i) {
    const PyObject* mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
    if ((const PyObject*)Py_TYPE(mode) != device_context) return true;
  }
  return false;
}

// Calls some mode or transform means to see operator by operator.
bool watched() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || function_mode() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         at::tracer::impl::is_dispatch_enabled();
}

// The i-th argument as a plain tensor on `like`'s device (if given); false: not this path.
bool take(PyObject* o, Tensor& t, const Tensor* like = nullptr) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return plain(t) && (like == nullptr || t.device() == like->device());
}

bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

bool last_contiguous(const Tensor& t) { return t.stride(-1) == 1; }

// Rows the attention and norm-rope kernels read with 16-byte loads.
bool aligned_rows(const Tensor& t) {
  if (t.stride(-1) != 1 || !aligned(t)) return false;
  const int64_t unit = 16 / t.element_size();
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if (t.stride(i) % unit != 0 || t.stride(i) < 0) return false;
  return true;
}
Tensor make_aligned_rows(const Tensor& t) {
  if (aligned_rows(t)) return t;
  Tensor c = t.contiguous();
  return aligned(c) ? c : c.clone();
}

// What a saved-tensor hook hands back has the values it was given, but may have another layout.
Tensor unpacked(const torch::autograd::Variable& t) { return t.defined() ? t.contiguous() : t; }

bool dense(const Tensor& t) { return t.is_contiguous() && aligned(t); }  // weights and tables

Tensor empty(at::IntArrayRef sizes, ScalarType dtype, const Tensor& like) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}
Tensor scratch(int64_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>(bytes, 16)}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool tracks(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// An absent tensor as autograd's functions take it.
std::optional<Tensor> given(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// The cotangent at the output's type, contiguous.
Tensor cotangent(const Tensor& g, ScalarType dtype) { return g.to(dtype).contiguous(); }

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* out(Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const float* fptr(const Tensor& t) { return static_cast<const float*>(ptr(t)); }
float* fout(Tensor& t) { return static_cast<float*>(out(t)); }

// A state that saved_data keeps as one value.
void keep(AutogradContext* ctx, std::vector<int64_t> v) { ctx->saved_data["i"] = c10::IValue(std::move(v)); }
std::vector<int64_t> kept(AutogradContext* ctx) { return ctx->saved_data["i"].toIntVector(); }

// ---------------------------------------------------------------- rms_norm

Tensor rms_norm_fwd(const Tensor& x, const Tensor& w, const Tensor& b, double eps, Tensor* rstd) {
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const c10::DeviceGuard guard(x.device());
  Tensor y = empty(x.sizes(), w.scalar_type(), x);
  if (rstd) *rstd = empty({rows}, at::kFloat, x);
  check(pk_rmsnorm_fwd(ptr(x), ptr(w), ptr(b), out(y), rstd ? fout(*rstd) : nullptr, rows, cols, (float)eps,
                       code_of(x.scalar_type()), code_of(w.scalar_type()), stream_of(x)));
  return y;
}

struct RmsNorm : Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const std::optional<Tensor>& bias,
                        double eps) {
    const Tensor b = bias.value_or(Tensor());
    Tensor rstd;
    Tensor y = rms_norm_fwd(x, w, b, eps, &rstd);
    ctx->save_for_backward({x, w, rstd});
    keep(ctx, {b.defined()});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor x = unpacked(saved[0]), w = unpacked(saved[1]), rstd = unpacked(saved[2]);
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    const c10::DeviceGuard guard(x.device());
    const Tensor dy = cotangent(grads[0], w.scalar_type());
    Tensor dx = empty(x.sizes(), x.scalar_type(), x), dw = empty(w.sizes(), w.scalar_type(), w), db;
    if (kept(ctx)[0]) db = empty(w.sizes(), w.scalar_type(), w);
    const int64_t bytes = pk_rmsnorm_bwd_workspace(rows, cols, code_of(x.scalar_type()));
    Tensor ws = scratch(bytes, x);
    check(pk_rmsnorm_bwd(ptr(x), ptr(w), fptr(rstd), ptr(dy), out(dx), out(dw), out(db), out(ws), bytes,
                         rows, cols, code_of(x.scalar_type()), code_of(w.scalar_type()), stream_of(x)));
    return {dx, dw, db, Tensor()};
  }
};

bool norm_types(const Tensor& x, const Tensor& w) {
  return x.scalar_type() == w.scalar_type() || (is_half(x.scalar_type()) && w.scalar_type() == at::kFloat);
}
bool norm_vector(const Tensor& w, const Tensor& x) {
  return w.dim() == 1 && w.size(0) == x.size(-1) && w.is_contiguous();
}

// ---------------------------------------------------------------- add_rms_norm

std::pair<Tensor, Tensor> add_rms_norm_fwd(const Tensor& x, const Tensor& r, const Tensor& w, double eps, double offset,
                                           Tensor& rstd) {
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const c10::DeviceGuard guard(x.device());
  Tensor y = empty(x.sizes(), w.scalar_type(), x), s = empty(x.sizes(), x.scalar_type(), x);
  rstd = empty({rows}, at::kFloat, x);
  check(pk_add_rmsnorm_fwd(ptr(x), ptr(r), ptr(w), out(y), out(s), fout(rstd), rows, cols, (float)eps,
                           (float)offset, code_of(x.scalar_type()), code_of(w.scalar_type()), stream_of(x)));
  return {y, s};
}

struct AddRmsNorm : Function<AddRmsNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r, const Tensor& w, double eps,
                               double offset) {
    Tensor rstd;
    auto [y, s] = add_rms_norm_fwd(x, r, w, eps, offset, rstd);
    ctx->save_for_backward({s, w, rstd});
    ctx->saved_data["o"] = offset;
    ctx->set_materialize_grads(false);
    return {y, s};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor s = unpacked(saved[0]), w = unpacked(saved[1]), rstd = unpacked(saved[2]);
    const int64_t cols = s.size(-1), rows = s.numel() / cols;
    const c10::DeviceGuard guard(s.device());
    if (!grads[0].defined()) {  // only the residual stream was used downstream
      const Tensor sum = grads[1].defined() ? grads[1].to(s.scalar_type()) : at::zeros_like(s);
      return {sum, sum, at::zeros_like(w), Tensor(), Tensor()};
    }
    const Tensor dy = cotangent(grads[0], w.scalar_type());
    const Tensor ds = grads[1].defined() ? cotangent(grads[1], s.scalar_type()) : Tensor();
    Tensor sum = empty(s.sizes(), s.scalar_type(), s), dw = empty(w.sizes(), w.scalar_type(), w);
    const int64_t bytes = pk_rmsnorm_bwd_workspace(rows, cols, code_of(s.scalar_type()));
    Tensor ws = scratch(bytes, s);
    check(pk_add_rmsnorm_bwd(ptr(s), ptr(w), fptr(rstd), ptr(dy), ptr(ds), out(sum), out(dw), out(ws),
                             bytes, rows, cols, (float)ctx->saved_data["o"].toDouble(), code_of(s.scalar_type()),
                             code_of(w.scalar_type()), stream_of(s)));
    return {sum, sum, dw, Tensor(), Tensor()};  // s = x + residual: one gradient for both
  }
};

// ---------------------------------------------------------------- swiglu

// Elements between consecutive rows when one stride reaches them all; -1 when none does.
int64_t row_stride(const Tensor& t) {
  if (t.is_contiguous()) return t.dim() ? t.size(-1) : 1;
  if (t.dim() < 2 || t.stride(-1) != 1) return -1;
  int64_t stride = -1, span = 1;
  for (int64_t i = t.dim() - 2; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (stride < 0) stride = t.stride(i);
    else if (t.stride(i) != stride * span) return -1;
    span *= t.size(i);
  }
  return stride < 0 ? t.size(-1) : stride;
}

Tensor swiglu_fwd(const Tensor& a, const Tensor& b) {
  const int64_t cols = a.dim() ? a.size(-1) : 1, rows = a.numel() / cols;
  const c10::DeviceGuard guard(a.device());
  Tensor y = empty(a.sizes(), a.scalar_type(), a);
  check(pk_swiglu_rows_fwd(ptr(a), ptr(b), out(y), rows, cols, row_stride(a), row_stride(b), code_of(a.scalar_type()),
                           stream_of(a)));
  return y;
}

struct SwiGlu : Function<SwiGlu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b) {
    ctx->save_for_backward({a, b});
    return swiglu_fwd(a, b);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Tensor a = saved[0], b = saved[1];
    if (row_stride(a) < 0 || row_stride(b) < 0) {
      a = a.contiguous();
      b = b.contiguous();
    }
    const int64_t cols = a.dim() ? a.size(-1) : 1, rows = a.numel() / cols;
    const c10::DeviceGuard guard(a.device());
    const Tensor g = cotangent(grads[0], a.scalar_type());
    Tensor da = empty(a.sizes(), a.scalar_type(), a), db = empty(b.sizes(), b.scalar_type(), b);
    check(pk_swiglu_rows_bwd(ptr(g), ptr(a), ptr(b), out(da), out(db), rows, cols, row_stride(a), row_stride(b),
                             code_of(a.scalar_type()), stream_of(a)));
    return {da, db};
  }
};

// ---------------------------------------------------------------- rotary_embedding

Tensor rotate(const Tensor& x, const Tensor& cs, const Tensor& sn, bool interleaved, bool conjugate) {
  const c10::DeviceGuard guard(x.device());
  Tensor y = empty(x.sizes(), x.scalar_type(), x);
  const int64_t strides[6] = {x.stride(0), x.stride(1), x.stride(2), y.stride(0), y.stride(1), y.stride(2)};
  check(pk_rotary(ptr(x), ptr(cs), ptr(sn), out(y), strides, x.size(0), x.size(1), x.size(2), x.size(3), cs.size(1),
                  code_of(x.scalar_type()), code_of(cs.scalar_type()), interleaved, conjugate, stream_of(x)));
  return y;
}

struct Rotary : Function<Rotary> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cs, const Tensor& sn, bool interleaved) {
    ctx->save_for_backward({cs, sn});
    keep(ctx, {interleaved});
    return rotate(x, cs, sn, interleaved, false);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor g = last_contiguous(grads[0]) ? grads[0] : grads[0].contiguous();
    return {rotate(g, unpacked(saved[0]), unpacked(saved[1]), kept(ctx)[0], true), Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------- rope

std::pair<Tensor, Tensor> rope_call(const Tensor& q, const Tensor& k, const Tensor& cs, const Tensor& sn, bool transpose,
                                    ScalarType dtype) {
  const c10::DeviceGuard guard(q.device());
  Tensor yq = empty(q.sizes(), dtype, q), yk = empty(k.sizes(), dtype, k);
  int64_t strides[12];
  const Tensor* ts[4] = {&q, &k, &yq, &yk};
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i) strides[3 * t + i] = ts[t]->stride(i);
  check(pk_rope(ptr(q), ptr(k), ptr(cs), ptr(sn), out(yq), out(yk), strides, q.size(0), q.size(1), k.size(1), q.size(2),
                q.size(3), cs.size(0), code_of(q.scalar_type()), code_of(dtype), code_of(cs.scalar_type()), transpose,
                stream_of(q)));
  return {yq, yk};
}

struct Rope : Function<Rope> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& cs, const Tensor& sn) {
    const ScalarType dtype = promoted(q.scalar_type(), cs.scalar_type());
    auto [yq, yk] = rope_call(q, k, cs, sn, false, dtype);
    ctx->save_for_backward({cs, sn});
    keep(ctx, {(int64_t)q.scalar_type(), (int64_t)dtype});
    return {yq, yk};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {  // undefined cotangents come as zeros
    const auto saved = ctx->get_saved_variables();
    const auto types = kept(ctx);
    Tensor g[2];
    for (int t = 0; t < 2; ++t) {
      g[t] = grads[t].to((ScalarType)types[1]);
      if (!last_contiguous(g[t])) g[t] = g[t].contiguous();
    }
    auto [dq, dk] = rope_call(g[0], g[1], unpacked(saved[0]), unpacked(saved[1]), true, (ScalarType)types[0]);
    return {dq, dk, Tensor(), Tensor()};
  }
};

// q [b, hq, s, d], k [b, hkv, s, d], tables [1 or b, s, d] of one type each
bool rope_shapes(const Tensor& q, const Tensor& k, const Tensor& cs, const Tensor& sn) {
  return q.dim() == 4 && k.dim() == 4 && cs.dim() == 3 && cs.sizes() == sn.sizes() && q.scalar_type() == k.scalar_type() &&
         cs.scalar_type() == sn.scalar_type() && q.size(0) == k.size(0) && q.size(2) == k.size(2) &&
         q.size(3) == k.size(3) && q.size(3) % 2 == 0 && cs.size(1) == q.size(2) && cs.size(2) == q.size(3) &&
         (cs.size(0) == 1 || cs.size(0) == q.size(0)) && cs.is_contiguous() && sn.is_contiguous() && last_contiguous(q) &&
         last_contiguous(k);
}

// ---------------------------------------------------------------- qk_norm_rope

struct NormRopeOut {
  Tensor yq, yk, rq, rk;
};

NormRopeOut norm_rope_fwd(const Tensor& q, const Tensor& k, const Tensor& qw, const Tensor& kw, const Tensor& cs,
                          const Tensor& sn, double eps) {
  const c10::DeviceGuard guard(q.device());
  const ScalarType dtype = promoted(promoted(q.scalar_type(), qw.scalar_type()), cs.scalar_type());
  NormRopeOut o;
  o.yq = empty(q.sizes(), dtype, q);
  o.yk = empty(k.sizes(), dtype, k);
  o.rq = empty(q.sizes().slice(0, 3), at::kFloat, q);
  o.rk = empty(k.sizes().slice(0, 3), at::kFloat, k);
  int64_t strides[12];
  const Tensor* ts[4] = {&q, &k, &o.yq, &o.yk};
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i) strides[3 * t + i] = ts[t]->stride(i);
  check(pk_qk_norm_rope_fwd(ptr(q), ptr(k), ptr(qw), ptr(kw), ptr(cs), ptr(sn), out(o.yq), out(o.yk),
                            fout(o.rq), fout(o.rk), strides, q.size(0), q.size(1), k.size(1),
                            q.size(2), q.size(3), cs.size(0), (float)eps, code_of(q.scalar_type()), code_of(dtype),
                            code_of(cs.scalar_type()), code_of(qw.scalar_type()), stream_of(q)));
  return o;
}

struct QkNormRope : Function<QkNormRope> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& qw, const Tensor& kw,
                               const Tensor& cs, const Tensor& sn, double eps) {
    NormRopeOut o = norm_rope_fwd(q, k, qw, kw, cs, sn, eps);
    ctx->save_for_backward({q, k, qw, kw, cs, sn, o.rq, o.rk});
    return {o.yq, o.yk};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {  // undefined cotangents come as zeros
    auto s = ctx->get_saved_variables();
    for (size_t i = 2; i < s.size(); ++i) s[i] = unpacked(s[i]);
    const Tensor q = make_aligned_rows(s[0]), k = make_aligned_rows(s[1]), &qw = s[2], &cs = s[4];
    const c10::DeviceGuard guard(q.device());
    const ScalarType dtype = promoted(promoted(q.scalar_type(), qw.scalar_type()), cs.scalar_type());
    const Tensor gq = make_aligned_rows(grads[0].to(dtype)), gk = make_aligned_rows(grads[1].to(dtype));
    Tensor dq = empty(q.sizes(), q.scalar_type(), q), dk = empty(k.sizes(), k.scalar_type(), k);
    Tensor dw = empty({2, q.size(3)}, qw.scalar_type(), q);
    const int64_t bytes =
        pk_qk_norm_rope_bwd_workspace(q.size(0), q.size(1), k.size(1), q.size(2), q.size(3), code_of(q.scalar_type()));
    Tensor ws = scratch(bytes, q);
    int64_t strides[18];
    const Tensor* ts[6] = {&q, &k, &gq, &gk, &dq, &dk};
    for (int t = 0; t < 6; ++t)
      for (int i = 0; i < 3; ++i) strides[3 * t + i] = ts[t]->stride(i);
    check(pk_qk_norm_rope_bwd(ptr(q), ptr(k), ptr(qw), ptr(s[3]), ptr(cs), ptr(s[5]), fptr(s[6]),
                              fptr(s[7]), ptr(gq), ptr(gk), out(dq), out(dk), out(dw), out(ws), bytes,
                              strides, q.size(0), q.size(1), k.size(1), q.size(2), q.size(3), cs.size(0),
                              code_of(q.scalar_type()), code_of(dtype), code_of(cs.scalar_type()),
                              code_of(qw.scalar_type()), stream_of(q)));
    return {dq, dk, dw.select(0, 0), dw.select(0, 1), Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------- attention

// Dense tensors [batch, seq, heads, dim], or packed ones [total, heads, dim]
// with their sequences' offsets.
struct Packing {
  Tensor cu;  // undefined: dense
  int64_t seqs = 0, longest = 0;
};

template <int N> std::array<int64_t, 3 * N> strides_of(const std::array<const Tensor*, N>& ts) {
  std::array<int64_t, 3 * N> st{};
  const int lead = (int)ts[0]->dim() - 1;
  for (int t = 0; t < N; ++t)
    for (int i = 0; i < lead; ++i) st[lead * t + i] = ts[t]->stride(i);
  return st;
}

std::pair<Tensor, Tensor> attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Packing& p, bool causal,
                                   float scale, bool want_lse) {
  const c10::DeviceGuard guard(q.device());
  const int64_t hq = q.size(-2), hkv = k.size(-2), d = q.size(-1);
  Tensor o = empty(q.sizes(), q.scalar_type(), q), lse;
  const auto st = strides_of<4>({&q, &k, &v, &o});
  const int code = code_of(q.scalar_type());
  if (p.cu.defined()) {
    if (want_lse) lse = empty({hq, q.size(0)}, at::kFloat, q);
    check(pk_attn_varlen_fwd(ptr(q), ptr(k), ptr(v), out(o), fout(lse), static_cast<const int*>(ptr(p.cu)),
                             st.data(), p.seqs, q.size(0), p.longest, hq, hkv, d, scale, causal, code, stream_of(q)));
  } else {
    if (want_lse) lse = empty({q.size(0), hq, q.size(1)}, at::kFloat, q);
    check(pk_attn_fwd(ptr(q), ptr(k), ptr(v), out(o), fout(lse), st.data(), q.size(0), q.size(1), hq,
                      hkv, d, scale, causal, code, stream_of(q)));
  }
  return {o, lse};
}

struct Attention : Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const std::optional<Tensor>& offsets, int64_t seqs, int64_t longest, bool causal, double scale) {
    const Tensor cu = offsets.value_or(Tensor());
    auto [o, lse] = attn_fwd(q, k, v, {cu, seqs, longest}, causal, (float)scale, true);
    ctx->save_for_backward({q, k, v, o, lse, cu});
    keep(ctx, {seqs, longest, causal});
    ctx->saved_data["s"] = scale;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor q = make_aligned_rows(saved[0]), k = make_aligned_rows(saved[1]), v = make_aligned_rows(saved[2]),
                 o = make_aligned_rows(saved[3]), lse = unpacked(saved[4]), cu = unpacked(saved[5]);
    const auto m = kept(ctx);
    const c10::DeviceGuard guard(q.device());
    const int64_t hq = q.size(-2), hkv = k.size(-2), d = q.size(-1);
    const Tensor g = make_aligned_rows(grads[0].to(q.scalar_type()));
    Tensor dq = empty(q.sizes(), q.scalar_type(), q), dk = empty(k.sizes(), k.scalar_type(), k),
           dv = empty(v.sizes(), v.scalar_type(), v);
    const auto st = strides_of<8>({&q, &k, &v, &o, &g, &dq, &dk, &dv});
    const float scale = (float)ctx->saved_data["s"].toDouble();
    const int code = code_of(q.scalar_type());
    if (cu.defined()) {
      const int64_t bytes = pk_attn_varlen_bwd_workspace(m[0], q.size(0), m[1], hq, hkv, d);
      Tensor ws = scratch(bytes, q);
      check(pk_attn_varlen_bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr(g), fptr(lse), out(ws), ws.numel(),
                               out(dq), out(dk), out(dv), static_cast<const int*>(ptr(cu)), st.data(), m[0], q.size(0), m[1], hq,
                               hkv, d, scale, m[2], code, stream_of(q)));
    } else {
      const int64_t bytes = pk_attn_bwd_workspace(q.size(0), q.size(1), hq, hkv, d);
      Tensor ws = scratch(bytes, q);
      check(pk_attn_bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr(g), fptr(lse), out(ws), ws.numel(), out(dq),
                        out(dk), out(dv), st.data(), q.size(0), q.size(1), hq, hkv, d, scale, m[2], code, stream_of(q)));
    }
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// q [.., hq, d] and k, v [.., hkv, d] of one type that the kernels read in place
bool attn_operands(const Tensor& q, const Tensor& k, const Tensor& v, int64_t dims) {
  if (q.dim() != dims || k.dim() != dims || k.sizes() != v.sizes()) return false;
  for (int64_t i = 0; i + 2 < dims; ++i)
    if (k.size(i) != q.size(i)) return false;
  const int64_t d = q.size(-1);
  return k.size(-1) == d && d % 8 == 0 && d <= 256 && q.size(-2) % k.size(-2) == 0 && q.scalar_type() == k.scalar_type() &&
         q.scalar_type() == v.scalar_type() && aligned_rows(q) && aligned_rows(k) && aligned_rows(v);
}

bool take_scale(PyObject* o, int64_t head_dim, double& scale) {
  if (o == Py_None) scale = std::pow((double)head_dim, -0.5);
  else if (PyFloat_CheckExact(o)) scale = PyFloat_AS_DOUBLE(o);
  else return false;
  return true;
}

// ---------------------------------------------------------------- the functions impls.py calls

PyObject* decline() { Py_RETURN_NOTIMPLEMENTED; }

PyObject* pair(Tensor a, Tensor b) {
  PyObject* t = PyTuple_New(2);
  if (t == nullptr) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(a)));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(b)));
  return t;
}

bool is_bool(PyObject* o) { return o == Py_True || o == Py_False; }

PyObject* py_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, b;
  if (n != 4 || watched() || !take(a[0], x) || x.dim() < 1 || !x.is_contiguous() || !take(a[1], w, &x) ||
      !norm_types(x, w) || !norm_vector(w, x) || !PyFloat_CheckExact(a[3]))
    return decline();
  if (a[2] != Py_None && !(take(a[2], b, &x) && b.scalar_type() == w.scalar_type() && norm_vector(b, x))) return decline();
  const double eps = PyFloat_AS_DOUBLE(a[3]);
  Tensor y;
  {
    pybind11::gil_scoped_release free;
    y = tracks({&x, &w, &b}) ? RmsNorm::apply(x, w, given(b), eps) : rms_norm_fwd(x, w, b, eps, nullptr);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyObject* py_add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, r, w;
  if (n != 5 || watched() || !take(a[0], x) || x.dim() < 1 || !x.is_contiguous() || !take(a[1], r, &x) ||
      r.sizes() != x.sizes() || r.scalar_type() != x.scalar_type() || !r.is_contiguous() || !take(a[2], w, &x) ||
      !norm_types(x, w) || !norm_vector(w, x) || !PyFloat_CheckExact(a[3]) || !PyFloat_CheckExact(a[4]))
    return decline();
  const double eps = PyFloat_AS_DOUBLE(a[3]), offset = PyFloat_AS_DOUBLE(a[4]);
  Tensor y, s;
  {
    pybind11::gil_scoped_release free;
    if (tracks({&x, &r, &w})) {
      auto o = AddRmsNorm::apply(x, r, w, eps, offset);
      y = o[0];
      s = o[1];
    } else {
      Tensor rstd;
      std::tie(y, s) = add_rms_norm_fwd(x, r, w, eps, offset, rstd);
    }
  }
  return pair(std::move(y), std::move(s));
  END_HANDLE_TH_ERRORS
}

PyObject* py_swiglu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor a, b;
  if (n != 2 || watched() || !take(args[0], a) || !take(args[1], b, &a) || a.sizes() != b.sizes() ||
      a.scalar_type() != b.scalar_type() || row_stride(a) < 0 || row_stride(b) < 0)
    return decline();
  Tensor y;
  {
    pybind11::gil_scoped_release free;
    y = tracks({&a, &b}) ? SwiGlu::apply(a, b) : swiglu_fwd(a, b);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyObject* py_rotary(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, cs, sn;
  if (n != 4 || watched() || !take(a[0], x) || x.dim() != 4 || !last_contiguous(x) || !take(a[1], cs, &x) ||
      !take(a[2], sn, &x) || cs.dim() != 2 || cs.sizes() != sn.sizes() || cs.scalar_type() != sn.scalar_type() ||
      cs.size(0) != x.size(1) || 2 * cs.size(1) > x.size(3) || !cs.is_contiguous() || !sn.is_contiguous() || !is_bool(a[3]))
    return decline();
  const bool interleaved = a[3] == Py_True;
  Tensor y;
  {
    pybind11::gil_scoped_release free;
    y = tracks({&x}) ? Rotary::apply(x, cs, sn, interleaved) : rotate(x, cs, sn, interleaved, false);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyObject* py_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, cs, sn;
  if (n != 4 || watched() || !take(a[0], q) || !take(a[1], k, &q) || !take(a[2], cs, &q) || !take(a[3], sn, &q) ||
      !rope_shapes(q, k, cs, sn))
    return decline();
  Tensor yq, yk;
  {
    pybind11::gil_scoped_release free;
    if (tracks({&q, &k})) {
      auto o = Rope::apply(q, k, cs, sn);
      yq = o[0];
      yk = o[1];
    } else {
      std::tie(yq, yk) = rope_call(q, k, cs, sn, false, promoted(q.scalar_type(), cs.scalar_type()));
    }
  }
  return pair(std::move(yq), std::move(yk));
  END_HANDLE_TH_ERRORS
}

PyObject* py_qk_norm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, qw, kw, cs, sn;
  if (n != 7 || watched() || !take(a[0], q) || !take(a[1], k, &q) || !take(a[2], qw, &q) || !take(a[3], kw, &q) ||
      !take(a[4], cs, &q) || !take(a[5], sn, &q) || !rope_shapes(q, k, cs, sn) || !PyFloat_CheckExact(a[6]))
    return decline();
  const int64_t d = q.size(3);
  const at::IntArrayRef width(&d, 1);
  if (qw.scalar_type() != kw.scalar_type() || !norm_types(q, qw) || qw.sizes() != width || kw.sizes() != width ||
      !dense(qw) || !dense(kw) || !dense(cs) || !dense(sn) || !aligned_rows(q) || !aligned_rows(k) ||
      pk_qk_norm_rope_bwd_workspace(q.size(0), q.size(1), k.size(1), q.size(2), d, code_of(q.scalar_type())) < 0)
    return decline();
  const double eps = PyFloat_AS_DOUBLE(a[6]);
  Tensor yq, yk;
  {
    pybind11::gil_scoped_release free;
    if (tracks({&q, &k, &qw, &kw})) {
      auto o = QkNormRope::apply(q, k, qw, kw, cs, sn, eps);
      yq = o[0];
      yk = o[1];
    } else {
      NormRopeOut o = norm_rope_fwd(q, k, qw, kw, cs, sn, eps);
      yq = o.yq;
      yk = o.yk;
    }
  }
  return pair(std::move(yq), std::move(yk));
  END_HANDLE_TH_ERRORS
}

PyObject* py_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v;
  double scale;
  if (n != 5 || watched() || !take(a[0], q) || !take(a[1], k, &q) || !take(a[2], v, &q) || !attn_operands(q, k, v, 4) ||
      !is_bool(a[3]) || !take_scale(a[4], q.size(3), scale))
    return decline();
  const bool causal = a[3] == Py_True;
  Tensor o;
  {
    pybind11::gil_scoped_release free;
    o = tracks({&q, &k, &v}) ? Attention::apply(q, k, v, std::optional<Tensor>(), (int64_t)0, (int64_t)0, causal, scale)
                             : attn_fwd(q, k, v, {}, causal, (float)scale, false).first;
  }
  return THPVariable_Wrap(std::move(o));
  END_HANDLE_TH_ERRORS
}

// q, k, v, the offsets on their device (int32, contiguous), number of sequences, longest, causal, scale
PyObject* py_attn_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v;
  Packing p;
  double scale;
  if (n != 8 || watched() || !take(a[0], q) || !take(a[1], k, &q) || !take(a[2], v, &q) || !attn_operands(q, k, v, 3) ||
      !THPVariable_CheckExact(a[3]) || !is_bool(a[6]) || !take_scale(a[7], q.size(2), scale))
    return decline();
  p.cu = THPVariable_Unpack(a[3]);
  p.seqs = PyLong_AsLongLong(a[4]);
  p.longest = PyLong_AsLongLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (p.cu.device() != q.device() || p.cu.scalar_type() != at::kInt || !p.cu.is_contiguous() ||
      p.cu.numel() != p.seqs + 1)
    return decline();
  const bool causal = a[6] == Py_True;
  Tensor o;
  {
    pybind11::gil_scoped_release free;
    o = tracks({&q, &k, &v}) ? Attention::apply(q, k, v, given(p.cu), p.seqs, p.longest, causal, scale)
                             : attn_fwd(q, k, v, p, causal, (float)scale, false).first;
  }
  return THPVariable_Wrap(std::move(o));
  END_HANDLE_TH_ERRORS
}

// The exception to raise, and torch's mode of a default device.
PyObject* py_set_types(PyObject*, PyObject* args) {
  PyObject *error, *context;
  if (!PyArg_ParseTuple(args, "OO", &error, &context)) return nullptr;
  Py_INCREF(error);
  Py_INCREF(context);
  Py_XSETREF(kernel_error, error);
  Py_XSETREF(device_context, context);
  Py_RETURN_NONE;
}

#define PK_FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    PK_FAST("rms_norm", py_rms_norm),         PK_FAST("add_rms_norm", py_add_rms_norm), PK_FAST("swiglu", py_swiglu),
    PK_FAST("rotary_embedding", py_rotary),   PK_FAST("rope", py_rope),                 PK_FAST("qk_norm_rope", py_qk_norm_rope),
    PK_FAST("attn", py_attn),                 PK_FAST("attn_varlen", py_attn_varlen),
    {"set_types", py_set_types, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "popcorn_amd._native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// With the library and torch this was compiled against, for the importer to compare.
PyMODINIT_FUNC PyInit__native() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && (PyModule_AddIntConstant(m, "ABI_VERSION", PK_ABI_VERSION) < 0 ||
                       PyModule_AddStringConstant(m, "TORCH_VERSION", PK_TORCH_VERSION) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
