// Native eager path of the public attention functions: the argument checks, the output and
// workspace allocations, the autograd nodes and the C ABI calls of flash_attn,
// flash_attn_varlen, flash_attn_decode and qk_norm_rope, in C++.
//
// Why: a training pass of the custom ops (torch.library ops whose bodies and autograd
// formulas are Python) costs about 175 us of host time on an MI355X host, most of it in the
// Python layers of the ops and of their backward, which runs on the autograd engine's device
// thread; the kernels of a 112M-model layer take 150-160 us, those of small batches 20-80.
//
// Each function takes a call only where plain eager mode gives it no meaning but the kernels
// themselves: exact torch.Tensor (or Parameter) arguments with the ordinary GPU dispatch
// keys, no dispatch or function mode, functorch transform, tracer or forward-mode tangent,
// and arguments inside the kernels' contract.  Otherwise it returns None and the caller goes
// on to the custom op, which serves every other case and raises every input error.  The
// autograd nodes save their tensors with save_for_backward (saved-tensor hooks and version
// checks apply), and a backward that is itself recorded or traced (create_graph, compiled
// autograd, modes) goes through the custom backward ops.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "ttfa.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using c10::DispatchKeySet;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------- when to take a call

// Keys of an ordinary GPU tensor; any other (functorch wrappers, Python subclasses, fake,
// functional, conjugate or negative views) sends the call to the custom op.
bool plain_tensor(const Tensor &t) {
  static const DispatchKeySet ordinary({DispatchKey::CUDA, DispatchKey::ADInplaceOrView,
                                        DispatchKey::AutogradCUDA, DispatchKey::AutocastCUDA});
  return t.defined() && t.is_cuda() && (t.key_set() | ordinary) == ordinary &&
         !t._fw_grad(/*level=*/0).defined();
}

bool plain_mode() {
  static const DispatchKeySet special(
      {DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::PythonDispatcher,
       DispatchKey::PreDispatch, DispatchKey::Functionalize, DispatchKey::Tracer,
       DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
       DispatchKey::FuncTorchVmapMode, DispatchKey::VmapMode, DispatchKey::DeferredInit});
  return !c10::impl::tls_local_dispatch_key_set().included_.has_any(special) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0;
}

// Whether autograd records the call: as the dispatcher would decide it.
bool recorded(std::initializer_list<const Tensor *> ts) {
  if (!c10::GradMode::is_enabled() ||
      c10::impl::tls_is_dispatch_key_excluded(DispatchKey::AutogradCUDA))
    return false;
  for (const Tensor *t : ts)
    if (t->requires_grad()) return true;
  return false;
}

// ------------------------------------------------------------------------------- helpers

void *stream_of(const Tensor &t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Raises the package's TTFAError for a nonzero status.
void check(int rc) {
  if (rc == 0) return;
  pybind11::gil_scoped_acquire gil;
  pybind11::module_::import("tinytrain_amd._lib").attr("check")(rc);
}

Tensor f32(const Tensor &like, at::IntArrayRef shape) {
  return at::empty(shape, like.options().dtype(at::kFloat));
}

// What empty_like gives for the contiguous tensors of these calls.
Tensor same(const Tensor &like) { return at::empty(like.sizes(), like.options()); }

float scale_of(int64_t D) { return (float)(1.0 / std::sqrt((double)D)); }

constexpr int64_t kIntMax = 0x7fffffff;

bool all_int(at::IntArrayRef sizes) {
  for (int64_t s : sizes)
    if (s > kIntMax) return false;
  return true;
}

// A backward pass that nothing records or traces.
bool plain_backward() { return !c10::GradMode::is_enabled() && plain_mode(); }

template <class Sig>
const c10::TypedOperatorHandle<Sig> op(const char *name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}

using Grads3 = std::tuple<Tensor, Tensor, Tensor>;

// ---------------------------------------------------------------------- batched attention

bool takes_attn(const Tensor &q, const Tensor &k, const Tensor &v) {
  if (!plain_tensor(q) || !plain_tensor(k) || !plain_tensor(v)) return false;
  if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes()) return false;
  if (k.size(0) != q.size(0) || k.size(2) != q.size(2) || k.size(3) != q.size(3)) return false;
  const auto dt = q.scalar_type();
  return k.size(1) >= 1 && q.size(1) % k.size(1) == 0 && (q.size(3) == 64 || q.size(3) == 128) &&
         (dt == at::kBFloat16 || dt == at::kFloat) && k.scalar_type() == dt &&
         v.scalar_type() == dt && k.device() == q.device() && v.device() == q.device() &&
         q.is_contiguous() && k.is_contiguous() && v.is_contiguous() && all_int(q.sizes());
}

int dtype_of(const Tensor &t) { return t.scalar_type() == at::kFloat ? TTFA_F32 : TTFA_BF16; }

std::pair<Tensor, Tensor> attn_fwd(const Tensor &q, const Tensor &k, const Tensor &v) {
  RECORD_FUNCTION("tinytrain::flash_attn_fwd", c10::ArrayRef<const c10::IValue>());
  const c10::DeviceGuard on(q.device());
  Tensor o = same(q), M = f32(q, {q.size(0), q.size(1), q.size(2)});
  check(ttfa_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                 o.mutable_data_ptr(), M.mutable_data_ptr<float>(), (int)q.size(0),
                 (int)q.size(1), (int)k.size(1), (int)q.size(2), (int)q.size(3), dtype_of(q),
                 scale_of(q.size(3)), stream_of(q)));
  return {o, M};
}

Grads3 attn_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o,
                const Tensor &dout, const Tensor &M) {
  RECORD_FUNCTION("tinytrain::flash_attn_bwd", c10::ArrayRef<const c10::IValue>());
  const c10::DeviceGuard on(q.device());
  const Tensor g = dout.contiguous();
  const int B = (int)q.size(0), Hq = (int)q.size(1), Hkv = (int)k.size(1), T = (int)q.size(2),
            D = (int)q.size(3), dt = dtype_of(q);
  const long long bytes = ttfa_bwd_workspace_bytes(B, Hq, Hkv, T, D, dt);
  Tensor ws = f32(q, {std::max<int64_t>(bytes / 4, 1)});
  Tensor dq = same(q), dk = same(k), dv = same(v);
  check(ttfa_bwd_ws(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                    o.const_data_ptr(), g.const_data_ptr(), M.const_data_ptr<float>(),
                    ws.mutable_data_ptr<float>(), dq.mutable_data_ptr(), dk.mutable_data_ptr(),
                    dv.mutable_data_ptr(), B, Hq, Hkv, T, D, dt, scale_of(D), stream_of(q)));
  return {dq, dk, dv};
}

// A gradient of shape `sizes` and type dt beside q; any strides (it is made contiguous).
bool grad_of(const Tensor &g, const Tensor &q, at::IntArrayRef sizes, at::ScalarType dt) {
  return plain_tensor(g) && g.sizes() == sizes && g.scalar_type() == dt && g.device() == q.device();
}

// A saved tensor as the forward made it: saved-tensor hooks may hand back others, which the
// custom op makes contiguous or refuses.
bool saved_as(const Tensor &t, const Tensor &q, at::IntArrayRef sizes, at::ScalarType dt) {
  return grad_of(t, q, sizes, dt) && t.is_contiguous();
}

struct FlashAttn : torch::autograd::Function<FlashAttn> {
  static constexpr bool is_traceable = true;

  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v) {
    auto [o, M] = attn_fwd(q, k, v);
    ctx->save_for_backward({q, k, v, o, M});
    return o;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &g = grads[0];
    const Tensor &q = s[0];
    const bool native = plain_backward() && takes_attn(q, s[1], s[2]) &&
                        grad_of(g, q, q.sizes(), q.scalar_type()) &&
                        saved_as(s[3], q, q.sizes(), q.scalar_type()) &&
                        saved_as(s[4], q, q.sizes().slice(0, 3), at::kFloat);
    Grads3 d = native
                   ? attn_bwd(s[0], s[1], s[2], s[3], g, s[4])
                   : op<Grads3(const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                               const Tensor &, const Tensor &)>("tinytrain::flash_attn_bwd")
                         .call(s[0], s[1], s[2], s[3], g, s[4]);
    return {std::get<0>(d), std::get<1>(d), std::get<2>(d)};
  }
};

// -------------------------------------------------------------- packed sequences (varlen)

bool takes_varlen(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu,
                  int64_t max_seqlen) {
  if (!plain_tensor(q) || !plain_tensor(k) || !plain_tensor(v) || !plain_tensor(cu)) return false;
  if (q.dim() != 3 || k.dim() != 3 || k.sizes() != v.sizes()) return false;
  if (k.size(1) != q.size(1) || k.size(2) != q.size(2)) return false;
  const auto bf = at::kBFloat16;
  return k.size(0) >= 1 && q.size(0) % k.size(0) == 0 && (q.size(2) == 64 || q.size(2) == 128) &&
         q.scalar_type() == bf && k.scalar_type() == bf && v.scalar_type() == bf &&
         cu.dim() == 1 && cu.numel() >= 2 && cu.scalar_type() == at::kInt && cu.is_contiguous() &&
         max_seqlen >= 1 && max_seqlen <= kIntMax && q.size(1) >= 1 &&
         k.device() == q.device() && v.device() == q.device() && cu.device() == q.device() &&
         q.is_contiguous() && k.is_contiguous() && v.is_contiguous() && all_int(q.sizes()) &&
         all_int(cu.sizes());
}

std::pair<Tensor, Tensor> varlen_fwd(const Tensor &q, const Tensor &k, const Tensor &v,
                                     const Tensor &cu, int64_t max_seqlen) {
  RECORD_FUNCTION("tinytrain::flash_attn_varlen_fwd", c10::ArrayRef<const c10::IValue>());
  const c10::DeviceGuard on(q.device());
  Tensor o = same(q), M = f32(q, {q.size(0), q.size(1)});
  check(ttfa_varlen_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                        o.mutable_data_ptr(), M.mutable_data_ptr<float>(),
                        cu.const_data_ptr<int>(), (int)cu.numel() - 1, (int)q.size(1),
                        (int)max_seqlen, (int)q.size(0), (int)k.size(0), (int)q.size(2),
                        TTFA_BF16, scale_of(q.size(2)), stream_of(q)));
  return {o, M};
}

Grads3 varlen_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o,
                  const Tensor &dout, const Tensor &M, const Tensor &cu, int64_t max_seqlen) {
  RECORD_FUNCTION("tinytrain::flash_attn_varlen_bwd", c10::ArrayRef<const c10::IValue>());
  const c10::DeviceGuard on(q.device());
  const Tensor g = dout.contiguous();
  Tensor delta = f32(q, {q.size(0), q.size(1)});
  Tensor dq = same(q), dk = same(k), dv = same(v);
  check(ttfa_varlen_bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                        o.const_data_ptr(), g.const_data_ptr(), M.const_data_ptr<float>(),
                        delta.mutable_data_ptr<float>(), dq.mutable_data_ptr(),
                        dk.mutable_data_ptr(), dv.mutable_data_ptr(), cu.const_data_ptr<int>(),
                        (int)cu.numel() - 1, (int)q.size(1), (int)max_seqlen, (int)q.size(0),
                        (int)k.size(0), (int)q.size(2), TTFA_BF16, scale_of(q.size(2)),
                        stream_of(q)));
  return {dq, dk, dv};
}

struct FlashAttnVarlen : torch::autograd::Function<FlashAttnVarlen> {
  static constexpr bool is_traceable = true;

  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                        const Tensor &cu, int64_t max_seqlen) {
    auto [o, M] = varlen_fwd(q, k, v, cu, max_seqlen);
    ctx->save_for_backward({q, k, v, o, M, cu});
    ctx->saved_data["max_seqlen"] = max_seqlen;
    return o;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const int64_t longest = ctx->saved_data["max_seqlen"].toInt();
    const Tensor &g = grads[0], &q = s[0];
    const bool native = plain_backward() && takes_varlen(q, s[1], s[2], s[5], longest) &&
                        grad_of(g, q, q.sizes(), q.scalar_type()) &&
                        saved_as(s[3], q, q.sizes(), q.scalar_type()) &&
                        saved_as(s[4], q, q.sizes().slice(0, 2), at::kFloat);
    Grads3 d =
        native
            ? varlen_bwd(s[0], s[1], s[2], s[3], g, s[4], s[5], longest)
            : op<Grads3(const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                        const Tensor &, const Tensor &, const Tensor &, c10::SymInt)>(
                  "tinytrain::flash_attn_varlen_bwd")
                  .call(s[0], s[1], s[2], s[3], g, s[4], s[5], c10::SymInt(longest));
    return {std::get<0>(d), std::get<1>(d), std::get<2>(d), Tensor(), Tensor()};
  }
};

// --------------------------------------------------------------------------------- decode

bool takes_decode(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &lens) {
  if (!plain_tensor(q) || !plain_tensor(k) || !plain_tensor(v) || !plain_tensor(lens)) return false;
  if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes()) return false;
  if (k.size(0) != q.size(0) || k.size(3) != q.size(3)) return false;
  const auto bf = at::kBFloat16;
  const int64_t Hkv = k.size(1);
  return Hkv >= 1 && q.size(1) % Hkv == 0 && (q.size(3) == 64 || q.size(3) == 128) &&
         (q.size(1) / Hkv) * q.size(2) <= 32 && q.scalar_type() == bf && k.scalar_type() == bf &&
         v.scalar_type() == bf && q.is_contiguous() && k.is_contiguous() && v.is_contiguous() &&
         lens.dim() == 1 && lens.size(0) == q.size(0) && lens.scalar_type() == at::kInt &&
         k.device() == q.device() && v.device() == q.device() && lens.device() == q.device() &&
         all_int(q.sizes()) && all_int(k.sizes());
}

// ------------------------------------------------------------------------------- prologue

struct Prologue {
  Tensor q, k, v, wq, wk, cos, sin;

  bool takes() const {
    for (const Tensor *t : {&q, &k, &v, &wq, &wk, &cos, &sin})
      if (!plain_tensor(*t) || t->device() != q.device()) return false;
    if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes()) return false;
    const int64_t T = q.size(1), D = q.size(3), Hkv = k.size(2);
    const auto bf = at::kBFloat16;
    if (k.size(0) != q.size(0) || k.size(1) != T || k.size(3) != D || Hkv < 1 ||
        q.size(2) % Hkv != 0 || (D != 64 && D != 128))
      return false;
    for (const Tensor *w : {&wq, &wk})
      if (w->dim() != 1 || w->size(0) != D || !w->is_floating_point()) return false;
    return cos.sizes() == sin.sizes() && cos.dim() == 2 && cos.size(0) >= T && cos.size(1) == D &&
           cos.is_floating_point() && sin.is_floating_point() && q.scalar_type() == bf &&
           k.scalar_type() == bf && v.scalar_type() == bf && q.is_contiguous() &&
           k.is_contiguous() && v.is_contiguous() && all_int(q.sizes());
  }
};

// Rows 0..T-1 of the RoPE tables: fp32 ones go to the kernels as they are (rounded to bf16
// there, the reference's cos.to(x.dtype)); anything else is cast to bf16 first.
struct Tables {
  Tensor cos, sin;
  int dtype;

  Tables(const Tensor &c, const Tensor &s, int64_t T) {
    auto direct = [](const Tensor &t) {
      return t.scalar_type() == at::kFloat && t.is_contiguous() &&
             ((uintptr_t)t.const_data_ptr() & 15) == 0;
    };
    auto cast = [&](const Tensor &t) { return t.narrow(0, 0, T).to(at::kBFloat16).contiguous(); };
    const bool as_is = direct(c) && direct(s);
    cos = as_is ? c : cast(c);
    sin = as_is ? s : cast(s);
    dtype = as_is ? TTFA_F32 : TTFA_BF16;
  }
};

Tensor weight(const Tensor &w) { return w.to(at::kFloat).contiguous(); }

struct PrologueOut {
  Tensor q, k, v, rq, rk;
};

PrologueOut prologue_fwd(const Prologue &p, double eps) {
  RECORD_FUNCTION("tinytrain::qk_norm_rope_fwd", c10::ArrayRef<const c10::IValue>());
  const int64_t B = p.q.size(0), T = p.q.size(1), Hq = p.q.size(2), D = p.q.size(3);
  const int64_t Hkv = p.k.size(2);
  const c10::DeviceGuard on(p.q.device());
  const Tables tab(p.cos, p.sin, T);
  const Tensor wq = weight(p.wq), wk = weight(p.wk);
  PrologueOut r{at::empty({B, Hq, T, D}, p.q.options()), at::empty({B, Hkv, T, D}, p.q.options()),
                at::empty({B, Hkv, T, D}, p.q.options()), f32(p.q, {B, T, Hq}),
                f32(p.q, {B, T, Hkv})};
  check(ttfa_qk_prologue_fwd_tables(
      p.q.const_data_ptr(), p.k.const_data_ptr(), p.v.const_data_ptr(), wq.const_data_ptr<float>(),
      wk.const_data_ptr<float>(), tab.cos.const_data_ptr(), tab.sin.const_data_ptr(), tab.dtype,
      r.q.mutable_data_ptr(), r.k.mutable_data_ptr(), r.v.mutable_data_ptr(), r.rq.mutable_data_ptr<float>(),
      r.rk.mutable_data_ptr<float>(), (int)B, (int)T, (int)Hq, (int)Hkv, (int)D, (float)eps,
      stream_of(p.q)));
  return r;
}

using Grads5 = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;

Grads5 prologue_bwd(const Tensor &gq, const Tensor &gk, const Tensor &gv, const Prologue &p,
                    const Tensor &rq, const Tensor &rk) {
  RECORD_FUNCTION("tinytrain::qk_norm_rope_bwd", c10::ArrayRef<const c10::IValue>());
  const int64_t B = p.q.size(0), T = p.q.size(1), Hq = p.q.size(2), D = p.q.size(3);
  const int64_t Hkv = p.k.size(2);
  const c10::DeviceGuard on(p.q.device());
  const Tables tab(p.cos, p.sin, T);
  const Tensor wq = weight(p.wq), wk = weight(p.wk);
  const Tensor dq = gq.contiguous(), dk = gk.contiguous(), dv = gv.contiguous();
  Tensor dq_raw = same(p.q), dk_raw = same(p.k), dv_raw = same(p.k);
  Tensor dwq = f32(p.q, {D}), dwk = f32(p.q, {D});
  const long long bytes =
      ttfa_qk_prologue_workspace_bytes((int)B, (int)T, (int)Hq, (int)Hkv, (int)D);
  if (bytes < 0) check(TTFA_E_SEQ);
  Tensor ws = f32(p.q, {std::max<int64_t>(bytes / 4, 4)});
  check(ttfa_qk_prologue_bwd_tables(
      dq.const_data_ptr(), dk.const_data_ptr(), dv.const_data_ptr(), p.q.const_data_ptr(),
      p.k.const_data_ptr(), wq.const_data_ptr<float>(), wk.const_data_ptr<float>(),
      tab.cos.const_data_ptr(), tab.sin.const_data_ptr(), tab.dtype, rq.const_data_ptr<float>(),
      rk.const_data_ptr<float>(), dq_raw.mutable_data_ptr(), dk_raw.mutable_data_ptr(),
      dv_raw.mutable_data_ptr(), dwq.mutable_data_ptr<float>(), dwk.mutable_data_ptr<float>(),
      ws.mutable_data_ptr<float>(), (int)B, (int)T, (int)Hq, (int)Hkv, (int)D, stream_of(p.q)));
  return {dq_raw, dk_raw, dv_raw, dwq.to(p.wq.scalar_type()), dwk.to(p.wk.scalar_type())};
}

struct QkNormRope : torch::autograd::Function<QkNormRope> {
  static constexpr bool is_traceable = true;

  static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k,
                               const Tensor &v, const Tensor &wq, const Tensor &wk,
                               const Tensor &cos, const Tensor &sin, double eps) {
    PrologueOut r = prologue_fwd({q, k, v, wq, wk, cos, sin}, eps);
    ctx->save_for_backward({q, k, wq, wk, cos, sin, r.rq, r.rk});
    return {r.q, r.k, r.v};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Prologue p{s[0], s[1], s[1], s[2], s[3], s[4], s[5]};
    const Tensor &gq = grads[0], &gk = grads[1], &gv = grads[2];
    const Tensor &q = s[0], &k = s[1];
    bool native = plain_backward() && p.takes();
    if (native) {
      const int64_t B = q.size(0), T = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
      const auto bf = at::kBFloat16;
      native = grad_of(gq, q, {B, Hq, T, D}, bf) && grad_of(gk, q, {B, Hkv, T, D}, bf) &&
               grad_of(gv, q, {B, Hkv, T, D}, bf) && saved_as(s[6], q, {B, T, Hq}, at::kFloat) &&
               saved_as(s[7], q, {B, T, Hkv}, at::kFloat);
    }
    Grads5 d = native ? prologue_bwd(gq, gk, gv, p, s[6], s[7])
                      : op<Grads5(const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                                  const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                                  const Tensor &, const Tensor &, const Tensor &)>(
                            "tinytrain::qk_norm_rope_bwd")
                            .call(gq, gk, gv, s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]);
    return {std::get<0>(d), std::get<1>(d), std::get<2>(d), std::get<3>(d), std::get<4>(d),
            Tensor(), Tensor(), Tensor()};
  }
};

// ------------------------------------------------------------------------ Python bindings

// The first n arguments as tensors; false when one of them is not an exact Tensor.
template <size_t N>
bool unpack(PyObject *const *args, Tensor (&out)[N]) {
  for (size_t i = 0; i < N; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;
    out[i] = THPVariable_Unpack(args[i]);
  }
  return true;
}

bool arity(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
  return false;
}

PyObject *pack(std::initializer_list<Tensor> ts) {
  PyObject *r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) throw python_error();
  Py_ssize_t i = 0;
  for (const Tensor &t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t));
  return r;
}

PyObject *py_flash_attn(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arity(n, 3)) return nullptr;
  Tensor t[3];
  if (!unpack(args, t) || !plain_mode() || !takes_attn(t[0], t[1], t[2])) Py_RETURN_NONE;
  return THPVariable_Wrap(recorded({&t[0], &t[1], &t[2]}) ? FlashAttn::apply(t[0], t[1], t[2])
                                                          : attn_fwd(t[0], t[1], t[2]).first);
  END_HANDLE_TH_ERRORS
}

PyObject *py_flash_attn_varlen(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arity(n, 5)) return nullptr;
  Tensor t[4];
  const int64_t longest = PyLong_AsLongLong(args[4]);
  if (longest == -1 && PyErr_Occurred()) return nullptr;
  if (!unpack(args, t) || !plain_mode() || !takes_varlen(t[0], t[1], t[2], t[3], longest))
    Py_RETURN_NONE;
  return THPVariable_Wrap(recorded({&t[0], &t[1], &t[2]})
                              ? FlashAttnVarlen::apply(t[0], t[1], t[2], t[3], longest)
                              : varlen_fwd(t[0], t[1], t[2], t[3], longest).first);
  END_HANDLE_TH_ERRORS
}

PyObject *py_flash_attn_decode(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arity(n, 4)) return nullptr;
  Tensor t[4];
  if (!unpack(args, t) || !plain_mode() || !takes_decode(t[0], t[1], t[2], t[3]) ||
      recorded({&t[0], &t[1], &t[2]}))
    Py_RETURN_NONE;
  const Tensor &q = t[0], &k = t[1], &v = t[2], lens = t[3].contiguous();
  const int B = (int)q.size(0), Hq = (int)q.size(1), Tq = (int)q.size(2), D = (int)q.size(3);
  const int Hkv = (int)k.size(1), L = (int)k.size(2);
  const long long bytes = ttfa_decode_workspace_bytes(B, Hq, Hkv, Tq, L, D);
  if (bytes < 0) Py_RETURN_NONE;
  RECORD_FUNCTION("tinytrain::flash_attn_decode", c10::ArrayRef<const c10::IValue>());
  const c10::DeviceGuard on(q.device());
  Tensor ws = f32(q, {bytes / 4 + 4}), o = same(q), lse = f32(q, {B, Hq, Tq});
  check(ttfa_decode_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                        lens.const_data_ptr<int>(), o.mutable_data_ptr(),
                        lse.mutable_data_ptr<float>(), ws.mutable_data_ptr<float>(), B, Hq, Hkv,
                        Tq, L, D, TTFA_BF16, scale_of(D), stream_of(q)));
  return pack({o, lse});
  END_HANDLE_TH_ERRORS
}

PyObject *py_qk_norm_rope(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arity(n, 8)) return nullptr;
  Tensor t[7];
  const double eps = PyFloat_AsDouble(args[7]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  if (!unpack(args, t) || !plain_mode()) Py_RETURN_NONE;
  const Prologue p{t[0], t[1], t[2], t[3], t[4], t[5], t[6]};
  if (!p.takes()) Py_RETURN_NONE;
  if (recorded({&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6]})) {
    const auto r = QkNormRope::apply(t[0], t[1], t[2], t[3], t[4], t[5], t[6], eps);
    return pack({r[0], r[1], r[2]});
  }
  const PrologueOut r = prologue_fwd(p, eps);
  return pack({r.q, r.k, r.v});
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"flash_attn", (PyCFunction)(void (*)(void))py_flash_attn, METH_FASTCALL,
     "o of flash_attn(q, k, v), or None where the custom op has to take the call."},
    {"flash_attn_varlen", (PyCFunction)(void (*)(void))py_flash_attn_varlen, METH_FASTCALL,
     "o of flash_attn_varlen(q, k, v, cu_seqlens, max_seqlen), or None."},
    {"flash_attn_decode", (PyCFunction)(void (*)(void))py_flash_attn_decode, METH_FASTCALL,
     "(o, lse) of flash_attn_decode(q, k_cache, v_cache, cache_seqlens), or None."},
    {"qk_norm_rope", (PyCFunction)(void (*)(void))py_qk_norm_rope, METH_FASTCALL,
     "(q, k, v) of qk_norm_rope(q, k, v, wq, wk, cos, sin, eps), or None."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ttfa_torch",
                      "Native eager path of the attention functions.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__ttfa_torch() { return PyModule_Create(&module); }
