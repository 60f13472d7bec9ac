// torch_ops.cpp — the operators' host path: argument checks, output
// allocation, the C ABI call and the autograd node, in native code.
//
// In Python one forward and backward of an operator (torch.autograd.Function,
// ctypes argument lists) costs 55-155 us of host time on two threads, more than
// the kernels of most calls take.  The functions below do the same work for a
// plain call (measured, forward and backward, us: the attention block of a
// GPT-2-small layer 184 -> 95, its kernels' time; rope_qk 121 -> 57; add_rms_norm
// 153 -> 65; swiglu 107 -> 71, its kernels' time; the fp32 forward of B1 H12 S256
// 15 -> 8): exact torch.Tensor (or Parameter) arguments on one GPU, shapes,
// dtypes and layouts the kernels take, no dispatch or function mode, functorch
// transform, forward-mode tangent or tracing in effect.  For anything else they
// return None and do nothing, and the caller takes the Python operator, which
// handles or refuses the call as always; so every error message comes from
// there.  The nodes keep what the Python operators keep, through SavedVariable
// (saved-tensor hooks and in-place checks apply; what a hook hands back is checked
// before a kernel indexes it).
//
// Host code only.  The entry points of libmi_attn.so are bound by address
// (bind()), so that this module runs whichever copy of it Python loaded.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <optional>

#include "../../include/mi_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

#define MI_BOUND(X)                                                                        \
  X(mi_status_str) X(mi_last_error) X(mi_attn_fwd) X(mi_attn_bwd) X(mi_attn_bwd_rope)      \
  X(mi_rope) X(mi_rope_qk) X(mi_xent_fwd) X(mi_xent_bwd) X(mi_rmsnorm_fwd)                 \
  X(mi_rmsnorm_bwd_workspace) X(mi_rmsnorm_bwd) X(mi_rmsnorm_bwd_acc)                      \
  X(mi_rmsnorm_add_fwd) X(mi_rmsnorm_add_bwd) X(mi_rmsnorm_add_bwd_acc) X(mi_swiglu_fwd)   \
  X(mi_swiglu_bwd) X(mi_wgrad_suits) X(mi_wgrad_workspace) X(mi_wgrad)

struct Bound {
#define X(f) decltype(&::f) f = nullptr;
  MI_BOUND(X)
#undef X
  PyObject* error = nullptr;  // MiError
} lib;

// A non-OK status as the Python binding reports it: MiError("what: name (text)").
void check(mi_status st, const char* what) {
  if (st == MI_OK) return;
  const std::string text =
      std::string(what) + ": " + lib.mi_status_str(st) + " (" + lib.mi_last_error() + ")";
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(lib.error, text.c_str());
  python_error e;
  e.persist();
  throw std::move(e);
}

// ---------------------------------------------------------------------------
// Plain calls
// ---------------------------------------------------------------------------
bool plain_context() {
  return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
         !torch::jit::tracer::isTracing() &&
         !c10::impl::tls_is_dispatch_key_included(
             c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool plain(PyObject* o, Tensor& t) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::ZeroTensor, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::Negative});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.numel() > 0 &&
         !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined();
}

// The C ABI's dtype code, -1 for others.
int code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return MI_F32;
    case at::kHalf: return MI_F16;
    case at::kBFloat16: return MI_BF16;
    default: return -1;
  }
}
mi_dtype dt(const Tensor& t) { return (mi_dtype)code(t); }

template <typename... T>
bool one_device(const Tensor& a, const T&... rest) {
  return ((rest.device() == a.device()) && ...);
}

void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef sizes, const Tensor& like) { return at::empty(sizes, like.options()); }
Tensor empty_f32(at::IntArrayRef sizes, const Tensor& like) {
  return at::empty(sizes, like.options().dtype(at::kFloat));
}

// Rows over the last dim as the C ABI takes them: count and stride; nothing if
// the leading dims are not one row axis or rows overlap.  The strides of a
// contiguous tensor's size-1 dims mean nothing: its rows lie one behind the other.
struct Rows {
  int64_t n, stride;
};
std::optional<Rows> rows_of(const Tensor& t) {
  const int64_t d = t.dim(), h = t.size(-1);
  if (t.is_contiguous()) return Rows{h ? t.numel() / h : 0, h};
  if (t.stride(-1) != 1) return std::nullopt;
  const int64_t rs = t.stride(-2);
  int64_t n = 1, expect = rs;
  for (int64_t i = d - 2; i >= 0; --i) {
    if (t.size(i) != 1 && t.stride(i) != expect) return std::nullopt;
    expect *= t.size(i);
    n *= t.size(i);
  }
  if (n > 1 && rs < h) return std::nullopt;
  return Rows{n, rs};
}
Tensor as_rows(const Tensor& t) { return rows_of(t) ? t : t.contiguous(); }
Rows rows(const Tensor& t) {
  const auto r = rows_of(t);
  TORCH_CHECK_VALUE(r, "the last dim must have unit stride and the leading dims one row axis; got ",
                    t.sizes(), " / ", t.strides());
  return *r;
}

// A tensor that a backward indexes as dense: what was saved may come back
// through a saved-tensor hook as something else.
void dense(const char* name, const Tensor& t, at::IntArrayRef sizes, at::ScalarType type,
           const Tensor& like) {
  TORCH_CHECK_VALUE(t.defined() && t.sizes() == sizes && t.scalar_type() == type &&
                        t.is_contiguous() && t.device() == like.device(),
                    "saved ", name, " must be a contiguous ", type, " ", sizes, " tensor on ",
                    like.device(), "; got ", t.scalar_type(), " ", t.sizes(), " / ", t.strides(),
                    " on ", t.device());
}
// The same for one that is read through its strides.
void strided(const char* name, const Tensor& t, at::IntArrayRef sizes, at::ScalarType type,
             const Tensor& like) {
  TORCH_CHECK_VALUE(t.defined() && t.sizes() == sizes && t.scalar_type() == type &&
                        t.device() == like.device(),
                    name, " must be a ", type, " ", sizes, " tensor on ", like.device(), "; got ",
                    t.scalar_type(), " ", t.sizes(), " on ", t.device());
}

// ---------------------------------------------------------------------------
// Flash attention
// ---------------------------------------------------------------------------
// t, or a copy if the kernels cannot read it in place (flash_attn._kernel_ready).
bool rows16(const Tensor& t) {
  if (((uintptr_t)t.data_ptr()) % 16) return false;
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if ((t.stride(i) * t.element_size()) % 16) return false;
  return true;
}
Tensor kernel_ready(const Tensor& t) {
  return t.stride(-1) == 1 && rows16(t) ? t : t.contiguous();
}

bool attn_ok(const Tensor& q, const Tensor& k, const Tensor& v) {
  return q.dim() == 4 && q.sizes() == k.sizes() && q.sizes() == v.sizes() && code(q) >= 0 &&
         q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type() &&
         one_device(q, k, v) && q.size(3) > 1;
}

struct AttnOut {
  Tensor o, lse;
};
AttnOut attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, bool causal) {
  const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
  AttnOut r{empty({B, H, S, D}, q), empty_f32({B, H, S}, q)};
  check(lib.mi_attn_fwd(dt(q), B, H, S, D, causal, 1.0 / std::sqrt((double)D), q.data_ptr(),
                        q.strides().data(), k.data_ptr(), k.strides().data(), v.data_ptr(),
                        v.strides().data(), r.o.data_ptr(), r.o.strides().data(),
                        r.lse.data_ptr<float>(), stream(q)),
        "mi_attn_fwd");
  return r;
}

struct FlashAttn : torch::autograd::Function<FlashAttn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_,
                        bool causal) {
    const Tensor q = kernel_ready(q_), k = kernel_ready(k_), v = kernel_ready(v_);
    AttnOut r = attn_fwd(q, k, v, causal);
    ctx->save_for_backward({q, k, v, r.lse, r.o});
    ctx->saved_data["causal"] = causal;
    return r.o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &lse = s[3], &o = s[4];
    Tensor go = kernel_ready(grads[0]);
    if (go.scalar_type() != q.scalar_type()) go = go.to(q.scalar_type());
    const at::ScalarType type = q.scalar_type();
    strided("saved q", q, go.sizes(), go.scalar_type(), go);
    strided("saved k", k, q.sizes(), type, q);
    strided("saved v", v, q.sizes(), type, q);
    strided("saved o", o, q.sizes(), type, q);
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
    dense("lse", lse, {B, H, S}, at::kFloat, q);
    Tensor ws = empty_f32({2, B, H, S}, q);
    Tensor dq = empty({B, H, S, D}, q), dk = empty({B, H, S, D}, q), dv = empty({B, H, S, D}, q);
    check(lib.mi_attn_bwd(dt(q), B, H, S, D, ctx->saved_data["causal"].toBool(),
                          1.0 / std::sqrt((double)D), q.data_ptr(), q.strides().data(),
                          k.data_ptr(), k.strides().data(), v.data_ptr(), v.strides().data(),
                          o.data_ptr(), o.strides().data(), go.data_ptr(), go.strides().data(),
                          lse.data_ptr<float>(), ws.data_ptr<float>(), dq.data_ptr(),
                          dq.strides().data(), dk.data_ptr(), dk.strides().data(), dv.data_ptr(),
                          dv.strides().data(), stream(q)),
          "mi_attn_bwd");
    return {dq, dk, dv, Tensor()};
  }
};

// ---------------------------------------------------------------------------
// Rotary embedding
// ---------------------------------------------------------------------------
bool tables_ok(const Tensor& cos, const Tensor& sin, int64_t S, int64_t D) {
  for (const Tensor* t : {&cos, &sin})
    if (t->dim() != 2 || t->size(0) < S || t->size(1) < D / 2 || code(*t) < 0) return false;
  return cos.scalar_type() == sin.scalar_type() && D % 2 == 0;
}

void check_tables(const variable_list& s, const Tensor& g) {
  TORCH_CHECK_VALUE(tables_ok(s[0], s[1], g.size(0), g.size(3)) && one_device(g, s[0], s[1]),
                    "saved cos / sin no longer fit the gradient");
}

void rope(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& out, bool inverse) {
  check(lib.mi_rope(dt(x), dt(cos), x.size(0), x.size(1), x.size(2), x.size(3), inverse,
                    x.data_ptr(), x.strides().data(), cos.data_ptr(), cos.strides().data(),
                    sin.data_ptr(), sin.strides().data(), out.data_ptr(), out.strides().data(),
                    stream(x)),
        "mi_rope");
}
void rope_qk(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin,
             const Tensor& qo, const Tensor& ko, bool inverse) {
  check(lib.mi_rope_qk(dt(q), dt(cos), q.size(0), q.size(1), q.size(2), q.size(3), inverse,
                       q.data_ptr(), q.strides().data(), k.data_ptr(), k.strides().data(),
                       cos.data_ptr(), cos.strides().data(), sin.data_ptr(), sin.strides().data(),
                       qo.data_ptr(), qo.strides().data(), ko.data_ptr(), ko.strides().data(),
                       stream(q)),
        "mi_rope_qk");
}

struct RoPE : torch::autograd::Function<RoPE> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cos,
                        const Tensor& sin) {
    Tensor out = at::empty_like(x);
    rope(x, cos, sin, out, false);
    ctx->save_for_backward({cos, sin});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    check_tables(s, grads[0]);
    Tensor dx = at::empty_like(grads[0]);
    rope(grads[0], s[0], s[1], dx, true);
    return {dx, Tensor(), Tensor()};
  }
};

struct RoPEQK : torch::autograd::Function<RoPEQK> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k,
                               const Tensor& cos, const Tensor& sin) {
    Tensor qo = at::empty_like(q), ko = at::empty_like(k);
    rope_qk(q, k, cos, sin, qo, ko, false);
    ctx->save_for_backward({cos, sin});
    return {qo, ko};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &gq = grads[0], &gk = grads[1];
    check_tables(s, gq);
    strided("the gradient of k", gk, gq.sizes(), gq.scalar_type(), gq);
    Tensor dq = at::empty_like(gq), dk = at::empty_like(gk);
    rope_qk(gq, gk, s[0], s[1], dq, dk, true);
    return {dq, dk, Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// The attention block: [S, B, 3 H D] -> RoPE(q, k) -> attention -> [S, B, H D]
// ---------------------------------------------------------------------------
// Strides of a [S, B, ..., H, D] tensor's slice in the kernels' [B, H, S, D] order.
struct BHSD {
  int64_t s[4];
  BHSD(int64_t S, int64_t B, int64_t H, int64_t D = 1) : s{B, H, S, D} {}
};

struct Block : torch::autograd::Function<Block> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cos,
                        const Tensor& sin, int64_t H, bool causal) {
    const int64_t S = qkv.size(0), B = qkv.size(1), D = qkv.size(2) / (3 * H);
    const int64_t esz = qkv.element_size();
    const Tensor x = qkv.view({S, B, 3, H, D});
    const int64_t sbhd[4] = {x.stride(0), x.stride(1), x.stride(3), x.stride(4)};
    char* xp = (char*)x.data_ptr();
    const int64_t part = x.stride(2) * esz;
    Tensor rot = empty({S, B, 2, H, D}, qkv);
    const int64_t rst[4] = {B * 2 * H * D, 2 * H * D, D, 1};
    char* rp = (char*)rot.data_ptr();
    check(lib.mi_rope_qk(dt(qkv), dt(cos), S, B, H, D, 0, xp, sbhd, xp + part, sbhd,
                         cos.data_ptr(), cos.strides().data(), sin.data_ptr(),
                         sin.strides().data(), rp, rst, rp + H * D * esz, rst, stream(qkv)),
          "mi_rope_qk");
    Tensor o = empty({S, B, H * D}, qkv), lse = empty_f32({B, H, S}, qkv);
    const BHSD rs(rst[0], rst[1], rst[2]), vs(sbhd[0], sbhd[1], sbhd[2]), os(B * H * D, H * D, D);
    check(lib.mi_attn_fwd(dt(qkv), B, H, S, D, causal, 1.0 / std::sqrt((double)D), rp, rs.s,
                          rp + H * D * esz, rs.s, xp + 2 * part, vs.s, o.data_ptr(), os.s,
                          lse.data_ptr<float>(), stream(qkv)),
          "mi_attn_fwd");
    ctx->save_for_backward({rot, qkv, o, lse, cos, sin});
    ctx->saved_data["heads"] = H;
    ctx->saved_data["causal"] = causal;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &rot = s[0], &qkv = s[1], &o = s[2], &lse = s[3], &cos = s[4], &sin = s[5];
    const int64_t H = ctx->saved_data["heads"].toInt();
    Tensor go = grads[0];
    const int64_t S = go.size(0), B = go.size(1), D = go.size(2) / H;
    const int64_t esz = go.element_size();
    const at::ScalarType type = go.scalar_type();
    strided("saved qkv", qkv, {S, B, 3 * H * D}, type, go);
    dense("rotated q and k", rot, {S, B, 2, H, D}, type, go);
    dense("output", o, {S, B, H * D}, type, go);
    dense("lse", lse, {B, H, S}, at::kFloat, go);
    TORCH_CHECK_VALUE(tables_ok(cos, sin, S, D) && one_device(go, cos, sin),
                      "saved cos / sin no longer fit the gradient");
    const Tensor x = qkv.view({S, B, 3, H, D});
    const std::vector<int64_t> shape{S, B, H, D};
    if (!at::detail::computeStride(go.sizes(), go.strides(), shape)) go = go.contiguous();
    go = go.view(shape);
    if (go.stride(-1) != 1 || !rows16(go)) go = go.contiguous();
    Tensor dqkv = empty({S, B, 3 * H * D}, qkv), ws = empty_f32({2, B, H, S}, qkv);
    // the saved qkv may have come back in another layout: its own strides, which
    // the C ABI checks
    const BHSD rs(B * 2 * H * D, 2 * H * D, D),
        vs(x.stride(0), x.stride(1), x.stride(3), x.stride(4)),
        os(B * H * D, H * D, D), gs(go.stride(0), go.stride(1), go.stride(2)),
        ds(B * 3 * H * D, 3 * H * D, D);
    char *rp = (char*)rot.data_ptr(), *dp = (char*)dqkv.data_ptr();
    const int64_t part = H * D * esz;
    check(lib.mi_attn_bwd_rope(
              dt(qkv), B, H, S, D, ctx->saved_data["causal"].toBool(),
              1.0 / std::sqrt((double)D), rp, rs.s, rp + part, rs.s,
              (char*)x.data_ptr() + 2 * x.stride(2) * esz, vs.s, o.data_ptr(), os.s,
              go.data_ptr(), gs.s, lse.data_ptr<float>(), ws.data_ptr<float>(), dp, ds.s,
              dp + part, ds.s, dp + 2 * part, ds.s, dt(cos), cos.data_ptr(),
              cos.strides().data(), sin.data_ptr(), sin.strides().data(), stream(qkv)),
          "mi_attn_bwd_rope");
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// Vocabulary cross entropy
// ---------------------------------------------------------------------------
struct Xent : torch::autograd::Function<Xent> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& target) {
    const Tensor z = as_rows(logits), tgt = target.to(at::kLong).contiguous();
    const auto lead = z.sizes().slice(0, z.dim() - 1);
    Tensor loss = empty(lead, z), lse = empty_f32(lead, z);
    const Rows r = rows(z);
    check(lib.mi_xent_fwd(dt(z), r.n, z.size(-1), z.data_ptr(), r.stride, tgt.data_ptr<int64_t>(),
                          loss.data_ptr(), lse.data_ptr<float>(), stream(z)),
          "mi_xent_fwd");
    ctx->save_for_backward({z, tgt, lse});
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &z = s[0], &tgt = s[1], &lse = s[2];
    const Tensor g = grads[0].to(z.scalar_type()).contiguous();
    const auto lead = z.sizes().slice(0, z.dim() - 1);
    dense("gradient of the loss", g, lead, z.scalar_type(), z);
    dense("target", tgt, lead, at::kLong, z);
    dense("lse", lse, lead, at::kFloat, z);
    Tensor grad = empty(z.sizes(), z);
    const Rows r = rows(z);
    check(lib.mi_xent_bwd(dt(z), r.n, z.size(-1), z.data_ptr(), r.stride, tgt.data_ptr<int64_t>(),
                          lse.data_ptr<float>(), g.data_ptr(), grad.data_ptr(), z.size(-1),
                          stream(z)),
          "mi_xent_bwd");
    return {grad, Tensor()};
  }
};

// ---------------------------------------------------------------------------
// RMSNorm, alone and with the residual add in front
// ---------------------------------------------------------------------------
// The weight in the dtype the kernels take for x (normalization._norm_weight).
Tensor norm_weight(const Tensor& x, const Tensor& weight) {
  Tensor w = weight;
  const bool f32 = w.scalar_type() == at::kFloat;
  if (!f32 && (w.scalar_type() != x.scalar_type() || x.scalar_type() == at::kFloat))
    w = w.to(at::kFloat);
  return w.contiguous();
}

// The weight's existing gradient, when the backward may add into it
// (normalization._grad_target); undefined otherwise.
Tensor grad_target(const Tensor& w, at::ScalarType weight_dtype) {
  if (w.grad_fn() || at::GradMode::is_enabled()) return Tensor();
  const Tensor g = w.grad();
  if (!g.defined() || g.scalar_type() != w.scalar_type() || w.scalar_type() != weight_dtype ||
      g.sizes() != w.sizes() || !g.is_contiguous())
    return Tensor();
  return g;
}

bool norm_ok(const Tensor& x, const Tensor& w) {
  return x.dim() >= 1 && w.dim() == 1 && x.size(-1) == w.size(0) && code(x) >= 0 && code(w) >= 0 &&
         one_device(x, w);
}

Tensor norm_out(const Tensor& x, const Tensor& w) {
  return at::empty(x.sizes(),
                   x.options().dtype(w.scalar_type() == at::kFloat ? at::kFloat : x.scalar_type()));
}

// dweight as autograd returns it: undefined where it went into the gradient.
Tensor norm_bwd(const Tensor& x, const Tensor& w, const Tensor& rstd, const Tensor& dy_,
                const Tensor& dsum_, const Tensor& dx, bool grad_into,
                at::ScalarType weight_dtype) {
  const Tensor dy = as_rows(dy_);
  const int64_t H = x.size(-1), n = rstd.numel();
  dense("rstd", rstd, x.sizes().slice(0, x.dim() - 1), at::kFloat, dy);
  dense("weight", w, {H}, w.scalar_type(), dy);
  // dy is read in the dtype that x and the weight gave y
  strided("the gradient", dy, x.sizes(),
          w.scalar_type() == at::kFloat ? at::kFloat : x.scalar_type(), x);
  const int64_t nws = lib.mi_rmsnorm_bwd_workspace(n, H);
  Tensor ws = empty_f32({nws}, x);
  const Tensor g = grad_into ? grad_target(w, weight_dtype) : Tensor();
  Tensor dw = g.defined() ? g : empty(w.sizes(), w);
  const Rows xr = rows(x), yr = rows(dy), dr = rows(dx);
  if (dsum_.defined()) {
    const Tensor dsum = as_rows(dsum_.to(x.scalar_type()));
    strided("the gradient of the sum", dsum, x.sizes(), x.scalar_type(), x);
    check((g.defined() ? lib.mi_rmsnorm_add_bwd_acc : lib.mi_rmsnorm_add_bwd)(
              dt(x), dt(w), n, H, x.data_ptr(), xr.stride, w.data_ptr(),
              rstd.data_ptr<float>(), dy.data_ptr(), yr.stride, dsum.data_ptr(),
              rows(dsum).stride, dx.data_ptr(), dr.stride, dw.data_ptr(),
              ws.data_ptr<float>(), nws, stream(x)),
          g.defined() ? "mi_rmsnorm_add_bwd_acc" : "mi_rmsnorm_add_bwd");
  } else {
    check((g.defined() ? lib.mi_rmsnorm_bwd_acc : lib.mi_rmsnorm_bwd)(
              dt(x), dt(w), n, H, x.data_ptr(), xr.stride, w.data_ptr(),
              rstd.data_ptr<float>(), dy.data_ptr(), yr.stride, dx.data_ptr(), dr.stride,
              dw.data_ptr(), ws.data_ptr<float>(), nws, stream(x)),
          g.defined() ? "mi_rmsnorm_bwd_acc" : "mi_rmsnorm_bwd");
  }
  return g.defined() ? Tensor() : dw.to(weight_dtype);
}

struct RMSNorm : torch::autograd::Function<RMSNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& weight, double eps,
                        bool grad_into) {
    const Tensor x = as_rows(x_), w = norm_weight(x_, weight);
    Tensor y = norm_out(x_, w), rstd = empty_f32(x_.sizes().slice(0, x_.dim() - 1), x_);
    const Rows r = rows(x);
    check(lib.mi_rmsnorm_fwd(dt(x), dt(w), r.n, x.size(-1), eps, x.data_ptr(), r.stride,
                             w.data_ptr(), y.data_ptr(), rows(y).stride,
                             rstd.data_ptr<float>(), stream(x)),
          "mi_rmsnorm_fwd");
    ctx->save_for_backward({x, w, rstd});
    ctx->saved_data["weight"] = (int64_t)weight.scalar_type();
    ctx->saved_data["into"] = grad_into;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    Tensor dx = empty(s[0].sizes(), s[0]);
    Tensor dw = norm_bwd(s[0], s[1], s[2], grads[0], Tensor(), dx,
                         ctx->saved_data["into"].toBool(),
                         (at::ScalarType)ctx->saved_data["weight"].toInt());
    return {dx, dw, Tensor(), Tensor()};
  }
};

struct AddRMSNorm : torch::autograd::Function<AddRMSNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_, const Tensor& res_,
                               const Tensor& weight, double eps, bool grad_into) {
    const Tensor x = as_rows(x_), res = as_rows(res_), w = norm_weight(x_, weight);
    Tensor sum = empty(x_.sizes(), x_), y = norm_out(x_, w);
    Tensor rstd = empty_f32(x_.sizes().slice(0, x_.dim() - 1), x_);
    const Rows r = rows(x);
    check(lib.mi_rmsnorm_add_fwd(dt(x), dt(w), r.n, x.size(-1), eps, x.data_ptr(), r.stride,
                                 res.data_ptr(), rows(res).stride, w.data_ptr(),
                                 sum.data_ptr(), rows(sum).stride, y.data_ptr(),
                                 rows(y).stride, rstd.data_ptr<float>(), stream(x)),
          "mi_rmsnorm_add_fwd");
    ctx->save_for_backward({sum, w, rstd});
    ctx->saved_data["weight"] = (int64_t)weight.scalar_type();
    ctx->saved_data["into"] = grad_into;
    ctx->set_materialize_grads(false);
    return {sum, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &sum = s[0], &w = s[1], &ds = grads[0], &dy = grads[1];
    const auto wd = (at::ScalarType)ctx->saved_data["weight"].toInt();
    if (!dy.defined()) {  // only the sum is used: the norm contributes nothing
      Tensor dx = ds.to(sum.scalar_type());
      return {dx, dx, at::zeros(w.sizes(), w.options().dtype(wd)), Tensor(), Tensor()};
    }
    Tensor dx = empty(sum.sizes(), sum);
    Tensor dw = norm_bwd(sum, w, s[2], dy, ds, dx, ctx->saved_data["into"].toBool(), wd);
    return {dx, dx, dw, Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// SwiGLU, and the linear whose weight gradient goes into the existing one
// ---------------------------------------------------------------------------
struct SwiGLU : torch::autograd::Function<SwiGLU> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate_up) {
    const Tensor gu = as_rows(gate_up);
    std::vector<int64_t> shape = gu.sizes().vec();
    shape.back() /= 2;
    Tensor h = empty(shape, gu);
    const Rows r = rows(gu);
    check(lib.mi_swiglu_fwd(dt(gu), r.n, shape.back(), gu.data_ptr(), r.stride, h.data_ptr(),
                            shape.back(), stream(gu)),
          "mi_swiglu_fwd");
    ctx->save_for_backward({gu});
    return h;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor gu = ctx->get_saved_variables()[0];
    const Tensor dh = as_rows(grads[0].to(gu.scalar_type()));
    std::vector<int64_t> shape = dh.sizes().vec();
    shape.back() *= 2;
    strided("saved gate_up", gu, shape, dh.scalar_type(), dh);
    Tensor dgu = empty(gu.sizes(), gu);
    const Rows r = rows(gu);
    check(lib.mi_swiglu_bwd(dt(gu), r.n, gu.size(-1) / 2, gu.data_ptr(), r.stride, dh.data_ptr(),
                            rows(dh).stride, dgu.data_ptr(), gu.size(-1), stream(gu)),
          "mi_swiglu_bwd");
    return {dgu};
  }
};

// dy^T x added to g, or in a new tensor (_lib.wgrad); undefined where a general
// GEMM is to be used.  The C ABI takes the sizes from dy and x: operands that do
// not fit each other (a saved x may have changed) are left to the GEMM, which
// refuses them.
Tensor wgrad(const Tensor& dy, const Tensor& x, const Tensor& g) {
  if (dy.dim() != 2 || x.dim() != 2 || x.size(0) != dy.size(0) ||
      (g.defined() &&
       (g.dim() != 2 || g.size(0) != dy.size(1) || g.size(1) != x.size(1) || !g.is_contiguous())))
    return Tensor();
  if (!dy.is_cuda() || x.device() != dy.device() || dy.scalar_type() != x.scalar_type() ||
      (code(dy) != MI_BF16 && code(dy) != MI_F16) ||
      !lib.mi_wgrad_suits(dy.size(0), dy.size(1), x.size(1)))
    return Tensor();
  for (const Tensor* t : {&dy, &x})
    if (t->stride(1) != 1 || t->stride(0) < t->size(1) || t->stride(0) >= 1 << 24 ||
        t->stride(0) % 8 || t->size(1) % 8 || (uintptr_t)t->data_ptr() % 16)
      return Tensor();
  if (g.defined() && (g.scalar_type() != dy.scalar_type() || g.device() != dy.device() ||
                      (uintptr_t)g.data_ptr() % 8))
    return Tensor();
  const int64_t n = lib.mi_wgrad_workspace(dy.size(0), dy.size(1), x.size(1));
  Tensor dw = g.defined() ? g : empty({dy.size(1), x.size(1)}, dy), ws = empty_f32({n}, dy);
  check(lib.mi_wgrad(dt(dy), dy.size(0), dy.size(1), x.size(1), dy.data_ptr(), dy.stride(0),
                     x.data_ptr(), x.stride(0), dw.data_ptr(), g.defined(), ws.data_ptr<float>(),
                     n, stream(dy)),
        "mi_wgrad");
  if (g.defined()) g.unsafeGetTensorImpl()->bump_version();  // as addmm_ would
  return dw;
}

struct LinearGradInto : torch::autograd::Function<LinearGradInto> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, bool into) {
    // as F.linear, only what a gradient needs (and w where its .grad takes dw)
    ctx->save_for_backward({w.requires_grad() ? x : Tensor(),
                            x.requires_grad() || into ? w : Tensor()});
    ctx->saved_data["into"] = into;
    return at::linear(x, w);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w = s[1], &gy = grads[0];
    const Tensor gx = ctx->needs_input_grad(0) ? gy.matmul(w) : Tensor();
    if (!ctx->needs_input_grad(1)) return {gx, Tensor(), Tensor()};
    const Tensor gy2 = gy.reshape({-1, gy.size(-1)}), x2 = x.reshape({-1, x.size(-1)});
    if (at::GradMode::is_enabled()) return {gx, gy2.t().matmul(x2), Tensor()};
    Tensor g = ctx->saved_data["into"].toBool() ? w.grad() : Tensor();
    if (!g.defined() || g.scalar_type() != gy.scalar_type() || g.sizes() != w.sizes() ||
        !g.is_contiguous()) {
      const Tensor dw = wgrad(gy2, x2, Tensor());
      return {gx, dw.defined() ? dw : gy2.t().matmul(x2), Tensor()};
    }
    if (!wgrad(gy2, x2, g).defined()) g.addmm_(gy2.t(), x2);
    return {gx, Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// The module's functions: None for a call that is not plain
// ---------------------------------------------------------------------------
using Args = PyObject* const*;

bool truth(PyObject* o, bool& v) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) PyErr_Clear();
  v = r > 0;
  return r >= 0;
}
bool number(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// f() without the interpreter lock: a launch may wait for room in its queue.
template <typename F>
auto released(F f) {
  pybind11::gil_scoped_release no_gil;
  return f();
}

PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* t = PyTuple_New(2);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
  return t;
}

#define PLAIN(cond) \
  if (!(cond)) Py_RETURN_NONE

PyObject* py_flash_attn(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v;
  bool causal;
  PLAIN(n == 4 && plain(a[0], q) && plain(a[1], k) && plain(a[2], v) && plain_context() &&
        attn_ok(q, k, v) && truth(a[3], causal));
  return THPVariable_Wrap(released([&] { return FlashAttn::apply(q, k, v, causal); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_flash_attn_forward(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v;
  bool causal;
  PLAIN(n == 4 && plain(a[0], q) && plain(a[1], k) && plain(a[2], v) && plain_context() &&
        attn_ok(q, k, v) && truth(a[3], causal));
  const AttnOut r = released(
      [&] { return attn_fwd(kernel_ready(q), kernel_ready(k), kernel_ready(v), causal); });
  return pair(r.o, r.lse);
  END_HANDLE_TH_ERRORS
}

PyObject* py_attention_block(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor qkv, cos, sin;
  bool causal;
  PLAIN(n == 5 && plain(a[0], qkv) && plain(a[1], cos) && plain(a[2], sin) && plain_context() &&
        PyLong_CheckExact(a[3]) && truth(a[4], causal));
  const long heads = PyLong_AsLong(a[3]);
  if (heads == -1 && PyErr_Occurred()) PyErr_Clear();
  PLAIN(heads > 0 && heads < (1 << 20) && qkv.dim() == 3 && qkv.size(2) % (3 * heads) == 0 &&
        qkv.stride(2) == 1 && code(qkv) >= 0 && one_device(qkv, cos, sin) &&
        tables_ok(cos, sin, qkv.size(0), qkv.size(2) / (3 * heads)));
  return THPVariable_Wrap(released([&] { return Block::apply(qkv, cos, sin, (int64_t)heads, causal); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_rope(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, cos, sin;
  PLAIN(n == 3 && plain(a[0], x) && plain(a[1], cos) && plain(a[2], sin) && plain_context() &&
        x.dim() == 4 && code(x) >= 0 && one_device(x, cos, sin) &&
        tables_ok(cos, sin, x.size(0), x.size(3)));
  return THPVariable_Wrap(released([&] { return RoPE::apply(x, cos, sin); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_rope_qk(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, cos, sin;
  PLAIN(n == 4 && plain(a[0], q) && plain(a[1], k) && plain(a[2], cos) && plain(a[3], sin) &&
        plain_context() && q.dim() == 4 && q.sizes() == k.sizes() &&
        q.scalar_type() == k.scalar_type() && code(q) >= 0 && one_device(q, k, cos, sin) &&
        tables_ok(cos, sin, q.size(0), q.size(3)));
  const variable_list r = released([&] { return RoPEQK::apply(q, k, cos, sin); });
  return pair(r[0], r[1]);
  END_HANDLE_TH_ERRORS
}

PyObject* py_xent(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor z, t;
  PLAIN(n == 2 && plain(a[0], z) && plain(a[1], t) && plain_context() && z.dim() >= 1 &&
        t.sizes() == z.sizes().slice(0, z.dim() - 1) && code(z) >= 0 && one_device(z, t) &&
        (t.scalar_type() == at::kLong || t.scalar_type() == at::kInt ||
         t.scalar_type() == at::kShort || t.scalar_type() == at::kByte ||
         t.scalar_type() == at::kChar));
  return THPVariable_Wrap(released([&] { return Xent::apply(z, t); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_rms_norm(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w;
  double eps;
  bool into;
  PLAIN(n == 4 && plain(a[0], x) && plain(a[1], w) && plain_context() && norm_ok(x, w) &&
        number(a[2], eps) && truth(a[3], into));
  return THPVariable_Wrap(released([&] { return RMSNorm::apply(x, w, eps, into); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_add_rms_norm(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, res, w;
  double eps;
  bool into;
  PLAIN(n == 5 && plain(a[0], x) && plain(a[1], res) && plain(a[2], w) && plain_context() &&
        norm_ok(x, w) && res.sizes() == x.sizes() && res.scalar_type() == x.scalar_type() &&
        one_device(x, res) && number(a[3], eps) && truth(a[4], into));
  const variable_list r = released([&] { return AddRMSNorm::apply(x, res, w, eps, into); });
  return pair(r[0], r[1]);
  END_HANDLE_TH_ERRORS
}

PyObject* py_swiglu(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor gu;
  PLAIN(n == 1 && plain(a[0], gu) && plain_context() && gu.dim() >= 1 && gu.size(-1) % 2 == 0 &&
        code(gu) >= 0);
  return THPVariable_Wrap(released([&] { return SwiGLU::apply(gu); }));
  END_HANDLE_TH_ERRORS
}

PyObject* py_linear_into_grad(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w;
  bool into;
  PLAIN(n == 3 && plain(a[0], x) && plain(a[1], w) && plain_context() && x.dim() >= 1 &&
        w.dim() == 2 && x.size(-1) == w.size(1) && one_device(x, w) && truth(a[2], into) &&
        !at::autocast::is_autocast_enabled(at::kCUDA) &&
        (into || (x.scalar_type() == w.scalar_type() && (code(x) == MI_BF16 || code(x) == MI_F16))));
  return THPVariable_Wrap(released([&] { return LinearGradInto::apply(x, w, into); }));
  END_HANDLE_TH_ERRORS
}

// bind({name: address}, MiError)
PyObject* py_bind(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 2 && PyDict_Check(a[0]), "bind(addresses, error)");
#define X(f)                                                                   \
  {                                                                            \
    PyObject* p = PyDict_GetItemString(a[0], #f);                              \
    TORCH_CHECK(p, "libmi_attn: no address for " #f);                          \
    void* v = PyLong_AsVoidPtr(p);                                             \
    if (!v && PyErr_Occurred()) throw python_error();                          \
    std::memcpy(&lib.f, &v, sizeof(v));                                        \
  }
  MI_BOUND(X)
#undef X
  Py_INCREF(a[1]);
  lib.error = a[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define FN(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FN(bind),       FN(flash_attn),  FN(flash_attn_forward),
                         FN(attention_block), FN(rope),   FN(rope_qk),
                         FN(xent),       FN(rms_norm),    FN(add_rms_norm),
                         FN(swiglu),     FN(linear_into_grad), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() { return PyModule_Create(&module); }
