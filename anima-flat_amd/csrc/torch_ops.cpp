// Native torch kernels of the package's ops: the CUDA and AutogradCUDA entries
// that take a call of the usual form from the dispatcher to libanima_attn.so
// without entering Python.
//
// The ops themselves (schemas, fake kernels, the kernels of every other
// dispatch key) are registered in Python by torch.library.custom_op; attach()
// adds these two keys to one of them. Reached through Python, an op costs
// 25-30 us of host time per call, and a training step's autograd wiring 320 us
// for prologue + attention forward and backward, more than their kernels take
// at 1024 tokens (about 105 us); through here 8-15 and 78 us.
//
// A call that a kernel here does not take as it is (an odd stride or
// alignment that needs a copy, another dtype, a shape error) goes to the op's
// Python function, which owns every such case and its error message.
#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <algorithm>
#include <cmath>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/anima_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using T2 = std::tuple<Tensor, Tensor>;
using T3 = std::tuple<Tensor, Tensor, Tensor>;

// ---------------------------------------------------------------- fallback --

// The ops' Python functions. Never destroyed: ops may outlive the interpreter.
std::map<std::string, PyObject*>& python_impls() {
  static auto* m = new std::map<std::string, PyObject*>();
  return *m;
}

template <class R, class... A>
R python_impl(const char* name, const A&... args) {
  pybind11::gil_scoped_acquire gil;
  const pybind11::handle fn(python_impls().at(name));
  return fn(args...).template cast<R>();
}

// ------------------------------------------------------------------ helpers --

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// bf16 on the GPU of `like`.
bool bf16_on(const Tensor& t, const Tensor& like) {
  return t.scalar_type() == at::kBFloat16 && t.is_cuda() && t.device() == like.device();
}

// A [B, S, H, hd] view that the attention kernels read in place.
bool kernel_ready(const Tensor& t) {
  return t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 &&
         aligned16(t);
}

// True when done; false (nothing launched) sends the call to the Python
// function, which raises the library's message.
bool launched(int rc, const char* what) {
  if (rc == AA_OK) return true;
  TORCH_CHECK(rc != AA_EHIP, what, ": ", aa_last_error(), " (code ", rc, ")");
  return false;
}

void set_strides(int64_t (&dst)[3], const Tensor& t) {
  for (int i = 0; i < 3; ++i) dst[i] = t.stride(i);
}

Tensor f32(const Tensor& t) { return t.to(at::kFloat).contiguous(); }

// ---------------------------------------------------------------- attention --

bool attention_ready(const Tensor& q, const Tensor& k, const Tensor& v, int64_t hd) {
  return q.dim() == 4 && k.dim() == 4 && v.dim() == 4 && k.sizes() == v.sizes() &&
         q.size(0) == k.size(0) && q.size(2) == k.size(2) && q.size(3) == hd && k.size(3) == hd &&
         bf16_on(q, q) && bf16_on(k, q) && bf16_on(v, q) && q.numel() > 0 && k.numel() > 0 &&
         kernel_ready(q) && kernel_ready(k) && kernel_ready(v);
}

bool lengths_ready(const Tensor& t, const Tensor& q, at::ScalarType dtype) {
  return t.dim() == 1 && t.size(0) == q.size(0) && t.scalar_type() == dtype &&
         t.device() == q.device() && t.is_contiguous();
}

// out (and lse when wanted); false: for the Python function.
bool forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor* seqused,
             const Tensor* ln_pad, int64_t hd, Tensor& out, Tensor* lse) {
  if (!attention_ready(q, k, v, hd)) return false;
  if (seqused && !lengths_ready(*seqused, q, at::kInt)) return false;
  if (ln_pad && !lengths_ready(*ln_pad, q, at::kFloat)) return false;
  const c10::DeviceGuard guard(q.device());
  const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), Sk = k.size(1);
  out = at::empty({B, Sq, H, hd}, q.options());
  if (lse) *lse = at::empty({B, H, Sq}, q.options().dtype(at::kFloat));
  aa_attn_fwd_args a = {};
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.out = out.data_ptr();
  a.lse = lse ? lse->data_ptr<float>() : nullptr;
  a.seqused_k = seqused ? seqused->data_ptr<int32_t>() : nullptr;
  a.ln_pad = ln_pad ? ln_pad->data_ptr<float>() : nullptr;
  set_strides(a.q_stride, q);
  set_strides(a.k_stride, k);
  set_strides(a.v_stride, v);
  set_strides(a.out_stride, out);
  a.B = B;
  a.Sq = Sq;
  a.Sk = Sk;
  a.H = H;
  a.hd = hd;
  a.softmax_scale = (float)(1.0 / std::sqrt((double)hd));
  a.dtype = AA_DTYPE_BF16;
  const size_t bytes = aa_attn_fwd_workspace(B, Sq, Sk, H, hd);
  Tensor ws;
  if (bytes) {
    ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    a.workspace = ws.data_ptr();
    a.workspace_bytes = bytes;
  }
  return launched(aa_attn_fwd(&a, stream_of(q)), "attn_fwd");
}

T2 fa_fwd(const Tensor& q, const Tensor& k, const Tensor& v) {
  Tensor out, lse;
  if (forward(q, k, v, nullptr, nullptr, 128, out, &lse)) return {out, lse};
  return python_impl<T2>("fa_fwd", q, k, v);
}

Tensor fa_fwd_nolse(const Tensor& q, const Tensor& k, const Tensor& v) {
  Tensor out;
  if (forward(q, k, v, nullptr, nullptr, 128, out, nullptr)) return out;
  return python_impl<Tensor>("fa_fwd_nolse", q, k, v);
}

T2 fa_fwd_k(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& seqused) {
  Tensor out, lse;
  if (forward(q, k, v, &seqused, nullptr, 128, out, &lse)) return {out, lse};
  return python_impl<T2>("fa_fwd_k", q, k, v, seqused);
}

Tensor fa_fwd_k_ctx(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& seqused,
                    const Tensor& ln_pad) {
  Tensor out;
  if (forward(q, k, v, &seqused, &ln_pad, 128, out, nullptr)) return out;
  return python_impl<Tensor>("fa_fwd_k_ctx", q, k, v, seqused, ln_pad);
}

Tensor attend_d384(const Tensor& q, const Tensor& k, const Tensor& v) {
  Tensor out;
  if (forward(q, k, v, nullptr, nullptr, 384, out, nullptr)) return out;
  return python_impl<Tensor>("attend_d384", q, k, v);
}

T3 fa_bwd(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
          const Tensor& lse) {
  const auto slow = [&] { return python_impl<T3>("fa_bwd", dout, q, k, v, out, lse); };
  if (!attention_ready(q, k, v, 128) || !dout.sizes().equals(q.sizes()) ||
      !out.sizes().equals(q.sizes()) || !bf16_on(dout, q) || !bf16_on(out, q) ||
      !dout.is_contiguous() || !aligned16(dout) || !kernel_ready(out))
    return slow();
  const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), Sk = k.size(1);
  if (lse.dim() != 3 || lse.size(0) != B || lse.size(1) != H || lse.size(2) != Sq ||
      lse.scalar_type() != at::kFloat || lse.device() != q.device() || !lse.is_contiguous())
    return slow();
  const c10::DeviceGuard guard(q.device());
  Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  if (!kernel_ready(dq) || !kernel_ready(dk) || !kernel_ready(dv)) return slow();
  aa_attn_bwd_args a = {};
  a.dout = dout.data_ptr();
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.out = out.data_ptr();
  a.lse = lse.data_ptr<float>();
  a.dq = dq.data_ptr();
  a.dk = dk.data_ptr();
  a.dv = dv.data_ptr();
  set_strides(a.dout_stride, dout);
  set_strides(a.q_stride, q);
  set_strides(a.k_stride, k);
  set_strides(a.v_stride, v);
  set_strides(a.out_stride, out);
  set_strides(a.dq_stride, dq);
  set_strides(a.dk_stride, dk);
  set_strides(a.dv_stride, dv);
  a.B = B;
  a.Sq = Sq;
  a.Sk = Sk;
  a.H = H;
  a.hd = 128;
  a.softmax_scale = (float)(1.0 / std::sqrt(128.0));
  a.dtype = AA_DTYPE_BF16;
  const size_t bytes = aa_attn_bwd_workspace(B, Sq, Sk, H, 128);
  const Tensor ws = at::empty({std::max<int64_t>((int64_t)bytes / 4, 1)}, q.options().dtype(at::kFloat));
  if (!launched(aa_attn_bwd(&a, ws.data_ptr(), bytes, stream_of(q)), "attn_bwd")) return slow();
  return {dq, dk, dv};
}

// ----------------------------------------------------------------- prologue --

bool on_gpu(const Tensor& t, const Tensor& like) { return t.device() == like.device(); }

bool qkv_ready(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
               const Tensor& sin, int64_t heads) {
  return qkv.dim() == 3 && bf16_on(qkv, qkv) && qkv.is_contiguous() && qkv.numel() > 0 &&
         cos.dim() == 2 && cos.size(1) == 64 && sin.sizes() == cos.sizes() &&
         cos.size(0) == qkv.size(1) && qkv.size(2) == 3 * heads * 128 && qw.numel() == 128 &&
         kw.numel() == 128 && on_gpu(qw, qkv) && on_gpu(kw, qkv) && on_gpu(cos, qkv) &&
         on_gpu(sin, qkv);
}

bool qkv_forward(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
                 const Tensor& sin, int64_t heads, double eps, Tensor& q, Tensor& k, Tensor* v) {
  if (!qkv_ready(qkv, qw, kw, cos, sin, heads)) return false;
  const c10::DeviceGuard guard(qkv.device());
  const int64_t B = qkv.size(0), S = qkv.size(1);
  q = at::empty({B, S, heads, 128}, qkv.options());
  k = at::empty_like(q);
  if (v) *v = at::empty_like(q);
  const Tensor qw32 = f32(qw), kw32 = f32(kw), c32 = f32(cos), s32 = f32(sin);
  return launched(aa_qkv_norm_rope_fwd(qkv.data_ptr(), q.data_ptr(), k.data_ptr(),
                                       v ? v->data_ptr() : nullptr, qw32.data_ptr<float>(),
                                       kw32.data_ptr<float>(), c32.data_ptr<float>(),
                                       s32.data_ptr<float>(), B, S, heads, 128, (float)eps,
                                       AA_DTYPE_BF16, stream_of(qkv)),
                  "qkv_norm_rope");
}

T2 qkv_norm_rope(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
                 const Tensor& sin, int64_t heads, double eps) {
  Tensor q, k;
  if (qkv_forward(qkv, qw, kw, cos, sin, heads, eps, q, k, nullptr)) return {q, k};
  return python_impl<T2>("qkv_norm_rope", qkv, qw, kw, cos, sin, heads, eps);
}

T3 qkv_norm_rope_v(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
                   const Tensor& sin, int64_t heads, double eps) {
  Tensor q, k, v;
  if (qkv_forward(qkv, qw, kw, cos, sin, heads, eps, q, k, &v)) return {q, k, v};
  return python_impl<T3>("qkv_norm_rope_v", qkv, qw, kw, cos, sin, heads, eps);
}

T3 qkv_norm_rope_bwd(const Tensor& qkv, const Tensor& dq_, const Tensor& dk_, const Tensor& dv_,
                     const Tensor& qw, const Tensor& kw, const Tensor& cos, const Tensor& sin,
                     int64_t heads, double eps) {
  const auto slow = [&] {
    return python_impl<T3>("qkv_norm_rope_bwd", qkv, dq_, dk_, dv_, qw, kw, cos, sin, heads, eps);
  };
  if (!qkv_ready(qkv, qw, kw, cos, sin, heads)) return slow();
  const int64_t B = qkv.size(0), S = qkv.size(1);
  for (const Tensor* t : {&dq_, &dk_, &dv_})
    if (!bf16_on(*t, qkv) || t->numel() != B * S * heads * 128) return slow();
  const c10::DeviceGuard guard(qkv.device());
  const Tensor dq = dq_.contiguous(), dk = dk_.contiguous(), dv = dv_.contiguous();
  Tensor dqkv = at::empty_like(qkv);
  const auto fopt = qkv.options().dtype(at::kFloat);
  Tensor dqw = at::empty({128}, fopt), dkw = at::empty({128}, fopt);
  const size_t bytes = aa_qkv_norm_rope_bwd_workspace(B, S, heads, 128);
  const Tensor ws = at::empty({std::max<int64_t>((int64_t)bytes / 4, 1)}, fopt);
  const Tensor qw32 = f32(qw), kw32 = f32(kw), c32 = f32(cos), s32 = f32(sin);
  if (!launched(aa_qkv_norm_rope_bwd(qkv.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                     dqkv.data_ptr(), qw32.data_ptr<float>(),
                                     kw32.data_ptr<float>(), c32.data_ptr<float>(),
                                     s32.data_ptr<float>(), dqw.data_ptr<float>(),
                                     dkw.data_ptr<float>(), ws.data_ptr(), bytes, B, S, heads, 128,
                                     (float)eps, AA_DTYPE_BF16, stream_of(qkv)),
                "qkv_norm_rope_bwd"))
    return slow();
  return {dqkv, dqw.to(qw.scalar_type()), dkw.to(kw.scalar_type())};
}

bool head_norm_ready(const Tensor& x, const Tensor& w, int64_t heads) {
  return x.dim() == 3 && bf16_on(x, x) && x.is_contiguous() && x.numel() > 0 && w.numel() == 128 &&
         x.size(2) == heads * 128 && on_gpu(w, x);
}

Tensor head_norm(const Tensor& x, const Tensor& w, int64_t heads, double eps) {
  if (head_norm_ready(x, w, heads)) {
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), S = x.size(1);
    Tensor y = at::empty({B, S, heads, 128}, x.options());
    const Tensor w32 = f32(w);
    if (launched(aa_head_norm_fwd(x.data_ptr(), y.data_ptr(), w32.data_ptr<float>(), B, S, heads,
                                  128, (float)eps, AA_DTYPE_BF16, stream_of(x)),
                 "head_norm"))
      return y;
  }
  return python_impl<Tensor>("head_norm", x, w, heads, eps);
}

T2 head_norm_bwd(const Tensor& x, const Tensor& dy_, const Tensor& w, int64_t heads, double eps) {
  const auto slow = [&] { return python_impl<T2>("head_norm_bwd", x, dy_, w, heads, eps); };
  if (!head_norm_ready(x, w, heads) || !bf16_on(dy_, x) || dy_.numel() != x.numel()) return slow();
  const c10::DeviceGuard guard(x.device());
  const int64_t B = x.size(0), S = x.size(1);
  const Tensor dy = dy_.contiguous();
  Tensor dx = at::empty_like(x);
  const auto fopt = x.options().dtype(at::kFloat);
  Tensor dw = at::empty({128}, fopt);
  const size_t bytes = aa_head_norm_bwd_workspace(B, S, heads, 128);
  const Tensor ws = at::empty({std::max<int64_t>((int64_t)bytes / 4, 1)}, fopt);
  const Tensor w32 = f32(w);
  if (!launched(aa_head_norm_bwd(x.data_ptr(), dy.data_ptr(), dx.data_ptr(), w32.data_ptr<float>(),
                                 dw.data_ptr<float>(), ws.data_ptr(), bytes, B, S, heads, 128,
                                 (float)eps, AA_DTYPE_BF16, stream_of(x)),
                "head_norm_bwd"))
    return slow();
  return {dx, dw.to(w.scalar_type())};
}

// -------------------------------------------------------------- projections --

// [B, S, K] rows at one row stride (what the C ABI addresses) and a weight of
// `cols` rows; false for the forms that take one launch per batch item.
bool proj_ready(const Tensor& x, const Tensor& w, int64_t cols) {
  return x.dim() == 3 && bf16_on(x, x) && x.numel() > 0 && x.size(1) > 1 && x.stride(2) == 1 &&
         (x.size(0) == 1 || x.stride(0) == x.size(1) * x.stride(1)) && bf16_on(w, x) &&
         w.is_contiguous() && w.dim() == 2 && w.size(0) == cols && w.size(1) == x.size(2);
}

T3 qkv_proj_norm_rope(const Tensor& x, const Tensor& w, const Tensor& qw, const Tensor& kw,
                      const Tensor& cos, const Tensor& sin, int64_t heads, double eps) {
  if (proj_ready(x, w, 3 * heads * 128) && x.size(2) == heads * 128 && cos.dim() == 2 &&
      cos.size(1) == 64 && cos.size(0) == x.size(1) && sin.sizes() == cos.sizes() &&
      qw.numel() == 128 && kw.numel() == 128 && on_gpu(qw, x) && on_gpu(kw, x) && on_gpu(cos, x) &&
      on_gpu(sin, x)) {
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), S = x.size(1);
    Tensor q = at::empty({B, S, heads, 128}, x.options());
    Tensor k = at::empty_like(q), v = at::empty_like(q);
    const Tensor qw32 = f32(qw), kw32 = f32(kw), c32 = f32(cos), s32 = f32(sin);
    if (launched(aa_qkv_proj_norm_rope(x.data_ptr(), x.stride(1), w.data_ptr(), q.data_ptr(),
                                       k.data_ptr(), v.data_ptr(), qw32.data_ptr<float>(),
                                       kw32.data_ptr<float>(), c32.data_ptr<float>(),
                                       s32.data_ptr<float>(), B, S, heads, 128, (float)eps,
                                       AA_DTYPE_BF16, stream_of(x)),
                 "qkv_proj_norm_rope"))
      return {q, k, v};
  }
  return python_impl<T3>("qkv_proj_norm_rope", x, w, qw, kw, cos, sin, heads, eps);
}

Tensor proj_head_norm(const Tensor& x, const Tensor& w, const Tensor& nw, int64_t heads, double eps) {
  if (proj_ready(x, w, heads * 128) && nw.numel() == 128 && on_gpu(nw, x)) {
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), S = x.size(1);
    Tensor y = at::empty({B, S, heads, 128}, x.options());
    const Tensor nw32 = f32(nw);
    if (launched(aa_proj_head_norm(x.data_ptr(), x.stride(1), w.data_ptr(), x.size(2), y.data_ptr(),
                                   nw32.data_ptr<float>(), B, S, heads, 128, (float)eps,
                                   AA_DTYPE_BF16, stream_of(x)),
                 "proj_head_norm"))
      return y;
  }
  return python_impl<Tensor>("proj_head_norm", x, w, nw, heads, eps);
}

T2 kv_proj_norm(const Tensor& x, const Tensor& w, const Tensor& kw, int64_t heads, double eps) {
  if (proj_ready(x, w, 2 * heads * 128) && kw.numel() == 128 && on_gpu(kw, x)) {
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), S = x.size(1);
    Tensor k = at::empty({B, S, heads, 128}, x.options());
    Tensor v = at::empty_like(k);
    const Tensor kw32 = f32(kw);
    if (launched(aa_kv_proj_norm(x.data_ptr(), x.stride(1), w.data_ptr(), x.size(2), k.data_ptr(),
                                 v.data_ptr(), kw32.data_ptr<float>(), B, S, heads, 128, (float)eps,
                                 AA_DTYPE_BF16, stream_of(x)),
                 "kv_proj_norm"))
      return {k, v};
  }
  return python_impl<T2>("kv_proj_norm", x, w, kw, heads, eps);
}

// ----------------------------------------------------------------- autograd --

// The dispatcher's handle of one op, called below or above autograd.
template <class R, class... A>
struct Op {
  c10::TypedOperatorHandle<R(A...)> handle;
  explicit Op(const char* name)
      : handle(c10::Dispatcher::singleton().findSchemaOrThrow(name, "").template typed<R(A...)>()) {}
  R operator()(A... args) const { return handle.call(args...); }
  R below(A... args) const {
    at::AutoDispatchBelowADInplaceOrView guard;
    return handle.call(args...);
  }
};

#define ANIMA_OP(fn, name, ...)            \
  const Op<__VA_ARGS__>& fn() {            \
    static const Op<__VA_ARGS__> op(name); \
    return op;                             \
  }
using CT = const Tensor&;
ANIMA_OP(op_fa_fwd, "anima_flat::fa_fwd", T2, CT, CT, CT)
ANIMA_OP(op_fa_fwd_nolse, "anima_flat::fa_fwd_nolse", Tensor, CT, CT, CT)
ANIMA_OP(op_fa_fwd_k, "anima_flat::fa_fwd_k", T2, CT, CT, CT, CT)
ANIMA_OP(op_fa_bwd, "anima_flat::fa_bwd", T3, CT, CT, CT, CT, CT, CT)
ANIMA_OP(op_fa_fwd_k_ctx, "anima_flat_amd::fa_fwd_k_ctx", Tensor, CT, CT, CT, CT, CT)
ANIMA_OP(op_attend_d384, "anima_flat_amd::attend_d384", Tensor, CT, CT, CT)
ANIMA_OP(op_qkv_norm_rope, "anima_flat::qkv_norm_rope", T2, CT, CT, CT, CT, CT, int64_t, double)
ANIMA_OP(op_qkv_norm_rope_v, "anima_flat::qkv_norm_rope_v", T3, CT, CT, CT, CT, CT, int64_t, double)
ANIMA_OP(op_qkv_norm_rope_bwd, "anima_flat::qkv_norm_rope_bwd", T3, CT, CT, CT, CT, CT, CT, CT, CT,
         int64_t, double)
ANIMA_OP(op_head_norm, "anima_flat::head_norm", Tensor, CT, CT, int64_t, double)
ANIMA_OP(op_head_norm_bwd, "anima_flat::head_norm_bwd", T2, CT, CT, CT, int64_t, double)
ANIMA_OP(op_qkv_proj_norm_rope, "anima_flat_amd::qkv_proj_norm_rope", T3, CT, CT, CT, CT, CT, CT,
         int64_t, double)
ANIMA_OP(op_proj_head_norm, "anima_flat_amd::proj_head_norm", Tensor, CT, CT, CT, int64_t, double)
ANIMA_OP(op_kv_proj_norm, "anima_flat_amd::kv_proj_norm", T2, CT, CT, CT, int64_t, double)
#undef ANIMA_OP

// Whether a call is recorded for the backward; no op here has a forward-mode
// derivative.
template <class... A>
bool needs_grad(const A&... args) {
  const auto any = [&](auto pred) {
    const auto one = [&](const auto& a) {
      if constexpr (std::is_same_v<std::decay_t<decltype(a)>, Tensor>) return pred(a);
      else return false;
    };
    return (one(args) || ...);
  };
  if (!c10::GradMode::is_enabled() || !any([](const Tensor& t) { return t.requires_grad(); }))
    return false;
  TORCH_CHECK_NOT_IMPLEMENTED(
      !any([](const Tensor& t) { return t._fw_grad(0).defined(); }),
      "You must implement the jvp function for custom autograd.Function to use it with forward "
      "mode AD.");
  return true;
}

// An op without a backward, reached with inputs that need one: its outputs
// need grad too, and asking for it raises what torch.library's own autograd
// kernel raises.
struct NoBackward : torch::autograd::Function<NoBackward> {
  static constexpr bool is_traceable = true;
  // The inputs are there for autograd to find (it does not look into lists).
  template <class... A>
  static variable_list forward(AutogradContext* ctx, const std::function<variable_list()>& run,
                               const std::string& name, const A&...) {
    ctx->saved_data["op"] = name;
    return run();
  }
  static variable_list backward(AutogradContext* ctx, const variable_list&) {
    TORCH_CHECK(false, "Trying to backward through ", ctx->saved_data["op"].toStringRef(),
                " but no autograd formula was registered. Please use register_autograd to add one.");
  }
};

variable_list as_list(const Tensor& t) { return {t}; }
variable_list as_list(const T2& t) { return {std::get<0>(t), std::get<1>(t)}; }
variable_list as_list(const T3& t) { return {std::get<0>(t), std::get<1>(t), std::get<2>(t)}; }
void from_list(const variable_list& l, Tensor& t) { t = l[0]; }
void from_list(const variable_list& l, T2& t) { t = {l[0], l[1]}; }
void from_list(const variable_list& l, T3& t) { t = {l[0], l[1], l[2]}; }

// AutogradCUDA kernel of an op without a backward.
template <auto OpFn, class R, class... A>
struct Plain {
  static R call(A... args) {
    if (!needs_grad(args...)) return OpFn().below(args...);
    std::string name = OpFn().handle.operator_name().name;
    name.replace(name.find("::"), 2, ".");
    const std::function<variable_list()> run = [&] { return as_list(OpFn().below(args...)); };
    R result;
    from_list(NoBackward::apply(run, name + ".default", args...), result);
    return result;
  }
};

// One output: the LSE, which has no derivative, is handed past the node (a node
// with an output marked as such cannot be traced by compiled autograd).
struct FaFwd : torch::autograd::Function<FaFwd> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, CT q, CT k, CT v, Tensor* lse) {
    Tensor out;
    std::tie(out, *lse) = op_fa_fwd().below(q, k, v);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, out, *lse});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    variable_list g = as_list(op_fa_bwd()(grads[0], s[0], s[1], s[2], s[3], s[4]));
    g.emplace_back();
    return g;
  }
};

T2 fa_fwd_autograd(CT q, CT k, CT v) {
  if (!needs_grad(q, k, v)) return op_fa_fwd().below(q, k, v);
  Tensor lse;
  Tensor out = FaFwd::apply(q, k, v, &lse);
  return {out, lse};
}

struct QkvNormRopeV : torch::autograd::Function<QkvNormRopeV> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, CT qkv, CT qw, CT kw, CT cos, CT sin,
                               int64_t heads, double eps) {
    auto [q, k, v] = op_qkv_norm_rope_v().below(qkv, qw, kw, cos, sin, heads, eps);
    ctx->save_for_backward({qkv, qw, kw, cos, sin});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["eps"] = eps;
    return {q, k, v};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    auto [dqkv, dqw, dkw] =
        op_qkv_norm_rope_bwd()(s[0], g[0], g[1], g[2], s[1], s[2], s[3], s[4],
                               ctx->saved_data["heads"].toInt(), ctx->saved_data["eps"].toDouble());
    return {dqkv, dqw, dkw, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

T3 qkv_norm_rope_v_autograd(CT qkv, CT qw, CT kw, CT cos, CT sin, int64_t heads, double eps) {
  if (!needs_grad(qkv, qw, kw, cos, sin))
    return op_qkv_norm_rope_v().below(qkv, qw, kw, cos, sin, heads, eps);
  T3 r;
  from_list(QkvNormRopeV::apply(qkv, qw, kw, cos, sin, heads, eps), r);
  return r;
}

struct HeadNorm : torch::autograd::Function<HeadNorm> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, CT x, CT w, int64_t heads, double eps) {
    Tensor y = op_head_norm().below(x, w, heads, eps);
    ctx->save_for_backward({x, w});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    auto [dx, dw] = op_head_norm_bwd()(s[0], g[0], s[1], ctx->saved_data["heads"].toInt(),
                                       ctx->saved_data["eps"].toDouble());
    return {dx, dw, Tensor(), Tensor()};
  }
};

Tensor head_norm_autograd(CT x, CT w, int64_t heads, double eps) {
  if (!needs_grad(x, w)) return op_head_norm().below(x, w, heads, eps);
  return HeadNorm::apply(x, w, heads, eps);
}

// ------------------------------------------------------------- registration --

// Registrations live as long as the process, as torch.library's do.
std::vector<std::unique_ptr<torch::Library>>& libraries() {
  static auto* v = new std::vector<std::unique_ptr<torch::Library>>();
  return *v;
}

template <class Cuda, class Autograd>
void add(const std::string& ns, const char* name, Cuda cuda, Autograd autograd) {
  for (const auto key : {c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA}) {
    libraries().push_back(std::make_unique<torch::Library>(torch::Library::IMPL, ns, key, __FILE__, __LINE__));
    if (key == c10::DispatchKey::CUDA) libraries().back()->impl(name, cuda);
    else libraries().back()->impl(name, autograd);
  }
}

#define ANIMA_ADD(fn, autograd) \
  if (name == #fn) return add(ns, #fn, TORCH_FN(fn), autograd)
#define ANIMA_PLAIN(fn, ...) \
  if (name == #fn) return add(ns, #fn, TORCH_FN(fn), &Plain<&op_##fn, __VA_ARGS__>::call)

void add_kernels(const std::string& ns, const std::string& name) {
  ANIMA_ADD(fa_fwd, &fa_fwd_autograd);
  ANIMA_ADD(qkv_norm_rope_v, &qkv_norm_rope_v_autograd);
  ANIMA_ADD(head_norm, &head_norm_autograd);
  ANIMA_PLAIN(fa_fwd_nolse, Tensor, CT, CT, CT);
  ANIMA_PLAIN(fa_fwd_k, T2, CT, CT, CT, CT);
  ANIMA_PLAIN(fa_bwd, T3, CT, CT, CT, CT, CT, CT);
  ANIMA_PLAIN(fa_fwd_k_ctx, Tensor, CT, CT, CT, CT, CT);
  ANIMA_PLAIN(attend_d384, Tensor, CT, CT, CT);
  ANIMA_PLAIN(qkv_norm_rope, T2, CT, CT, CT, CT, CT, int64_t, double);
  ANIMA_PLAIN(qkv_norm_rope_bwd, T3, CT, CT, CT, CT, CT, CT, CT, CT, int64_t, double);
  ANIMA_PLAIN(head_norm_bwd, T2, CT, CT, CT, int64_t, double);
  ANIMA_PLAIN(qkv_proj_norm_rope, T3, CT, CT, CT, CT, CT, CT, int64_t, double);
  ANIMA_PLAIN(proj_head_norm, Tensor, CT, CT, CT, int64_t, double);
  ANIMA_PLAIN(kv_proj_norm, T2, CT, CT, CT, int64_t, double);
  TORCH_CHECK(false, "no native kernels for ", ns, "::", name);
}

// Gives op ns::name its native CUDA and AutogradCUDA kernels; `impl` is the
// op's Python function, for the calls they do not take.
void attach(const std::string& qualname, pybind11::function impl) {
  const size_t at = qualname.find("::");
  TORCH_CHECK(at != std::string::npos, "expected ns::name, got ", qualname);
  const std::string ns = qualname.substr(0, at), name = qualname.substr(at + 2);
  python_impls()[name] = impl.release().ptr();
  add_kernels(ns, name);
}

}  // namespace

PYBIND11_MODULE(_anima_torch, m) {
  m.def("attach", &attach, "Native dispatcher kernels for one op of the package");
  // What this file's argument structs are laid out for; the library may be newer.
  m.def("abi_version", [] { return AA_ABI_VERSION; }, "Of the header it was compiled with");
  m.def("library_abi_version", &aa_abi_version, "Of the libanima_attn.so it is linked to");
}
