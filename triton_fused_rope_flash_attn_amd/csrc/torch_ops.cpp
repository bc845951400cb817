// Native kernels of the torch ops farope::attn_fwd, farope::attn_bwd and their
// packed-layout forms farope::attn_qkv_fwd, farope::attn_qkv_bwd.
//
// The ops, their schemas, fake kernels and CPU errors are defined in
// attention.py.  This library adds their GPU kernels (dispatch keys CUDA and
// AutogradCUDA, which take precedence over the definitions there): argument
// checks, allocation and the C ABI call without the interpreter, and an
// autograd node whose backward runs on the engine's thread without taking the
// interpreter lock.  Small calls are bound by exactly that host work: a
// training pass of 96 planes of 197 rows took 226 us around 43 us of kernels
// with the Python kernels, 70 to 75 us with these (box to box).
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/library.h>

#include <sstream>

#include "farope.h"

namespace {

using at::Tensor;
using torch::autograd::variable_list;
using Three = std::tuple<Tensor, Tensor, Tensor>;

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? FAROPE_F32 : t == at::kHalf ? FAROPE_F16 : t == at::kBFloat16 ? FAROPE_BF16 : -1;
}
std::string shape_str(const Tensor& t) {
  std::ostringstream s;
  s << '(';
  for (int64_t i = 0; i < t.dim(); ++i) s << (i ? ", " : "") << t.size(i);
  s << (t.dim() == 1 ? ",)" : ")");
  return s.str();
}
std::string dtype_str(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return "torch.float32";
    case at::kHalf: return "torch.float16";
    case at::kBFloat16: return "torch.bfloat16";
    case at::kDouble: return "torch.float64";
    default: return std::string("torch.") + c10::toString(t.scalar_type());
  }
}

void check_qkv(const Tensor& q, const Tensor& k, const Tensor& v) {
  TORCH_CHECK_VALUE(q.dim() == 4, "Q must be [B, H, N, D]; got shape ", shape_str(q));
  TORCH_CHECK_VALUE(k.sizes() == q.sizes() && v.sizes() == q.sizes(), "Q, K, V must have the same shape; got ",
                    shape_str(q), ", ", shape_str(k), ", ", shape_str(v));
  TORCH_CHECK_TYPE(dtype_code(q.scalar_type()) >= 0, "farope: unsupported tensor dtype ", dtype_str(q));
  TORCH_CHECK_TYPE(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(),
                   "farope: Q, K, V must share one dtype; got ", dtype_str(q), ", ", dtype_str(k), ", ", dtype_str(v));
  TORCH_CHECK(q.is_cuda(), "farope runs on ROCm GPUs only (hand-written gfx950 kernels); got a ", q.device(), " tensor");
  TORCH_CHECK(k.device() == q.device() && v.device() == q.device(), "farope: Q, K, V must be on the same device");
}

void check_rope(const Tensor& rope, int64_t n_pos, int64_t d, const at::Device& device) {
  const int64_t want = (n_pos + 1) * (d / 2) * 2;
  TORCH_CHECK_VALUE(rope.scalar_type() == at::kFloat && rope.dim() == 1 && rope.numel() == want && rope.is_contiguous(),
                    "farope: packed RoPE table must be contiguous fp32 of ", want, " elements for n_pos=", n_pos, ", D=", d,
                    "; got ", dtype_str(rope), " ", shape_str(rope));
  TORCH_CHECK(rope.device() == device, "farope: RoPE table on ", rope.device(), ", tensors on ", device);
}

farope_attn_desc make_desc(int64_t B, int64_t H, int64_t N, int64_t D, at::ScalarType io, int64_t n_pos, bool has_cls,
                           double scale, int64_t comp) {
  // (sizes past 32 bits are refused, not wrapped)
  for (int64_t s : {B, H, N, D, n_pos, comp})
    TORCH_CHECK_VALUE(s >= 0 && s <= INT32_MAX, "farope: sizes must fit 32 bits");
  farope_attn_desc d;
  d.batch = (int32_t)B;
  d.heads = (int32_t)H;
  d.seq_len = (int32_t)N;
  d.head_dim = (int32_t)D;
  d.n_pos = (int32_t)n_pos;
  d.has_cls = has_cls ? 1 : 0;
  d.io_dtype = dtype_code(io);
  d.compute_dtype = (int32_t)comp;
  d.softmax_scale = (float)scale;
  return d;
}

void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == FAROPE_OK, what, ": ", farope_strerror(rc), " (status ", rc, ")");
}

const int64_t* strides(const Tensor& t) { return t.strides().data(); }
float* floats(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr<float>() : nullptr; }
void* data(const Tensor& t) { return t.numel() ? t.data_ptr() : nullptr; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }
Tensor workspace(const Tensor& like, size_t elems) {
  return elems ? at::empty({(int64_t)elems}, like.options().dtype(at::kFloat)) : Tensor();
}

Three attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& rope, int64_t n_pos, bool has_cls,
               double scale, int64_t comp) {
  check_qkv(q, k, v);
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
  check_rope(rope, n_pos, D, q.device());
  const c10::DeviceGuard guard(q.device());
  const farope_attn_desc desc = make_desc(B, H, N, D, q.scalar_type(), n_pos, has_cls, scale, comp);
  const Tensor o = at::empty({B, H, N, D}, q.options());
  const Tensor lse = at::empty({B, H, N}, q.options().dtype(at::kFloat));
  const bool res = farope_attn_residual_elems(&desc) != 0;
  const Tensor o_res = res ? at::empty({B, H, N, D}, q.options()) : at::empty({0}, q.options());
  const Tensor ws = workspace(q, farope_attn_fwd_workspace_elems(&desc));
  check_rc(farope_attn_fwd_ws(&desc, q.data_ptr(), strides(q), k.data_ptr(), strides(k), v.data_ptr(), strides(v),
                              floats(rope), (size_t)rope.numel(), o.data_ptr(), strides(o), data(o_res),
                              lse.data_ptr<float>(), floats(ws), stream_of(q)),
           "farope_attn_fwd");
  return {o, lse, o_res};
}

Three attn_bwd(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
               const Tensor& rope, int64_t n_pos, bool has_cls, double scale, int64_t comp, const Tensor& o_res) {
  check_qkv(q, k, v);
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
  check_rope(rope, n_pos, D, q.device());
  TORCH_CHECK_VALUE(dout.sizes() == q.sizes() && o.sizes() == q.sizes(), "farope: dO and O must have Q's shape");
  TORCH_CHECK(dout.device() == q.device() && o.device() == q.device() && lse.device() == q.device() &&
                  o_res.device() == q.device(),
              "farope: dO, O, LSE and O_res must be on Q's device");
  const Tensor g = dout.scalar_type() == q.scalar_type() ? dout : dout.to(q.scalar_type());
  TORCH_CHECK_TYPE(o.scalar_type() == q.scalar_type(), "farope: O must have Q's dtype; got ", dtype_str(o));
  TORCH_CHECK_VALUE(lse.scalar_type() == at::kFloat && lse.dim() == 3 && lse.size(0) == B && lse.size(1) == H &&
                        lse.size(2) == N && lse.is_contiguous(),
                    "farope: LSE must be contiguous fp32 [B, H, N]");
  TORCH_CHECK_VALUE(!o_res.numel() || (o_res.sizes() == q.sizes() && o_res.scalar_type() == q.scalar_type() &&
                                       o_res.is_contiguous()),
                    "farope: O_res must be contiguous with Q's shape and dtype, or empty");
  const c10::DeviceGuard guard(q.device());
  const farope_attn_desc desc = make_desc(B, H, N, D, q.scalar_type(), n_pos, has_cls, scale, comp);
  const Tensor dq = at::empty({B, H, N, D}, q.options());
  const Tensor dk = at::empty({B, H, N, D}, q.options());
  const Tensor dv = at::empty({B, H, N, D}, q.options());
  const Tensor ws = workspace(q, farope_attn_bwd_workspace_elems(&desc));
  check_rc(farope_attn_bwd(&desc, q.data_ptr(), strides(q), k.data_ptr(), strides(k), v.data_ptr(), strides(v),
                           o.data_ptr(), strides(o), data(o_res), g.data_ptr(), strides(g), lse.data_ptr<float>(),
                           floats(rope), (size_t)rope.numel(), dq.data_ptr(), strides(dq), dk.data_ptr(), strides(dk),
                           dv.data_ptr(), strides(dv), floats(ws), stream_of(q)),
           "farope_attn_bwd");
  return {dq, dk, dv};
}

// ---------------------------------------------------------------------------
// Packed layout: q, k, v are thirds of one [B, N, 3 H D] projection output and
// O is [B, N, H D], as an attention layer's two projections hold them.  The
// kernels read and write those places directly, so neither pass copies.
// ---------------------------------------------------------------------------
struct Heads {   // [B, H, N, D] view of part `third` of a [B, N, parts H D] tensor
  void* ptr;
  int64_t st[4];
  Heads(const Tensor& t, int64_t third, int64_t H, int64_t D)
      : ptr(static_cast<char*>(t.data_ptr()) + third * H * D * t.stride(2) * (int64_t)t.element_size()),
        st{t.stride(0), D * t.stride(2), t.stride(1), t.stride(2)} {}
};

int64_t check_packed(const Tensor& qkv, const Tensor& rope, int64_t heads, int64_t n_pos) {
  TORCH_CHECK_VALUE(qkv.dim() == 3 && heads > 0 && qkv.size(2) % (3 * heads) == 0,
                    "farope: qkv must be [B, N, 3 * heads * head_dim]; got ", shape_str(qkv), " for ", heads, " heads");
  TORCH_CHECK_TYPE(dtype_code(qkv.scalar_type()) >= 0, "farope: unsupported tensor dtype ", dtype_str(qkv));
  TORCH_CHECK(qkv.is_cuda(), "farope runs on ROCm GPUs only (hand-written gfx950 kernels); got a ", qkv.device(), " tensor");
  const int64_t D = qkv.size(2) / (3 * heads);
  check_rope(rope, n_pos, D, qkv.device());
  return D;
}

Three attn_qkv_fwd(const Tensor& qkv, const Tensor& rope, int64_t heads, int64_t n_pos, bool has_cls, double scale,
                   int64_t comp) {
  const int64_t D = check_packed(qkv, rope, heads, n_pos), B = qkv.size(0), N = qkv.size(1);
  const c10::DeviceGuard guard(qkv.device());
  const farope_attn_desc desc = make_desc(B, heads, N, D, qkv.scalar_type(), n_pos, has_cls, scale, comp);
  const Tensor out = at::empty({B, N, heads * D}, qkv.options());
  const Tensor lse = at::empty({B, heads, N}, qkv.options().dtype(at::kFloat));
  const bool res = farope_attn_residual_elems(&desc) != 0;
  const Tensor o_res = res ? at::empty({B, heads, N, D}, qkv.options()) : at::empty({0}, qkv.options());
  const Tensor ws = workspace(qkv, farope_attn_fwd_workspace_elems(&desc));
  const Heads q(qkv, 0, heads, D), k(qkv, 1, heads, D), v(qkv, 2, heads, D), o(out, 0, heads, D);
  check_rc(farope_attn_fwd_ws(&desc, q.ptr, q.st, k.ptr, k.st, v.ptr, v.st, floats(rope), (size_t)rope.numel(), o.ptr, o.st,
                              data(o_res), lse.data_ptr<float>(), floats(ws), stream_of(qkv)),
           "farope_attn_fwd");
  return {out, lse, o_res};
}

Tensor attn_qkv_bwd(const Tensor& dout, const Tensor& qkv, const Tensor& out, const Tensor& lse, const Tensor& rope,
                    int64_t heads, int64_t n_pos, bool has_cls, double scale, int64_t comp, const Tensor& o_res) {
  const int64_t D = check_packed(qkv, rope, heads, n_pos), B = qkv.size(0), N = qkv.size(1);
  TORCH_CHECK_VALUE(out.dim() == 3 && out.size(0) == B && out.size(1) == N && out.size(2) == heads * D &&
                        dout.sizes() == out.sizes(),
                    "farope: dO and O must be [B, N, heads * head_dim]");
  TORCH_CHECK(dout.device() == qkv.device() && out.device() == qkv.device() && lse.device() == qkv.device() &&
                  o_res.device() == qkv.device(),
              "farope: dO, O, LSE and O_res must be on qkv's device");
  const Tensor g = dout.scalar_type() == qkv.scalar_type() ? dout : dout.to(qkv.scalar_type());
  TORCH_CHECK_TYPE(out.scalar_type() == qkv.scalar_type(), "farope: O must have qkv's dtype; got ", dtype_str(out));
  TORCH_CHECK_VALUE(lse.scalar_type() == at::kFloat && lse.dim() == 3 && lse.size(0) == B && lse.size(1) == heads &&
                        lse.size(2) == N && lse.is_contiguous(),
                    "farope: LSE must be contiguous fp32 [B, H, N]");
  TORCH_CHECK_VALUE(!o_res.numel() || (o_res.dim() == 4 && o_res.numel() == out.numel() && o_res.size(1) == heads &&
                                       o_res.scalar_type() == qkv.scalar_type() && o_res.is_contiguous()),
                    "farope: O_res must be contiguous [B, H, N, D] of qkv's dtype, or empty");
  const c10::DeviceGuard guard(qkv.device());
  const farope_attn_desc desc = make_desc(B, heads, N, D, qkv.scalar_type(), n_pos, has_cls, scale, comp);
  const Tensor dqkv = at::empty({B, N, 3 * heads * D}, qkv.options());
  const Tensor ws = workspace(qkv, farope_attn_bwd_workspace_elems(&desc));
  const Heads q(qkv, 0, heads, D), k(qkv, 1, heads, D), v(qkv, 2, heads, D), o(out, 0, heads, D), d(g, 0, heads, D);
  const Heads dq(dqkv, 0, heads, D), dk(dqkv, 1, heads, D), dv(dqkv, 2, heads, D);
  check_rc(farope_attn_bwd(&desc, q.ptr, q.st, k.ptr, k.st, v.ptr, v.st, o.ptr, o.st, data(o_res), d.ptr, d.st,
                           lse.data_ptr<float>(), floats(rope), (size_t)rope.numel(), dq.ptr, dq.st, dk.ptr, dk.st, dv.ptr,
                           dv.st, floats(ws), stream_of(qkv)),
           "farope_attn_bwd");
  return dqkv;
}

// ---------------------------------------------------------------------------
// Autograd.  n_pos and compute_dtype stay symbolic, as in the ops' schemas, so
// that tracing with symbolic sizes sees them unchanged.
// ---------------------------------------------------------------------------
using FwdSig = Three(const Tensor&, const Tensor&, const Tensor&, const Tensor&, c10::SymInt, bool, double, c10::SymInt);
using BwdSig = Three(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                     c10::SymInt, bool, double, c10::SymInt, const Tensor&);
const c10::TypedOperatorHandle<FwdSig>& fwd_op() {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("farope::attn_fwd", "").typed<FwdSig>();
  return op;
}
const c10::TypedOperatorHandle<BwdSig>& bwd_op() {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("farope::attn_bwd", "").typed<BwdSig>();
  return op;
}
variable_list list3(const Three& t) { return {std::get<0>(t), std::get<1>(t), std::get<2>(t)}; }

struct AttnFwdNode : torch::autograd::Function<AttnFwdNode> {
  static variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const Tensor& rope, c10::SymInt n_pos, bool has_cls, double scale, c10::SymInt comp) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Three r = fwd_op().call(q, k, v, rope, n_pos, has_cls, scale, comp);
    const auto& [o, lse, o_res] = r;
    ctx->mark_non_differentiable({lse, o_res});
    // LSE's and the residual's incoming gradients are never used: no zero
    // tensors are made for them
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, o, lse, rope, o_res});
    ctx->saved_data["n_pos"] = n_pos;
    ctx->saved_data["has_cls"] = has_cls;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["comp"] = comp;
    return list3(r);
  }
  static variable_list backward(torch::autograd::AutogradContext* ctx, variable_list grads) {
    variable_list out(8);
    if (!grads[0].defined()) return out;   // O received no gradient
    const variable_list s = ctx->get_saved_variables();
    const Three g = bwd_op().call(grads[0], s[0], s[1], s[2], s[3], s[4], s[5], ctx->saved_data["n_pos"].toSymInt(),
                                  ctx->saved_data["has_cls"].toBool(), ctx->saved_data["scale"].toDouble(),
                                  ctx->saved_data["comp"].toSymInt(), s[6]);
    std::tie(out[0], out[1], out[2]) = g;
    return out;
  }
};

// The gradients are not differentiable again.
struct AttnBwdNode : torch::autograd::Function<AttnBwdNode> {
  static variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& dout, const Tensor& q, const Tensor& k,
                               const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& rope, c10::SymInt n_pos,
                               bool has_cls, double scale, c10::SymInt comp, const Tensor& o_res) {
    at::AutoDispatchBelowADInplaceOrView below;
    return list3(bwd_op().call(dout, q, k, v, o, lse, rope, n_pos, has_cls, scale, comp, o_res));
  }
  static variable_list backward(torch::autograd::AutogradContext*, variable_list) {
    TORCH_CHECK(false,
                "Trying to backward through farope.attn_bwd.default but no autograd formula was registered "
                "(the attention's gradients are not differentiable again).");
  }
};

bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

Three attn_fwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& rope, c10::SymInt n_pos, bool has_cls,
                        double scale, c10::SymInt comp) {
  if (at::GradMode::is_enabled() && any_requires_grad({&q, &k, &v, &rope})) {
    const variable_list r = AttnFwdNode::apply(q, k, v, rope, n_pos, has_cls, scale, comp);
    return {r[0], r[1], r[2]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  return fwd_op().call(q, k, v, rope, n_pos, has_cls, scale, comp);
}

Three attn_bwd_autograd(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                        const Tensor& lse, const Tensor& rope, c10::SymInt n_pos, bool has_cls, double scale, c10::SymInt comp,
                        const Tensor& o_res) {
  if (at::GradMode::is_enabled() && any_requires_grad({&dout, &q, &k, &v, &o, &lse, &rope, &o_res})) {
    const variable_list r = AttnBwdNode::apply(dout, q, k, v, o, lse, rope, n_pos, has_cls, scale, comp, o_res);
    return {r[0], r[1], r[2]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  return bwd_op().call(dout, q, k, v, o, lse, rope, n_pos, has_cls, scale, comp, o_res);
}

using QkvFwdSig = Three(const Tensor&, const Tensor&, c10::SymInt, c10::SymInt, bool, double, c10::SymInt);
using QkvBwdSig = Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, c10::SymInt, c10::SymInt,
                         bool, double, c10::SymInt, const Tensor&);
const c10::TypedOperatorHandle<QkvFwdSig>& qkv_fwd_op() {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("farope::attn_qkv_fwd", "").typed<QkvFwdSig>();
  return op;
}
const c10::TypedOperatorHandle<QkvBwdSig>& qkv_bwd_op() {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("farope::attn_qkv_bwd", "").typed<QkvBwdSig>();
  return op;
}

struct QkvFwdNode : torch::autograd::Function<QkvFwdNode> {
  static variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& qkv, const Tensor& rope, c10::SymInt heads,
                               c10::SymInt n_pos, bool has_cls, double scale, c10::SymInt comp) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Three r = qkv_fwd_op().call(qkv, rope, heads, n_pos, has_cls, scale, comp);
    const auto& [o, lse, o_res] = r;
    ctx->mark_non_differentiable({lse, o_res});
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({qkv, o, lse, rope, o_res});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["n_pos"] = n_pos;
    ctx->saved_data["has_cls"] = has_cls;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["comp"] = comp;
    return list3(r);
  }
  static variable_list backward(torch::autograd::AutogradContext* ctx, variable_list grads) {
    variable_list out(7);
    if (!grads[0].defined()) return out;
    const variable_list s = ctx->get_saved_variables();
    out[0] = qkv_bwd_op().call(grads[0], s[0], s[1], s[2], s[3], ctx->saved_data["heads"].toSymInt(),
                               ctx->saved_data["n_pos"].toSymInt(), ctx->saved_data["has_cls"].toBool(),
                               ctx->saved_data["scale"].toDouble(), ctx->saved_data["comp"].toSymInt(), s[4]);
    return out;
  }
};

struct QkvBwdNode : torch::autograd::Function<QkvBwdNode> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& dout, const Tensor& qkv, const Tensor& o,
                        const Tensor& lse, const Tensor& rope, c10::SymInt heads, c10::SymInt n_pos, bool has_cls, double scale,
                        c10::SymInt comp, const Tensor& o_res) {
    at::AutoDispatchBelowADInplaceOrView below;
    return qkv_bwd_op().call(dout, qkv, o, lse, rope, heads, n_pos, has_cls, scale, comp, o_res);
  }
  static variable_list backward(torch::autograd::AutogradContext*, variable_list) {
    TORCH_CHECK(false,
                "Trying to backward through farope.attn_qkv_bwd.default but no autograd formula was registered "
                "(the attention's gradients are not differentiable again).");
  }
};

Three attn_qkv_fwd_autograd(const Tensor& qkv, const Tensor& rope, c10::SymInt heads, c10::SymInt n_pos, bool has_cls,
                            double scale, c10::SymInt comp) {
  if (at::GradMode::is_enabled() && any_requires_grad({&qkv, &rope})) {
    const variable_list r = QkvFwdNode::apply(qkv, rope, heads, n_pos, has_cls, scale, comp);
    return {r[0], r[1], r[2]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  return qkv_fwd_op().call(qkv, rope, heads, n_pos, has_cls, scale, comp);
}

Tensor attn_qkv_bwd_autograd(const Tensor& dout, const Tensor& qkv, const Tensor& o, const Tensor& lse, const Tensor& rope,
                             c10::SymInt heads, c10::SymInt n_pos, bool has_cls, double scale, c10::SymInt comp,
                             const Tensor& o_res) {
  if (at::GradMode::is_enabled() && any_requires_grad({&dout, &qkv, &o, &lse, &rope, &o_res}))
    return QkvBwdNode::apply(dout, qkv, o, lse, rope, heads, n_pos, has_cls, scale, comp, o_res);
  at::AutoDispatchBelowADInplaceOrView below;
  return qkv_bwd_op().call(dout, qkv, o, lse, rope, heads, n_pos, has_cls, scale, comp, o_res);
}

}  // namespace

TORCH_LIBRARY_IMPL(farope, CUDA, m) {
  m.impl("attn_fwd", attn_fwd);
  m.impl("attn_bwd", attn_bwd);
  m.impl("attn_qkv_fwd", attn_qkv_fwd);
  m.impl("attn_qkv_bwd", attn_qkv_bwd);
}

TORCH_LIBRARY_IMPL(farope, AutogradCUDA, m) {
  m.impl("attn_fwd", attn_fwd_autograd);
  m.impl("attn_bwd", attn_bwd_autograd);
  m.impl("attn_qkv_fwd", attn_qkv_fwd_autograd);
  m.impl("attn_qkv_bwd", attn_qkv_bwd_autograd);
}
