// Autograd functions of the training kernels for tensors that nothing stands between: where the kernels are short the host
// bounds a step, and a function written in Python takes it longer. Attention over 8 x 197 tokens, 12 heads of 64, forward and
// backward: 100 us with the Python function, 78 with this one; a training step of two 512-wide layers 1130 and 1030. What
// a transform, a mode or a tracer wants to see goes to the Python functions (the result is empty here).
#include <torch/extension.h>

#include "plain.h"

namespace cai {

std::vector<at::Tensor> rmsnorm_fwd(at::Tensor input, at::Tensor weight, double eps, bool save_inv_rms);
std::vector<at::Tensor> rmsnorm_fused_add_fwd(at::Tensor input, at::Tensor residual, at::Tensor weight, double eps,
                                              bool save_inv_rms, c10::optional<at::Tensor> res_out);
std::vector<at::Tensor> rmsnorm_bwd(at::Tensor dy, at::Tensor x, at::Tensor weight, at::Tensor inv_rms,
                                    c10::optional<at::Tensor> dres, bool cast_dw);
at::Tensor swiglu_fwd(at::Tensor gate_up);
at::Tensor swiglu_bwd(at::Tensor dout, at::Tensor gate_up);
void rope_inplace(at::Tensor q, c10::optional<at::Tensor> k, at::Tensor table, c10::optional<at::Tensor> positions, bool backward);
std::vector<at::Tensor> flash_attn_fwd(at::Tensor q, at::Tensor k, at::Tensor v, bool causal, double scale,
                                       c10::optional<at::Tensor> seqlens, c10::optional<at::Tensor> seqlens_k);
std::vector<at::Tensor> flash_attn_bwd(at::Tensor dout, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor out, at::Tensor lse,
                                       bool causal, double scale, at::Tensor dq, at::Tensor dk, at::Tensor dv,
                                       c10::optional<at::Tensor> seqlens, c10::optional<at::Tensor> seqlens_k);
std::vector<at::Tensor> flash_attn_varlen_fwd(at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor cu_seqlens, long max_seqlen,
                                              bool causal, double scale);
std::vector<at::Tensor> flash_attn_varlen_bwd(at::Tensor dout, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor out,
                                              at::Tensor lse, at::Tensor cu_seqlens, long max_seqlen, bool causal, double scale);

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using Maybe = c10::optional<at::Tensor>;

const at::Tensor none;

Maybe maybe(const at::Tensor& t) { return t.defined() ? Maybe(t) : c10::nullopt; }

struct RMSNorm : torch::autograd::Function<RMSNorm> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x_in, const at::Tensor& weight, double eps) {
    const at::Tensor x = x_in.contiguous();
    auto r = rmsnorm_fwd(x, weight.contiguous(), eps, true);
    ctx->save_for_backward({x, weight, r[1]});
    return r[0];
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto r = rmsnorm_bwd(grads[0].contiguous(), s[0], s[1], s[2], c10::nullopt, true);
    return {r[0], r[1].to(s[1].scalar_type()), none};
  }
};

struct FusedAddRMSNorm : torch::autograd::Function<FusedAddRMSNorm> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& residual_in, const at::Tensor& weight, double eps) {
    const at::Tensor residual = residual_in.contiguous(), res = at::empty_like(residual);
    auto r = rmsnorm_fused_add_fwd(x.contiguous(), residual, weight.contiguous(), eps, true, res);
    ctx->save_for_backward({res, weight, r[1]});
    return {r[0], res};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const at::Tensor &h = s[0], &weight = s[1], &dres = grads[1];
    // the residual stream's gradient rides along, unless the backward is part of a graph itself (create_graph): the
    // kernel's result would end it
    const bool fused = dres.defined() && dres.scalar_type() == h.scalar_type() && !at::GradMode::is_enabled();
    auto r = rmsnorm_bwd(grads[0].contiguous(), h, weight, s[2], fused ? Maybe(dres.contiguous()) : c10::nullopt, true);
    const at::Tensor total = dres.defined() && !fused ? r[0] + dres : r[0];
    return {total, total, r[1].to(weight.scalar_type()), none};
  }
};

struct SwiGLU : torch::autograd::Function<SwiGLU> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& gate_up) {
    ctx->save_for_backward({gate_up});
    return swiglu_fwd(gate_up.contiguous());
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return {swiglu_bwd(grads[0].contiguous(), ctx->get_saved_variables()[0].contiguous())};
  }
};

struct FlashAttention : torch::autograd::Function<FlashAttention> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal,
                            double scale, const Maybe& seqlens, const Maybe& seqlens_k) {
    auto r = flash_attn_fwd(q, k, v, causal, scale, seqlens, seqlens_k);
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->save_for_backward({q, k, v, r[0], r[1], seqlens.value_or(none), seqlens_k.value_or(none)});
    return r[0];
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto r = flash_attn_bwd(grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4], ctx->saved_data["causal"].toBool(),
                            ctx->saved_data["scale"].toDouble(), none, none, none, maybe(s[5]), maybe(s[6]));
    return {r[0], r[1], r[2], none, none, none, none};
  }
};

struct FlashAttentionVarlen : torch::autograd::Function<FlashAttentionVarlen> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                            const at::Tensor& cu, int64_t longest, bool causal, double scale) {
    auto r = flash_attn_varlen_fwd(q, k, v, cu, longest, causal, scale);
    ctx->saved_data["longest"] = longest;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->save_for_backward({q, k, v, r[0], r[1], cu});
    return r[0];
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto r = flash_attn_varlen_bwd(grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4], s[5], ctx->saved_data["longest"].toInt(),
                                   ctx->saved_data["causal"].toBool(), ctx->saved_data["scale"].toDouble());
    return {r[0], r[1], r[2], none, none, none, none};
  }
};

// the queries, keys and values of [B, S, (Hq + 2 Hkv) D]
struct Heads {
  at::Tensor q, k, v;
  Heads(const at::Tensor& t, int64_t Hq, int64_t Hkv, int64_t D) {
    const int64_t B = t.size(0), S = t.size(1);
    q = t.slice(2, 0, Hq * D).view({B, S, Hq, D});
    k = t.slice(2, Hq * D, (Hq + Hkv) * D).view({B, S, Hkv, D});
    v = t.slice(2, (Hq + Hkv) * D).view({B, S, Hkv, D});
  }
};

struct FusedRopeAttention : torch::autograd::Function<FusedRopeAttention> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& qkv, const at::Tensor& table, const Maybe& positions, int64_t Hq,
                            int64_t Hkv, int64_t D, bool causal, double scale, const Maybe& seqlens) {
    const Heads h(qkv, Hq, Hkv, D);
    rope_inplace(h.q, h.k, table, positions, false);
    auto r = flash_attn_fwd(h.q, h.k, h.v, causal, scale, seqlens, c10::nullopt);
    ctx->saved_data["heads"] = std::vector<int64_t>{Hq, Hkv, D, causal};
    ctx->saved_data["scale"] = scale;
    ctx->save_for_backward({qkv, r[0], r[1], table, positions.value_or(none), seqlens.value_or(none)});
    return r[0];
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const auto n = ctx->saved_data["heads"].toIntVector();
    const at::Tensor dqkv = at::empty_like(s[0]);
    const Heads h(s[0], n[0], n[1], n[2]), d(dqkv, n[0], n[1], n[2]);
    flash_attn_bwd(grads[0].contiguous(), h.q, h.k, h.v, s[1], s[2], n[3], ctx->saved_data["scale"].toDouble(), d.q, d.k, d.v,
                   maybe(s[5]), c10::nullopt);
    rope_inplace(d.q, d.k, s[3], maybe(s[4]), true);
    return {dqkv, none, none, none, none, none, none, none, none};
  }
};

bool direct(at::TensorList tensors) {
  for (const at::Tensor& t : tensors)
    if (!t.is_cuda() || !plain(t) || has_tangent(t)) return false;
  return true;
}

}  // namespace

Maybe native_rms_norm(const at::Tensor& x, const at::Tensor& weight, double eps) {
  if (!direct({x, weight})) return c10::nullopt;
  return RMSNorm::apply(x, weight, eps);
}

c10::optional<std::tuple<at::Tensor, at::Tensor>> native_fused_add_rms_norm(const at::Tensor& x, const at::Tensor& residual,
                                                                           const at::Tensor& weight, double eps) {
  if (!direct({x, residual, weight})) return c10::nullopt;
  auto r = FusedAddRMSNorm::apply(x, residual, weight, eps);
  return std::make_tuple(r[0], r[1]);
}

Maybe native_swiglu(const at::Tensor& gate_up) {
  if (!direct({gate_up})) return c10::nullopt;
  return SwiGLU::apply(gate_up);
}

Maybe native_flash_attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal, double scale,
                             const Maybe& seqlens, const Maybe& seqlens_k) {
  if (!direct({q, k, v})) return c10::nullopt;
  return FlashAttention::apply(q, k, v, causal, scale, seqlens, seqlens_k);
}

Maybe native_flash_attention_varlen(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cu,
                                    int64_t longest, bool causal, double scale) {
  if (!direct({q, k, v})) return c10::nullopt;
  return FlashAttentionVarlen::apply(q, k, v, cu, longest, causal, scale);
}

Maybe native_fused_rope_attention(const at::Tensor& qkv, const at::Tensor& table, const Maybe& positions, int64_t Hq, int64_t Hkv,
                                  int64_t D, bool causal, double scale, const Maybe& seqlens) {
  if (!direct({qkv})) return c10::nullopt;
  return FusedRopeAttention::apply(qkv, table, positions, Hq, Hkv, D, causal, scale, seqlens);
}

}  // namespace cai
