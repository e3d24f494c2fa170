// Linear layers without a bias: weight gradients and small products are csrc/products.hip's, the others the library's.
#include <ATen/autocast_mode.h>
#include <torch/extension.h>

#include "plain.h"

namespace cai {

at::Tensor weight_grad(const at::Tensor& dy, const at::Tensor& x, const c10::optional<at::Tensor>& add, bool keep);
bool weight_grad_serves(const at::Tensor& dy, const at::Tensor& x);
at::Tensor multiply(const at::Tensor& x, const at::Tensor& w, bool slow);
std::vector<at::Tensor> linear_grads(const at::Tensor& dy, const at::Tensor& w, const at::Tensor& x);

namespace {

// not under autocast either, which casts the operands of the library's products
bool plain_here(const at::Tensor& t) { return plain(t) && !at::autocast::is_autocast_enabled(at::kCUDA); }

struct Linear : torch::autograd::Function<Linear> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& weight) {
    // as the built-in layer: each gradient's factor is kept only if that gradient is wanted
    ctx->save_for_backward({x, x.requires_grad() ? weight : at::Tensor()});
    if (x.size(-1) != weight.size(1) || weight.dim() != 2) return at::linear(x, weight);   // which says what is wrong
    auto sizes = x.sizes().vec();
    sizes.back() = weight.size(0);
    return at::_unsafe_view(multiply(x.reshape({-1, x.size(-1)}), weight, false), sizes);   // no view, which may not be changed in place
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &x = saved[0], &weight = saved[1], &dy = grads[0];
    if (!dy.defined()) return {at::Tensor(), at::Tensor()};
    const at::Tensor dy2 = dy.reshape({-1, dy.size(-1)});
    at::Tensor dx, dw;
    // a backward that is part of a graph itself (create_graph), or that something watches, takes operations it can see
    const bool closed = !at::GradMode::is_enabled() && plain_here(dy2);
    if (closed && ctx->needs_input_grad(0) && ctx->needs_input_grad(1) && plain_here(weight) && plain_here(x)) {
      const auto both = linear_grads(dy2, weight, x.reshape({-1, x.size(-1)}));
      if (!both.empty()) return {both[0].view(x.sizes()), both[1]};
    }
    if (ctx->needs_input_grad(0)) dx = (closed && plain_here(weight) ? multiply(dy2, weight, true) : at::mm(dy2, weight)).view(x.sizes());
    if (ctx->needs_input_grad(1)) {
      const at::Tensor x2 = x.reshape({-1, x.size(-1)});
      if (closed && plain_here(x2) && weight_grad_serves(dy2, x2)) dw = weight_grad(dy2, x2, c10::nullopt, false);
      else dw = at::mm(dy2.t(), x2);
    }
    return {dx, dw};
  }
};

}  // namespace

at::Tensor linear(const at::Tensor& x, const at::Tensor& weight) {
  if (x.dim() < 2 || x.numel() == 0 || !plain_here(x) || !plain_here(weight) || has_tangent(x) || has_tangent(weight)) return at::linear(x, weight);
  return Linear::apply(x, weight);
}

}  // namespace cai
