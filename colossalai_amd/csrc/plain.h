// Whether a tensor may go to a kernel at once.
#pragma once

#include <ATen/TensorSubclassLikeUtils.h>
#include <torch/csrc/jit/frontend/tracer.h>

namespace cai {

// nothing that watches or rewrites single operations stands between this tensor and a kernel
inline bool plain(const at::Tensor& t) {
  return !at::isTensorSubclassLike(t) && !torch::jit::tracer::isTracing()
      && !c10::impl::tls_is_dispatch_key_included(at::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

inline bool has_tangent(const at::Tensor& t) { return t._fw_grad(0).defined(); }

}  // namespace cai
