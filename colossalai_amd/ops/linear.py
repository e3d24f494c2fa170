"""Linear layers in training: the weight gradient and small products of a plain bfloat16 ``nn.Linear`` by
csrc/products.hip, the table's gradient of a plain ``nn.Embedding`` by csrc/embedding.hip.

The layer stays an ``nn.Linear`` that parallel policies, LoRA or the zero-bubble schedule replace or change; ``project``
calls whatever it has become.
"""

from typing import Optional

import torch
import torch.nn as nn
from torch.nn.modules import module as _hooks

from ._kernels import kernels

__all__ = ["embed", "multiply", "project", "weight_grad"]


def multiply(x: torch.Tensor, w: torch.Tensor, slow: bool = False) -> torch.Tensor:
    """x [M, K] times w [N, K]^T, or with ``slow`` times w [K, N]; outside autograd."""
    if x.is_cuda:
        return kernels().multiply(x, w, slow)
    return x @ (w if slow else w.t())


def weight_grad(dy: torch.Tensor, x: torch.Tensor, add: Optional[torch.Tensor] = None, keep: bool = False) -> torch.Tensor:
    """dy [K, M], x [K, N] -> dy^T x (+ ``add``, float32) in their type, or in float32 with ``keep``: then in ``add`` if given."""
    if dy.is_cuda:
        return kernels().weight_grad(dy, x, add, keep)
    part = dy.t() @ x
    if add is not None:
        part = add.add_(part) if keep else add + part
    return part.to(torch.float32 if keep else dy.dtype)


def _bare(layer: nn.Module) -> bool:
    """Whether calling the layer is its own forward and nothing else: no hooks, no forward of the instance's own."""
    return not (layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks or layer._backward_pre_hooks
                or _hooks._global_forward_hooks or _hooks._global_forward_pre_hooks
                or _hooks._global_backward_hooks or _hooks._global_backward_pre_hooks or "forward" in layer.__dict__)


def project(layer: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``layer(x)``. Plain bfloat16 layers whose weight is trained take the native form; layers of other types or with
    hooks, tensor subclasses, other data types, function modes, compilation and anything under autocast are called."""
    if (type(layer) is nn.Linear and type(x) is torch.Tensor and x.is_cuda and x.dtype is torch.bfloat16
            and not torch.compiler.is_compiling() and torch.is_grad_enabled()):
        weight = layer.weight
        if (layer.bias is None and type(weight) is nn.Parameter and weight.requires_grad and weight.dtype is torch.bfloat16
                and weight.device == x.device and _bare(layer) and not torch._C._len_torch_function_stack()):
            return kernels().linear(x, weight)
    return layer(x)


def embed(layer: nn.Module, tokens: torch.Tensor) -> torch.Tensor:
    """``layer(tokens)``. Plain bfloat16 tables that are trained take the native form, others are called, as in ``project``; so are
    tables of less than 2^20 elements, whose gradients the host bounds either way (1024 rows of 512, 512 tokens: 41 us both)."""
    if (type(layer) is nn.Embedding and type(tokens) is torch.Tensor and tokens.is_cuda and tokens.dtype is torch.int64
            and not torch.compiler.is_compiling() and torch.is_grad_enabled()):
        weight = layer.weight
        if (layer.padding_idx is None and layer.max_norm is None and not layer.scale_grad_by_freq and not layer.sparse
                and type(weight) is nn.Parameter and weight.numel() >= 1 << 20 and weight.requires_grad and weight.dtype is torch.bfloat16
                and weight.device == tokens.device and _bare(layer) and not torch._C._len_torch_function_stack()):
            return kernels().embedding(tokens, weight)
    return layer(tokens)
