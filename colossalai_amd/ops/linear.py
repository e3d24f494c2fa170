"""Linear layers in training: the weight gradient of a plain bfloat16 ``nn.Linear`` by csrc/weight_grad.hip.

The layer stays an ``nn.Linear`` that parallel policies, LoRA or the zero-bubble schedule replace or change; ``project``
calls whatever it has become.
"""

import torch
import torch.nn as nn
from torch.nn.modules import module as _hooks

from ._kernels import kernels

__all__ = ["project"]


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
