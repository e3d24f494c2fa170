"""The autograd functions of csrc/functions.cpp against the Python ones that they stand for."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from colossalai_amd.ops import attention, build_rope_table, norm, swiglu
from colossalai_amd.ops._kernels import kernels

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _randn(*shape):
    return torch.randn(*shape, device="cuda").to(BF16)


def _calls():
    """name -> (native, Python function, inputs that take gradients)"""
    from colossalai_amd.ops.swiglu import _SwiGLU

    torch.manual_seed(0)
    q, k, v = _randn(2, 96, 4, 64), _randn(2, 96, 2, 64), _randn(2, 96, 2, 64)
    lens = torch.tensor([96, 33], dtype=torch.int32, device="cuda")
    cu = torch.tensor([0, 60, 96], dtype=torch.int32, device="cuda")
    table = build_rope_table(128, 64, 10000.0, torch.device("cuda"))
    positions = torch.arange(192, device="cuda", dtype=torch.int32) % 96
    x, r, w = _randn(3, 50, 256), _randn(3, 50, 256), _randn(256)
    n = kernels()
    return {
        "rms_norm": (lambda *a: n.native_rms_norm(*a, 1e-5), lambda *a: norm._RMSNorm.apply(*a, 1e-5), (x[:, ::2], w)),
        "add_norm": (lambda *a: n.native_fused_add_rms_norm(*a, 1e-5), lambda *a: norm._FusedAddRMSNorm.apply(*a, 1e-5), (x, r, w)),
        "swiglu": (n.native_swiglu, _SwiGLU.apply, (x.transpose(0, 1),)),
        "dense": (lambda *a: n.native_flash_attention(*a, True, 0.125, None, None),
                  lambda *a: attention._FlashAttention.apply(*a, True, 0.125, None), (q, k, v)),
        "padded": (lambda *a: n.native_flash_attention(*a, False, 0.2, lens, None),
                   lambda *a: attention._FlashAttention.apply(*a, False, 0.2, lens), (q, k, v)),
        "packed": (lambda *a: n.native_flash_attention_varlen(*a, cu, 60, True, 0.125),
                   lambda *a: attention._FlashAttentionVarlen.apply(*a, cu, 60, True, 0.125), (q[0], k[0], v[0])),
        "rope": (lambda a: n.native_fused_rope_attention(a + 0, table, None, 4, 2, 64, True, 0.125, None),
                 lambda a: attention._FusedRopeAttention.apply(a + 0, table, None, 4, 2, 64, True, 0.125, None), (_randn(2, 96, 512),)),
        "rope_at": (lambda a: n.native_fused_rope_attention(a + 0, table, positions, 4, 2, 64, True, 0.125, lens),
                    lambda a: attention._FusedRopeAttention.apply(a + 0, table, positions, 4, 2, 64, True, 0.125, lens), (_randn(2, 96, 512),)),
    }


def _run(call, inputs, kept):
    inputs = [t.detach().requires_grad_() for t in inputs]
    out = call(*inputs)
    out = out if isinstance(out, tuple) else (out,)
    grads = torch.autograd.grad(out[:kept], inputs, [torch.ones_like(t).cumsum(-1) for t in out[:kept]])
    return [t.detach() for t in out] + list(grads)


@pytest.mark.parametrize("name", ["rms_norm", "add_norm", "swiglu", "dense", "padded", "packed", "rope", "rope_at"])
@pytest.mark.parametrize("kept", [1, 2])   # gradients of the first result only, of both
def test_same_bits_as_the_python_function(name, kept):
    native, python, inputs = _calls()[name]
    for a, b in zip(_run(native, inputs, kept), _run(python, inputs, kept)):
        assert a.dtype == b.dtype and torch.equal(a, b)


NAMES = ["rms_norm", "add_norm", "swiglu", "dense", "padded", "packed", "rope", "rope_at"]


def _backward(call, inputs, form):
    inputs = [t.detach().requires_grad_() for t in inputs]
    out = call(*inputs)
    out = out if isinstance(out, tuple) else (out,)
    if form == "last result":
        return torch.autograd.grad(out[-1], inputs, torch.ones_like(out[-1]), allow_unused=True)
    douts = [torch.ones((), device="cuda", dtype=t.dtype).expand_as(t) if form == "one for all" else torch.ones_like(t).cumsum(-1) for t in out]
    if form == "some inputs":
        return torch.autograd.grad(out, inputs[-1:], douts)
    if form == "twice":
        torch.autograd.grad(out, inputs, douts, retain_graph=True)
    return torch.autograd.grad(out, inputs, douts, create_graph=form == "graph", retain_graph=True)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("form", ["one for all", "last result", "some inputs", "twice", "graph"])
def test_backward_forms_of_both(name, form):
    native, python, inputs = _calls()[name]
    for a, b in zip(_backward(native, inputs, form), _backward(python, inputs, form)):
        if b is None:
            assert a is None
            continue
        assert a.dtype == b.dtype and a.requires_grad == b.requires_grad and torch.equal(a, b)


@pytest.mark.parametrize("name", NAMES)
def test_results_are_changed_in_place_alike(name):
    """Accepted or refused, forward and backward."""
    def told(call, inputs):
        inputs = [t.detach().requires_grad_() for t in inputs]
        try:
            out = call(*inputs)
            out = out if isinstance(out, tuple) else (out,)
            for t in out:
                t.mul_(2.0)
            return torch.autograd.grad(out, inputs, [torch.ones_like(t) for t in out])
        except RuntimeError as e:
            return "in place" in str(e) or "inplace" in str(e)

    native, python, inputs = _calls()[name]
    a, b = told(native, inputs), told(python, inputs)
    if isinstance(b, bool):
        assert a is b is True
    else:
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_what_watches_or_rewrites_goes_to_python():
    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    n, x = kernels(), _randn(4, 64)
    assert n.native_swiglu(x) is not None and n.native_swiglu(x.cpu()) is None
    with Watch():
        assert n.native_swiglu(x) is None
    seen = []
    torch.func.vmap(lambda t: seen.append(n.native_swiglu(t)) or t)(x)
    torch.func.grad(lambda t: seen.append(n.native_swiglu(t)) or t.sum().float())(x)
    with torch.autograd.forward_ad.dual_level():
        seen.append(n.native_swiglu(torch.autograd.forward_ad.make_dual(x, x)))
    assert seen == [None, None, None]
    packed = []
    x.requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        y = swiglu(x)
    assert len(packed) == 1 and y.requires_grad
    with torch.no_grad():
        assert not swiglu(x).requires_grad
