"""Tables of embeddings: their gradient by csrc/embedding.hip, and what goes to the layer itself.

The bound: a gradient's row is a sum in float32 of bfloat16 rows, rounded once: 2^-9 of a value, and 2^-24 of the sum of the magnitudes for
each of its additions.
"""

import pytest
import torch
import torch.nn as nn

from colossalai_amd.ops.linear import embed


def _native(layer, tokens):
    from colossalai_amd import _C

    return _C.embedding(tokens, layer.weight)


def _check(layer, tokens, embed=_native):
    torch.manual_seed(0)
    out = embed(layer, tokens)
    dy = torch.randn_like(out)
    layer.zero_grad(set_to_none=True)
    out.backward(dy)
    V, W = layer.weight.shape
    assert torch.equal(out, nn.functional.embedding(tokens, layer.weight))
    flat, rows = tokens.flatten(), dy.reshape(-1, W).double()
    want = torch.zeros(V, W, dtype=torch.float64, device=dy.device).index_add_(0, flat, rows)
    size = torch.zeros_like(want).index_add_(0, flat, rows.abs())
    count = torch.bincount(flat, minlength=V)[:, None]
    bound = want.abs() * 2.0 ** -8 + size * count * 2.0 ** -24 if dy.dtype is torch.bfloat16 else size * 1e-5
    assert ((layer.weight.grad.double() - want).abs() <= bound).all()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("V,W,T", [(1, 8, 1), (127, 64, 63), (128, 512, 64), (129, 520, 65), (1000, 768, 1025), (32000, 4096, 700), (300, 1032, 5000)])
@pytest.mark.parametrize("spread", ["even", "few", "one"])
def test_gradient(V, W, T, spread):
    """Rows and channels that end inside a block, parts of the tokens; rows without a token, with one, with 64 and 65, and with all of them."""
    layer = nn.Embedding(V, W, device="cuda", dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(V + T)
    tokens = torch.randint(0, V, (T,), generator=g)
    if spread == "few":
        tokens = torch.cat([torch.full((64,), V // 2), torch.full((65,), V - 1), tokens % 3 % V])[torch.randperm(T + 129, generator=g)]
    elif spread == "one":
        tokens = torch.full((T,), V - 1)
    out = _check(layer, tokens.cuda())
    assert type(out.grad_fn).__name__ == "CppFunction"   # the kernels'


@pytest.mark.gpu
def test_repeats_and_second_derivatives():
    layer = nn.Embedding(500, 64, device="cuda", dtype=torch.bfloat16)
    tokens = torch.randint(0, 500, (3, 2000), device="cuda")
    grads = []
    for _ in range(2):
        out = _native(layer, tokens)
        torch.manual_seed(1)
        grads.append(torch.autograd.grad(out, layer.weight, torch.randn_like(out))[0])
    assert torch.equal(*grads)   # sums in the order of the tokens
    out = _native(layer, tokens)
    dy = torch.randn_like(out).requires_grad_()
    (dw,) = torch.autograd.grad(out, layer.weight, dy, create_graph=True)
    (ddy,) = torch.autograd.grad(dw.float().square().sum(), dy)
    assert torch.allclose(ddy.float(), 2 * dw.float()[tokens], rtol=1e-2, atol=1e-2)


def _is_native(V, W, T):
    weight = torch.zeros(V, W, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    from colossalai_amd import _C

    out = _C.embedding(torch.randint(0, V, (T,), device="cuda"), weight)
    dy = torch.ones_like(out)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        torch.autograd.grad(out, weight, dy)
        torch.cuda.synchronize()
    return any("list_kernel" in e.key for e in seen.key_averages())


@pytest.mark.gpu
@pytest.mark.parametrize("V,W,T,native", [
    (2048, 512, 16384, True), (2048, 512, 16385, False), (50304, 1016, 16385, False),   # narrow
    (31999, 1024, 16385, False), (32000, 1024, 16385, True), (1024, 2040, 16385, False), (512, 2048, 16385, True),   # few rows
])
def test_many_tokens(V, W, T, native):
    """Over many tokens one row's are too many for the few blocks that a narrow or a small table has for it: the library's."""
    assert _is_native(V, W, T) == native
    if V < 32000:
        layer = nn.Embedding(V, W, device="cuda", dtype=torch.bfloat16)
        _check(layer, (torch.rand(T, device="cuda") * 7).exp().long().clamp(max=V - 1))   # by frequency


@pytest.mark.gpu
def test_what_a_layer_takes():
    tokens = torch.randint(0, 2048, (3, 50), device="cuda")
    layer = nn.Embedding(2048, 512, device="cuda", dtype=torch.bfloat16)
    assert type(_check(layer, tokens, embed).grad_fn).__name__ == "CppFunction"
    small = nn.Embedding(2048, 504, device="cuda", dtype=torch.bfloat16)
    assert type(embed(small, tokens).grad_fn).__name__ == "EmbeddingBackward0"
    layer.register_forward_hook(lambda *a: None)
    assert type(embed(layer, tokens).grad_fn).__name__ == "EmbeddingBackward0"
    with torch.no_grad():
        assert embed(layer, tokens).grad_fn is None


@pytest.mark.gpu
@pytest.mark.parametrize("make", [
    lambda: nn.Embedding(2048, 512, padding_idx=3, device="cuda", dtype=torch.bfloat16),
    lambda: nn.Embedding(2048, 512, device="cuda"),
    lambda: nn.Embedding(40, 30003, device="cuda", dtype=torch.bfloat16),
])
def test_others_are_the_layers(make):
    """A row of padding, other data types and channels that loads of 16 bytes do not divide."""
    layer = make()
    tokens = torch.randint(0, 40, (7, 9), device="cuda")
    embed(layer, tokens).float().square().sum().backward()
    got = layer.weight.grad.clone()
    layer.zero_grad(set_to_none=True)
    layer(tokens).float().square().sum().backward()
    assert torch.allclose(got.float(), layer.weight.grad.float(), rtol=1e-2, atol=1e-2)


def test_on_the_cpu():
    _check(nn.Embedding(50, 12), torch.randint(0, 50, (4, 11)), embed)
