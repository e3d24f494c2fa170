"""Weight gradients and small products of linear layers (csrc/products.hip) and the layer that uses them (csrc/linear.cpp)."""

import json

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from colossalai_amd.ops._kernels import has_kernels, kernels
from colossalai_amd.ops.linear import project

BF16 = torch.bfloat16
needs_extension = pytest.mark.skipif(not has_kernels(), reason="extension not built")


def _close(got, dy, x, add=None, keep=False):
    """Within a rounding of the result's type and the float32 sums of K products, in any order."""
    a, b = dy.double(), x.double()
    ref, size = a.t() @ b, a.abs().t() @ b.abs()
    if add is not None:
        ref, size = ref + add.double(), size + add.double().abs()
    limit = size * (dy.shape[0] + 2) * 2.0 ** -24 + (0 if keep else ref.abs() * 2.0 ** -8) + 1e-30
    assert got.dtype == (torch.float32 if keep else BF16)
    assert ((got.double() - ref).abs() <= limit).all()


# edges of both tile sizes, of the steps of 32 tokens and of the parts
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(8, 8, 1), (128, 136, 31), (120, 256, 33), (264, 248, 300), (768, 768, 4100), (1032, 776, 1500),
                                   (512, 512, 512), (4096, 4104, 65), (8, 2048, 16384), (5120, 4096, 1000),
                                   (4096, 768, 8190), (760, 2056, 8192), (2312, 776, 4100)])
def test_against_64_bits(M, N, K):
    torch.manual_seed(M + N + K)
    dy, x = (torch.randn(K, n, device="cuda").to(BF16) for n in (M, N))
    _close(kernels().weight_grad(dy, x), dy, x)
    first = kernels().weight_grad(dy, x, None, True)
    _close(first, dy, x, None, True)
    add = torch.randn(M, N, device="cuda")
    before = add.clone()
    _close(kernels().weight_grad(dy, x, add, False), dy, x, before)
    again = kernels().weight_grad(dy, x, add, True)
    assert again.data_ptr() == add.data_ptr()
    _close(again, dy, x, before, True)


# one round of the tiles of 256 x 256 and of 256 x 128, whose ring of four steps is left behind each of them
@pytest.mark.gpu
@pytest.mark.parametrize("N", [4088, 2040])
@pytest.mark.parametrize("K", [1, 33, 65, 97, 129, 160, 192, 223, 256, 261])
def test_large_tiles_over_few_steps(N, K):
    torch.manual_seed(N + K)
    dy, x = (torch.randn(K, n, device="cuda").to(BF16) for n in (4088, N))
    _close(kernels().weight_grad(dy, x, None, True), dy, x, None, True)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(128, 136, 31), (264, 248, 300), (768, 768, 4100), (12, 20, 33)])
@pytest.mark.parametrize("offset", [1, 2, 3, 5])
@pytest.mark.parametrize("keep", [False, True])
def test_sums_at_odd_addresses(M, N, K, offset, keep):
    torch.manual_seed(offset)
    dy, x = (torch.randn(K, n, device="cuda").to(BF16) for n in (M, N))
    flat = torch.randn(M * N + 16, device="cuda")
    add = flat[offset: offset + M * N].view(M, N)
    before = flat.clone()
    got = kernels().weight_grad(dy, x, add, keep)
    if keep:
        assert got.data_ptr() == add.data_ptr()
    # sizes that the library multiplies round the product to bfloat16 before it is added
    wide = 0 if M % 8 == 0 else (dy.double().t() @ x.double()).abs() * 2.0 ** -8
    ref = before[offset: offset + M * N].view(M, N).double() + dy.double().t() @ x.double()
    size = before.abs().max() + dy.double().abs().t() @ x.double().abs()
    assert ((got.double() - ref).abs() <= size * (K + 2) * 2.0 ** -24 + wide + (0 if keep else ref.abs() * 2.0 ** -8 + 1e-30)).all()
    assert torch.equal(flat[:offset], before[:offset]) and torch.equal(flat[offset + M * N:], before[offset + M * N:])


def _formed_here(call):
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        call()
        torch.cuda.synchronize()
    return any("product_kernel" in e.key for e in seen.key_averages())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,here", [(4096, 4096, 64, False), (4096, 2056, 1024, False), (2304, 4096, 1599, False),
                                        (2304, 4096, 1600, True), (4096, 2048, 100, True), (512, 512, 512, True)])
def test_few_tokens_are_the_librarys(M, N, K, here):
    """Storing a large result is most of such a product, which the library does faster; a float32 sum is formed here in any case."""
    torch.manual_seed(K)
    dy, x = (torch.randn(K, n, device="cuda").to(BF16) for n in (M, N))
    _close(kernels().weight_grad(dy, x), dy, x)
    assert _formed_here(lambda: kernels().weight_grad(dy, x)) == here
    assert _formed_here(lambda: kernels().weight_grad(dy, x, None, True))


@pytest.mark.gpu
def test_strides_and_sizes_of_other_forms():
    torch.manual_seed(0)
    wide = torch.randn(300, 1000, device="cuda").to(BF16)
    x = torch.randn(300, 264, device="cuda").to(BF16)
    forms = [wide[:, 8:272], wide[:, 3:267], wide.t()[:300, :264], wide[:1, :264].expand(300, 264), wide[:, :250], wide[::2, :264]]
    for dy in forms:
        for a, b in ((dy, x[: dy.shape[0]]), (x[: dy.shape[0]], dy)):
            _close(kernels().weight_grad(a, b), a, b)


@pytest.mark.gpu
def test_what_is_not_finite_stays_in_its_row():
    dy, x = torch.ones(100, 264, device="cuda", dtype=BF16), torch.ones(100, 136, device="cuda", dtype=BF16)
    dy[99, 7], x[0, 135] = float("nan"), float("inf")
    got = kernels().weight_grad(dy, x)
    rows = torch.arange(264, device="cuda") != 7
    assert got[7].isnan().all() and (got[rows][:, 135] == float("inf")).all() and (got[rows][:, :135] == 100).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 32), (127, 136, 64), (129, 128, 96), (510, 1024, 512), (300, 264, 1056), (512, 512, 2048),
                                   (2048, 2048, 512), (33, 40, 40), (8192, 512, 64)])
def test_products_against_64_bits(M, N, K):
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K, device="cuda").to(BF16), torch.randn(N, K, device="cuda").to(BF16)
    for a in (x, torch.randn(M, 2 * K + 8, device="cuda").to(BF16)[:, 8: K + 8]):
        _close(kernels().multiply(a, w, False), a.t(), w.t())
        _close(kernels().multiply(a, w.t().contiguous(), True), a.t(), w.t())
    x[M // 2, K - 1] = float("nan")
    got = kernels().multiply(x, w, False)
    assert got[M // 2].isnan().all() and got.isnan().sum() == N


# both of a small layer's gradients by one launch: either whole, cut in parts, with remainders; the last two are too large for it
@pytest.mark.gpu
@pytest.mark.parametrize("K,M,N,one", [(1, 32, 8, True), (127, 96, 136, True), (512, 2048, 512, True), (512, 1536, 512, True), (2000, 256, 520, True),
                                       (33, 4096, 264, True), (4096, 64, 128, True), (500, 4096, 4096, False), (512, 24, 64, False)])
def test_both_gradients_of_a_small_layer(K, M, N, one):
    torch.manual_seed(M + N + K)
    x, w, dy = (torch.randn(*s, device="cuda").to(BF16) for s in ((K, N), (M, N), (K, M)))
    x.requires_grad_(), w.requires_grad_()
    out = kernels().linear(x, w)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        dx, dw = torch.autograd.grad(out, (x, w), dy)
        torch.cuda.synchronize()
    assert any("product_pair" in e.key for e in seen.key_averages()) == one
    _close(dw, dy, x.detach())
    _close(dx, dy.t(), w.detach())
    only = torch.autograd.grad(kernels().linear(x, w), x, dy)[0]
    _close(only, dy.t(), w.detach())


@pytest.mark.gpu
@pytest.mark.parametrize("slow", [False, True])
@pytest.mark.parametrize("M,N,K,own", [(512, 3072, 1152, True), (2048, 768, 1152, True), (512, 3072, 1184, False),   # whole
                                       (512, 1024, 1024, True), (512, 1024, 2048, False), (256, 3072, 1536, False), (8, 2048, 4096, False)])   # would be cut
def test_which_products_are_small(M, N, K, own, slow):
    """Up to 14 us by the plan: a chain of calls waits 19 us for each of the library's, whose kernels take 10 where cut ones take 15."""
    x, w = (torch.randn(*s, device="cuda").to(BF16) for s in ((M, K), (K, N) if slow else (N, K)))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        y = kernels().multiply(x, w, slow)
        torch.cuda.synchronize()
    assert any("product_kernel" in e.key for e in seen.key_averages()) == own
    _close(y, x.t(), w if slow else w.t())


@pytest.mark.gpu
@pytest.mark.parametrize("K,M,N,most", [(9685, 168, 352, 22), (5463, 1328, 72, 9), (14360, 208, 480, 18), (11817, 552, 128, 25), (970, 952, 408, 3)])
def test_parts_of_few_tiles(K, M, N, most, tmp_path):
    """Each part costs the sum, which few tiles give to few blocks: up to half as many parts as their bytes alone would allow."""
    dy, x = (torch.randn(K, n, device="cuda").to(BF16) for n in (M, N))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        dw = kernels().weight_grad(dy, x)
        torch.cuda.synchronize()
    seen.export_chrome_trace(str(tmp_path / "trace.json"))
    with open(tmp_path / "trace.json") as f:
        (grid,) = [e["args"]["grid"][0] for e in json.load(f)["traceEvents"] if e.get("cat") == "kernel" and "::product_kernel" in e["name"]]
    tiles = -(-M // 128) * -(-N // 128)
    assert 1 < grid // tiles <= most
    _close(dw, dy, x)


def _step(call, x, w, g):
    x, w = x.detach().requires_grad_(), w.detach().requires_grad_()
    y = call(x, w)
    y.backward(g)
    return y.detach(), x.grad, w.grad


@needs_extension
@pytest.mark.parametrize("shape", [(5, 16), (2, 3, 16), (2, 2, 3, 16)])
def test_layer_is_the_builtin_one_on_the_cpu(shape):
    torch.manual_seed(1)
    x, w, g = torch.randn(*shape), torch.randn(24, 16), torch.randn(*shape[:-1], 24)
    for a, b in zip(_step(kernels().linear, x, w, g), _step(F.linear, x, w, g)):
        torch.testing.assert_close(a, b)


@needs_extension
@pytest.mark.parametrize("shape", [(5, 16), (2, 3, 16)])
@pytest.mark.parametrize("change", [lambda y: y.add_(1.0), lambda y: y[..., :4].mul_(2.0), lambda y: y.relu_()])
def test_result_may_be_changed_in_place(shape, change):
    torch.manual_seed(4)
    x, w, g = torch.randn(*shape), torch.randn(24, 16), torch.randn(*shape[:-1], 24)

    def changed(lin):
        def call(x, w):
            y = lin(x, w)
            change(y)
            return y
        return call

    for a, b in zip(_step(changed(kernels().linear), x, w, g), _step(changed(F.linear), x, w, g)):
        torch.testing.assert_close(a, b)


@needs_extension
def test_layer_under_transforms():
    torch.manual_seed(2)
    x, w = torch.randn(4, 16, dtype=torch.float64), torch.randn(8, 16, dtype=torch.float64)
    lin = kernels().linear
    assert torch.autograd.gradcheck(lin, (x.requires_grad_(), w.requires_grad_()))
    assert torch.autograd.gradgradcheck(lin, (x, w))
    x, w = x.detach(), w.detach()
    torch.testing.assert_close(torch.func.vmap(lin, (0, None))(x.expand(3, 4, 16), w), F.linear(x.expand(3, 4, 16), w))
    torch.testing.assert_close(torch.func.jacrev(lin, 1)(x, w), torch.func.jacrev(F.linear, 1)(x, w))
    torch.testing.assert_close(torch.func.jvp(lambda t: lin(t, w), (x,), (x,)), torch.func.jvp(lambda t: F.linear(t, w), (x,), (x,)))
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x, x)
        assert torch.autograd.forward_ad.unpack_dual(lin(d, w.requires_grad_())).tangent is not None
    w, kept = w.detach().requires_grad_(), []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
        y = lin(x, w)
    assert len(kept) == 1   # the input; the weight's own factor is not wanted
    torch.testing.assert_close(torch.autograd.grad(y, w, torch.ones(3, 4, 8, dtype=torch.float64), is_grads_batched=True)[0],
                               x.sum(0).expand(3, 8, 16))


@pytest.mark.gpu
def test_projection_takes_the_native_form_only_for_plain_layers():
    torch.manual_seed(3)
    layer = nn.Linear(264, 136, bias=False, device="cuda", dtype=BF16)
    x = torch.randn(2, 50, 264, device="cuda").to(BF16).requires_grad_()
    seen = []

    assert "CppNode" in project(layer, x).grad_fn.name()
    handle = layer.register_forward_hook(lambda *a: seen.append(1))
    project(layer, x)
    handle.remove()
    assert seen == [1]
    layer.forward = lambda t: seen.append(2) or F.linear(t, layer.weight)
    project(layer, x)
    del layer.forward
    assert seen == [1, 2]
    with torch.autocast("cuda", torch.float16):
        assert project(layer, x).dtype == torch.float16
    y, g = project(layer, x), torch.randn(2, 50, 136, device="cuda").to(BF16)
    got = torch.autograd.grad(y, (x, layer.weight), g)
    ref = torch.autograd.grad(layer(x), (x, layer.weight), g)
    torch.testing.assert_close(got[0], ref[0], rtol=0, atol=0)
    _close(got[1], g.view(-1, 136), x.detach().view(-1, 264))
    graph = torch.autograd.grad(project(layer, x), layer.weight, g, create_graph=True)[0]
    assert graph.requires_grad
    layer.weight.requires_grad_(False)
    project(layer, x).backward(g)
    assert layer.weight.grad is None and x.grad is not None


@pytest.mark.gpu
def test_a_mode_that_counts_operations_sees_every_product():
    from torch.utils.flop_counter import FlopCounterMode

    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    x, w = torch.randn(96, 64, device="cuda").to(BF16).requires_grad_(), torch.randn(136, 64, device="cuda").to(BF16).requires_grad_()
    labels = torch.arange(96, device="cuda")
    layer = nn.Linear(64, 136, bias=False, device="cuda", dtype=BF16)
    for call, rows in ((lambda: fused_linear_cross_entropy(x, w, labels), 3 * 96), (lambda: project(layer, x).sum(), 3 * 96),
                       (lambda: fused_linear_cross_entropy(x, w, labels, chunk_size=20), 3 * 96 + 16)):   # 16 rows' logits twice
        with FlopCounterMode(display=False) as counter:
            call().backward()
        assert counter.get_total_flops() == 2 * rows * 64 * 136
