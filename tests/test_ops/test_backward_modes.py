"""Backward passes of the fused loss and the fused norm where autograd is asked for more than one gradient: graphs of the
backward itself, and autocast to another type. The kernels are replaced by stand-ins that, like them, work outside
autograd, so that the choice of the path is what is tested; the same cases run on the GPU with the kernels."""

import pytest
import torch

from colossalai_amd.ops import fused_add_rms_norm, fused_ce, norm


class StandIns:
    """What the extension offers to these ops, in torch."""

    @staticmethod
    def ce_fwd(logits, labels, ignore_index, lse, nll):
        assert logits.dtype == torch.bfloat16
        with torch.no_grad():
            x = logits.float()
            lse.copy_(torch.logsumexp(x, 1))
            valid = labels != ignore_index
            nll.copy_((lse - x.gather(1, labels.masked_fill(~valid, 0)[:, None])[:, 0]) * valid)

    @staticmethod
    def ce_loss(nll, labels, ignore_index):
        n = (labels != ignore_index).sum().clamp(min=1).float()
        return torch.stack([nll.sum() / n, n])

    @staticmethod
    def ce_bwd(logits, labels, ignore_index, lse, grad, loss):
        assert logits.dtype == torch.bfloat16
        with torch.no_grad():
            ds = torch.exp(logits.float() - lse[:, None])
            valid = labels != ignore_index
            ds[torch.arange(len(ds)), labels.masked_fill(~valid, 0)] -= 1.0
            logits.detach().copy_(ds * (valid[:, None] * grad / loss[1]))

    @staticmethod
    def rmsnorm_fused_add_fwd(x, residual, weight, eps, save, out):
        with torch.no_grad():
            out.copy_(x.float() + residual.float())
            inv = torch.rsqrt(out.float().pow(2).mean(-1) + eps)
            return (out.float() * inv[:, None] * weight.float()).to(x.dtype), inv

    @staticmethod
    def rmsnorm_bwd(dy, x, weight, inv, dres=None, cast_dw=False):
        with torch.no_grad():
            xf, g = x.float(), dy.float() * weight.float()
            dx = inv[:, None] * (g - xf * (g * xf).mean(-1, keepdim=True) * inv[:, None] ** 2)
            if dres is not None:
                dx = dx + dres.float()
            return dx.to(x.dtype), (dy.float() * xf * inv[:, None]).sum(0).to(weight.dtype)


@pytest.fixture(params=["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def device(request, monkeypatch):
    if request.param == "cpu":
        for module in (fused_ce, norm):
            monkeypatch.setattr(module, "use_hip", lambda *tensors: True)
            monkeypatch.setattr(module, "kernels", lambda: StandIns)
    return request.param


def _loss_inputs(device, N=37, V=80, H=64):
    torch.manual_seed(0)
    hidden = torch.randn(N, H).bfloat16().to(device).requires_grad_()
    weight = (0.3 * torch.randn(V, H)).bfloat16().to(device).requires_grad_()
    labels = torch.randint(0, V, (N,))
    labels[::5] = -100
    return hidden, weight, labels.to(device)


def _near(got, want):
    # both round the gradients of the logits and the result to bfloat16, 2^-9 of a value at most each
    assert (got.double() - want.double()).norm() < 4 * 2.0 ** -9 * want.double().norm()


@pytest.mark.parametrize("chunk", [16, 4096])
def test_loss_gradients_under_create_graph(device, chunk):
    hidden, weight, labels = _loss_inputs(device)
    loss = fused_ce.fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk)
    plain = torch.autograd.grad(loss, (hidden, weight), retain_graph=True)
    graph = torch.autograd.grad(loss, (hidden, weight), create_graph=True)
    for a, b in zip(graph, plain):
        _near(a.detach(), b)
        assert a.grad_fn is not None  # part of a graph: nothing is dropped from a second derivative in silence


@pytest.mark.parametrize("where", ["forward", "backward", "both"])
def test_loss_under_autocast_to_half(device, where):
    hidden, weight, labels = _loss_inputs(device)
    kind = hidden.device.type
    loss = fused_ce.fused_linear_cross_entropy(hidden, weight, labels)
    want = (loss, *torch.autograd.grad(loss, (hidden, weight)))
    with torch.autocast(kind, dtype=torch.float16, enabled=where != "backward"):
        loss = fused_ce.fused_linear_cross_entropy(hidden, weight, labels)
    with torch.autocast(kind, dtype=torch.float16, enabled=where != "forward"):
        got = (loss, *torch.autograd.grad(loss, (hidden, weight)))
    for a, b in zip(got, want):
        assert a.dtype == b.dtype
        _near(a.detach(), b.detach())


def test_loss_in_a_checkpoint(device):
    """Saved tensors of a checkpointed segment may be taken once only."""
    from torch.utils.checkpoint import checkpoint

    hidden, weight, labels = _loss_inputs(device)
    loss = fused_ce.fused_linear_cross_entropy(hidden, weight, labels)
    want = torch.autograd.grad(loss, (hidden, weight))
    loss = checkpoint(fused_ce.fused_linear_cross_entropy, hidden, weight, labels, use_reentrant=False)
    for a, b in zip(torch.autograd.grad(loss, (hidden, weight)), want):
        assert torch.equal(a, b)


def test_residual_gradient_keeps_its_graph(device):
    """The gradient that flows past the norm is a function of the stream: its derivative is part of a second one."""
    torch.manual_seed(0)
    x, res = (torch.randn(9, 64).bfloat16().to(device) for _ in range(2))
    w = torch.ones(64, dtype=torch.bfloat16, device=device)
    x.requires_grad_()
    _, h = fused_add_rms_norm(x, res, w, 1e-6)
    (first,) = torch.autograd.grad(h.float().pow(3).sum(), x, create_graph=True)
    _near(first.detach(), 3 * h.detach().float() ** 2)
    (second,) = torch.autograd.grad(first.float().sum(), x)
    _near(second, 6 * h.detach().float())
