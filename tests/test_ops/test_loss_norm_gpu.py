"""Cross entropy over bf16 logits and RMSNorm at the edges of their kernels, against float32 (norm) and float64 (loss)
references of the same bfloat16 inputs."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ROUND = 2.0 ** -8  # of a value at most, by rounding it to bfloat16 (8 significant bits)


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("N,V,H,chunk", [(1, 8, 64, 4096), (37, 1000, 64, 4096), (130, 50257, 64, 64), (257, 32000, 128, 256),
                                         (64, 1023, 32, 17)])
def test_linear_cross_entropy(N, V, H, chunk):
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    torch.manual_seed(0)
    hidden = torch.randn(N, H, device="cuda").bfloat16().requires_grad_()
    weight = (0.2 * torch.randn(V, H, device="cuda")).bfloat16().requires_grad_()
    labels = torch.randint(0, V, (N,), device="cuda")
    if N > 2:
        labels[::3] = -100
    loss = fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk)
    dh, dw = torch.autograd.grad(3.0 * loss, (hidden, weight))

    h, w = hidden.detach().double().requires_grad_(), weight.detach().double().requires_grad_()
    want = torch.nn.functional.cross_entropy(h @ w.t(), labels, ignore_index=-100)
    wh, ww = torch.autograd.grad(3.0 * want, (h, w))
    # the logits are rounded to bfloat16, at most ROUND of the largest each way, and a loss is a difference of two of them
    top = (h @ w.t()).abs().max().item()
    assert abs(loss.item() - want.item()) < 2 * ROUND * top
    # a logit's rounding moves its probability by that share of it, and the gradient is rounded once more
    assert _rel(dh, wh) < 2 * ROUND * (top + 1)
    assert _rel(dw, ww) < 2 * ROUND * (top + 1)


@pytest.mark.parametrize("rows,V", [(4096, 32000), (1000, 50257), (2048, 512)])
def test_loss_keeps_float32_precision(rows, V):
    from colossalai_amd.ops._kernels import kernels

    torch.manual_seed(1)
    logits = torch.randn(rows, V, device="cuda").bfloat16()
    labels = torch.randint(0, V, (rows,), device="cuda")
    lse = torch.empty(rows, device="cuda")
    nll = torch.empty_like(lse)
    kernels().ce_fwd(logits, labels, -100, lse, nll)
    loss = kernels().ce_loss(nll, labels, -100)[0].item()
    want = torch.nn.functional.cross_entropy(logits.double(), labels).item()
    # rows' own roundings (three of values below 16, half of 2^-20 each at most) go either way and average out; what is
    # left is a lean of the exponentials, 1e-7 of the sum, and the rounding of the loss itself, half of 2^-20
    assert abs(loss - want) < 2.0 ** -20


def test_a_chunk_of_very_many_rows():
    """More rows than one launch holds threads for."""
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    N, V, H = (1 << 24) + 5, 8, 8
    torch.manual_seed(0)
    hidden = torch.randn(N, H, device="cuda").bfloat16().requires_grad_()
    weight = torch.randn(V, H, device="cuda").bfloat16()
    labels = torch.randint(0, V, (N,), device="cuda")
    got = []
    for chunk in (1 << 16, N):
        loss = fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk)
        got.append((loss, torch.autograd.grad(loss * N, hidden)[0]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_cross_entropy_without_a_row_that_counts():
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    hidden = torch.randn(9, 64, device="cuda").bfloat16().requires_grad_()
    weight = torch.randn(80, 64, device="cuda").bfloat16().requires_grad_()
    loss = fused_linear_cross_entropy(hidden, weight, torch.full((9,), -100, device="cuda"))
    assert loss.item() == 0.0
    assert all((g == 0).all() for g in torch.autograd.grad(loss, (hidden, weight)))


@pytest.mark.parametrize("V", [64, 1003])
def test_row_statistics_with_infinities(V):
    from colossalai_amd.ops import kernels

    x = torch.randn(5, V, device="cuda").bfloat16()
    x[0, : V // 2] = float("-inf")
    x[1, 3] = float("inf")
    x[2] = float("-inf")
    x[3] *= 300
    labels = torch.tensor([V - 1, 0, 1, 2, -100], device="cuda")
    lse, nll = torch.empty(5, device="cuda"), torch.empty(5, device="cuda")
    kernels().ce_fwd(x, labels, -100, lse, nll)
    want = torch.logsumexp(x.double(), 1)
    # float32: a sum of V terms and the reference's own rounding
    torch.testing.assert_close(lse.double(), want, rtol=V * 2.0 ** -24, atol=V * 2.0 ** -24)
    assert nll[4] == 0 and nll[1] == float("inf") and torch.isnan(nll[2])
    labels[0] = V  # outside the row: nothing is read there
    kernels().ce_fwd(x, labels, -100, lse, nll)
    assert torch.isnan(nll[0])


@pytest.mark.parametrize("V", [64, 1003, 32000])
def test_row_statistics_with_nan(V):
    """A NaN anywhere in a row is in its statistics: the columns that a thread reads first and last, whole groups of eight, and
    beside infinities."""
    from colossalai_amd.ops import kernels

    spots = [(0, 1), (0, 8), (V - 1, V), (V - 8, V), (V // 2, V // 2 + 1), (0, V)]
    x = torch.randn(len(spots) + 2, V, device="cuda").bfloat16()
    for row, (lo, hi) in enumerate(spots):
        x[row, lo:hi] = float("nan")
    x[-2] = float("-inf")
    x[-2, 0] = float("nan")
    x[-1, : V // 2] = float("-inf")
    x[-1, 1] = float("nan")
    labels = torch.full((len(x),), V // 4, device="cuda")
    lse, nll = torch.empty(len(x), device="cuda"), torch.empty(len(x), device="cuda")
    kernels().ce_fwd(x, labels, -100, lse, nll)
    assert torch.isnan(lse).all() and torch.isnan(nll).all()


def test_ignored_rows_show_what_is_not_finite():
    """As in the general form, where an ignored row's loss and gradient are multiplied by 0."""
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    hidden = torch.randn(6, 64, device="cuda").bfloat16()
    hidden[2] = float("nan")
    weight = torch.randn(80, 64, device="cuda").bfloat16()
    labels = torch.tensor([1, 2, -100, 3, -100, 4], device="cuda")
    assert torch.isnan(fused_linear_cross_entropy(hidden, weight, labels))
    hidden[2] = 0.0
    hidden.requires_grad_()
    loss = fused_linear_cross_entropy(hidden, weight, labels)
    (dh,) = torch.autograd.grad(loss, hidden, torch.full_like(loss, float("inf")), retain_graph=True)
    assert torch.isnan(dh[2]).all() and torch.isnan(dh[4]).all()
    (dh,) = torch.autograd.grad(loss, hidden)
    assert (dh[2] == 0).all() and torch.isfinite(dh).all()


@pytest.mark.parametrize("V", [80, 1003])
@pytest.mark.parametrize("label", [-1, -7, None])
def test_a_label_outside_the_row_spoils_its_gradient(V, label):
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    hidden = torch.randn(5, 64, device="cuda").bfloat16().requires_grad_()
    weight = torch.randn(V, 64, device="cuda").bfloat16()
    labels = torch.tensor([1, 2, V if label is None else label, 3, -100], device="cuda")
    loss = fused_linear_cross_entropy(hidden, weight, labels)
    (dh,) = torch.autograd.grad(loss, hidden)
    assert torch.isnan(loss) and torch.isnan(dh[2]).all()
    assert torch.isfinite(dh[[0, 1, 3, 4]]).all()


@pytest.mark.parametrize("rows,H", [(1, 8), (3, 512), (5, 520), (130, 768), (9, 1032), (33, 2048), (6, 2056), (7, 4104), (5, 8192),
                                    (5000, 64)])
def test_add_norm_and_its_gradients(rows, H):
    from colossalai_amd.ops import fused_add_rms_norm, rms_norm

    torch.manual_seed(0)
    x, res, dy, dh = (torch.randn(rows, H, device="cuda").bfloat16() for _ in range(4))
    w = (1 + 0.1 * torch.randn(H, device="cuda")).bfloat16()
    for t in (x, res, w):
        t.requires_grad_()
    kept = res.detach().clone()
    y, h = fused_add_rms_norm(x, res, w, 1e-5)
    dx, dr, dw = torch.autograd.grad((y, h), (x, res, w), (dy, dh))
    assert torch.equal(res.detach(), kept)  # the old residual stream is left alone

    hf = (x.detach().float() + res.detach().float()).requires_grad_()
    wf = w.detach().float().requires_grad_()
    yf = hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + 1e-5) * wf
    gh, gw = torch.autograd.grad(yf, (hf, wf), dy.float())
    assert _rel(h, hf) < ROUND and _rel(y, yf) < ROUND
    # the backward starts from the rounded h: twice ROUND through the norm, and the result is rounded
    assert _rel(dx, gh + dh.float()) < 3 * ROUND and torch.equal(dx, dr)
    assert _rel(dw, gw) < 3 * ROUND

    y = rms_norm(x, w, 1e-5)
    (dx,) = torch.autograd.grad(y, (x,), dy)
    xf = x.detach().float().requires_grad_()
    yf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5) * w.detach().float()
    (gx,) = torch.autograd.grad(yf, (xf,), dy.float())
    assert _rel(y, yf) < ROUND and _rel(dx, gx) < 2 * ROUND


# rows in the kept part, in it and beyond it, and logits of which none fit
@pytest.mark.parametrize("N,V,chunk,kept_bytes,kept", [(37, 1000, 64, 1 << 30, 37), (300, 1024, 64, 1 << 30, 256),
                                                       (300, 1024, 64, 300000, 128), (300, 1003, 64, 100000, 0)])
def test_linear_cross_entropy_with_kept_logits(monkeypatch, N, V, chunk, kept_bytes, kept):
    from colossalai_amd.ops import fused_ce

    monkeypatch.setattr(fused_ce, "_KEPT_BYTES", kept_bytes)
    assert fused_ce._spans(N, V, chunk, True)[0] == kept
    torch.manual_seed(5)
    hidden = torch.randn(N, 64, device="cuda").bfloat16().requires_grad_()
    weight = (0.2 * torch.randn(V, 64, device="cuda")).bfloat16().requires_grad_()
    labels = torch.randint(0, V, (N,), device="cuda")
    loss = fused_ce.fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk)
    first = torch.autograd.grad(loss, (hidden, weight), retain_graph=True)
    again = torch.autograd.grad(loss, (hidden, weight))
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    h, w = hidden.detach().double().requires_grad_(), weight.detach().double().requires_grad_()
    want = torch.nn.functional.cross_entropy(h @ w.t(), labels)
    top = (h @ w.t()).abs().max().item()
    for got, ref in zip(first, torch.autograd.grad(want, (h, w))):
        assert _rel(got, ref) < 2 * ROUND * (top + 1)
    with torch.no_grad():
        assert abs(fused_ce.fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk).item() - want.item()) < 2 * ROUND * top


@pytest.mark.parametrize("kept_bytes,chunks", [(0, 0), (1 << 24, 2), (None, 4)])
def test_memory_of_kept_logits(kept_bytes, chunks):
    """What a loss holds until its backward, and the backward's peak, are bounded by what the caller allows."""
    from colossalai_amd.ops.fused_ce import fused_linear_cross_entropy

    N, V, H, chunk = 8192, 4096, 64, 1024
    a_chunk = chunk * V * 2
    torch.manual_seed(6)
    hidden = torch.randn(N, H, device="cuda").bfloat16().requires_grad_()
    weight = (0.2 * torch.randn(V, H, device="cuda")).bfloat16().requires_grad_()
    labels = torch.randint(0, V, (N,), device="cuda")
    want = torch.autograd.grad(fused_linear_cross_entropy(hidden, weight, labels), (hidden, weight))
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    loss = fused_linear_cross_entropy(hidden, weight, labels, chunk_size=chunk, kept_bytes=kept_bytes)
    few = 4 << 20   # statistics, gradients and the sums of the weight's
    assert torch.cuda.memory_allocated() - before <= chunks * a_chunk + few
    torch.cuda.reset_peak_memory_stats()
    got = torch.autograd.grad(loss, (hidden, weight))
    # the kept logits and their gradient, and two chunks: one is let go when the next is formed
    assert torch.cuda.max_memory_allocated() - before <= (2 * chunks + 2) * a_chunk + few
    for a, b in zip(got, want):
        assert _rel(a, b) < 2 * ROUND
