"""Chunked fused linear + cross-entropy.

Computes ``CE(hidden @ W^T, labels)`` without ever materializing the full
[N, V] logits: tokens are processed in chunks; backward recomputes each
chunk's logits and feeds the dW/dh GEMMs directly. At the flagship bench
size (147k tokens x 32k vocab) this replaces a ~50 GB fp32 logits+softmax
footprint with chunk buffers.
On the GPU the first rows, four chunks of at most 1 GiB of logits, are one chunk whose bfloat16 logits the
backward still finds: the activations of a decoder layer for as many tokens are larger, and forming
them again was 5 to 7 % of a training step of 8192 to 16384 tokens (16380 x 32000 at width 4096: 2.9 ms of 51;
its products over all rows at once take 6.9 ms for 7.7 in four chunks). They are held from the forward to the backward,
which takes as much again for their gradient; ``kept_bytes`` bounds them, or with 0 leaves one chunk at a time.

GEMMs run through hipBLASLt (torch.matmul), the weight gradient and small products in bfloat16
through csrc/products.hip; softmax math is fp32. In bfloat16 on
the GPU a chunk's logits are read once in the forward and overwritten by their
gradient in the backward (csrc/cross_entropy.hip).
Reference parity: the reference materializes logits and uses torch CE (or
DistCrossEntropy under TP); this op is our memory-optimized equivalent.
"""

from typing import Optional

import torch

from ._kernels import kernels, use_hip
from .linear import multiply, weight_grad

__all__ = ["fused_linear_cross_entropy"]


def _bf16_products(t: torch.Tensor) -> bool:
    """Whether bfloat16 operands give a bfloat16 product here: not under autocast to another type."""
    kind = t.device.type
    return not torch.is_autocast_enabled(kind) or torch.get_autocast_dtype(kind) == torch.bfloat16


_KEPT_CHUNKS, _KEPT_BYTES = 4, 1 << 30


def _spans(rows: int, vocab: int, chunk_size: int, keep: bool, kept_bytes: Optional[int] = None):
    """How many rows' bfloat16 logits stay for the backward, and the spans of rows that are worked on: those rows, if
    any, then chunks."""
    kept = 0
    if keep:
        most = _KEPT_BYTES if kept_bytes is None else max(kept_bytes, 0)
        fit = min(_KEPT_CHUNKS * chunk_size, most // (2 * max(vocab, 1)))
        kept = rows if rows <= fit else fit // chunk_size * chunk_size
    return kept, [(0, kept)] * (kept > 0) + [(s, min(s + chunk_size, rows)) for s in range(kept, rows, chunk_size)]


class _FusedLinearCE(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden, weight, labels, ignore_index, chunk_size, recorded=False, kept_bytes=None):
        # hidden [N, H] (bf16/fp32), weight [V, H], labels [N]
        N = hidden.shape[0]
        ctx.chunk_size = chunk_size
        ctx.ignore_index = ignore_index
        ctx.hip = (hidden.dtype == weight.dtype == torch.bfloat16 and labels.dtype == torch.int64
                   and use_hip(hidden, weight, labels) and _bf16_products(hidden))
        if ctx.hip:
            labels = labels.contiguous()
            lse = torch.empty(N, dtype=torch.float32, device=hidden.device)
            nll = torch.empty_like(lse)
            ctx.kept, ctx.spans = _spans(N, weight.shape[0], chunk_size, recorded and hidden.is_cuda, kept_bytes)
            kept = []
            for s, e in ctx.spans:
                logits = multiply(hidden[s:e], weight)
                kernels().ce_fwd(logits, labels[s:e], ignore_index, lse[s:e], nll[s:e])
                if e <= ctx.kept:
                    kept.append(logits)
            loss = kernels().ce_loss(nll, labels, ignore_index)
            ctx.save_for_backward(hidden, weight, labels, lse, loss, *kept)
            return loss[0].clone()  # a tensor of its own: what is saved is not handed out
        lse = torch.empty(N, dtype=torch.float32, device=hidden.device)
        picked = torch.empty(N, dtype=torch.float32, device=hidden.device)
        valid = labels != ignore_index
        safe_labels = labels.masked_fill(~valid, 0)
        for s in range(0, N, chunk_size):
            e = min(s + chunk_size, N)
            logits = (hidden[s:e] @ weight.t()).float()
            lse[s:e] = torch.logsumexp(logits, dim=-1)
            picked[s:e] = logits.gather(-1, safe_labels[s:e].unsqueeze(-1)).squeeze(-1)
        n_valid = valid.sum().clamp(min=1)
        loss = ((lse - picked) * valid).sum() / n_valid
        ctx.save_for_backward(hidden, weight, safe_labels, valid, lse, n_valid)
        return loss

    @staticmethod
    def backward(ctx, grad_out):
        # the kernel works on bfloat16 logits, in place and outside autograd: a backward that is part of a graph itself
        # (create_graph) or under autocast to another type takes the general form
        if ctx.hip and not torch.is_grad_enabled() and _bf16_products(grad_out):
            return _backward_hip(ctx, grad_out)
        if ctx.hip:
            hidden, weight, labels, lse, loss, *_ = ctx.saved_tensors
            valid = labels != ctx.ignore_index
            safe_labels, n_valid = labels.masked_fill(~valid, 0), loss[1]
        else:
            hidden, weight, safe_labels, valid, lse, n_valid = ctx.saved_tensors
        N, H = hidden.shape
        chunk_size = ctx.chunk_size
        dh = torch.empty_like(hidden)
        dw = torch.zeros_like(weight, dtype=torch.float32)
        scale = (grad_out / n_valid).float()
        for s in range(0, N, chunk_size):
            e = min(s + chunk_size, N)
            logits = (hidden[s:e] @ weight.t()).float()
            ds = torch.exp(logits - lse[s:e].unsqueeze(-1))
            ds.scatter_add_(
                -1, safe_labels[s:e].unsqueeze(-1),
                -torch.ones(e - s, 1, dtype=torch.float32, device=ds.device),
            )
            ds *= (valid[s:e].unsqueeze(-1) * scale)
            ds = ds.to(hidden.dtype)
            dh[s:e] = ds @ weight
            dw += (ds.t() @ hidden[s:e]).float()
        return dh, dw.to(weight.dtype), None, None, None, None, None


def _backward_hip(ctx, grad_out):
    hidden, weight, labels, lse, loss, *kept = ctx.saved_tensors
    N = hidden.shape[0]
    grad = grad_out.float()
    dh = torch.empty_like(hidden)
    dw = None
    for s, e in ctx.spans:
        if e <= ctx.kept:
            ds = torch.empty_like(kept[0])  # not in the logits' place: the graph may be gone through again
            kernels().ce_bwd(kept[0], labels[s:e], ctx.ignore_index, lse[s:e], grad, loss, ds)
        else:
            ds = multiply(hidden[s:e], weight)
            kernels().ce_bwd(ds, labels[s:e], ctx.ignore_index, lse[s:e], grad, loss)
        if e - s == N:
            dh = multiply(ds, weight, True)
        else:
            torch.mm(ds, weight, out=dh[s:e])
        # chunks are summed in float32, by the product itself
        dw = weight_grad(ds, hidden[s:e], dw, e < N)
    if dw is None:
        dw = torch.zeros_like(weight)
    return dh, dw.to(weight.dtype), None, None, None, None, None


def fused_linear_cross_entropy(
    hidden: torch.Tensor,
    weight: torch.Tensor,
    labels: torch.Tensor,
    ignore_index: int = -100,
    chunk_size: int = 4096,
    kept_bytes: Optional[int] = None,
) -> torch.Tensor:
    """hidden [.., H], weight [V, H], labels [..] -> mean CE over valid tokens.

    Memory beyond the inputs and gradients, in bfloat16 on the GPU: the logits of ``chunk_size`` rows at a time, and, where a
    gradient is recorded, those of the first rows (four chunks, ``kept_bytes`` at most, 1 GiB if it is None) from the
    forward to the backward and as much again during the backward. Losses that are summed before one backward hold theirs
    each. ``kept_bytes=0`` keeps none: the backward forms every chunk's logits again."""
    H = hidden.shape[-1]
    recorded = torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad)
    return _FusedLinearCE.apply(hidden.reshape(-1, H), weight, labels.reshape(-1), ignore_index, chunk_size, recorded, kept_bytes)
