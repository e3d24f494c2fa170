"""Parallel residual streams ("hyper-connections").

A token carries ``S`` residual rows ``x_1 .. x_S`` (float32 ``[N, S, W]``) instead of
one. A sublayer reads ``u = sum_s read[s] x_s``; from its output ``y`` every stream is
formed anew, all at once from the old ones:

    x_t <- sum_s mix[s, t] x_s + write[t] * y        (mix indexed [from, to]).

``streams_start`` makes every stream the token's (scaled) embedding row and forms the first
sublayer's normed input. ``streams_update`` does one sublayer's write, in place,
together with the read and RMS norm of whatever comes next — the next sublayer,
or the output head, which reads the plain sum (``read=None``) — so each stream
element is read and written once per sublayer.

A layer of two sublayers need not write the streams in between: ``streams_read`` forms what the second one reads,
and ``streams_update_two`` writes both. Before the first write the streams may be ``Rows``: every one of
them the token's embedding row, which is then read in their place.
"""

from dataclasses import dataclass
from typing import Optional, Tuple, Union

import torch

from ._kernels import serving_kernels, use_serving_hip as use_hip
from .group_norm import grouped_rms_norm_ref

__all__ = ["Rows", "streams_start", "streams_start_ref", "streams_update", "streams_update_ref", "streams_begin", "streams_pairs",
           "streams_read", "streams_update_two"]


@dataclass
class Rows:
    """Streams that all are their token's row of ``table`` [vocab, W] so far."""

    table: torch.Tensor
    tokens: torch.Tensor
    streams: int

    def select(self, which: torch.Tensor) -> "Rows":
        return Rows(self.table, self.tokens.index_select(0, which), self.streams)

    def filled(self) -> torch.Tensor:
        return self.table[self.tokens].float()[:, None, :].repeat(1, self.streams, 1)


def _read_norm(x, read, weight, eps, out_dtype):
    u = x.sum(1) if read is None else torch.einsum("nsw,s->nw", x, read.float())
    return grouped_rms_norm_ref(u, weight, 1, eps, None, out_dtype)


def streams_start_ref(table, tokens, streams: int, read, weight, eps: float, scale: float = 1.0):
    x = (table[tokens].float() * scale)[:, None, :].repeat(1, streams, 1)
    return x, _read_norm(x, read, weight, eps, table.dtype)


def streams_start(table, tokens, streams: int, read, weight, eps: float, scale: float = 1.0):
    """table [vocab, W], tokens [N] int64 -> (streams [N, S, W] float32 = ``scale`` times the rows, ``rms_norm(u) *
    weight`` in the table's dtype). With one stream that is the start of an ordinary pre-norm model."""
    if use_hip(table):
        return tuple(serving_kernels().streams_start(table, tokens, streams, read, weight, eps, float(scale)))
    return streams_start_ref(table, tokens, streams, read, weight, eps, scale)


def streams_update_ref(x, y, mix, write, read, weight, eps: float, out_dtype=None):
    x.copy_(torch.einsum("nsw,st->ntw", x, mix.float()) + write.float()[None, :, None] * y.float()[:, None, :])
    return None if weight is None else _read_norm(x, read, weight, eps, out_dtype or y.dtype)


def streams_update(x, y, mix, write, read: Optional[torch.Tensor], weight: Optional[torch.Tensor], eps: float,
                   out_dtype=None):
    """x [N, S, W] float32, updated in place from the sublayer's output y [N, W]; ``mix`` [S, S], ``write`` [S]. Returns
    ``rms_norm(sum_s read[s] x_s) * weight`` of the new streams in ``out_dtype`` (``read=None``: the plain sum), or
    None when ``weight`` is None."""
    if use_hip(x):
        return serving_kernels().streams_update(x, y.contiguous(), mix, write, read, weight, eps, out_dtype or y.dtype)
    return streams_update_ref(x, y, mix, write, read, weight, eps, out_dtype)


def streams_pairs(y, streams: int) -> bool:
    """Whether ``streams_read`` and ``streams_update_two`` have kernels for rows like ``y``; without, updates one by one are faster."""
    return use_hip(y) and serving_kernels().streams_pairs(streams, y.shape[1])


def _base(x: Union[torch.Tensor, Rows], y) -> Tuple:
    return (x, None, None) if not isinstance(x, Rows) else (None, x.table, x.tokens) if x.table.dtype == y.dtype else (x.filled(), None, None)


def streams_begin(table, tokens, streams: int, read, weight, eps: float):
    """``streams_start`` with unit scale that leaves the streams as ``Rows`` where the other ops take them: ``(streams, input)``."""
    if streams_pairs(table, streams):
        h = serving_kernels().streams_start(table, tokens, streams, read, weight, eps, 1.0, False)[1]
        return Rows(table, tokens, streams), h
    return streams_start(table, tokens, streams, read, weight, eps)


def streams_read(x: Union[torch.Tensor, Rows], y, mix, write, read, weight, eps: float, out_dtype=None):
    """What ``streams_update`` returns, with the streams left as they are."""
    y = y.contiguous()
    if streams_pairs(y, write.numel()):
        h = serving_kernels().streams_pass(*_base(x, y), None, None, None, y, mix, write, read, weight, eps, out_dtype or y.dtype)
        if h is not None:
            return h
    x = x.filled() if isinstance(x, Rows) else x.clone()
    return streams_update(x, y, mix, write, read, weight, eps, out_dtype)


def streams_update_two(x: Union[torch.Tensor, Rows], first: Tuple, y, mix, write, read, weight, eps: float, out_dtype=None):
    """Two updates, of ``first`` = (y, mix, write) and of the others: ``(streams, input)``, the streams written in place unless they were
    ``Rows``."""
    y1, y = first[0].contiguous(), y.contiguous()
    if streams_pairs(y, write.numel()):
        new, table, tokens = _base(x, y)
        if new is None:
            new = torch.empty(y.shape[0], write.numel(), y.shape[1], dtype=torch.float32, device=y.device)
        h = serving_kernels().streams_pass(new, table, tokens, y1, first[1], first[2], y, mix, write, read, weight, eps, out_dtype or y.dtype)
        if h is not None:
            return new, h
    x = x.filled() if isinstance(x, Rows) else x
    streams_update(x, y1, first[1], first[2], None, None, eps)
    return x, streams_update(x, y, mix, write, read, weight, eps, out_dtype)
