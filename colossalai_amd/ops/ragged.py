"""Ragged serving batch descriptor shared by the sequence-state ops.

One engine step runs ``N`` new tokens that belong to ``B`` live sequences:
a prompt portion of any length next to single decode tokens. Every op that
carries per-sequence memory (paged keys/values, recurrent matrices, the tail
of a short convolution, the previous token of a token shift) takes this
descriptor instead of a dense ``[B, S]`` layout, so that a result does not
depend, but for the order of float32 sums, on how a prompt was cut or on what
else shares the step.
"""

from dataclasses import dataclass
from typing import List, Optional, Sequence

import torch

from ._kernels import serving_kernels

__all__ = ["RaggedBatch", "to_device"]

LISTED_TOKENS = 32  # up to here a step's per-token vectors are made on the host: a launch takes as long


_COPIES = {}  # device index -> the stream of complete()


def complete(make, device) -> torch.Tensor:
    """The tensor that ``make()`` fills on a GPU from host numbers, complete for every stream when this returns, as one copied from pageable
    memory is. Such a copy waits for all the work ahead of it, so that the GPU then waits for what the host does next; this one has a
    stream of its own, and the host waits for nothing else."""
    index = torch.device(device).index
    index = torch.cuda.current_device() if index is None else index
    if index not in _COPIES:
        _COPIES[index] = torch.cuda.Stream(index)
    current, copies = torch.cuda.current_stream(index), _COPIES[index]
    with torch.cuda.stream(copies):
        made = make()
    made.record_stream(current)  # the memory is of the other stream's: not to be used again before this one's work is done
    copies.synchronize()
    return made


def refuse_capture() -> None:
    """A captured copy from pinned memory would be repeated by every replay, from memory that holds something else by then."""
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("tensors of host numbers cannot be made while a graph is captured")


def to_device(values: Sequence, dtype, device, ordered: bool = False) -> torch.Tensor:
    """A tensor of host numbers on `device`, complete for every stream; `ordered`: for the current one, as any work of the device, with nothing
    that the host waits for (15 to 20 us). Not while a graph is captured."""
    if torch.device(device).type != "cuda":
        return torch.tensor(values, dtype=dtype).to(device)
    refuse_capture()

    def copy():
        return torch.tensor(values, dtype=dtype, pin_memory=True).to(device, non_blocking=True)

    return copy() if ordered else complete(copy, device)


@dataclass
class RaggedBatch:
    # device tensors (int32)
    cu: torch.Tensor          # [B + 1] offsets of each sequence's new tokens in the flat token axis
    start: torch.Tensor       # [B] tokens the sequence already holds (= position of its first new token)
    slots: torch.Tensor       # [B] state slot of each sequence
    tok_seq: torch.Tensor     # [N] which sequence (0..B-1) a token belongs to
    positions: torch.Tensor   # [N] absolute position of a token in its sequence
    block_tables: Optional[torch.Tensor]  # [B, max_blocks] page ids (None when no layer keeps keys)
    kv_rows: Optional[torch.Tensor]       # [N] flat pool row (page * page_size + offset) of each token
    # host mirrors
    cu_host: List[int]
    start_host: List[int]
    slots_host: List[int]
    page_size: int = 0
    ordered: bool = False  # vectors are for the stream they were made on
    _dense: Optional[dict] = None  # memo of dense_context(), by window
    _chunk_tables: Optional[dict] = None  # memo of chunk_tables(), by chunk size
    _tiles: Optional[tuple] = None  # memo of tile_counts()
    _singles: Optional[tuple] = None  # memo of single_tokens()
    _even: Optional[dict] = None  # memo of key_lengths(), by window and fewest

    @property
    def num_seqs(self) -> int:
        return len(self.start_host)

    @property
    def num_tokens(self) -> int:
        return self.cu_host[-1]

    @property
    def max_new(self) -> int:
        return max(self.cu_host[i + 1] - self.cu_host[i] for i in range(self.num_seqs))

    def tile_counts(self):
        """Tiles of 32, 64 and 128 tokens of the prompt portions (all 0 for a pure decode step): the grids of the matrix-core
        attention kernel when every key head has three or more, two or a single query head."""
        if self._tiles is None:
            cu = self.cu_host
            new = [b - a for a, b in zip(cu, cu[1:])]
            decode = cu[-1] == len(new)   # every sequence brings a token
            self._tiles = tuple(0 if decode else sum((n + size - 1) // size for n in new) for size in (32, 64, 128))
        return self._tiles

    def single_tokens(self, window: int = 0):
        """Of a step with prompt portions: how many sequences bring one token, and whether the longest of them sees at least
        half as many keys as the longest portion's last token."""
        if self._singles is None:
            new = [b - a for a, b in zip(self.cu_host, self.cu_host[1:])]
            single = [s + 1 for n, s in zip(new, self.start_host) if n == 1]
            self._singles = len(single), max(single, default=0), max((s + n for n, s in zip(new, self.start_host) if n > 1), default=0)
        count, short, long = self._singles
        if window > 0:
            short, long = min(short, window), min(long, window)
        return count, 2 * short >= long

    def key_lengths(self, window: int = 0, fewest: int = 1):
        """Of the tiles of 32 new tokens of the sequences that bring `fewest` or more: ``(mean / most, most)`` of the keys that a tile's last token
        sees, about (a sequence's tiles count as its first and last one's mean), and the most that one sees."""
        if self._even is None:
            self._even = {}
        if (window, fewest) not in self._even:
            total = most = tiles = 0.0
            for a, b, s in zip(self.cu_host, self.cu_host[1:], self.start_host):
                if b - a < fewest:
                    continue
                lo, hi, n = s + min(32, b - a), s + b - a, (b - a + 31) // 32
                if window <= 0 or hi <= window:
                    mean = (lo + hi) / 2
                elif lo >= window:
                    mean = window
                else:   # grows up to the window, then stays
                    mean = ((lo + window) / 2 * (window - lo) + window * (hi - window)) / (hi - lo)
                total += mean * n
                tiles += n
                most = max(most, min(hi, window) if window > 0 else hi)
            self._even[window, fewest] = (total / (tiles * most), int(most)) if tiles else (0.5, 0)
        return self._even[window, fewest]

    @property
    def num_tiles32(self) -> int:
        """32-token tiles of the prompt portions (0 for a pure decode step):
        the grid of the matrix-core attention kernel."""
        return self.tile_counts()[0]

    @property
    def max_total(self) -> int:
        """Longest sequence after this step (cached + new tokens)."""
        return max(self.start_host[i] + self.cu_host[i + 1] - self.cu_host[i] for i in range(self.num_seqs))

    def dense_context(self, window: int = 0):
        """For ops that lay the whole context of the step's sequences (cached and new tokens) out densely, each
        sequence padded to whole pages: ``(rows, tables, total)`` with ``rows`` [total] the pool row of every place
        of that layout (a padding place repeats the sequence's last row) and ``tables`` [B, max_pages] int32 the page
        table of the dense layout itself (consecutive pages, sequence after sequence). With a sliding ``window`` the
        layout of a sequence starts with the page (and 32-key tile) of the first key that its first new token still
        sees; table entries ahead of it are not meant to be read. Built on the device from the step's own index
        vectors, once per step and window, on the stream that is the current one then."""
        if self._dense is None:
            self._dense = {}
        if window not in self._dense:
            ps, dev = self.page_size, self.cu.device
            shift = ps.bit_length() - 1
            lens = [self.start_host[i] + self.cu_host[i + 1] - self.cu_host[i] for i in range(self.num_seqs)]
            align = max(ps, 32)
            skip = [max(0, s - window + 1) // align * align // ps if window > 0 else 0 for s in self.start_host]
            pages = [(n + ps - 1) // ps - k for n, k in zip(lens, skip)]
            first, total_pages = [], 0
            for n in pages:
                first.append(total_pages)
                total_pages += n
            width = max(n + k for n, k in zip(pages, skip))
            host = to_device([first, pages, lens, skip], torch.int32, dev, self.ordered)   # one copy
            total = total_pages * ps
            if self.block_tables.is_cuda:
                rows = torch.empty(total, dtype=torch.long, device=dev)
                tables = torch.empty(self.num_seqs, width, dtype=torch.int32, device=dev)
                serving_kernels().dense_context(rows, tables, self.block_tables, host, ps)
                self._dense[window] = (rows, tables, total)
                return self._dense[window]
            first_d, pages_d, lens_d, skip_d = (host[i].long() for i in range(4))
            seq = torch.repeat_interleave(torch.arange(self.num_seqs, device=dev), pages_d * ps, output_size=total)
            pos = torch.arange(total, device=dev) - (first_d - skip_d)[seq] * ps
            pos = torch.minimum(pos, lens_d[seq] - 1)
            rows = (self.block_tables[seq, pos >> shift].long() << shift) + (pos & (ps - 1))
            cols = torch.arange(width, device=dev)[None, :] - skip_d[:, None]
            tables = torch.where((cols >= 0) & (cols < pages_d[:, None]), first_d[:, None] + cols, 0).int()
            self._dense[window] = (rows, tables.contiguous(), total)
        return self._dense[window]

    def chunk_tables(self, size: int):
        """Cut every sequence's new tokens into chunks of ``size``: ``(chunks, seq_chunks)`` with ``chunks`` [K, 4] int32
        = (sequence, first token, end token, 0) in sequence order and ``seq_chunks`` [B + 1] each sequence's range of
        chunks, on the device (one copy). Built once per step and size, shared by the step's layers."""
        if self._chunk_tables is None:
            self._chunk_tables = {}
        if size not in self._chunk_tables:
            rows, ranges = [], [0]
            for b in range(self.num_seqs):
                lo, hi = self.cu_host[b], self.cu_host[b + 1]
                for t in range(lo, hi, size):
                    rows += [b, t, min(t + size, hi), 0]
                ranges.append(len(rows) // 4)
            buf = to_device(rows + ranges, torch.int32, self.cu.device, self.ordered)
            self._chunk_tables[size] = (buf[: len(rows)].view(-1, 4), buf[len(rows):])
        return self._chunk_tables[size]

    @staticmethod
    def _fit_int32(starts, new_counts, pages, page_size) -> bool:
        """Whether positions and pool rows are numbers that the device's 32-bit arithmetic makes, as they nearly always are; the
        host's lists refuse others."""
        return (min(starts) >= 0 and max(s + n for s, n in zip(starts, new_counts)) < 2 ** 31
                and (not pages or (min(pages) >= 0 and (max(pages) + 1) * page_size <= 2 ** 31)))

    @classmethod
    def build(cls, new_counts: Sequence[int], starts: Sequence[int], slots: Sequence[int], device,
              tables: Optional[Sequence[Sequence[int]]] = None, page_size: int = 0, *, ordered: bool = False) -> "RaggedBatch":
        """The vectors are complete for every stream when this returns; with `ordered` for the current one, and so are those made later
        from host numbers: for a step that is used there and nowhere else."""
        cu = [0]
        for n in new_counts:
            assert n > 0, "a sequence in a step brings at least one token"
            cu.append(cu[-1] + n)
        B, N, width = len(new_counts), cu[-1], 0
        if tables is not None:
            for i, n in enumerate(new_counts):
                assert len(tables[i]) * page_size >= starts[i] + n, "block table does not cover the new tokens"
            width = max(len(t) for t in tables)
        # one host-to-device copy for all index vectors of the step; the fields are views into it
        parts = [cu, list(starts), list(slots), [p for t in tables or () for p in list(t) + [0] * (width - len(t))]]
        sizes = [B + 1, B, B, B * width, N, N, N if tables is not None else 0]
        if torch.device(device).type == "cuda" and N > LISTED_TOKENS and cls._fit_int32(starts, new_counts, parts[3], page_size):
            refuse_capture()

            def fill():   # a token's own entries on the device
                buf = torch.empty(sum(sizes), dtype=torch.int32, device=device)
                head = torch.tensor([v for part in parts for v in part], dtype=torch.int32, pin_memory=True)
                buf[: head.numel()].copy_(head, non_blocking=True)
                serving_kernels().ragged_index(buf, B, N, width, page_size)
                return buf

            buf = fill() if ordered else complete(fill, device)
        else:
            tok_seq, pos, rows = [], [], []
            for i, n in enumerate(new_counts):
                tok_seq += [i] * n
                pos += list(range(starts[i], starts[i] + n))
                if tables is not None:
                    t = tables[i]
                    rows += [t[p // page_size] * page_size + p % page_size for p in range(starts[i], starts[i] + n)]
            buf = to_device([v for part in parts + [tok_seq, pos, rows] for v in part], torch.int32, device, ordered)
        cu_d, start_d, slots_d, tables_d, tok_seq_d, pos_d, rows_d = buf.split(sizes)
        return cls(
            cu=cu_d, start=start_d, slots=slots_d, tok_seq=tok_seq_d, positions=pos_d,
            block_tables=tables_d.view(B, width) if tables is not None else None,
            kv_rows=rows_d if tables is not None else None,
            cu_host=cu, start_host=list(starts), slots_host=list(slots), page_size=page_size, ordered=ordered,
        )
