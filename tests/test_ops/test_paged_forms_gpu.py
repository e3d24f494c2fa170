"""Paged attention over the edges of its kernels: token and key tile remainders, sequences of a few tokens beside long
ones, scales of either sign and zero, with and without the parts that put scores into the base-2 domain early.

The bound: float32 scores and weights; the output is rounded to bfloat16 once (at most 2^-8 of a value) and a score
error of a few float32 roundings of the largest score moves a weight by less than that."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -8


def _batch(counts, starts, page, seed=0):
    from colossalai_amd.ops.ragged import RaggedBatch

    need = [(a + b + page - 1) // page for a, b in zip(counts, starts)]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(order[at: at + n])
        at += n
    return RaggedBatch.build(counts, starts, list(range(len(counts))), "cuda", tables, page), sum(need)


def _check(counts, starts, H, G, D, Dv, page, scale, **kw):
    from colossalai_amd.ops.paged_attention import distance_slopes, paged_attention, paged_attention_ref

    torch.manual_seed(1)
    batch, pages = _batch(counts, starts, page)
    k = torch.randn(pages, page, G, D, device="cuda").bfloat16()
    v = torch.randn(pages, page, G, Dv, device="cuda").bfloat16()
    q = torch.randn(sum(counts), H, D, device="cuda").bfloat16()
    if kw.pop("slopes", False):
        kw["slopes"] = distance_slopes(H, "cuda")
    if kw.pop("gate", False):
        kw["gate"] = torch.randn(sum(counts), H, device="cuda").bfloat16()
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(H, device="cuda") + 2.0
    if kw.pop("factors", False):
        kw["key_factors"] = torch.rand(pages, page, G, device="cuda") + 0.5
    got = paged_attention(q, k, v, batch, scale, **kw)
    kw.setdefault("window", 0)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, scale, **{n: (t.float() if n == "gate" else t)
                                                                                  for n, t in kw.items()})
    err = (got.double() - want.double()).norm() / want.double().norm()
    assert err < BOUND, f"{err:.2e}"
    assert torch.isfinite(got.float()).all()


@pytest.mark.parametrize("scale", [0.1, -0.1, 0.0])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0, sink=True), dict(slopes=True, window=70, keep_first=4), dict(chunk=64)])
def test_portions_and_scales(scale, kw):
    _check([33, 1, 96, 65], [0, 130, 31, 64], 8, 2, 128, 128, 16, scale, **dict(kw))


@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 64), (256, 256), (72, 40), (320, 256)])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0, sink=True), dict(sink_logits=True, gate=True), dict(factors=True),
                                dict(slopes=True, window=1500, keep_first=4)])
def test_decode_with_keys_in_parts(D, Dv, kw):
    """Long contexts beside one that leaves most parts empty, one that ends a part exactly, and a token that sees itself only."""
    _check([1, 1, 1, 1], [4999, 0, 2047, 600], 4, 2, D, Dv, 16, 0.1, **dict(kw))


@pytest.mark.parametrize("H,G,starts", [(16, 4, [9000]), (6, 2, [8200, 100]), (8, 8, [3000, 511, 512, 513])])
def test_decode_heads_and_parts(H, G, starts):
    _check([1] * len(starts), starts, H, G, 128, 128, 64, 0.09)


@pytest.mark.parametrize("H,G,starts", [(8, 2, [4000, 37]), (4, 2, [8191]), (4, 2, [8200]), (1, 1, [20000])])
def test_decode_in_float32(H, G, starts):
    """The last ones at and beyond the 64 parts that the merge takes."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(2)
    n = len(starts)
    batch, pages = _batch([1] * n, starts, 16)
    q, k, v = (torch.randn(*s, device="cuda") for s in ((n, H, 128), (pages, 16, G, 128), (pages, 16, G, 128)))
    got = paged_attention(q, k, v, batch, 0.09, softcap=7.0, sink=True)
    want = paged_attention_ref(q, k, v, batch, 0.09, softcap=7.0, sink=True)
    # float32 sums over the weights: keys^0.5 roundings of 2^-24 at most on average, and as much again in the reference
    assert (got - want).norm() / want.norm() < 2 * max(starts) ** 0.5 * 2.0 ** -24


# One sequence whose heads fill one or two blocks: its keys would go into more than the 64 parts that the merge takes from
# 16384 keys on (32768 with a single head); one page more, twice as many and on, and shared heads.
@pytest.mark.parametrize("H,G,start", [(4, 2, 16383), (4, 2, 16384), (4, 1, 16400), (2, 2, 40000), (1, 1, 32767), (1, 1, 33000),
                                       (2, 1, 70000)])
def test_decode_with_most_parts(H, G, start):
    _check([1], [start], H, G, 128, 128, 16, 0.09)


@pytest.mark.parametrize("start", [4095, 4096, 9000])
def test_latent_rows_with_most_parts(start):
    """Values that are the leading channels of wide key rows, two query heads."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(3)
    batch, pages = _batch([1], [start], 16)
    k = torch.randn(pages, 16, 1, 576, device="cuda").bfloat16()
    q = torch.randn(1, 2, 576, device="cuda").bfloat16()
    got = paged_attention(q, k, k[..., :512], batch, 0.05)
    want = paged_attention_ref(q.float(), k.float(), k[..., :512].float(), batch, 0.05)
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("counts", [[1], [40]])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0), dict(softcap=5.0, sink=True)])
def test_nan_stays_nan(counts, kw):
    """A query or a key of NaN shows in what it touches, and nowhere else, also where a cap bounds the score. The other scores
    reach far beyond the cap's near form."""
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(4)
    batch, pages = _batch(counts, [100], 16)
    n = sum(counts)
    k, v = (torch.randn(pages, 16, 2, 64, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(n, 4, 64, device="cuda").bfloat16()
    q[n - 1, 0, 5] = float("nan")          # one token's first head: of key head 0
    k[batch.block_tables[0, 2], 3, 1, 7] = float("nan")   # position 35, which every token sees: key head 1
    bad = torch.isnan(paged_attention(q, k, v, batch, 1.0, **kw).float()).all(-1)
    some = torch.isnan(paged_attention(q, k, v, batch, 1.0, **kw).float()).any(-1)
    want = torch.zeros(n, 4, dtype=torch.bool, device="cuda")
    want[n - 1, 0] = True
    want[:, 2:] = True
    assert torch.equal(bad, want) and torch.equal(some, want)


@pytest.mark.parametrize("counts", [[1], [40]])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0, sink=True), dict(chunk=64)])
def test_a_scale_of_nan_shows(counts, kw):
    from colossalai_amd.ops.paged_attention import paged_attention

    batch, pages = _batch(counts, [100], 16)
    k, v = (torch.randn(pages, 16, 2, 64, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(sum(counts), 4, 64, device="cuda").bfloat16()
    assert torch.isnan(paged_attention(q, k, v, batch, float("nan"), **kw).float()).all()


@pytest.mark.parametrize("spread", [0.02, 0.1, 0.5])
def test_capped_scores_keep_float32_precision(spread):
    """A decode token that sees one key and the sink returns p = 1 / (1 + exp(-s)) of its value 1: s can be read back."""
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(5)
    n, H, D, cap = 512, 8, 64, 30.0
    batch, pages = _batch([1] * n, [0] * n, 1)
    q = torch.randn(n, H, D, device="cuda").bfloat16()
    k = torch.randn(pages, 1, H, D, device="cuda").bfloat16()
    v = torch.ones(pages, 1, H, D, device="cuda").bfloat16()
    dots = (q.double() * k[batch.block_tables[:, 0].long(), 0].double()).sum(-1)
    scale = spread * cap / dots.std().item()
    p = paged_attention(q, k, v, batch, scale, softcap=cap, sink=True, out_dtype=torch.float32)[..., 0].double()
    s = cap * torch.tanh(dots * scale / cap)
    mine = torch.log(p / (1 - p))
    seen = (s < 0) & (s > -12)   # there p's own rounding is at most 2^-23 of s
    err = (mine - s)[seen]
    # a score's roundings are relative to it (sums of the product, scale, quotient, tanh), those of exponential, sum and quotient of p
    # are not: four of half of 2^-23 at most either way
    assert err.pow(2).mean().sqrt() < 4 * 2.0 ** -24 * (1 + s[seen].pow(2).mean().sqrt())


@pytest.mark.parametrize("H,G,counts,starts,page", [
    (6, 2, [40, 1, 33], [0, 70, 31], 8),     # few blocks, two groups of waves: odd and even numbers of key tiles
    (4, 4, [300, 129], [0, 5], 16),          # a block of 128 tokens of one head
    (24, 3, [1100], [0], 64),                # 6 rows of heads: neither a divisor nor a multiple of the XCDs
    (16, 16, [2200, 17], [0, 0], 32),        # 16 rows, every block running at once
    (16, 16, [4700], [0], 32),               # 16 rows, more blocks than run at once
    (64, 8, [900], [100], 4),                # 16 rows of several heads, pages smaller than a wave's load
    (4, 1, [2500], [0], 64),                 # one row over all XCDs
    (8, 2, [2600, 31], [700, 0], 1),         # four XCDs a row
])
@pytest.mark.parametrize("D,Dv,kw", [(128, 128, {}), (64, 64, dict(softcap=5.0, sink=True)), (48, 64, {}),
                                     (72, 40, dict(slopes=True, window=200, keep_first=40))])
def test_every_tile_is_taken_once(H, G, counts, starts, page, D, Dv, kw):
    _check(counts, starts, H, G, D, Dv, page, 0.1, **dict(kw))


@pytest.mark.parametrize("softcap", [0.5, 50.0])
@pytest.mark.parametrize("scale", [1e-4, 0.03, 1.0])
def test_soft_caps_near_and_far(softcap, scale):
    """Scores far below the cap, about it and far above it: the two forms of tanh."""
    _check([64, 700], [10, 0], 16, 4, 64, 64, 16, scale, softcap=softcap, sink=True)


@pytest.mark.parametrize("ratio", [1e-9, 1e-6, 1e-5, 0.9e-4, 1.1e-4, 3e-3, 0.9e3, 1.1e3, 1e5, 1e6])
@pytest.mark.parametrize("D", [64, 128, 72])
@pytest.mark.parametrize("kw", [dict(sink=True), {}, dict(sink=True, slopes=True)])
def test_soft_caps_of_any_ratio(ratio, D, kw):
    """Scores about half the cap, whatever product of a scale and of queries they come from; queries of 0 are among them."""
    from colossalai_amd.ops.paged_attention import distance_slopes, paged_attention

    torch.manual_seed(12)
    n, start, H, G, cap = 70, 40, 8, 2, 30.0
    batch, pages = _batch([n], [start], 16)
    k, v = (torch.randn(pages, 16, G, D, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(n, H, D, device="cuda").bfloat16()
    q[..., 0], q[5] = 64.0, 0.0
    k[..., 0] = (2.0 + 2.0 * torch.rand(pages, 16, G, device="cuda")) * (-1.0 if kw else 1.0)   # a sink shows scores far below it
    kk, vv = (t[batch.block_tables[0].long()].flatten(0, 1)[: n + start].double().repeat_interleave(H // G, 1) for t in (k, v))
    most = torch.einsum("nhd,mhd->hnm", q.double(), kk).abs().max().item()
    up = 2.0 ** math.floor(math.log2(0.5 / ratio / most))    # exact
    q, ratio = q * up, 0.499 / (most * up)
    slopes = distance_slopes(H, "cuda") if kw.get("slopes") else None
    got = paged_attention(q, k, v, batch, ratio * cap, softcap=cap, sink=kw.get("sink", False), slopes=slopes, out_dtype=torch.float32)
    s = cap * torch.tanh(torch.einsum("nhd,mhd->hnm", q.double(), kk) * ratio)
    far = torch.arange(start, start + n, device="cuda")[:, None] - torch.arange(start + n, device="cuda")
    if slopes is not None:
        s -= slopes.double()[:, None, None] * far
    s = s.masked_fill(far < 0, float("-inf"))
    if kw.get("sink"):
        s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
    want = torch.einsum("hnm,mhd->nhd", torch.softmax(s, -1)[..., : n + start], vv)
    # weights have 16 bits or more (two bfloat16 halves), and a score of up to 15 nats some ten roundings of 2^-24
    err = (got - want).norm() / want.norm()
    assert err < 2.0 ** -16 + 15 * 10 * 2.0 ** -24, f"{err:.2e}"


# One, two, three and four or more query heads a key head: blocks of 128, 64 and 32 tokens. Head sizes that fill the pieces of 32 channels that
# tiles are loaded in, end inside one, or leave one of a pair out.
@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 128, 128), (4, 2, 128, 128), (4, 2, 64, 128), (3, 1, 64, 64), (5, 1, 128, 64), (4, 2, 96, 96),
                                      (2, 1, 48, 40), (4, 1, 24, 8), (4, 2, 72, 104)])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0, sink=True), dict(slopes=True, window=70, keep_first=4, gate=True),
                                dict(factors=True, chunk=100)])
def test_portions_of_head_counts_and_sizes(H, G, D, Dv, kw):
    _check([33, 1, 96, 65, 64, 129], [0, 130, 31, 64, 1, 500], H, G, D, Dv, 16, 0.1, **dict(kw))


@pytest.mark.parametrize("levels", [
    (0, 9, 18, 27, 36, 45),          # the nearest keys, which are taken first, have the largest scores
    (60, 40, 20, 0, -20, -40),       # every 64 keys' weights pass the reference of those before
    (-3000, 0, -3000, 4, 8, 1000),   # far below, far above
])
@pytest.mark.parametrize("kw", [{}, dict(sink_logits=True), dict(window=200, keep_first=5)])
@pytest.mark.parametrize("rows", [1, 16])
def test_scores_that_rise_and_fall(levels, kw, rows):
    """Keys 64 at a time have scores of a level of their own (in nats): the reference that a token's weights are taken against is left
    behind, raised, or stays. `rows` sequences: two groups of waves a block, or one."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(6)
    n, scale = 64 * len(levels), 128 ** -0.5
    batch, pages = _batch([n - 10] * rows, [10] * rows, 64)
    k, v = (torch.randn(pages, 64, 4, 128, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(rows * (n - 10), 16, 128, device="cuda").bfloat16()
    q[..., 0] = 8.0
    for b in range(rows):
        for i, level in enumerate(levels):
            k[batch.block_tables[b, i].long(), :, :, 0] = level / (8.0 * scale)
    kw = dict(kw)
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(16, device="cuda") + 2.0
    got = paged_attention(q, k, v, batch, scale, **kw)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, scale, **kw)
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("levels", [
    (0, 9, 18, 27, 36, 45, 54, 63),  # from the farthest tile of 32 keys to the nearest, which is taken first
    (63, 54, 45, 36, 27, 18, 9, 0),  # every tile passes the reference of those before it
    (125, 100, 75, 50, 25, 0),
    (56, 42, 42, 28, 28, 14, 14, 0),   # every second one does
    (42, 42, 28, 28, 14, 14, 0),
    (9, 0, 27, 36, 54, 45, 63),
])
@pytest.mark.parametrize("kw", [{}, dict(sink_logits=True), dict(window=150, keep_first=40)])
@pytest.mark.parametrize("rows", [1, 32])
def test_tiles_that_rise(levels, kw, rows):
    """Keys 32 at a time have scores of a level of their own: the reference is raised after the first or the second of a step's two
    tiles, while the other's weights are on their way to the values. `rows` sequences: two groups of waves a block, or one."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(13)
    n, scale = 32 * len(levels), 128 ** -0.5
    batch, pages = _batch([n - 10] * rows, [10] * rows, 32)
    k, v = (torch.randn(pages, 32, 4, 128, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(rows * (n - 10), 16, 128, device="cuda").bfloat16()
    q[..., 0] = 8.0
    for i, level in enumerate(levels):
        k[batch.block_tables[:, i].long(), :, :, 0] = level / (8.0 * scale)
    kw = dict(kw)
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(16, device="cuda") + 2.0
    got = paged_attention(q, k, v, batch, scale, **kw)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, scale, **kw)
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("D", [64, 128, 72])
@pytest.mark.parametrize("rows", [1, 40])
def test_large_values_of_rising_scores(D, rows):
    """Values of about 2^104: a weight is taken again before it passes 2^12, so that its product stays below 2^128."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(14)
    n, scale = 256, D ** -0.5
    batch, pages = _batch([n] * rows, [0] * rows, 64)
    k, v = (torch.randn(pages, 64, 4, D, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(rows * n, 16, D, device="cuda").bfloat16()
    q[..., 0] = 8.0
    for i, level in enumerate((16, 16, 16, 0)):   # the nearest keys are taken first
        k[batch.block_tables[:, i].long(), :, :, 0] = level / (8.0 * scale)
    v = v * 2.0 ** 104
    got = paged_attention(q, k, v, batch, scale)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, scale)
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("rows,H", [(1, 2), (40, 16)])
@pytest.mark.parametrize("keep_first,key,clean", [(0, 270, 364), (4, 290, 396)])
def test_values_outside_a_window_of_several_token_tiles(bad, rows, H, keep_first, key, clean):
    """Blocks of 128 tokens: a step whose keys all lie before a wave's window adds nothing to it, whatever they hold, and the kept first keys
    behind it are seen again. One and two groups of waves."""
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(15)
    batch, pages = _batch([128] * rows, [300] * rows, 16)
    k, v = (torch.randn(pages, 16, H, 64, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(128 * rows, H, 64, device="cuda").bfloat16()
    want = paged_attention(q, k, v, batch, 0.1, 40, keep_first)
    v[batch.block_tables[:, key // 16].long(), key % 16] = bad
    got = paged_attention(q, k, v, batch, 0.1, 40, keep_first)
    sees = (batch.positions >= key) & (batch.positions < key + 40)
    assert not torch.isfinite(got[sees].float()).any()
    assert torch.equal(got[batch.positions >= clean], want[batch.positions >= clean])


@pytest.mark.parametrize("which", ["keys", "values"])
def test_pools_at_an_odd_address(which):
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(7)
    batch, pages = _batch([40, 1], [100, 3], 16)
    k, v = (torch.randn(pages, 16, 2, 64, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(41, 4, 64, device="cuda").bfloat16()
    want = paged_attention(q, k, v, batch, 0.1)
    t = k if which == "keys" else v
    odd = torch.empty(t.numel() + 1, device="cuda", dtype=t.dtype)[1:].view(t.shape).copy_(t)
    got = paged_attention(q, odd if which == "keys" else k, odd if which == "values" else v, batch, 0.1)
    assert (got.double() - want.double()).norm() / want.double().norm() < 2 * BOUND


@pytest.mark.parametrize("counts,starts", [([40, 1], [100, 3]), ([200], [0]), ([33, 1, 96], [0, 130, 31])])
@pytest.mark.parametrize("kw", [{}, dict(window=70, keep_first=4), dict(sink_logits=True)])
@pytest.mark.parametrize("offset", [1, 4])
def test_portions_of_pools_at_odd_addresses_take_the_same_kernel(counts, starts, kw, offset):
    """The same bits; the pages beside a sequence's own may be numbered anyhow."""
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(12)
    batch, pages = _batch(counts, starts, 16)
    k, v = (torch.randn(pages, 16, 2, 64, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(sum(counts), 4, 64, device="cuda").bfloat16()
    kw = dict(kw)
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(4, device="cuda")
    odd = [torch.empty(t.numel() + offset, device="cuda", dtype=t.dtype)[offset:].view(t.shape).copy_(t) for t in (k, v)]
    want = paged_attention(q, k, v, batch, 0.1, **kw)
    own = torch.tensor([(a + b + 15) // 16 for a, b in zip(counts, starts)], device="cuda")
    batch.block_tables[torch.arange(batch.block_tables.shape[1], device="cuda") >= own[:, None]] = 1 << 20
    assert torch.equal(paged_attention(q, *odd, batch, 0.1, **kw), want)


# Decode tokens: groups of 1 to 16 query heads (17: another kernel), key and value sizes that differ, last tiles of one key and of 32,
# windows and blocks that begin inside a page and a tile, kept keys that end in the middle of a page.
@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 128, 128), (6, 2, 64, 128), (16, 1, 128, 64), (17, 1, 64, 64), (10, 2, 64, 64)])
@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0), dict(sink_logits=True, gate=True), dict(chunk=1000),
                                dict(slopes=True, window=333, keep_first=37), dict(window=2300, keep_first=5, sink=True)])
def test_decode_of_head_counts_and_sizes(H, G, D, Dv, page, kw):
    _check([1] * 7, [0, 30, 31, 32, 340, 1999, 4100], H, G, D, Dv, page, 0.1, **dict(kw))


@pytest.mark.parametrize("levels", [(0, 9, 18, 27, 36, 45), (60, 40, 20, 0, -20, -40), (-3000, 0, -3000, 4, 8, 1000)])
@pytest.mark.parametrize("parts", [False, True])
def test_decode_scores_that_rise_and_fall(levels, parts):
    """Levels (in nats) of 256 or 2048 keys each: inside a wave's tiles, and from part to part."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(8)
    each, scale = 2048 if parts else 256, 128 ** -0.5
    batch, pages = _batch([1, 1], [each * len(levels) - 1, 100], 64)
    k, v = (torch.randn(pages, 64, 2, 128, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(2, 8, 128, device="cuda").bfloat16()
    q[..., 0] = 8.0
    for i, level in enumerate(levels):
        k[batch.block_tables[0, i * each // 64: (i + 1) * each // 64].long(), :, :, 0] = level / (8.0 * scale)
    got = paged_attention(q, k, v, batch, scale)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, scale)
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


# decode tokens beside portions that fill the chip alone, first, last and between them: they go to the decode kernel, whole and
# in parts; in the last two cases they stay (short contexts, few enough blocks)
@pytest.mark.parametrize("counts,starts", [([1, 1000, 1, 990, 1], [900, 40, 1500, 0, 3]), ([1, 1, 1, 1990], [2100, 1025, 0, 3]),
                                           ([1, 1000, 1, 990], [300, 40, 100, 0]), ([1, 500, 1], [700, 0, 600])])
@pytest.mark.parametrize("H,G,D,Dv", [(16, 4, 128, 128), (16, 8, 64, 64), (16, 4, 64, 128)])
@pytest.mark.parametrize("kw", [dict(window=1024, keep_first=4, slopes=True, gate=True), dict(softcap=5.0, sink=True)])
def test_decode_tokens_beside_long_portions(counts, starts, H, G, D, Dv, kw):
    _check(counts, starts, H, G, D, Dv, 16, D ** -0.5, **dict(kw))


@pytest.mark.parametrize("D,group", [(64, 1), (128, 1), (64, 16), (128, 4)])
def test_decode_weights_are_whole(D, group):
    """256 keys of value v_a and 256 of -1, whose weights p differ from head to head and whose sums nearly cancel: 2^-13 of them is
    left. A weight's error of 2^-18, what two bfloat16 halves leave, would be up to a twentieth of the result; weights of 24 bits,
    their exponential (2^-22) and the result's own rounding make less than 2^-7 of it."""
    from colossalai_amd.ops.paged_attention import paged_attention

    heads, n, page = 32, 512, 16
    batch, pages = _batch([1], [n - 1], page)
    k, v = torch.zeros(n, heads, D), torch.zeros(n, heads, D)
    q = torch.zeros(1, heads, D)
    q[0, :, 3] = 1.0
    below = -(0.05 + torch.arange(heads) / 50.0).bfloat16().double()      # scores of the second half; those of the first are 0
    k[n // 2:, :, 3] = below.float()
    v[n // 2:] = -1.0
    p = torch.exp(below)
    v[: n // 2] = p.bfloat16().float()[:, None]
    for i in range(3):   # the first keys' values bring the sums together
        gap = (n // 2) * (p * (1 + 2.0 ** -13)) - v[: n // 2, :, 0].double().sum(0)
        v[i] = (v[i, :, 0].double() + gap).bfloat16().float()[:, None]
    want = (v[: n // 2, :, 0].double().sum(0) - (n // 2) * p) / ((n // 2) * (1 + p))
    assert (want.abs() / p).max() < 2.0 ** -12 and want.abs().min() > 0
    order = batch.block_tables[0].long().cpu()
    pool = lambda t: t.view(pages, page, heads, D)[torch.argsort(order)].cuda().bfloat16()
    q = q.repeat_interleave(group, 1).cuda().bfloat16()   # all heads of a key head alike
    got = paged_attention(q, pool(k), pool(v), batch, 1.0)[0, :, 0].double().cpu().view(heads, group)
    assert ((got - want[:, None]).abs() <= 2.0 ** -6 * want.abs().max()).all()


@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (8, 1, 64, 128), (16, 1, 64, 64), (2, 2, 64, 64)])
@pytest.mark.parametrize("start", [300, 335, 3000])
@pytest.mark.parametrize("kw", [{}, dict(window=290, keep_first=3), dict(sink=True, softcap=5.0)])
def test_decode_values_that_are_infinite(H, G, D, Dv, start, kw):
    """A visible value of inf is the result of its channel, one of each sign or a NaN give NaN; the other channels, and keys that are
    not seen, keep theirs."""
    from colossalai_amd.ops.paged_attention import paged_attention

    torch.manual_seed(9)
    n = 34   # enough for groups of any size
    batch, pages = _batch([1] * n, [start] + [start - 7] * (n - 1), 16)
    k, v = torch.randn(pages, 16, G, D, device="cuda").bfloat16(), torch.randn(pages, 16, G, Dv, device="cuda").bfloat16()
    q = torch.randn(n, H, D, device="cuda").bfloat16()
    want = paged_attention(q, k, v, batch, 0.1, **kw)
    row = lambda pos: (batch.block_tables[0, pos // 16].long(), pos % 16)
    inf = float("inf")
    for pos, channel, value in [(start, 1, inf), (start - 40, 2, -inf), (start - 280, 3, inf), (start - 280, 4, inf),
                                (start, 4, -inf), (start - 1, 5, float("nan"))]:
        v[row(pos)][G - 1, channel] = value
    hidden = row(start + 1 if (start + 1) % 16 else 5)   # behind the token, or ahead of the window if there is one
    if (start + 1) % 16 or "window" in kw:
        v[hidden][:, 6] = inf
    got = paged_attention(q, k, v, batch, 0.1, **kw)
    last = got[0, -1]
    assert last[1] == inf and last[2] == -inf and last[3] == inf and last[4].isnan() and last[5].isnan()
    want[0, (G - 1) * (H // G):, 1:6] = got[0, (G - 1) * (H // G):, 1:6]
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("start", [100, 299, 3000])
@pytest.mark.parametrize("size", [1.2e19, 3e9, -1.5e10])
@pytest.mark.parametrize("kw", [{}, dict(window=290), dict(slopes=True)])
def test_decode_scores_of_any_size(start, size, kw):
    """Equal scores as large as float32 holds them (-3.2e38 in base 2), or so large that a rounding of theirs is more than the exponential
    can take: a token is the mean of the values that it sees."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(10)
    batch, pages = _batch([1], [start], 16)
    q, k = torch.zeros(1, 4, 64, device="cuda"), torch.zeros(pages, 16, 2, 64, device="cuda")
    q[..., 0] = 2.0 ** 64 if size > 1e15 else 1.0
    k[..., 0] = -size
    v = torch.randn(pages, 16, 2, 64, device="cuda").bfloat16()
    kw = dict(kw)
    if kw.pop("slopes", False):
        kw["slopes"] = torch.full((4,), 2.0 ** -60, device="cuda")   # nothing beside such a score
    got = paged_attention(q.bfloat16(), k.bfloat16(), v, batch, 1.0, **kw)
    kw.setdefault("window", 0)
    want = paged_attention_ref(q * 0, k, v.float(), batch, 1.0, **kw)   # equal scores, of any size
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("start", [299, 3000])
@pytest.mark.parametrize("H,D", [(4, 64), (32, 128)])
@pytest.mark.parametrize("kw", [{}, dict(softcap=5.0), dict(softcap=5.0, sink=True), dict(sink_logits=True), dict(slopes=True, window=280)])
def test_decode_nan_stays_nan(start, H, D, kw):
    """As test_nan_stays_nan, over more keys than the form for short contexts takes, whole and in parts: a query, a key that one wave
    of many meets, a slope, and a scale of NaN."""
    from colossalai_amd.ops.paged_attention import distance_slopes, paged_attention

    torch.manual_seed(4)
    n = 17   # enough for groups of 16 heads
    batch, pages = _batch([1] * n, [start] + [start - 20] * (n - 1), 16)
    k, v = (torch.randn(pages, 16, 2, D, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(n, H, D, device="cuda").bfloat16()
    kw = dict(kw)
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(H, device="cuda")
    if kw.pop("slopes", False):
        kw["slopes"] = distance_slopes(H, "cuda")
        kw["slopes"][1] = float("nan")
    clean = paged_attention(q, k, v, batch, 1.0, **kw)
    q[1, 0, 5] = float("nan")
    k[batch.block_tables[0, (start - 200) // 16], (start - 200) % 16, 1, 7] = float("nan")
    got = paged_attention(q, k, v, batch, 1.0, **kw)
    bad = torch.zeros(n, H, dtype=torch.bool, device="cuda")
    bad[1, 0] = True
    bad[0, H // 2:] = True
    if "slopes" in kw:
        bad[:, 1] = True
    assert torch.equal(got.isnan().all(-1), bad) and torch.equal(got.isnan().any(-1), bad)
    # heads of a block raise their references together: roundings of the others may differ
    assert (got[~bad].double() - clean[~bad].double()).norm() < BOUND * clean[~bad].double().norm()
    assert paged_attention(q, k, v, batch, float("nan"), **kw).isnan().all()


@pytest.mark.parametrize("starts", [[299, 700], [3000]])
@pytest.mark.parametrize("H,G,D,Dv", [(8, 4, 64, 128), (16, 2, 128, 64), (12, 12, 128, 128)])
@pytest.mark.parametrize("kw", [{}, dict(chunk=600), dict(sink_logits=True, gate=True)])
def test_decode_with_shared_value_heads(starts, H, G, D, Dv, kw):
    """Two key heads (all of them where there are two) read the same values."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(11)
    n = len(starts)
    batch, pages = _batch([1] * n, starts, 16)
    k, v = torch.randn(pages, 16, G, D, device="cuda").bfloat16(), torch.randn(pages, 16, G // 2, Dv, device="cuda").bfloat16()
    q = torch.randn(n, H, D, device="cuda").bfloat16()
    kw = dict(kw)
    if kw.pop("gate", False):
        kw["gate"] = torch.randn(n, H, device="cuda").bfloat16()
    if kw.pop("sink_logits", False):
        kw["sink_logits"] = torch.randn(H, device="cuda") + 2.0
    got = paged_attention(q, k, v, batch, 0.1, **kw)
    want = paged_attention_ref(q.float(), k.float(), v.float(), batch, 0.1, 0, **{a: (t.float() if a == "gate" else t)
                                                                                for a, t in kw.items()})
    assert (got.double() - want.double()).norm() / want.double().norm() < BOUND


@pytest.mark.parametrize("H,G,D,Dv", [(16, 4, 128, 128), (16, 1, 64, 128), (4, 4, 64, 64)])
@pytest.mark.parametrize("starts", [[20, 0], [255, 100, 31], [700] * 5, [1300, 900] * 8, [9000], [30000, 3]])
def test_decode_parts_meet_whoever_ends_last(H, G, D, Dv, starts):
    """The parts of a token's keys are put together by one of their own blocks, in an order that does not depend on which: every
    repetition has the same bits, also from a graph, whose launches repeat themselves over memory that others have used."""
    from colossalai_amd.ops.paged_attention import paged_attention, paged_attention_ref

    torch.manual_seed(6)
    n = len(starts)
    batch, pages = _batch([1] * n, starts, 16)
    k, v = (torch.randn(pages, 16, G, d, device="cuda").bfloat16() for d in (D, Dv))
    gate = torch.randn(n, H, device="cuda").bfloat16()
    qs = [torch.randn(n, H, D, device="cuda").bfloat16() for _ in range(3)]

    def call(q):
        return paged_attention(q, k, v, batch, D ** -0.5, gate=gate, softcap=20.0, sink=True)

    want = [call(q) for q in qs]
    for q, w in zip(qs, want):
        ref = paged_attention_ref(q.float(), k.float(), v.float(), batch, D ** -0.5, gate=gate.float(), softcap=20.0, sink=True)
        assert (w.double() - ref.double()).norm() / ref.double().norm() < BOUND
    torch.cuda.synchronize()
    q = qs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        first, second = call(q), call(q)
    for i in range(30):
        q.copy_(qs[i % 3])
        first.zero_()
        second.zero_()
        graph.replay()
        assert torch.equal(first, want[i % 3]) and torch.equal(second, want[i % 3])
        assert torch.equal(call(q), want[i % 3])


@pytest.mark.parametrize("seqs", [17, 64, 65, 130])
def test_portions_of_many_sequences_find_theirs(seqs):
    """A block looks for its sequence 64 at a time: decode tokens, short and longer portions on either side of that."""
    counts = [1 if i % 5 else 33 + i % 40 for i in range(seqs)]
    _check(counts, [(7 * i) % 90 for i in range(seqs)], 8, 2, 64, 64, 16, 0.1, window=64, keep_first=3)


@pytest.mark.parametrize("counts,starts", [([1000] * 4, [0] * 4), ([700, 33, 1, 1100, 150, 1], [0, 900, 700, 100, 1500, 0]), ([300] * 9, list(range(0, 1800, 200))),
                                           ([65] * 40, [31 * i for i in range(40)]), ([40] * 70, [0] * 70)])
@pytest.mark.parametrize("H,G,kw", [(16, 4, {}), (8, 8, dict(window=300, keep_first=5)), (16, 8, dict(softcap=5.0, sink=True))])
def test_tiles_by_length_are_all_taken(counts, starts, H, G, kw):
    """More blocks than CUs: the longest tiles of all sequences start first, of up to 64 sequences."""
    _check(counts, starts, H, G, 64, 64, 16, 0.1, **dict(kw))
