"""Flash attention where its launch takes another form: forward blocks of two and four waves, tile remainders,
key/value tiles whose heads several backward blocks share (float32 sums), strided outputs, a negative scale.

The bound: rounding to bfloat16 is 2^-8 of a value at most, 2^-8 / sqrt(3) of a tensor in the 2-norm. An output or a
gradient is rounded itself and is a product of two operands of which at most two were rounded before (probabilities or
their gradients, the output in delta): three such errors add up to 2^-8 in the 2-norm, and half as much again
is left for their not being independent.
"""

import json

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 3 * 2.0 ** -9


def _near(got, want, what, lone=False):
    if lone and what in ("dq", "dk"):
        # a softmax over one key is constant: these vanish but for dout · v and dout · out, both about sqrt(D), being
        # rounded to bfloat16 apart
        assert got.float().abs().max() < 2.0 ** -7 * got.shape[-1] ** 0.5, what
        return
    err = (got.double() - want.double()).norm() / want.double().norm().clamp_min(1e-20)
    assert err < BOUND, f"{what}: {err:.2e}"


def _reference(q, k, v, dout, causal, scale):
    """Float32 outputs and gradients, one head at a time."""
    B, S, H, D = q.shape
    G = k.shape[2]
    q, k, v, dout = (t.float() for t in (q, k, v, dout))
    out, dq, dk, dv = torch.zeros_like(q), torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    hidden = torch.ones(S, k.shape[1], dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(B):
        for h in range(H):
            g = h // (H // G)
            s = (q[b, :, h] @ k[b, :, g].t()) * scale
            if causal:
                s = s.masked_fill(hidden, float("-inf"))
            p = torch.softmax(s, 1)
            out[b, :, h] = p @ v[b, :, g]
            ds = p * (dout[b, :, h] @ v[b, :, g].t() - (dout[b, :, h] * out[b, :, h]).sum(1, keepdim=True)) * scale
            dq[b, :, h] = ds @ k[b, :, g]
            dk[b, :, g] += ds.t() @ q[b, :, h]
            dv[b, :, g] += p.t() @ dout[b, :, h]
    return out, dq, dk, dv


def _inputs(B, S, H, G, D, seed=0):
    torch.manual_seed(seed)
    return [torch.randn(B, S, h, D, device="cuda").bfloat16() for h in (H, G, G, H)]


@pytest.mark.parametrize("B,S,H,G,D,causal,scale", [
    (1, 1, 2, 1, 128, True, None),
    (2, 31, 4, 4, 64, True, None),
    (1, 33, 4, 2, 128, False, None),
    (3, 129, 12, 12, 64, False, None),      # remainder rows of a block of four waves, small grid
    (4, 300, 32, 32, 128, True, None),      # blocks of four waves
    (1, 512, 8, 2, 128, True, None),        # four blocks share a tile's heads
    (1, 520, 6, 2, 64, True, None),         # three do
    (2, 640, 4, 1, 64, False, None),        # without a mask, too few blocks for the CUs
    (1, 520, 71, 1, 64, True, None),        # a prime group: one head a block
    (2, 1100, 71, 1, 64, True, None),       # blocks of three and of two heads
    (1, 1100, 71, 1, 128, False, None),     # and of two and of one
    (1, 200, 4, 2, 64, True, -0.2),
    (1, 130, 2, 2, 128, False, -0.1),
    (1, 100, 2, 2, 64, True, 0.0),          # every visible key counts the same; no gradient of the scores
])
def test_dense(B, S, H, G, D, causal, scale):
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(B, S, H, G, D)
    want = _reference(q, k, v, dout, causal, D ** -0.5 if scale is None else scale)
    for t in (q, k, v):
        t.requires_grad_()
    out = flash_attention(q, k, v, causal=causal, scale=scale)
    got = (out, *torch.autograd.grad(out, (q, k, v), dout))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        if scale == 0.0 and name in ("dq", "dk"):
            assert (a == 0).all(), name
        else:
            _near(a, b, name, lone=S == 1)


@pytest.mark.parametrize("H,G,S,causal", [(71, 1, 8192, True), (28, 4, 8192, True), (71, 1, 8192, False), (8, 2, 8192, True)])
def test_workspace_of_shared_heads_is_bounded(H, G, S, causal):
    """The float32 sums of blocks that share a tile's heads stay below 8 bytes for each channel of 1024 tiles of 128 rows, also
    where a group has no small divisor; every head still counts."""
    from colossalai_amd.ops import kernels

    D = 64
    q, k, v, dout = _inputs(1, S, H, G, D)
    out, lse = kernels().flash_attn_fwd(q, k, v, causal, D ** -0.5)
    none = q.new_empty(0)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grads = kernels().flash_attn_bwd(dout, q, k, v, out, lse, causal, D ** -0.5, none, none, none)
    kept = sum(g.nbytes for g in grads) + lse.nbytes
    assert torch.cuda.max_memory_allocated() - before - kept <= 1024 * 128 * D * 8 + (4 << 20)
    # a group's dV is linear in its heads' dout: all heads together are the sum of the heads one by one
    want = torch.zeros_like(v, dtype=torch.float32)
    for h in range(H):
        o1, l1 = kernels().flash_attn_fwd(q[:, :, h: h + 1].contiguous(), k[:, :, h // (H // G)][:, :, None].contiguous(),
                                          v[:, :, h // (H // G)][:, :, None].contiguous(), causal, D ** -0.5)
        d1 = kernels().flash_attn_bwd(dout[:, :, h: h + 1].contiguous(), q[:, :, h: h + 1].contiguous(),
                                      k[:, :, h // (H // G)][:, :, None].contiguous(),
                                      v[:, :, h // (H // G)][:, :, None].contiguous(), o1, l1, causal, D ** -0.5, none, none, none)
        want[:, :, h // (H // G)] += d1[2][:, :, 0].float()
    _near(grads[2], want, "dv")


def test_padded_rows_with_shared_heads():
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(2, 512, 8, 2, 128)
    lens = [512, 333]
    for t in (q, k, v):
        t.requires_grad_()
    out = flash_attention(q, k, v, causal=True, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    got = (out, *torch.autograd.grad(out, (q, k, v), dout))
    for b, n in enumerate(lens):
        want = _reference(*(t[b: b + 1, :n].detach() for t in (q, k, v, dout)), True, 128 ** -0.5)
        for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
            _near(a[b: b + 1, :n], w, name)
            assert (a[b, n:] == 0).all(), name


@pytest.mark.parametrize("lens,H,G,D", [([512, 1, 0, 300], 4, 2, 128), ([700], 8, 2, 64), ([64, 128, 129, 31], 2, 2, 64),
                                        ([300 - 7 * i for i in range(40)], 8, 2, 128)])  # the last by tile
def test_packed(lens, H, G, D):
    from colossalai_amd.ops import flash_attention_varlen

    total = sum(lens)
    q, k, v, dout = (t[0] for t in _inputs(1, total, H, G, D))
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    for t in (q, k, v):
        t.requires_grad_()
    out = flash_attention_varlen(q, k, v, cu, max(lens), causal=True)
    got = (out, *torch.autograd.grad(out, (q, k, v), dout))
    at = 0
    for n in lens:
        if n:
            want = _reference(*(t[None, at: at + n].detach() for t in (q, k, v, dout)), True, D ** -0.5)
            for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
                _near(a[None, at: at + n], w, name, lone=n == 1)
        at += n


@pytest.mark.parametrize("causal", [True, False])
def test_a_scale_of_nan_shows(causal):
    from colossalai_amd.ops import flash_attention

    q, k, v, _ = _inputs(1, 70, 2, 1, 64)
    assert torch.isnan(flash_attention(q, k, v, causal=causal, scale=float("nan")).float()).all()


def test_packed_backward_with_very_many_sequences():
    """More blocks than one grid dimension holds threads for: many short sequences beside one that is long."""
    from colossalai_amd.ops import flash_attention_varlen

    lens = [1] * 65000
    lens[30000] = 32768
    total, D = sum(lens), 64
    q, k, v, dout = (t[0] for t in _inputs(1, total, 1, 1, D))
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    for t in (q, k, v):
        t.requires_grad_()
    out = flash_attention_varlen(q, k, v, cu, max(lens), causal=True)
    got = torch.autograd.grad(out, (q, k, v), dout)
    # the long one by itself, through a batch of one
    one = slice(30000, 30000 + 32768)
    alone = [t[one].detach().requires_grad_() for t in (q, k, v)]
    out1 = flash_attention_varlen(*alone, torch.tensor([0, 32768], dtype=torch.int32, device="cuda"), 32768, causal=True)
    for name, a, w in zip(("dq", "dk", "dv"), got, torch.autograd.grad(out1, alone, dout[one])):
        _near(a[one], w, name)
    # a token that sees itself only: its value's gradient is dout
    short = torch.ones(total, dtype=torch.bool, device="cuda")
    short[one] = False
    assert torch.equal(got[2][short], dout[short])


def test_strided_gradients_with_shared_heads():
    """dk/dv as views into one packed buffer, filled by the kernel that adds the partial sums."""
    from colossalai_amd.ops import kernels

    B, S, H, G, D = 1, 512, 8, 2, 64
    q, k, v, dout = _inputs(B, S, H, G, D)
    want = _reference(q, k, v, dout, True, D ** -0.5)
    packed = torch.full((B, S, (H + 2 * G) * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    dq = packed[:, :, : H * D].view(B, S, H, D)
    dk = packed[:, :, H * D: (H + G) * D].view(B, S, G, D)
    dv = packed[:, :, (H + G) * D:].view(B, S, G, D)
    out, lse = kernels().flash_attn_fwd(q, k, v, True, D ** -0.5)
    kernels().flash_attn_bwd(dout, q, k, v, out, lse, True, D ** -0.5, dq, dk, dv)
    for name, a, b in zip(("out", "dq", "dk", "dv"), (out, dq, dk, dv), want):
        _near(a, b, name)


@pytest.mark.parametrize("S", [31, 32, 33, 63, 64, 65, 95, 96, 97, 159, 160, 161, 223, 225, 257])
@pytest.mark.parametrize("D,causal", [(64, True), (128, True), (128, False)])
def test_where_steps_without_a_mask_end(S, D, causal):
    """Steps of 64 keys do not look for a mask until the diagonal or the end of the keys is near: odd halves on either side of it,
    with whole sequences and with padded ones."""
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(2, S, 2, 1, D, S)
    lens = [S, S - 17]
    for padded in (False, True):
        a = [t.clone().requires_grad_() for t in (q, k, v)]
        o = flash_attention(*a, causal=causal, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda") if padded else None)
        got = [o] + list(torch.autograd.grad(o, a, dout))
        for b, n in enumerate(lens if padded else [S, S]):
            one = [t[b: b + 1, :n] for t in (q, k, v, dout)]
            for name, x, y in zip(("out", "dq", "dk", "dv"), got, _reference(*one, causal, D ** -0.5)):
                _near(x[b: b + 1, :n], y, f"{name} {padded} {b}")


@pytest.mark.parametrize("B,S,H,G", [(1, 700, 12, 12), (3, 300, 5, 5), (2, 1100, 7, 1), (1, 130, 20, 4), (1, 3000, 6, 2), (5, 257, 16, 16)])
def test_rows_dealt_to_the_chips_parts(B, S, H, G):
    """Causal rows, of numbers that eight parts of the chip share evenly or not, several side by side; remainders of either."""
    q, k, v, dout = _inputs(B, S, H, G, 64, S)
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    from colossalai_amd.ops import flash_attention

    o = flash_attention(*a, causal=True)
    for name, x, y in zip(("out", "dq", "dk", "dv"), [o] + list(torch.autograd.grad(o, a, dout)), _reference(q, k, v, dout, True, 0.125)):
        _near(x, y, name)


def _launches(call, tmp_path):
    """Template arguments and grids of the attention kernels that a call runs, and what it returns."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        out = call()
        torch.cuda.synchronize()
    seen.export_chrome_trace(str(tmp_path / "trace.json"))
    with open(tmp_path / "trace.json") as f:
        kernels = [e for e in json.load(f)["traceEvents"] if e.get("cat") == "kernel"]
    found = {k: [e for e in kernels if k in e["name"]] for k in ("fa_fwd_kernel", "fa_bwd_kernel")}
    return {k: (e[0]["name"].split("<")[1].split(">")[0].replace(" ", ""), e[0]["args"]["grid"]) for k, e in found.items() if e}, out


# more than 256 blocks of four waves, and from 513 on not all at once; rows a multiple of 8, of 4 and of 2, and odd ones: an XCD has whole ones, every
# second, fourth or eighth tile. In the last but one an XCD's rows are more than it would take together.
@pytest.mark.parametrize("B,S,H,G,D", [(2, 1100, 16, 4, 64), (1, 2900, 12, 12, 64), (1, 3600, 10, 5, 128), (1, 4100, 9, 3, 64),
                                       (4, 620, 32, 8, 128), (1, 3000, 28, 4, 64), (1, 4700, 14, 2, 64), (2, 4500, 5, 5, 128), (1, 4200, 17, 17, 64)])
@pytest.mark.parametrize("padded", [False, True])
def test_forward_rows_dealt_to_the_chips_parts(B, S, H, G, D, padded, tmp_path):
    """Causal batches beyond 256 blocks whose rows have tiles enough: the forward deals them too; padded ones go key head by key head."""
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(B, S, H, G, D, S)
    lens = [S - (S // 3 + 5) * ((b + 1) % 3) for b in range(B)] if padded else [S] * B
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    seen, o = _launches(lambda: flash_attention(*a, causal=True, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda") if padded else None), tmp_path)
    assert seen["fa_fwd_kernel"][0] == f"{D},4,false,true"
    got = [o] + list(torch.autograd.grad(o, a, dout))
    for b, n in enumerate(lens):
        for name, x, y in zip(("out", "dq", "dk", "dv"), got, _reference(*(t[b: b + 1, :n] for t in (q, k, v, dout)), True, D ** -0.5)):
            _near(x[b: b + 1, :n], y, f"{name} {b}")
            assert not x[b, n:].any()


@pytest.mark.parametrize("B,S,H,D,forward,backward", [
    (64, 100, 6, 64, False, False), (60, 200, 4, 64, False, True), (8, 384, 16, 128, True, True), (26, 300, 8, 64, False, True),   # one tile, two, three
    (8, 400, 16, 64, True, True),                                                                                                   # four
    (11, 300, 9, 64, False, False), (7, 600, 10, 128, False, False), (3, 1000, 14, 64, False, False), (9, 500, 12, 64, False, False),   # an XCD has a part of a row
    (2, 1000, 18, 64, True, True),
])
def test_rows_of_few_tiles_stay_in_order(B, S, H, D, forward, backward, tmp_path):
    """Rows that several XCDs would share are dealt if each gets four tiles of them or more, whole ones of four tiles or more (the backward's: of two),
    of three if all blocks run at once."""
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(B, S, H, H, D, S)
    a = [t.clone().requires_grad_() for t in (q, k, v)]

    def step():
        o = flash_attention(*a, causal=True)
        return [o] + list(torch.autograd.grad(o, a, dout))

    seen, got = _launches(step, tmp_path)
    tiles, rows = (S + 127) // 128, B * H
    parts = next(n for n in (1, 2, 4, 8) if rows * n % 8 == 0)
    assert tiles * rows > 256
    assert seen["fa_fwd_kernel"][0] == f"{D},4,false,{str(forward).lower()}"
    in_order = (tiles * rows + 7) // 8 * 8 + tiles * rows
    assert seen["fa_bwd_kernel"][1][0] == (2 * -(-tiles // parts) * parts * rows if backward else in_order)
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, _reference(q, k, v, dout, True, D ** -0.5)):
        _near(x, y, name)


@pytest.mark.parametrize("S", [100, 200, 300])
@pytest.mark.parametrize("H,G,causal", [(6, 6, False), (8, 2, True)])
def test_padded_batches_of_few_tiles(S, H, G, causal):
    """One tile: sequence by sequence. Two: so in the forward. Three: key head by key head."""
    from colossalai_amd.ops import flash_attention

    B = 50
    q, k, v, dout = _inputs(B, S, H, G, 64, S)
    lens = [0 if b == 7 else max(20, S - 37 * b % (3 * S // 4)) for b in range(B)]
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    o = flash_attention(*a, causal=causal, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    got = [o] + list(torch.autograd.grad(o, a, dout))
    for b, n in enumerate(lens):
        assert not any(x[b, n:].any() for x in got)
        if n:
            for name, x, y in zip(("out", "dq", "dk", "dv"), got, _reference(*(t[b: b + 1, :n] for t in (q, k, v, dout)), causal, 0.125)):
                _near(x[b: b + 1, :n], y, f"{name} {b}")


@pytest.mark.parametrize("lens,H,G,D,looked_up", [
    ([150, 60] * 30, 16, 4, 64, False), ([150, 60] * 30, 32, 4, 128, False),                                                # two tiles
    ([400, 250, 130] * 10, 32, 8, 64, False), ([400, 250, 130] * 5, 16, 8, 128, False), ([400, 250, 130] * 10, 32, 4, 128, True),
    ([150, 60] * 30, 12, 12, 64, True), ([1100, 250] * 5, 16, 4, 64, True),                                                  # ungrouped heads; long sequences
])
def test_packed_forward_tile_by_tile(lens, H, G, D, looked_up, tmp_path):
    """Grouped heads over short sequences: the forward looks tiles up with 128 channels, more than two tiles and 1024 blocks."""
    from colossalai_amd.ops import flash_attention_varlen

    T = sum(lens)
    q, k, v, dout = (t[0] for t in _inputs(1, T, H, G, D, T))
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    seen, o = _launches(lambda: flash_attention_varlen(*a, cu, max(lens), causal=True), tmp_path)
    assert (seen["fa_fwd_kernel"][1][1] == 1) == looked_up   # a line of blocks, or one of tiles for each sequence and head
    got = [o] + list(torch.autograd.grad(o, a, dout))
    at = 0
    for n in lens:
        for name, x, y in zip(("out", "dq", "dk", "dv"), got, _reference(*(t[None, at: at + n] for t in (q, k, v, dout)), True, D ** -0.5)):
            _near(x[at: at + n], y[0], f"{name} {n}")
        at += n


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("H,G,D", [(16, 16, 64), (18, 2, 64), (16, 4, 128), (20, 20, 128)])
def test_packed_tiles_by_lookup_at_their_edges(H, G, D, causal):
    """Equal lengths, an empty sequence ahead, between and behind, tiles that are just full and one row more."""
    from colossalai_amd.ops import flash_attention_varlen

    lens = [0, 900, 21, 0, 900, 129, 1500, 128, 640, 0]
    T = sum(lens)
    assert min(T // 128 + len(lens), 12 * len(lens)) * H > 512   # tiles by their bound and heads: beyond 512 blocks they are looked up
    q, k, v, dout = (t[0] for t in _inputs(1, T, H, G, D, T))
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    o = flash_attention_varlen(*a, torch.tensor([0] + lens).cumsum(0).int().cuda(), max(lens), causal=causal)
    got = [o] + list(torch.autograd.grad(o, a, dout))
    at = 0
    for n in lens:
        if n:
            want = _reference(*(t[None, at: at + n] for t in (q, k, v, dout)), causal, D ** -0.5)
            for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
                _near(x[at: at + n], y[0], f"{name} {n}")
        at += n


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lens,H,G", [
    ([900, 1, 0, 900, 129, 1500, 128, 640], 12, 12),               # equal lengths, an empty one, tiles that are just full
    ([5000], 16, 4), ([40, 300] * 32 + [1100], 6, 2),              # one; two a lane
    ([20] * 255 + [900], 9, 3), ([20] * 256 + [900], 9, 3),        # the most that are looked up, and one more
    ([300 + 37 * i for i in range(20)], 5, 5),
])
def test_packed_tiles_by_lookup(lens, H, G, causal):
    """Packed batches of more blocks than run at once: their blocks look their tiles up, longest sequences first."""
    from colossalai_amd.ops import flash_attention_varlen

    T, D = sum(lens), 64
    q, k, v, dout = (t[0] for t in _inputs(1, T, H, G, D, T))
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    o = flash_attention_varlen(*a, cu, max(lens), causal=causal)
    got = [o] + list(torch.autograd.grad(o, a, dout))
    want = [torch.zeros_like(t, dtype=torch.float32) for t in (q, q, k, v)]
    at = 0
    for n in lens:
        if n:
            for w, r in zip(want, _reference(*(t[None, at: at + n] for t in (q, k, v, dout)), causal, D ** -0.5)):
                w[at: at + n] = r[0]
        at += n
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
        _near(x, y, name)


@pytest.mark.parametrize("causal", [True, False])
# at least 20 keys: of two, a row's dq is one difference of dout · v and dout · out, whose roundings (2^-9 of about sqrt(D) each) are not small beside it
@pytest.mark.parametrize("S,H,G", [(20, 2, 2), (63, 4, 1), (64, 4, 1), (65, 4, 1), (255, 3, 3), (256, 2, 2), (257, 2, 2)])
def test_statistics_of_few_rows(S, H, G, causal):
    """64 channels, up to 8 tiles of 32 query rows a block: the backward's blocks form -lse and -delta themselves. Padded sequences too, one of them empty."""
    from colossalai_amd.ops import flash_attention

    q, k, v, dout = _inputs(3, S, H, G, 64, S)
    lens = [S, max(20, S - 40), 0]
    a = [t.clone().requires_grad_() for t in (q, k, v)]
    o = flash_attention(*a, causal=causal, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    got = [o] + list(torch.autograd.grad(o, a, dout))
    for b, n in enumerate(lens):
        for x in got:
            assert not x[b, n:].any()
        if n:
            want = _reference(*(t[b: b + 1, :n] for t in (q, k, v, dout)), causal, 0.125)
            for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
                _near(x[b: b + 1, :n], y, name)


@pytest.mark.parametrize("H", [31, 32, 33])
@pytest.mark.parametrize("D,causal", [(64, True), (128, False)])
@pytest.mark.parametrize("packed", [False, True])
def test_on_either_side_of_blocks_of_two_waves(H, D, causal, packed):
    """Four tiles of 128 rows a head: up to 128 blocks of four waves they are cut into blocks of two."""
    from colossalai_amd.ops import flash_attention, flash_attention_varlen

    q, k, v, dout = _inputs(1, 500, H, H, D)
    want = _reference(q, k, v, dout, causal, D ** -0.5)[0]
    if packed:
        cu = torch.tensor([0, 500], dtype=torch.int32, device="cuda")
        got = flash_attention_varlen(q[0], k[0], v[0], cu, 500, causal=causal)[None]
    else:
        got = flash_attention(q, k, v, causal=causal)
    _near(got, want, "out")


@pytest.mark.parametrize("levels", [
    (0, 9, 18, 27, 36, 45),          # every tile's weights pass the reference of the one before
    (0, 5, 10, 15, 20, 25),          # every second one's do
    (60, 40, 20, 0, -20, -40),       # the first tile has the largest scores
    (-3000, 0, -3000, 4, 8, 1000),   # far below, far above
])
@pytest.mark.parametrize("D,causal", [(128, False), (64, False), (128, True)])
def test_scores_that_rise_and_fall(levels, D, causal):
    """Scores of a level of their own (in nats) in each key tile of 64: the reference that the forward takes a row's weights
    against is left behind, raised, or stays."""
    from colossalai_amd.ops import flash_attention

    S = 64 * len(levels)
    q, k, v, dout = _inputs(1, S, 4, 2, D)
    scale = D ** -0.5
    q[..., 0] = 8.0
    k[..., 0] = torch.tensor(levels, device="cuda").repeat_interleave(64)[None, :, None] / (8.0 * scale)
    want = _reference(q, k, v, dout, causal, scale)
    for t in (q, k, v):
        t.requires_grad_()
    out = flash_attention(q, k, v, causal=causal)
    got = (out, *torch.autograd.grad(out, (q, k, v), dout))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        # dq and dk: not channel 0, whose partner is as large as a level, nor rows of a single key under a mask
        if name in ("dq", "dk"):
            if causal:
                continue
            a, b = a[..., 1:], b[..., 1:]
        _near(a, b, name)


# Levels of 32 keys: every half tile, every odd one, every even one passes the reference of those before it, or the first has the largest scores.
LEVELS_32 = [(0, 9, 18, 27, 36, 45, 54, 63), (0, 25, 50, 75, 100, 125), (0, 14, 14, 28, 28, 42, 42, 56), (0, 0, 14, 14, 28, 28, 42), (63, 45, 54, 36, 27, 0, 9)]


@pytest.mark.parametrize("levels", LEVELS_32)
@pytest.mark.parametrize("S", [None, 160, 200])
@pytest.mark.parametrize("D,causal", [(128, False), (64, False), (128, True)])
def test_half_tiles_that_rise(levels, S, D, causal):
    """The reference is raised after either half of a tile, while the weights of the half before it are on their way to the values."""
    from colossalai_amd.ops import flash_attention

    S = S or 32 * len(levels)
    q, k, v, dout = _inputs(1, S, 4, 2, D)
    q[..., 0] = 8.0
    level = torch.tensor(levels, device="cuda").repeat_interleave(32)[:S]
    k[..., 0] = torch.nn.functional.pad(level, (0, max(0, S - len(level))))[None, :, None] / (8.0 * D ** -0.5)
    _near(flash_attention(q, k, v, causal=causal), _reference(q, k, v, dout, causal, D ** -0.5)[0], "out")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("packed", [False, True])
def test_large_values_of_rising_scores(D, packed):
    """Values of about 2^104: a weight is taken again before it passes 2^12, so that its product stays below 2^128."""
    from colossalai_amd.ops import flash_attention, flash_attention_varlen

    S = 192
    q, k, v, dout = _inputs(1, S, 4, 2, D)
    q[..., 0] = 8.0
    k[:, :, :, 0] = torch.where(torch.arange(S, device="cuda") < 64, 0.0, 16.0)[None, :, None] / (8.0 * D ** -0.5)
    v = v * 2.0 ** 104
    want = _reference(q, k, v, dout, packed, D ** -0.5)[0]
    if packed:
        cu = torch.tensor([0, S], dtype=torch.int32, device="cuda")
        got = flash_attention_varlen(q[0], k[0], v[0], cu, S, causal=True)[None]
    else:
        got = flash_attention(q, k, v, causal=False)
    _near(got, want, "out")


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("D,causal", [(128, False), (64, False), (64, True)])
def test_rows_past_a_padded_sequence_may_hold_anything(bad, D, causal):
    """Ends in the first and in the second half of a tile and of a wave's rows; the rows past them are 0, and so are their gradients."""
    from colossalai_amd.ops import flash_attention

    lens = [130, 1, 33, 64, 95, 160, 97]
    q, k, v, dout = _inputs(len(lens), 160, 4, 2, D)
    past = torch.arange(160, device="cuda") >= torch.tensor(lens, device="cuda")[:, None]
    want = [torch.zeros_like(t, dtype=torch.float32) for t in (q, q, k, v)]
    for b, n in enumerate(lens):
        for t, r in zip(want, _reference(*[t[b: b + 1, :n] for t in (q, k, v, dout)], causal, D ** -0.5)):
            t[b, :n] = r[0]
    q, k, v = (t.masked_fill(past[..., None, None], bad).requires_grad_() for t in (q, k, v))
    out = flash_attention(q, k, v, causal=causal, seqlens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    got = (out, *torch.autograd.grad(out, (q, k, v), dout))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        _near(a, b, name)
        assert not a[past].any(), name


@pytest.mark.parametrize("place", ["odd address", "odd rows", "far rows", "one row for all"])
@pytest.mark.parametrize("packed", [False, True])
def test_inputs_that_tiles_cannot_be_loaded_from_as_they_lie(place, packed):
    from colossalai_amd.ops import flash_attention, flash_attention_varlen

    S, D = 150, 64
    q, k, v, dout = _inputs(1, S, 4, 2, D, seed=3)

    def lay(t):
        n = t.shape[2] * D
        if place == "odd address":
            return torch.empty(S * n + 1, device="cuda", dtype=t.dtype)[1:].view(t.shape).copy_(t)
        if place == "one row for all":
            return t[:, :1].expand(t.shape)
        step = n + 1 if place == "odd rows" else 1 << 23
        room = torch.empty((S - 1) * step + n, device="cuda", dtype=t.dtype)
        return room.as_strided(t.shape, (0, step, D, 1)).copy_(t)

    laid = [lay(t).detach().requires_grad_() for t in (q, k, v)]
    d = lay(dout) if place == "odd address" else dout
    want = _reference(*[t.detach() for t in laid], d, True, D ** -0.5)
    if packed:
        cu = torch.tensor([0, S], dtype=torch.int32, device="cuda")
        out = flash_attention_varlen(*[t[0] for t in laid], cu, S, causal=True)[None]
    else:
        out = flash_attention(*laid, causal=True)
    got = (out, *torch.autograd.grad(out, laid, d))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        if place == "one row for all" and name in ("dq", "dk"):
            # equal keys and values: dP - delta vanishes but for the output's rounding, 2^-9 of dout · v (4 sqrt(D) at most here),
            # times the scale, a key or query channel (4 at most), and for dk the sum of a key's weights (ln S + 1 at most)
            assert a.float().abs().max() < 2.0 ** -9 * 4 * 4 * (6 if name == "dk" else 1)
        else:
            _near(a, b, name)


def test_a_score_of_nan_is_not_lost():
    """The forward looks at a tile's sum to see whether its reference must be raised; NaN makes the rows that meet it NaN."""
    from colossalai_amd.ops import flash_attention

    q, k, v, _ = _inputs(1, 300, 4, 2, 64)
    k[0, 200, 1, 5] = float("nan")     # key head 1, seen from row 200 on
    q[0, 100, 0, 3] = float("nan")
    bad = flash_attention(q, k, v, causal=True)[0].isnan()
    want = torch.zeros_like(bad)
    want[200:, 2:] = True
    want[100, 0] = True
    assert torch.equal(bad, want)
