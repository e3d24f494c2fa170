"""The work whose speed this framework is judged by: what its users run most, through its public entry points.

Three kinds of program use the framework, and each has cases here:

* training a decoder (``LlamaForCausalLM``): one forward and backward pass over a batch, as the training loop of
  ``bench.py`` runs it ("step");
* attention by itself (``flash_attention``, ``flash_attention_varlen``), forward and backward, which the other model
  families call with shapes of their own: grouped heads over long sequences, packed fine-tuning samples, right-padded
  bidirectional batches, image patches ("dense", "packed");
* serving over paged keys: the attention of a ragged step (``paged_attention``: prompt portions, decode tokens or both)
  and a whole prompt through the continuous-batching engine ("paged", "prompt").

Everything is bfloat16 with float32 statistics, which is what training and serving run in.
"""

import math

import torch
from torch.utils.checkpoint import checkpoint

from colossalai_amd.inference.config import InferenceConfig
from colossalai_amd.inference.paged_engine import ContinuousBatchEngine
from colossalai_amd.models import BekulixForCausalLM, LlamaConfig, LlamaForCausalLM
from colossalai_amd.ops import flash_attention, flash_attention_varlen
from colossalai_amd.ops.paged_attention import distance_slopes, paged_attention
from colossalai_amd.ops.ragged import RaggedBatch

BF16, F64 = torch.bfloat16, torch.float64


def listed():
    return [
        # the smallest training step there is (the package's own smoke check): launches and latency
        dict(name="step_small", kind="step", layers=2, width=512, inner=1024, heads=4, kv_heads=4, vocab=1024, batch=2, seq=256),
        # a third of the 100M-parameter decoder: head size 64, a vocabulary that is large beside the width
        dict(name="step_100m", kind="step", layers=4, width=768, inner=2048, heads=12, kv_heads=12, vocab=32000, batch=8, seq=1024),
        # two layers of the 7B decoder at the headline sequence length
        dict(name="step_7b", kind="step", layers=2, width=4096, inner=11008, heads=32, kv_heads=32, vocab=32000, batch=4, seq=4096),
        # one long sequence with grouped heads (the 8B decoder's heads at its full context)
        dict(name="attn_long", kind="dense", batch=1, seq=8192, heads=32, kv_heads=8, dim=128, causal=True, padded=False),
        # packed fine-tuning samples of many lengths
        dict(name="attn_packed", kind="packed", tokens=16384, longest=4096, heads=32, kv_heads=8, dim=128),
        # a bidirectional encoder's batch, right-padded
        dict(name="attn_encoder", kind="dense", batch=16, seq=512, heads=12, kv_heads=12, dim=64, causal=False, padded=True),
        # image patches and a class token: an odd, short sequence
        dict(name="attn_patches", kind="dense", batch=8, seq=197, heads=12, kv_heads=12, dim=64, causal=False, padded=False),
        # one 4096-token prompt of a model with capped scores and a sink
        dict(name="prefill_4k", kind="paged", seqs=1, decode=0, new=4096, cached=0, heads=16, kv_heads=4, dim=128, page=64,
             window=0, softcap=30.0, sink=True),
        # a mixed step: chunks of two prompts beside 14 decode tokens, sliding window with kept first keys
        dict(name="mixed_window", kind="paged", seqs=16, decode=14, new=1000, cached=2100, heads=16, kv_heads=4, dim=128,
             page=16, window=1024, softcap=0.0, sink=False),
        # a decode step of 16 sequences
        dict(name="decode_1k", kind="paged", seqs=16, decode=16, new=0, cached=1024, heads=16, kv_heads=4, dim=128, page=64,
             window=0, softcap=30.0, sink=True),
        # a decode step of a few long sequences
        dict(name="decode_16k", kind="paged", seqs=4, decode=4, new=0, cached=16384, heads=16, kv_heads=4, dim=128, page=64,
             window=0, softcap=0.0, sink=False),
        # a whole prompt through the engine: three kinds of attention, residual streams, gated feed-forward
        dict(name="prompt_engine", kind="prompt", width=2048, layers=6, heads=16, kv_heads=4, dim=128, vocab=32000, new=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "dense", "dense", "packed", "paged", "paged", "paged", "prompt"])
    if kind == "step":
        dim, heads = rng.choice([64, 128]), rng.choice([4, 8, 12, 16, 32])
        width = dim * heads
        seq = _log_int(rng, 128, 4096)
        return dict(kind=kind, layers=2, width=width, inner=max(256, 8 * width // 3 // 256 * 256), heads=heads,
                    kv_heads=heads // rng.choice([1, 1, 2, 4]), vocab=rng.choice([1024, 8000, 32000]),
                    batch=max(1, _log_int(rng, 512, 16384) // seq), seq=seq)
    if kind in ("dense", "packed"):
        dim = rng.choice([64, 128])
        kv = rng.choice([1, 2, 4, 8, 12])
        heads = kv * rng.choice([1, 1, 2, 2 if kv > 8 else 4]) if kv > 1 else rng.choice([4, 8])
        if kind == "packed":
            return dict(kind=kind, tokens=_log_int(rng, 1024, 16384), longest=_log_int(rng, 128, 4096), heads=heads,
                        kv_heads=kv, dim=dim)
        seq = _log_int(rng, 128, 8192)
        return dict(kind=kind, batch=max(1, _log_int(rng, 512, 16384) // seq), seq=seq, heads=heads, kv_heads=kv,
                    dim=dim, causal=rng.random() < 0.6, padded=rng.random() < 0.4)
    if kind == "paged":
        kv = rng.choice([2, 4, 8])
        seqs = rng.randint(1, 16)
        decode = rng.choice([0, seqs, rng.randint(0, seqs)])
        portions = seqs - decode
        new = _log_int(rng, 64, 4096 // max(portions, 1)) if portions else 0
        window = rng.choice([0, 0, 512, 1024])
        cap = rng.random() < 0.4
        return dict(kind=kind, seqs=seqs, decode=decode, new=new, cached=_log_int(rng, 128, 8192 if portions == 0 else 2048),
                    heads=kv * rng.choice([2, 4]), kv_heads=kv, dim=rng.choice([64, 128]), page=rng.choice([16, 64]),
                    window=window, softcap=30.0 if cap else 0.0, sink=cap)
    return dict(kind=kind, width=rng.choice([1024, 2048]), layers=rng.choice([3, 6]), heads=16, kv_heads=4, dim=128,
                vocab=32000, new=_log_int(rng, 256, 4096))


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(1000003 * seed + 17)


def _lengths(case, seed):
    """Sample lengths of a packed or padded batch: between a sixteenth of the longest and the longest, one of them the
    longest."""
    g = _gen(seed, "cpu")
    if case["kind"] == "packed":
        left, out = case["tokens"], []
        while left > 0:
            u = torch.rand((), generator=g).item() if out else 1.0
            out.append(min(left, max(1, int(case["longest"] * 16 ** (u - 1)))))
            left -= out[-1]
        return out
    u = torch.rand(case["batch"], generator=g)
    out = [max(1, int(case["seq"] * (0.25 + 0.75 * float(x)))) for x in u]
    out[0] = case["seq"]
    return out


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(BF16)


def _llama(case):
    return LlamaConfig(vocab_size=case["vocab"], hidden_size=case["width"], intermediate_size=case["inner"],
                       num_hidden_layers=case["layers"], num_attention_heads=case["heads"],
                       num_key_value_heads=case["kv_heads"], max_position_embeddings=max(4096, case["seq"]))


def _llama_step(case, seed):
    with torch.device("cuda"):
        model = LlamaForCausalLM(_llama(case)).to(BF16)
    g = _gen(seed)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.copy_(1.0 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
            else:
                p.copy_(torch.randn(p.shape, generator=g, device="cuda") * 0.02)
    tokens = torch.randint(0, case["vocab"], (case["batch"], case["seq"]), generator=g, device="cuda")
    return model.train(), tokens


def _paged_rows(case):
    """New tokens and cached tokens of every sequence of a step; context lengths spread by a quarter around the case's."""
    n = case["seqs"]
    new = [1 if i < case["decode"] else max(1, case["new"] - 37 * (i - case["decode"])) for i in range(n)]
    spread = [1.0 + 0.25 * (2 * i / (n - 1) - 1) if n > 1 else 1.0 for i in range(n)]
    return new, [int(case["cached"] * s) for s in spread]


def _paged(case, seed):
    g = _gen(seed)
    new, start = _paged_rows(case)
    H, G, D, ps = case["heads"], case["kv_heads"], case["dim"], case["page"]
    need = [(a + b + ps - 1) // ps for a, b in zip(new, start)]
    order = torch.randperm(sum(need), generator=_gen(seed, "cpu")).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(order[at: at + n])
        at += n
    kpool, vpool = _randn(g, sum(need), ps, G, D), _randn(g, sum(need), ps, G, D)
    q = _randn(g, sum(new), H, D, std=1.5)
    gate = _randn(g, sum(new), H) if case["window"] else None
    slopes = distance_slopes(H, "cuda") if case["window"] else None
    batch = RaggedBatch.build(new, start, list(range(len(new))), "cuda", tables, ps)
    return q, kpool, vpool, batch, gate, slopes


def _engine_config(case):
    """Layers in turn: attention over one cached row per token, differential attention in blocks, latent attention in a
    window."""
    H, G, D, W = case["heads"], case["kv_heads"], case["dim"], case["width"]
    att = dict(dim=D, heads=H, kv_heads=G, vdim=D, scale=D ** -0.5, q_temp=dict(coef=0.1, every=512))
    dif = dict(dim=D // 2, heads=H, kv_heads=G, vdim=D, scale=(D // 2) ** -0.5, diff=0.4, mask=dict(size=2048))
    lat = dict(dim=D, heads=H, vdim=D, kv_rank=2 * D, scale=D ** -0.5, mask=dict(size=1024))
    kinds = [("attention", att), ("attention_2", dif), ("latent_attention", lat)]
    ff = (8 * W // 3 + 255) // 256 * 256
    return dict(architecture="Bekulix", vocab=case["vocab"], width=W, norm=dict(eps=1e-6), streams=4,
                layers=[dict(type=kinds[i % 3][0], mixer=kinds[i % 3][1], mlp=dict(kind="dense", ff=ff))
                        for i in range(case["layers"])])


def _engine_tensors(case, seed):
    cfg, g, P = _engine_config(case), _gen(seed), {}
    W, n = cfg["width"], cfg["streams"]

    def mat(name, rows, cols):
        P[name] = _randn(g, rows, cols, std=cols ** -0.5)

    def vec(name, size, mean=0.0, std=0.1):
        P[name] = (mean + std * torch.randn(size, generator=g, device="cuda")).to(BF16)

    mat("embed", cfg["vocab"], W)
    mat("head", cfg["vocab"], W)
    vec("final.norm", W)
    for i, spec in enumerate(cfg["layers"]):
        p, a, c = "l%d." % i, "l%d.mix." % i, spec["mixer"]
        H, D = c["heads"], c["dim"]
        for name in ("1", "2"):
            vec(p + "norm" + name, W)
            vec(p + "hc%s.in" % name, n, 1.0 / n, 0.3 / n)
            vec(p + "hc%s.out" % name, n, 0.8, 0.3)
            P[p + "hc%s.mix" % name] = (0.8 * torch.eye(n, device="cuda")
                                        + 0.2 / n * torch.randn(n, n, generator=g, device="cuda")).to(BF16)
        if spec["type"] == "attention":
            mat(a + "q", H * D, W)
            mat(a + "k", c["kv_heads"] * D, W)
            vec(a + "q.norm", D, 1.3)
            vec(a + "k.norm", D, 0.9)
        elif spec["type"] == "latent_attention":
            mat(a + "q", H * D, W)
            mat(a + "dkv", c["kv_rank"], W)
            vec(a + "dkv.norm", c["kv_rank"], 1.0)
            mat(a + "uk", H * D, c["kv_rank"])
            mat(a + "uv", H * c["vdim"], c["kv_rank"])
        else:
            for name, rows in (("q", 2 * H * D), ("k", 2 * c["kv_heads"] * D), ("v", c["kv_heads"] * c["vdim"])):
                mat(a + name, rows, W)
                vec(a + name + ".b", rows, 0.0, 0.3)
            for name in ("lq1", "lk1", "lq2", "lk2"):
                vec(a + name, D, 0.0, 0.05)
        mat(a + "o", W, H * c["vdim"])
        mat(p + "mlp.gate", spec["mlp"]["ff"], W)
        mat(p + "mlp.up", spec["mlp"]["ff"], W)
        mat(p + "mlp.down", W, spec["mlp"]["ff"])
    return cfg, P


def _prompt(case, seed):
    return torch.randint(0, case["vocab"], (case["new"],), generator=_gen(seed, "cpu")).tolist()


def _qkv(case, seed):
    g, H, G, D = _gen(seed), case["heads"], case["kv_heads"], case["dim"]
    lead = (case["tokens"],) if case["kind"] == "packed" else (case["batch"], case["seq"])
    return [_randn(g, *lead, h, D) for h in (H, G, G, H)]


def prepare(case, seed):
    if case["kind"] == "step":
        model, tokens = _llama_step(case, seed)
        return dict(case=case, model=model, tokens=tokens)
    if case["kind"] in ("dense", "packed"):
        q, k, v, dout = _qkv(case, seed)
        s = dict(case=case, q=q.requires_grad_(), k=k.requires_grad_(), v=v.requires_grad_(), dout=dout, lens=None)
        if case["kind"] == "packed":
            lens = _lengths(case, seed)
            s.update(cu=torch.tensor([0] + lens).cumsum(0).int().cuda(), longest=max(lens))
        elif case["padded"]:
            s.update(lens=torch.tensor(_lengths(case, seed), dtype=torch.int32, device="cuda"))
        return s
    if case["kind"] == "paged":
        q, kpool, vpool, batch, gate, slopes = _paged(case, seed)
        return dict(case=case, q=q, k=kpool, v=vpool, batch=batch, gate=gate, slopes=slopes)
    cfg, tensors = _engine_tensors(case, seed)
    with torch.device("cuda"):
        model = BekulixForCausalLM.from_checkpoint(cfg, tensors, dtype=BF16, device="cuda")
    engine = ContinuousBatchEngine(model, InferenceConfig(max_batch_size=1), num_blocks=case["new"] // 64 + 1, block_size=64)
    return dict(case=case, engine=engine, prompt=_prompt(case, seed))


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        model = state["model"]
        model.zero_grad(set_to_none=True)
        loss = model(state["tokens"], labels=state["tokens"])["loss"]
        loss.backward()
        return dict({name: p.grad for name, p in model.named_parameters()}, loss=loss.detach())
    if case["kind"] in ("dense", "packed"):
        q, k, v = state["q"], state["k"], state["v"]
        if case["kind"] == "packed":
            out = flash_attention_varlen(q, k, v, state["cu"], state["longest"], causal=True)
        else:
            out = flash_attention(q, k, v, causal=case["causal"], seqlens=state["lens"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return dict(out=out.detach(), dq=dq, dk=dk, dv=dv)
    if case["kind"] == "paged":
        return paged_attention(state["q"], state["k"], state["v"], state["batch"], case["dim"] ** -0.5, case["window"],
                               4 if case["window"] else 0, state["slopes"], state["gate"], case["softcap"], case["sink"])
    engine, prompt = state["engine"], state["prompt"]
    logits = engine.run_ragged([("p", prompt, [len(prompt) - 1])])
    engine.close_sequence("p")
    return logits


# ------------------------------------------------------------------------------------------------ work
def _pairs(n, start=0, window=0, kept=0):
    """Visible (query, key) pairs of n new causal tokens after ``start`` cached ones."""
    if window == 0:
        return n * start + n * (n + 1) // 2
    return sum(min(p + 1, window) + min(kept, max(0, p + 1 - window)) for p in range(start, start + n))


def work(case):
    if case["kind"] == "step":
        W, F, V, T = case["width"], case["inner"], case["vocab"], case["batch"] * case["seq"]
        D = W // case["heads"]
        matrices = case["layers"] * (W * D * (case["heads"] + 2 * case["kv_heads"]) + W * W + 3 * W * F) + V * W
        pairs = case["batch"] * case["layers"] * case["heads"] * _pairs(case["seq"])
        return dict(flops=6 * matrices * T + 14 * D * pairs, bytes=2 * 2 * (matrices + V * W) + 8 * T)
    if case["kind"] in ("dense", "packed"):
        H, G, D = case["heads"], case["kv_heads"], case["dim"]
        if case["kind"] == "packed":
            T, lens, causal = case["tokens"], _lengths(case, 1), True
        else:
            T, causal = case["batch"] * case["seq"], case["causal"]
            lens = _lengths(case, 1) if case["padded"] else [case["seq"]] * case["batch"]
        pairs = H * sum(_pairs(n) if causal else n * n for n in lens)
        return dict(flops=14 * D * pairs, bytes=2 * T * D * (4 * H + 4 * G))
    if case["kind"] == "paged":
        new, start = _paged_rows(case)
        H, G, D = case["heads"], case["kv_heads"], case["dim"]
        kept = 4 if case["window"] else 0
        keys = sum(min(a + b, case["window"] + a + kept) if case["window"] else a + b for a, b in zip(new, start))
        pairs = sum(_pairs(a, b, case["window"], kept) for a, b in zip(new, start))
        return dict(flops=4 * D * H * pairs, bytes=4 * keys * G * D + 4 * sum(new) * H * D)
    W, N, H, G, D = case["width"], case["new"], case["heads"], case["kv_heads"], case["dim"]
    matrices = flops = 0
    for spec in _engine_config(case)["layers"]:
        c, m = spec["mixer"], 3 * W * spec["mlp"]["ff"] + W * H * D
        if spec["type"] == "attention":
            m += W * D * (H + G)
            flops += 4 * D * H * _pairs(N)
        elif spec["type"] == "latent_attention":
            m += W * (H * D + c["kv_rank"]) + 2 * H * D * c["kv_rank"]
            flops += 4 * D * H * _pairs(N, 0, 1024)
        else:
            m += W * D * (H + 2 * G)
            flops += (2 * D + 4 * D) * H * (N // 2048 * _pairs(2048) + _pairs(N % 2048))
        matrices += m
    return dict(flops=flops + 2 * matrices * N + 2 * case["vocab"] * W, bytes=2 * (matrices + case["vocab"] * W) + 2 * N * W)


def tolerance(case):
    # about four times the largest relative error against 64 bits that was seen: weight gradients of a step 0.018, attention
    # and its gradients 0.0025, paged attention 0.0017, logits after all layers 0.015
    if case["kind"] == "step":
        return {"rel": 0.08}
    if case["kind"] in ("dense", "packed"):
        return {"rel": 0.01}
    if case["kind"] == "paged":
        return {"rel": 0.007}
    return {"rel": 0.06}


# ------------------------------------------------------------------------------------------------ 64 bits
def _visible(n, m, start, causal, window=0, kept=0, chunk=0):
    i = torch.arange(start, start + n, device="cuda")[:, None]
    j = torch.arange(m, device="cuda")[None, :]
    if not causal:
        return (j >= 0).expand(n, m)
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < kept))
    if chunk:
        seen = seen & (j >= i - i % chunk)
    return seen


def _head(q, k, v, scale, seen, softcap=0.0, sink=False, slope=None, start=0):
    """One head in 64 bits: q [n, D], k [m, D], v [m, Dv] -> [n, Dv]."""
    s = (q @ k.t()) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    if slope is not None:
        n, m = s.shape
        s = s - slope * (torch.arange(start, start + n, device="cuda")[:, None] - torch.arange(m, device="cuda")).to(F64)
    s = s.masked_fill(~seen, float("-inf"))
    if sink:
        s = torch.cat([s, torch.zeros_like(s[:, :1])], 1)
    return torch.softmax(s, 1)[:, : k.shape[0]] @ v


def _exact_attention(case, seed):
    q, k, v, dout = (t.to(F64) for t in _qkv(case, seed))
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    got = [torch.zeros_like(t) for t in (q, q, k, v)]
    if case["kind"] == "packed":
        spans, at = [], 0
        for n in _lengths(case, seed):
            spans.append((slice(at, at + n),))
            at += n
        causal = True
    else:
        lens = _lengths(case, seed) if case["padded"] else [case["seq"]] * case["batch"]
        spans, causal = [(b, slice(0, n)) for b, n in enumerate(lens)], case["causal"]
    for span in spans:
        n = span[-1].stop - span[-1].start
        seen = _visible(n, n, 0, causal)
        for h in range(H):
            at, kat = span + (h,), span + (h // (H // G),)
            qh, kh, vh, dh = q[at], k[kat], v[kat], dout[at]
            p = torch.softmax((qh @ kh.t() * D ** -0.5).masked_fill(~seen, float("-inf")), 1)
            out = p @ vh
            ds = p * (dh @ vh.t() - (dh * out).sum(1, keepdim=True)) * D ** -0.5
            got[0][at] = out
            got[1][at] = ds @ kh
            got[2][kat] += ds.t() @ qh
            got[3][kat] += p.t() @ dh
    return dict(out=got[0], dq=got[1], dk=got[2], dv=got[3])


def _exact_step(case, seed):
    model, tokens = _llama_step(case, seed)
    cfg = model.config
    P = {name: p.detach().to(F64).requires_grad_() for name, p in model.named_parameters()}
    H, G, D, half = case["heads"], case["kv_heads"], cfg.head_dim, cfg.head_dim // 2
    B, S = tokens.shape
    freq = cfg.rope_theta ** (-torch.arange(0, D, 2, dtype=F64, device="cuda") / D)
    angle = torch.arange(S, dtype=F64, device="cuda")[:, None] * freq
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    seen = _visible(S, S, 0, True)

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + cfg.rms_norm_eps) * w

    def turn(x):
        lo, hi = x[..., :half], x[..., half:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)

    def mix(y):  # [S, (H + 2G) D] of one sequence
        q, k, v = turn(y[:, : H * D].view(S, H, D)), turn(y[:, H * D: (H + G) * D].view(S, G, D)), y[:, (H + G) * D:].view(S, G, D)
        heads = [checkpoint(_head, q[:, h], k[:, h // (H // G)], v[:, h // (H // G)], D ** -0.5, seen, use_reentrant=False)
                 for h in range(H)]
        return torch.cat(heads, 1)

    def layer(x, p):
        y = norm(x, P[p + "input_layernorm_weight"]) @ P[p + "self_attn.qkv_proj.weight"].t()
        x = x + torch.stack([mix(r) for r in y]) @ P[p + "self_attn.o_proj.weight"].t()
        gu = norm(x, P[p + "post_attention_layernorm_weight"]) @ P[p + "mlp.gate_up_proj.weight"].t()
        gate, up = gu.chunk(2, -1)
        return x + (torch.nn.functional.silu(gate) * up) @ P[p + "mlp.down_proj.weight"].t()

    def nll(x, y):
        return torch.nn.functional.cross_entropy(x @ P["lm_head.weight"].t(), y, reduction="sum")

    x = P["model.embed_tokens.weight"][tokens]
    for i in range(case["layers"]):
        x = layer(x, "model.layers.%d." % i)
    x = norm(x, P["model.norm_weight"])[:, :-1]
    loss = sum(checkpoint(nll, x[b], tokens[b, 1:], use_reentrant=False) for b in range(B)) / (B * (S - 1))
    loss.backward()
    return dict({name: p.grad for name, p in P.items()}, loss=loss.detach())


def _exact_paged(case, seed):
    q, kpool, vpool, batch, gate, slopes = _paged(case, seed)
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    out = torch.empty(q.shape, dtype=F64, device="cuda")
    kept = 4 if case["window"] else 0
    for b, (lo, hi, start) in enumerate(zip(batch.cu_host, batch.cu_host[1:], batch.start_host)):
        m = start + hi - lo
        pages = batch.block_tables[b, : (m + case["page"] - 1) // case["page"]].long()
        k, v = (p[pages].reshape(-1, G, D)[:m].to(F64) for p in (kpool, vpool))
        seen = _visible(hi - lo, m, start, True, case["window"], kept)
        for h in range(H):
            g = h // (H // G)
            out[lo:hi, h] = _head(q[lo:hi, h].to(F64), k[:, g], v[:, g], D ** -0.5, seen, case["softcap"], case["sink"],
                                  None if slopes is None else slopes[h].to(F64), start)
    return out if gate is None else out * torch.sigmoid(gate.to(F64))[:, :, None]


def _exact_prompt(case, seed):
    cfg, P = _engine_tensors(case, seed)
    P = {k: v.to(F64) for k, v in P.items()}
    T, eps = case["new"], cfg["norm"]["eps"]

    def unit(x):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)

    def mixer(h, a, kind, c):
        H, D, Dv, scale = c["heads"], c["dim"], c["vdim"], c["scale"]
        if kind == "attention":
            r = H // c["kv_heads"]
            raw = (h @ P[a + "k"].t()).view(T, -1, D)
            pos = torch.arange(T, device="cuda", dtype=F64)
            temp = 1 + c["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / c["q_temp"]["every"]) + 1)
            q = unit((h @ P[a + "q"].t()).view(T, H, D)) * P[a + "q.norm"] * temp[:, None, None]
            k, seen = unit(raw) * P[a + "k.norm"], _visible(T, T, 0, True)
            y = [_head(q[:, x], k[:, x // r], raw[:, x // r], scale, seen) for x in range(H)]
        elif kind == "latent_attention":
            q, lat = (h @ P[a + "q"].t()).view(T, H, D), unit(h @ P[a + "dkv"].t()) * P[a + "dkv.norm"]
            k, v = (lat @ P[a + "uk"].t()).view(T, H, D), (lat @ P[a + "uv"].t()).view(T, H, Dv)
            seen = _visible(T, T, 0, True, c["mask"]["size"])
            y = [_head(q[:, x], k[:, x], v[:, x], scale, seen) for x in range(H)]
        else:
            r = H // c["kv_heads"]
            q, k, v = (h @ P[a + n].t() + P[a + n + ".b"] for n in ("q", "k", "v"))
            q, k, v = q.view(T, H, 2, D), k.view(T, -1, 2, D), v.view(T, -1, Dv)
            lam = (P[a + "lq1"] @ P[a + "lk1"]).exp() - (P[a + "lq2"] @ P[a + "lk2"]).exp() + c["diff"]
            seen, y = _visible(T, T, 0, True, chunk=c["mask"]["size"]), []
            for x in range(H):
                one, two = (_head(q[:, x, m], k[:, x // r, m], v[:, x // r], scale, seen) for m in (0, 1))
                y.append(unit(one - lam * two) * (1 - c["diff"]))
        return torch.cat(y, 1) @ P[a + "o"].t()

    X = P["embed"][torch.tensor(_prompt(case, seed), device="cuda")].expand(cfg["streams"], T, case["width"])
    for i, spec in enumerate(cfg["layers"]):
        p = "l%d." % i
        for part in ("1", "2"):
            h = unit(torch.einsum("s,stw->tw", P[p + "hc%s.in" % part], X)) * (1 + P[p + "norm" + part])
            if part == "1":
                y = mixer(h, p + "mix.", spec["type"], spec["mixer"])
            else:
                y = (torch.relu(h @ P[p + "mlp.gate"].t()) * (h @ P[p + "mlp.up"].t())) @ P[p + "mlp.down"].t()
            X = torch.einsum("stw,sr->rtw", X, P[p + "hc%s.mix" % part]) + P[p + "hc%s.out" % part][:, None, None] * y
    return unit(X[:, -1:].sum(0)) * (1 + P["final.norm"]) @ P["head"].t()


def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    if case["kind"] in ("dense", "packed"):
        with torch.no_grad():
            return _exact_attention(case, seed)
    with torch.no_grad():
        return _exact_paged(case, seed) if case["kind"] == "paged" else _exact_prompt(case, seed)
