"""The work that a user of this framework has it do, as cases to be timed and compared.

What runs behind a question is one chain: the encoder turns texts into vectors, the vector scan finds rows, a decoder
prefills the prompt and decodes the answer; ingest runs the same encoder and decoders in large batches.  The cases are
those parts through their public entry points:

  step     one engine step of a decoder, model.forward + compute_logits: a packed batch of prompt portions as the engine
           launches it, or one token for each of a batch of sequences, captured once in a graph and replayed as the engine
           does.  "qwen2" is the flagship family, "zofesun" the hybrid whose layers hold the attention, linear attention,
           recurrence and feed-forward that the hybrid families share.  Sizes "1b" and "7b" are the two bench sizes.
  experts  the mixture-of-experts feed-forward of the other hybrid families: router and the chosen experts
  mixer    a sequence mixer of those families from its fused projection to its output: the state-space scan, the gated
           delta rule, the selective scan, and windowed, block-local or capped attention over the paged cache
  embed    BertEncoder.encode_ids on ragged chunks (bge-base)
  search   score_topk: the exact scan of the vector index, with and without a metadata filter

The families with experts are timed by parts, since their routers choose: a step that rounds differently sends a token
elsewhere, and whole-model outputs could then not be compared.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from githubrepostorag_amd.models.configs import DecoderConfig, decoder_config, encoder_config
from githubrepostorag_amd.models.encoder import BertEncoder
from githubrepostorag_amd.models.qwen2 import Qwen2Model
from githubrepostorag_amd.models.zofesun import ZofesunModel
from githubrepostorag_amd.ops.attention import AttnMetadata, choose_splits, decode_mw_plan, sink_attention
from githubrepostorag_amd.ops.elementwise import rope_table, rope_vnorm_store
from githubrepostorag_amd.ops.gemm import WS
from githubrepostorag_amd.ops.moe import moe_experts, moe_route
from githubrepostorag_amd.ops.recurrent import (causal_conv, gated_delta, gated_rmsnorm, pad_step_matrix, selective_scan,
                                                ssm_scan)
from githubrepostorag_amd.ops.topk import Predicate, score_topk

DEV = "cuda"
BF = torch.bfloat16
BS = 16  # tokens per cache block: the engine's default
VOCAB = 32768
# width, heads, kv heads, head size, feed-forward, layers: the sizes of the hybrid bench
SIZES = {"1b": (1536, 12, 2, 128, 8960, 8), "7b": (3584, 28, 4, 128, 18944, 4)}
EXPERTS, TOP, GROUPS, KEEP = 16, 4, 4, 2


def listed():
    return [
        # an answer being written for one user: the smallest step, where latency and launches count
        dict(name="decode_one", kind="step", family="qwen2", size="7b", phase="decode", seqs=1, tokens=1100, past=0),
        # a serving batch: 64 sequences of 200 to 2000 keys
        dict(name="decode_64", kind="step", family="qwen2", size="7b", phase="decode", seqs=64, tokens=70000, past=0),
        # a full prefill step of the engine's budget: retrieval prompts of a few hundred to a few thousand tokens
        dict(name="prefill_8k", kind="step", family="qwen2", size="7b", phase="prefill", seqs=7, tokens=8192, past=0),
        # the same two steps of a hybrid decoder, and a lone medium prompt of its smaller size, of an odd length
        dict(name="hybrid_decode_64", kind="step", family="zofesun", size="7b", phase="decode", seqs=64, tokens=70000, past=0),
        dict(name="hybrid_prefill_8k", kind="step", family="zofesun", size="7b", phase="prefill", seqs=7, tokens=8192, past=0),
        dict(name="hybrid_prefill_1k", kind="step", family="zofesun", size="1b", phase="prefill", seqs=1, tokens=1187, past=0),
        # expert feed-forward: a prefill step's tokens, and a decode batch's
        dict(name="experts_4k", kind="experts", size="7b", unit="glu", tokens=4096, phase="prefill"),
        dict(name="experts_64", kind="experts", size="7b", unit="glu", tokens=64, phase="decode"),
        # sequence mixers of a prefill step
        dict(name="state_space_4k", kind="mixer", mixer="state_space", size="7b", seqs=3, tokens=4096),
        dict(name="window_attention_8k", kind="mixer", mixer="window", size="7b", seqs=2, tokens=8192),
        # ingest: a batch of code chunks to embed
        dict(name="embed_chunks", kind="embed", tokens=24000, seqs=128),
        # retrieval: the exact scan over a large table for a batch of questions
        dict(name="search_1m", kind="search", rows=1_000_000, queries=16, k=10, filter=False),
    ]


def _between(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm; odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "hybrid decode", "hybrid prefill", "experts", "mixer", "mixer", "embed", "search"])
    size = rng.choice(["1b", "7b"])
    family = "zofesun" if "hybrid" in kind else "qwen2"
    if kind.endswith("decode"):
        seqs = _between(rng, 1, 128)
        return dict(kind="step", family=family, size=size, phase="decode", seqs=seqs,
                    tokens=max(seqs * 64, min(130000, seqs * _between(rng, 100, 4000))), past=0)
    if kind.endswith("prefill"):
        tokens = _between(rng, 300, 8192)
        return dict(kind="step", family=family, size=size, phase="prefill", tokens=tokens,
                    seqs=rng.randint(1, max(1, tokens // 300)), past=rng.choice([0, 0, 1000]))
    if kind == "experts":
        phase = rng.choice(["prefill", "decode"])
        return dict(kind="experts", size=size, unit=rng.choice(["glu", "clamped", "relu2"]), phase=phase,
                    tokens=_between(rng, 1, 256) if phase == "decode" else _between(rng, 300, 4096))
    if kind == "mixer":
        tokens = _between(rng, 300, 8192)
        return dict(kind="mixer", size=size, tokens=tokens, seqs=rng.randint(1, max(1, tokens // 300)),
                    mixer=rng.choice(["state_space", "delta", "selective", "window", "block", "capped"]))
    if kind == "embed":
        seqs = _between(rng, 1, 128)
        return dict(kind="embed", seqs=seqs, tokens=seqs * rng.randint(20, 190))
    return dict(kind="search", rows=_between(rng, 20_000, 1_000_000), queries=_between(rng, 1, 64), k=rng.choice([5, 10, 30]),
                filter=rng.choice([False, True]))


# ---------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed * 9176 + 5)


def _randn(g, *shape, std=1.0, dtype=BF):
    return torch.empty(*shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _mat(g, n, k):
    """A projection matrix whose outputs have its inputs' scale."""
    return _randn(g, n, k, std=k ** -0.5)


def _around(g, v, n, std=0.1):
    return (v + _randn(g, n, std=std, dtype=torch.float32)).to(BF)


def _lengths(total, n, most=None):
    """n unequal lengths that sum to ``total``: of the case alone, so every state of a case has the same shapes."""
    rng = random.Random(total * 131 + n)
    w = [rng.uniform(0.2, 1.9) for _ in range(n)]
    got = [max(1, int(total * x / sum(w))) for x in w]
    got[-1] += max(0, total - sum(got))
    return [min(x, most) for x in got] if most else got


def _i32(v):
    return torch.tensor(v, dtype=torch.int32).to(DEV)


def _batch(c, g, kv_heads, heads, vdim):
    """The step's metadata over a cache whose blocks lie in no order.  decode: one new token per sequence, the last of its
    length; prefill: ``past`` tokens of each sequence are in the cache already."""
    decode = c.get("phase") == "decode"
    lens = _lengths(c["tokens"], c["seqs"])
    past = [n - 1 for n in lens] if decode else [c.get("past", 0)] * len(lens)
    ctx = lens if decode else [n + p for n, p in zip(lens, past)]
    width = -(-max(ctx) // BS)
    blocks = 1 + sum(-(-n // BS) for n in ctx)
    order = torch.randperm(blocks - 1, generator=torch.Generator().manual_seed(c["tokens"] + c["seqs"])) + 1
    bt = torch.zeros(len(ctx), width, dtype=torch.int32)
    at, pos, slots, q = 0, [], [], [0]
    for i, n in enumerate(ctx):
        k = -(-n // BS)
        bt[i, :k] = order[at:at + k]
        at += k
        p = torch.arange(past[i], n)
        pos.append(p)
        slots.append(bt[i][p // BS].long() * BS + p % BS)
        q.append(q[-1] + n - past[i])
    m = dict(q_start=_i32(q), ctx_len=_i32(ctx), block_tables=bt.to(DEV), slot_mapping=torch.cat(slots).to(torch.int32).to(DEV),
             max_q_len=1 if decode else max(n - p for n, p in zip(ctx, past)), num_seqs=len(ctx), num_tokens=q[-1],
             is_decode=decode, state_slots=torch.arange(len(ctx), dtype=torch.int32, device=DEV))
    if decode:
        plan = decode_mw_plan(len(ctx), kv_heads, max(ctx), max(ctx)) or choose_splits(max(ctx), len(ctx), kv_heads)
        m.update(num_splits=plan[0], split_len=plan[1],
                 part_o=torch.empty(plan[0] * len(ctx) * heads * vdim, dtype=torch.float32, device=DEV),
                 part_ml=torch.empty(plan[0] * len(ctx) * heads * 2, dtype=torch.float32, device=DEV))
    return dict(meta=AttnMetadata(**m), pos=torch.cat(pos).to(torch.int32).to(DEV), blocks=blocks, q=q, ctx=ctx, past=past, bt=bt)


def _captured(step, keep=()):
    """A graph of ``step`` and its outputs; the buffers of ``keep`` are as they were before."""
    ws, saved = {}, [t.clone() for t in keep]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), WS.owned_by(ws):
        step()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with WS.owned_by(ws), torch.cuda.graph(graph):
        out = step()
    for t, v in zip(keep, saved):
        t.copy_(v)
    return graph, out, ws


def _qwen2_weights(c, g):
    W, H, G, D, ff, nl = SIZES[c["size"]]
    sd = {"model.embed_tokens.weight": _randn(g, VOCAB, W, std=0.02), "lm_head.weight": _mat(g, VOCAB, W),
          "model.norm.weight": _around(g, 1.0, W)}
    for i in range(nl):
        p = f"model.layers.{i}."
        sd[p + "input_layernorm.weight"], sd[p + "post_attention_layernorm.weight"] = _around(g, 1.0, W), _around(g, 1.0, W)
        for n, r in (("q", H * D), ("k", G * D), ("v", G * D)):
            sd[p + f"self_attn.{n}_proj.weight"] = _mat(g, r, W)
            sd[p + f"self_attn.{n}_proj.bias"] = _randn(g, r, std=0.1)
        sd[p + "self_attn.o_proj.weight"] = _mat(g, W, H * D)
        sd[p + "mlp.gate_proj.weight"], sd[p + "mlp.up_proj.weight"] = _mat(g, ff, W), _mat(g, ff, W)
        sd[p + "mlp.down_proj.weight"] = _mat(g, W, ff)
    return sd


def _zofesun_weights(cfg, g):
    W = cfg.hidden_size
    sd = {"embed": _randn(g, cfg.vocab_size, W), "head": _mat(g, cfg.vocab_size, W)}

    def norm(name):
        sd[name], sd[name + ".b"] = _around(g, 1.0, W), _randn(g, W, std=0.02)
        sd[name + ".alpha"] = torch.tensor(0.5 + 0.1 * (len(sd) % 5), dtype=BF)

    norm("final.norm")
    for i, L in enumerate(cfg.layers):
        p, m = f"l{i}.", L.mixer
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            norm(p + n)
        if m.kind == "mingru":
            for n in "zxg":
                sd[p + "mix." + n] = _mat(g, m.width, W)
            sd[p + "mix.z.b"], sd[p + "mix.x.b"] = _randn(g, m.width, std=0.5), _randn(g, m.width, std=0.5)
            sd[p + "mix.o"] = _mat(g, W, m.width)
        else:
            a, r = m.left, m.right
            for n, rows in (("left.q", a.heads * a.dim), ("left.k", a.kv_heads * a.dim), ("left.v", a.kv_heads * a.vdim),
                            ("right.q", r.heads * r.dim), ("right.k", r.heads * r.dim), ("right.v", r.heads * r.vdim),
                            ("right.g", r.heads * r.vdim)):
                sd[p + "mix." + n] = _mat(g, rows, W)
            sd[p + "mix.left.sink"] = _randn(g, a.heads)
            sd[p + "mix.left.o"], sd[p + "mix.right.o"] = _mat(g, W, a.heads * a.vdim), _mat(g, W, r.heads * r.vdim)
            sd[p + "mix.right.norm"] = _around(g, 1.0, r.heads * r.vdim)
        sd[p + "mlp.gate"], sd[p + "mlp.up"] = _mat(g, L.mlp.ff, W), _mat(g, L.mlp.ff, W)
        sd[p + "mlp.down"] = _mat(g, W, L.mlp.ff)
    return sd


def _step_inputs(c, seed):
    """The weights, batch, token ids, cache and state of a step: what prepare() loads and exact() computes with."""
    g = _gen(seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    sd = _qwen2_weights(c, g) if c["family"] == "qwen2" else _zofesun_weights(decoder_config("zofesun-" + c["size"]), g)
    b = _batch(c, g, G, H, D)
    ids = torch.randint(0, VOCAB, (b["meta"].num_tokens,), generator=g, device=DEV, dtype=torch.int32)
    kv, state = [], []
    for i in range(nl):
        gru = c["family"] == "zofesun" and decoder_config("zofesun-" + c["size"]).layers[i].mixer.kind == "mingru"
        kv.append(None if gru else (_randn(g, b["blocks"], G, BS, D), _randn(g, b["blocks"], G, BS, D)))
        shape = (c["seqs"] + 1, W) if gru else (c["seqs"] + 1, H, D, D)
        state.append(_randn(g, *shape, dtype=torch.float32) if c["family"] == "zofesun" else None)
    return sd, b, ids, kv, state


def _prepare_step(c, seed):
    sd, b, ids, kv, state = _step_inputs(c, seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    if c["family"] == "qwen2":
        model = Qwen2Model(DecoderConfig("qwen2-" + c["size"], VOCAB, W, ff, nl, H, G, D, max_position=16384), state_dict=sd)
        more = {}
    else:
        model = ZofesunModel(decoder_config("zofesun-" + c["size"]), state_dict=sd)
        model.prepare(16384)
        more = {"state": state}
    meta = b["meta"]
    last = (meta.q_start[1:] - 1).long()

    def step():
        with torch.inference_mode():
            hidden = model.forward(ids, b["pos"], meta, kv, **more)
            rows = hidden if meta.is_decode else hidden.index_select(0, last)
            return {"hidden": hidden, "logits": model.compute_logits(rows), "kv": kv, "state": more.get("state")}

    if not meta.is_decode:
        return {"call": step}
    graph, out, ws = _captured(step, [t for t in state if t is not None])
    return {"graph": graph, "out": out, "ws": ws, "model": model, "call": step}


def _experts_inputs(c, seed):
    g = _gen(seed)
    W, _, _, _, ff, _ = SIZES[c["size"]]
    Fe = (ff // 5) // 64 * 64
    gu = Fe if c["unit"] == "relu2" else 2 * Fe
    return dict(h=_randn(g, c["tokens"], W), wr=_randn(g, EXPERTS + 1, W, std=2 * W ** -0.5, dtype=torch.float32),
                wgu=_randn(g, EXPERTS, gu, W, std=W ** -0.5), wd=_randn(g, EXPERTS, W, Fe, std=Fe ** -0.5))


def _prepare_experts(c, seed):
    x = _experts_inputs(c, seed)
    unit = dict(glu={}, clamped=dict(limit=7.0, alpha=1.702, shift=1.0), relu2=dict(unit="relu2"))[c["unit"]]

    def step():
        with torch.inference_mode():
            ids, wts, gate = moe_route(x["h"], x["wr"], EXPERTS, TOP, GROUPS, KEEP)
            return {"ids": ids, "weights": wts, "gate": gate, "experts": moe_experts(x["h"], ids, x["wgu"], x["wd"], **unit)}

    if c["phase"] == "prefill":
        return {"call": step}
    graph, out, ws = _captured(step)
    return {"graph": graph, "out": out, "ws": ws, "call": step}


def _mixer_inputs(c, seed):
    g = _gen(seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    b = _batch(c, g, G, H, D)
    T, S = b["meta"].num_tokens, c["seqs"] + 1
    x = dict(b=b, g=g, T=T)
    f32 = dict(dtype=torch.float32)
    if c["mixer"] == "state_space":  # z | x B C | dt, 64-wide heads, 128 state numbers
        P, N = 64, 128
        Hs = W // P
        ch = Hs * P + 2 * N
        x.update(Hs=Hs, N=N, P=P, ch=ch, proj=_randn(g, T, Hs * P + ch + Hs, std=0.7), w=_randn(g, ch, 4, std=0.5, **f32),
                 cb=_randn(g, ch, std=0.2, **f32), cst=torch.zeros(S, 3, ch, dtype=BF, device=DEV), dtb=_randn(g, Hs, **f32),
                 alog=torch.empty(Hs, device=DEV).uniform_(-1.5, 0.5, generator=g), skip=1 + _randn(g, Hs, std=0.3, **f32),
                 st=torch.zeros(S, Hs, N, P, device=DEV), norm=1 + _randn(g, Hs * P, std=0.1, **f32))
    elif c["mixer"] == "delta":  # q | k | v | g | b | a
        ch = 2 * G * D + H * D
        x.update(ch=ch, proj=_randn(g, T, ch + H * D + 2 * H), w=_randn(g, ch, 4, std=0.5, **f32),
                 cst=torch.zeros(S, 3, ch, dtype=BF, device=DEV),
                 alog=torch.empty(H, device=DEV).uniform_(-1.5, 0.5, generator=g), dtb=-3 + _randn(g, H, **f32),
                 st=torch.zeros(S, H, D, D, device=DEV), norm=(1 + _randn(g, D, std=0.1, **f32)).repeat(H))
    elif c["mixer"] == "selective":  # x | z, 16 state numbers per channel, step sizes from W / 16 numbers
        N, R, inner = 16, W // 16, W
        x.update(N=N, R=R, inner=inner, proj=_randn(g, T, 2 * inner), w=_randn(g, inner, 4, std=0.5, **f32),
                 cb=_randn(g, inner, std=0.2, **f32), cst=torch.zeros(S, 3, inner, dtype=BF, device=DEV),
                 low=_randn(g, T, R + 2 * N), wdt=pad_step_matrix(_randn(g, inner, R, std=R ** -0.5)),
                 dtb=-3 + _randn(g, inner, **f32), A=-torch.exp(_randn(g, inner, N, std=0.7, **f32)),
                 skip=1 + _randn(g, inner, std=0.3, **f32), st=torch.zeros(S, inner, N, device=DEV))
    else:
        x.update(proj=_randn(g, T, (H + 2 * G) * D), ones=torch.ones(D, device=DEV), rot=D // 2,
                 table=rope_table(max(b["ctx"]), D // 2, 1e4, DEV), temp=1 + _randn(g, H, std=0.2, **f32),
                 kv=[torch.zeros(b["blocks"], G, BS, D, dtype=BF, device=DEV) for _ in range(2)])
    return x


def _attention_form(c, x):
    """The keyword arguments of a mixer's attention."""
    return dict(window=dict(window=1024), capped=dict(window=1024, softcap=30.0), block=dict(chunk=1024, head_scale=x.get("temp")))[
        c["mixer"]]


def _prepare_mixer(c, seed):
    x = _mixer_inputs(c, seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    meta, p = x["b"]["meta"], x["proj"]

    def state_space():
        Hs, N, P, inner = x["Hs"], x["N"], x["P"], x["Hs"] * x["P"]
        xbc = causal_conv(p, inner, x["w"], x["cb"], x["cst"], meta)
        o = ssm_scan(xbc, p, inner + x["ch"], x["dtb"], x["alog"], x["skip"], x["st"], meta, Hs, 1, N, P)
        y = torch.empty(x["T"], inner, dtype=BF, device=DEV)
        gated_rmsnorm(o, x["norm"], p, 0, 1e-5, y, gate="silu", gate_first=True)
        return {"y": y, "conv": x["cst"], "state": x["st"]}

    def delta():
        vv = H * D
        xc = causal_conv(p, 0, x["w"], None, x["cst"], meta)
        y = gated_delta(xc, p, x["ch"] + vv, x["ch"] + vv + H, x["ch"], x["alog"], x["dtb"], x["norm"], 1e-5, x["st"], meta,
                        H, G, D, D)
        return {"y": y, "conv": x["cst"], "state": x["st"]}

    def selective():
        xc = causal_conv(p, 0, x["w"], x["cb"], x["cst"], meta)
        y = selective_scan(xc, x["low"], x["wdt"], x["R"], x["dtb"], x["A"], x["skip"], p, x["inner"], x["st"], meta)
        return {"y": y, "conv": x["cst"], "state": x["st"]}

    def attention():
        kc, vc = x["kv"]
        q = rope_vnorm_store(p, 0, H * D, (H + G) * D, x["b"]["pos"], x["table"], meta.slot_mapping, kc, vc, H, G, D, D,
                             x["rot"], 1e-5, vnorm=False, qw=x["ones"], kw=x["ones"])
        return {"y": sink_attention(q, kc, vc, meta, D ** -0.5, None, **_attention_form(c, x)), "kv": x["kv"]}

    call = dict(state_space=state_space, delta=delta, selective=selective).get(c["mixer"], attention)

    def step():
        with torch.inference_mode():
            return call()

    return {"call": step}


def _embed_inputs(c, seed):
    g = _gen(seed)
    cfg = encoder_config("bge-base-en-v1.5")
    W, ff = cfg.hidden_size, cfg.intermediate_size
    e = "embeddings."
    sd = {e + "word_embeddings.weight": _randn(g, cfg.vocab_size, W, std=0.05), e + "position_embeddings.weight": _randn(
        g, cfg.max_position, W, std=0.02), e + "token_type_embeddings.weight": _randn(g, cfg.type_vocab_size, W, std=0.02)}
    norms = [e + "LayerNorm"]
    for i in range(cfg.num_layers):
        p = f"encoder.layer.{i}."
        for n, r, k in (("attention.self.query", W, W), ("attention.self.key", W, W), ("attention.self.value", W, W),
                        ("attention.output.dense", W, W), ("intermediate.dense", ff, W), ("output.dense", W, ff)):
            sd[p + n + ".weight"], sd[p + n + ".bias"] = _mat(g, r, k), _randn(g, r, std=0.02)
        norms += [p + "attention.output.LayerNorm", p + "output.LayerNorm"]
    for n in norms:
        sd[n + ".weight"], sd[n + ".bias"] = _around(g, 1.0, W, 0.05), _randn(g, W, std=0.02)
    rng = random.Random(seed)
    ids = [[rng.randrange(999, cfg.vocab_size) for _ in range(n)] for n in _lengths(c["tokens"], c["seqs"], cfg.max_seq_length)]
    return cfg, sd, ids


def _prepare_embed(c, seed):
    cfg, sd, ids = _embed_inputs(c, seed)
    enc = BertEncoder(cfg, device=DEV, state_dict=sd)

    def call():
        f32, bf16 = enc.encode_ids(ids)
        return {"vectors": f32, "stored": bf16}

    return {"call": call}


def _search_inputs(c, seed):
    g = _gen(seed)
    d = 768
    centre = _randn(g, 64, d, dtype=torch.float32)  # the rows of a code base lie in groups
    X = torch.empty(c["rows"], d, dtype=BF, device=DEV)
    for a in range(0, c["rows"], 1 << 17):
        n = min(1 << 17, c["rows"] - a)
        x = _randn(g, n, d, dtype=torch.float32) + centre[torch.randint(0, 64, (n,), generator=g, device=DEV)]
        X[a:a + n] = F.normalize(x, dim=1)
    q = _randn(g, c["queries"], d, dtype=torch.float32) + centre[torch.randint(0, 64, (c["queries"],), generator=g, device=DEV)]
    col = torch.randint(0, 4, (c["rows"],), generator=g, device=DEV, dtype=torch.int32)
    return X, F.normalize(q, dim=1).to(BF), col


def _prepare_search(c, seed):
    X, q, col = _search_inputs(c, seed)
    preds = [Predicate(col, 1)] if c["filter"] else None

    def call():
        scores, ids = score_topk(X, q, c["k"], preds=preds)
        return {"scores": scores, "ids": ids}

    return {"call": call}


def prepare(case, seed):
    return dict(step=_prepare_step, experts=_prepare_experts, mixer=_prepare_mixer, embed=_prepare_embed,
                search=_prepare_search)[case["kind"]](case, seed)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _pairs(c, window=0, block=0):
    """Visible (query, key) pairs of the case's batch."""
    total = 0
    for n in _lengths(c["tokens"], c["seqs"]):
        if c.get("phase") == "decode":
            total += n
        elif block:
            total += (n // block) * block * (block + 1) // 2 + (n % block) * (n % block + 1) // 2
        else:
            w = min(window or n, n)
            total += w * (w + 1) // 2 + (n - w) * w + n * c.get("past", 0)
    return total


def work(c):
    if c["kind"] == "search":
        return {"bytes": c["rows"] * (768 * 2 + 4 * c["filter"]) + c["queries"] * (768 * 2 + c["k"] * 12),
                "flops": 2 * c["rows"] * 768 * c["queries"]}
    if c["kind"] == "embed":
        W, ff, nl = 768, 3072, 12
        lens = _lengths(c["tokens"], c["seqs"], 512)
        T, n = sum(lens), nl * (4 * W * W + 2 * W * ff)
        return {"bytes": 2 * n + T * W * 2 + c["seqs"] * W * 6, "flops": 2 * T * n + nl * 4 * W * sum(x * x for x in lens)}
    W, H, G, D, ff, nl = SIZES[c["size"]]
    if c["kind"] == "experts":
        T, Fe, m = c["tokens"], (ff // 5) // 64 * 64, 2 if c["unit"] == "relu2" else 3
        used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** T)
        return {"bytes": 2 * used * m * Fe * W + 4 * (EXPERTS + 1) * W + 2 * T * W * (1 + TOP) + 8 * T * TOP,
                "flops": 2 * m * T * TOP * Fe * W + 2 * T * (EXPERTS + 1) * W}
    if c["kind"] == "mixer":
        T = sum(_lengths(c["tokens"], c["seqs"]))
        if c["mixer"] == "state_space":  # the state update and read-out of every token
            Hs, N, P = W // 64, 128, 64
            return {"bytes": 2 * T * (3 * W + 2 * N + Hs) + 4 * c["seqs"] * Hs * N * P, "flops": 4 * T * Hs * N * P}
        if c["mixer"] == "delta":
            return {"bytes": 2 * T * (3 * H * D + 2 * G * D + 2 * H) + 4 * c["seqs"] * H * D * D, "flops": 6 * T * H * D * D}
        if c["mixer"] == "selective":
            return {"bytes": 2 * T * (3 * W + W // 16 + 32) + 4 * c["seqs"] * W * 16, "flops": 4 * T * W * 16 + 2 * T * W * (W // 16)}
        pairs = _pairs(c, block=1024) if c["mixer"] == "block" else _pairs(c, window=1024)
        return {"bytes": 2 * T * (2 * H + 4 * G) * D, "flops": 4 * pairs * H * D}
    decode = c["phase"] == "decode"
    lens = _lengths(c["tokens"], c["seqs"])
    T = len(lens) if decode else sum(lens)
    if c["family"] == "qwen2":
        n, att, state = nl * (2 * H * D * W + 2 * G * D * W + 3 * W * ff), nl, 0
    else:
        gru, ffw = nl // 4, nl * 3 * W * ff
        att = nl - gru
        n = att * ((H + 2 * G) * D * W + 4 * H * D * W + 2 * H * D * W) + gru * 4 * W * W + ffw
        state = 4 * len(lens) * (att * H * D * D + gru * W) * (2 if decode or c["past"] else 1)
    pairs, keys = _pairs(c), sum(lens) + (0 if decode else c["past"] * len(lens))
    scan = 0 if c["family"] == "qwen2" else 4 * T * att * H * D * D
    return {"bytes": 2 * (n + VOCAB * W) + att * 4 * keys * G * D + state + 2 * (2 * T * W + len(lens) * VOCAB),
            "flops": 2 * T * n + 2 * len(lens) * VOCAB * W + att * 4 * pairs * H * D + scan}


def tolerance(c):
    if c["kind"] == "search":  # fp32 sums of exact products; rows whose scores tie in fp32 may change places
        return {"rel": 1e-5, "differ": 0.005}
    if c["kind"] == "embed":  # twelve layers of bf16 activations
        return {"rel": 0.02, "max": 0.2}
    if c["kind"] == "experts":  # bf16 activations between the two products; the fp32 router may decide a tie otherwise
        return {"rel": 0.01, "max": 0.1, "differ": 0.002}
    if c["kind"] == "mixer":
        return {"rel": 0.01, "max": 0.2}
    if c["family"] == "zofesun":  # four to eight layers of bf16 activations on an fp32 residual stream
        return {"rel": 0.015, "max": 0.3}
    return {"rel": 0.03, "max": 0.5}  # a bf16 residual stream


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _d(t):
    return t.double()


def _rms(t, eps):
    return t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + eps)


def _rotate(t, pos, rot, base):
    """The first ``rot`` dims of [T, heads, d]: dim i with i + rot / 2."""
    h = rot // 2
    ang = pos.double()[:, None] * base ** (-torch.arange(h, dtype=torch.float64, device=DEV) / h)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = t[..., :h], t[..., h:rot]
    return torch.cat([a * c - b * s, b * c + a * s, t[..., rot:]], -1)


def _cached(cache, bt, n):
    """The first n cached rows of a sequence, [n, G, D]."""
    return _d(cache[bt[: -(-n // BS)].long().to(DEV)]).permute(0, 2, 1, 3).reshape(-1, cache.shape[1], cache.shape[3])[:n]


def _softmax_attention(q, k, v, past, scale, sink=None, window=0, chunk=0, softcap=0.0, head_scale=None):
    """q [n, H, d], k / v [past + n, G, d] -> [n, H, d]; some query rows at a time."""
    n, H, _ = q.shape
    R = H // k.shape[1]
    k, v = k.repeat_interleave(R, 1).permute(1, 2, 0).contiguous(), v.repeat_interleave(R, 1).permute(1, 0, 2).contiguous()
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device=DEV)
    keys = torch.arange(past + n, device=DEV)
    for a in range(0, n, 1024):
        e = min(n, a + 1024)
        s = torch.matmul(q[a:e].permute(1, 0, 2).contiguous(), k) * scale
        if head_scale is not None:
            s = s * _d(head_scale)[:, None, None]
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        pos = torch.arange(past + a, past + e, device=DEV)[:, None]
        hide = keys > pos
        if window:
            hide = hide | (keys <= pos - window)
        if chunk:
            hide = hide | (keys < pos - pos % chunk)
        s = s.masked_fill(hide, -math.inf)
        if sink is not None:
            s = torch.cat([s, _d(sink)[:, None, None].expand(H, e - a, 1)], -1)
        out[a:e] = torch.matmul(torch.softmax(s, -1)[..., : past + n], v).permute(1, 0, 2)
    return out


def _parts(b):
    """(rows, cached tokens, sequence) of each sequence of a batch."""
    return [(slice(b["q"][i], b["q"][i + 1]), b["past"][i], i) for i in range(len(b["ctx"]))]


def _paged(q, k, v, kv, b, scale, **more):
    """Attention of the step's rows over the cached rows and themselves."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device=DEV)
    for r, past, i in _parts(b):
        ks, vs = k[r], v[r]
        if past:
            ks, vs = torch.cat([_cached(kv[0], b["bt"][i], past), ks]), torch.cat([_cached(kv[1], b["bt"][i], past), vs])
        out[r] = _softmax_attention(q[r], ks, vs, past, scale, **more)
    return out


def _exact_qwen2(c, seed):
    sd, b, ids, kv, _ = _step_inputs(c, seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    get = lambda n: _d(sd[n])  # noqa: E731
    x = get("model.embed_tokens.weight")[ids.long()]
    for i in range(nl):
        p = f"model.layers.{i}."
        h = _rms(x, 1e-6) * get(p + "input_layernorm.weight")
        q, k, v = ((h @ get(p + f"self_attn.{n}_proj.weight").T + get(p + f"self_attn.{n}_proj.bias")).view(-1, m, D)
                   for n, m in (("q", H), ("k", G), ("v", G)))
        q, k = _rotate(q, b["pos"], D, 1e6), _rotate(k, b["pos"], D, 1e6)
        a = _paged(q, k, v, kv[i], b, D ** -0.5)
        x = x + a.reshape(-1, H * D) @ get(p + "self_attn.o_proj.weight").T
        h = _rms(x, 1e-6) * get(p + "post_attention_layernorm.weight")
        u = F.silu(h @ get(p + "mlp.gate_proj.weight").T) * (h @ get(p + "mlp.up_proj.weight").T)
        x = x + u @ get(p + "mlp.down_proj.weight").T
    x = _rms(x, 1e-6) * get("model.norm.weight")
    rows = [r.stop - 1 for r, _, _ in _parts(b)]
    return {"hidden": x, "logits": x[rows] @ get("lm_head.weight").T, "kv": None, "state": None}


def _exact_zofesun(c, seed):
    sd, b, ids, kv, state = _step_inputs(c, seed)
    cfg = decoder_config("zofesun-" + c["size"])
    get = lambda n: _d(sd[n].to(DEV))  # noqa: E731
    dyt = lambda t, n: torch.tanh(get(n + ".alpha") * t) * get(n) + get(n + ".b")  # noqa: E731
    x = get("embed")[ids.long()]
    final = []
    for i, L in enumerate(cfg.layers):
        p, m, S = f"l{i}.", L.mixer, _d(state[i])
        h = dyt(x, p + "norm1")
        lin = lambda n: h @ get(p + "mix." + n).T  # noqa: E731
        if m.kind == "mingru":
            z, u, gate = torch.sigmoid(lin("z") + get(p + "mix.z.b")), lin("x") + get(p + "mix.x.b"), F.silu(lin("g"))
            add, keep, y = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), 1 - z, torch.empty_like(z)
            for r, past, s in _parts(b):
                cur = S[s] if past else torch.zeros_like(S[s])
                for t in range(r.start, r.stop):
                    cur = torch.addcmul(add[t], keep[t], cur)
                    y[t] = cur
                S[s] = cur
            y = (y * gate) @ get(p + "mix.o").T
        else:
            a, w = m.left, m.right
            q, k, v = (lin("left." + n).view(-1, n_, a.dim) for n, n_ in (("q", a.heads), ("k", a.kv_heads), ("v", a.kv_heads)))
            q, k = _rotate(q, b["pos"], a.rot_dims, a.rot_base), _rotate(k, b["pos"], a.rot_dims, a.rot_base)
            o = _paged(q, k, _rms(v, cfg.norm_eps), kv[i], b, a.scale, sink=get(p + "mix.left.sink"))
            y = m.left_scale * o.reshape(-1, a.heads * a.vdim) @ get(p + "mix.left.o").T
            q, k, v = (F.silu(lin("right." + n)).view(-1, w.heads, w.dim).permute(1, 0, 2).contiguous() for n in "qkv")
            lam = torch.tensor(w.decay, dtype=torch.float32, device=DEV).double().log()[:, None, None]
            o = torch.empty_like(v)
            for r, past, s in _parts(b):
                cur = S[s] if past else torch.zeros_like(S[s])
                for e in range(r.start, r.stop, 1024):
                    t = slice(e, min(r.stop, e + 1024))
                    n = t.stop - e
                    step = torch.arange(n, device=DEV, dtype=torch.float64)
                    back = step[:, None] - step
                    pw = torch.where(back >= 0, torch.exp(lam * back.clamp_min(0)), 0.0)
                    o[:, t] = (q[:, t] @ k[:, t].transpose(1, 2).contiguous() * pw) @ v[:, t] + torch.exp(
                        lam * (step[:, None] + 1)) * (q[:, t] @ cur)
                    cur = torch.exp(lam * n) * cur + (k[:, t] * torch.exp(lam * (n - 1 - step[:, None]))).transpose(
                        1, 2).contiguous() @ v[:, t]
                S[s] = cur
            o = o.permute(1, 0, 2).reshape(-1, w.heads * w.vdim)
            o = _rms(o, cfg.norm_eps) * get(p + "mix.right.norm") * torch.sigmoid(lin("right.g")) * m.right_scale
            y = y + o @ get(p + "mix.right.o").T
        final.append(S)
        x = x + dyt(y, p + "norm1b")
        h = dyt(x, p + "norm2")
        gate = (h @ get(p + "mlp.gate").T).clamp(max=L.mlp.limit)
        up = (h @ get(p + "mlp.up").T).clamp(-L.mlp.limit, L.mlp.limit)
        x = x + dyt((gate * torch.sigmoid(1.702 * gate) * (up + 1)) @ get(p + "mlp.down").T, p + "norm2b")
    x = dyt(x, "final.norm")
    rows = [r.stop - 1 for r, _, _ in _parts(b)]
    return {"hidden": x, "logits": x[rows] @ get("head").T, "kv": None, "state": final}


def _exact_experts(c, seed):
    x = _experts_inputs(c, seed)
    h, wr = _d(x["h"]), _d(x["wr"])
    z = h @ wr.T
    s = torch.softmax(z[:, :EXPERTS], -1)
    best = s.view(-1, GROUPS, EXPERTS // GROUPS).amax(-1)
    shut = torch.ones_like(best, dtype=torch.bool).scatter_(1, best.topk(KEEP, -1).indices, False)
    wts, ids = s.masked_fill(shut.repeat_interleave(EXPERTS // GROUPS, 1), -1.0).topk(TOP, -1)
    out = torch.zeros(h.shape[0], TOP, h.shape[1], dtype=torch.float64, device=DEV)
    for e in range(EXPERTS):
        t, k = torch.where(ids == e)
        v = h[t] @ _d(x["wgu"][e]).T
        if c["unit"] == "relu2":
            u = v.clamp_min(0).pow(2)
        else:
            g, u = v.chunk(2, 1)
            if c["unit"] == "clamped":
                g = g.clamp(max=7.0)
                u = g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1)
            else:
                u = F.silu(g) * u
        out[t, k] = u @ _d(x["wd"][e]).T
    return {"ids": None, "weights": wts, "gate": torch.sigmoid(z[:, EXPERTS]), "experts": out}


def _exact_conv(x, off, ch, bias=None):
    """The causal convolution of every sequence from no past, and the last inputs that it keeps."""
    inp, w = _d(x["proj"][:, off:off + ch]), _d(x["w"])
    out, kept = torch.empty_like(inp), torch.zeros(x["cst"].shape, dtype=torch.float64, device=DEV)
    for r, _, s in _parts(x["b"]):
        full = torch.cat([torch.zeros(3, ch, dtype=torch.float64, device=DEV), inp[r]])
        n = r.stop - r.start
        out[r] = F.silu(sum(w[:, j] * full[j:j + n] for j in range(4)) + (0 if bias is None else _d(bias)))
        kept[s] = full[n:]
    return out, kept


def _exact_mixer(c, seed):
    x = _mixer_inputs(c, seed)
    W, H, G, D, ff, nl = SIZES[c["size"]]
    p, b, T = x["proj"], x["b"], x["T"]
    state = None if "st" not in x else torch.zeros(x["st"].shape, dtype=torch.float64, device=DEV)
    if c["mixer"] == "state_space":
        Hs, N, P = x["Hs"], x["N"], x["P"]
        inner = Hs * P
        u, kept = _exact_conv(x, inner, x["ch"], x["cb"])
        xs, B, C = u[:, :inner].view(T, Hs, P).permute(1, 0, 2), u[:, inner:inner + N], u[:, inner + N:]
        dt = F.softplus(_d(p[:, inner + x["ch"]:]) + _d(x["dtb"])).T
        lg = -torch.exp(_d(x["alog"]))[:, None] * dt  # [Hs, T] log of the decay
        y = torch.empty(Hs, T, P, dtype=torch.float64, device=DEV)
        for r, _, s in _parts(b):
            cur = state[s]
            for e in range(r.start, r.stop, 512):
                t = slice(e, min(r.stop, e + 512))
                cum = lg[:, t].cumsum(1)
                n = t.stop - e
                low = torch.ones(n, n, dtype=torch.bool, device=DEV).tril()
                L = torch.exp((cum[:, :, None] - cum[:, None]).masked_fill(~low, -math.inf))
                v = xs[:, t] * dt[:, t, None]
                y[:, t] = (L * (C[t] @ B[t].T)) @ v + torch.exp(cum)[:, :, None] * (C[t] @ cur)
                cur = torch.exp(cum[:, -1])[:, None, None] * cur + (
                    B[t].T[None] * torch.exp(cum[:, -1:] - cum)[:, None]) @ v
            state[s] = cur
        y = (y + _d(x["skip"])[:, None, None] * xs).permute(1, 0, 2).reshape(T, inner)
        y = _rms(y * F.silu(_d(p[:, :inner])), 1e-5) * _d(x["norm"])
        return {"y": y, "conv": kept, "state": state}
    if c["mixer"] == "delta":
        ch, vv = x["ch"], H * D
        u, kept = _exact_conv(x, 0, ch)
        unit = lambda t: t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q = (unit(u[:, :G * D].view(T, G, D)) * D ** -0.5).repeat_interleave(H // G, 1)
        k = unit(u[:, G * D:2 * G * D].view(T, G, D)).repeat_interleave(H // G, 1)
        v = u[:, 2 * G * D:].view(T, H, D)
        beta = torch.sigmoid(_d(p[:, ch + vv:ch + vv + H]))[:, :, None]
        g = torch.exp(-torch.exp(_d(x["alog"])) * F.softplus(_d(p[:, ch + vv + H:ch + vv + 2 * H]) + _d(x["dtb"])))
        o = torch.empty(T, H, D, dtype=torch.float64, device=DEV)
        g, kb = g[:, :, None, None], k * beta
        vb = v * beta
        for r, _, s in _parts(b):
            cur = state[s]
            for t in range(r.start, r.stop):
                cur = g[t] * cur
                add = vb[t][:, None] - torch.matmul(kb[t][:, None], cur)
                cur = torch.baddbmm(cur, k[t][:, :, None], add)
                o[t] = torch.matmul(q[t][:, None], cur)[:, 0]
            state[s] = cur
        y = (_rms(o, 1e-5)).reshape(T, vv) * _d(x["norm"]) * F.silu(_d(p[:, ch:ch + vv]))
        return {"y": y, "conv": kept, "state": state}
    if c["mixer"] == "selective":
        N, R, inner = x["N"], x["R"], x["inner"]
        u, kept = _exact_conv(x, 0, inner, x["cb"])
        low = _d(x["low"])
        dt = F.softplus(low[:, :R] @ _d(x["wdt"][:, :R]).T + _d(x["dtb"]))
        B, C, A, y = low[:, R:R + N], low[:, R + N:R + 2 * N], _d(x["A"]), torch.empty_like(u)
        du = dt * u
        for r, _, s in _parts(b):
            cur = state[s]
            for t in range(r.start, r.stop):
                cur = torch.exp(dt[t][:, None] * A) * cur + du[t][:, None] * B[t]
                y[t] = cur @ C[t]
            state[s] = cur
        return {"y": (y + _d(x["skip"]) * u) * F.silu(_d(p[:, inner:])), "conv": kept, "state": state}
    q, k, v = (_d(p[:, o:o + n * D]).view(T, n, D) for o, n in ((0, H), (H * D, G), ((H + G) * D, G)))
    q, k = _rotate(_rms(q, 1e-5), b["pos"], x["rot"], 1e4), _rotate(_rms(k, 1e-5), b["pos"], x["rot"], 1e4)
    return {"y": _paged(q, k, v, x["kv"], b, D ** -0.5, **_attention_form(c, x)).reshape(T, H * D), "kv": None}


def _exact_embed(c, seed):
    cfg, sd, batch = _embed_inputs(c, seed)
    get = lambda n: _d(sd[n])  # noqa: E731
    W, nh, D = cfg.hidden_size, cfg.num_heads, cfg.head_dim
    norm = lambda t, n: F.layer_norm(t, (W,), get(n + ".weight"), get(n + ".bias"), cfg.layer_norm_eps)  # noqa: E731
    ids = torch.tensor([t for s in batch for t in s], device=DEV)
    pos = torch.cat([torch.arange(len(s)) for s in batch]).to(DEV)
    starts = [0]
    for s in batch:
        starts.append(starts[-1] + len(s))
    x = norm(get("embeddings.word_embeddings.weight")[ids] + get("embeddings.position_embeddings.weight")[pos]
             + get("embeddings.token_type_embeddings.weight")[0], "embeddings.LayerNorm")
    for i in range(cfg.num_layers):
        p = f"encoder.layer.{i}."
        lin = lambda t, n: t @ get(p + n + ".weight").T + get(p + n + ".bias")  # noqa: E731
        q, k, v = (lin(x, "attention.self." + n).view(-1, nh, D).transpose(0, 1).contiguous() for n in ("query", "key", "value"))
        a = torch.empty_like(x)
        for s, e in zip(starts, starts[1:]):
            w = torch.softmax(q[:, s:e] @ k[:, s:e].transpose(1, 2).contiguous() * D ** -0.5, -1)
            a[s:e] = (w @ v[:, s:e]).transpose(0, 1).reshape(e - s, W)
        x = norm(x + lin(a, "attention.output.dense"), p + "attention.output.LayerNorm")
        x = norm(x + lin(F.gelu(lin(x, "intermediate.dense")), "output.dense"), p + "output.LayerNorm")
    v = F.normalize(x[starts[:-1]], dim=1)
    return {"vectors": v, "stored": v}


def _exact_search(c, seed):
    X, q, col = _search_inputs(c, seed)
    best = []
    for a in range(0, c["rows"], 1 << 17):
        s = _d(q) @ _d(X[a:a + (1 << 17)]).T
        if c["filter"]:
            s = s.masked_fill(col[a:a + (1 << 17)] != 1, -math.inf)
        best.append(s.topk(min(c["k"], s.shape[1]), 1).values)
    return {"scores": torch.cat(best, 1).topk(c["k"], 1).values, "ids": None}


def exact(case, seed):
    if case["kind"] == "step":
        return (_exact_qwen2 if case["family"] == "qwen2" else _exact_zofesun)(case, seed)
    return dict(experts=_exact_experts, mixer=_exact_mixer, embed=_exact_embed, search=_exact_search)[case["kind"]](case, seed)
